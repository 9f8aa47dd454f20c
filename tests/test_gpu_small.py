"""Solves of few columns (nh_small.hip: blocks of 16, 32 or 64 columns with all their levels in LDS) against
the tiled kernels (a forced tile height): the same solution bits, iteration counts and residual, at the
edges of the blocks' forms -- levels per thread, padded level batches, columns per block, rows per sum,
periodic sides of one to a few cells, the level limits -- with the ZW/ZP planes and the table, alone and in
a batch, and across warm-started steps; and the matvec and the line solve against the oracle.
"""
import numpy as np
import pytest

import oracle
from orctm_amd import abi, synth
from orctm_amd.nh import NHBatch, NHSolver, options

pytestmark = pytest.mark.gpu

# (nx, ny, nz, periodic x, periodic y)
SHAPES = [(1, 1, 1, 0, 0), (2, 1, 3, 1, 1), (15, 3, 8, 0, 1), (16, 2, 9, 1, 0), (17, 5, 47, 0, 0), (64, 4, 48, 1, 1),
          (65, 3, 49, 1, 0), (63, 4, 144, 0, 1), (33, 3, 145, 0, 0), (20, 2, 240, 0, 0), (20, 2, 241, 0, 0),
          (64, 70, 57, 0, 0), (70, 40, 73, 1, 0), (66, 33, 121, 0, 0), (64, 66, 36, 0, 1), (61, 67, 37, 0, 0),
          (130, 45, 61, 1, 0), (64, 130, 76, 0, 0), (64, 130, 77, 0, 0), (129, 256, 4, 0, 0), (64, 65, 109, 0, 0),
          (128, 65, 156, 0, 0), (64, 65, 157, 0, 0)]


def _grid(nx, ny, nz, cx, cy, seed=5):
    side = dict(cyclic_x=bool(cx), cyclic_y=bool(cy))
    if cx:
        side.update(open_w=False, open_e=False)
    if cy:
        side.update(open_n=False, open_s=False)
    return synth.build(synth.GridSpec(nx, ny, nz, smooth=2.0, seed=seed, **side))


def _solve(g, divg, steps=2, **kw):
    pnh = np.zeros((g.IE, g.JE, g.KE), order="F")
    with NHSolver(g, options(**kw)) as s:
        out = []
        for k in range(steps):
            if k:
                s.perturb_rhs(0.01, 40 + k)
            else:
                s.set_rhs(divg)
            st = s.solve_resident()
            out.append((st["status"], st["outer_iters"], st["inner_iters"], st["rel_res"], s.get_solution(pnh).copy()))
        return out


def _same(a, b):
    return a[:4] == b[:4] and np.array_equal(a[4].view(np.uint64), b[4].view(np.uint64))


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_few_columns_equal_the_tiled_kernels(shape, precision):
    print(f"[small] {shape} precision={precision}", flush=True)
    g, divg = _grid(*shape)
    for table in (-1, 1):
        kw = dict(precision=precision, zw_table=table, maxit=300)
        small, tiled = _solve(g, divg, **kw), _solve(g, divg, tile_rows=4, **kw)
        assert all(_same(a, b) for a, b in zip(small, tiled)), (table, [a[:4] for a in small], [a[:4] for a in tiled])


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
@pytest.mark.parametrize("shape", [SHAPES[5], SHAPES[11], SHAPES[16]], ids=lambda s: "x".join(map(str, s)))
def test_matvec_and_line_solve_against_the_oracle(shape, precision):
    print(f"[small operators] {shape} precision={precision}", flush=True)
    g, divg = _grid(*shape)
    A, S = oracle.assemble(g)
    dt = np.float32 if precision == abi.MIXED else np.float64
    C = oracle.inner_coef(A, S, dt, grid=g)
    invD, L = oracle.line_factor(g, C)
    x = synth.normal(98, 2, g.cells).astype(dt)
    u = np.uint32 if precision == abi.MIXED else np.uint64
    with NHSolver(g, options(precision=precision)) as s:
        assert np.array_equal(s.inner_apply(x).view(u), oracle.matvec(g, C, x).view(u))
        z, rho = s.inner_precond(x)
        z_ref, rho_ref = oracle.line_apply(g, invD, L, x)
        assert np.array_equal(z.view(u), z_ref.view(u))


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
def test_a_batch_of_few_columns_equals_each_alone(precision):
    print(f"[small batch] precision={precision}", flush=True)
    grids = [_grid(*s) for s in (SHAPES[4], SHAPES[6], SHAPES[14], SHAPES[3])]
    solvers = [NHSolver(g, options(precision=precision)) for g, _ in grids]
    for s, (_, d) in zip(solvers, grids):
        s.set_rhs(d)
    batch = NHBatch(solvers)
    _, stats = batch.solve()
    for s, st, (g, d) in zip(solvers, stats, grids):
        p = s.get_solution(np.zeros(s.shape, order="F"))
        assert _same((st["status"], st["outer_iters"], st["inner_iters"], st["rel_res"], p),
                     _solve(g, d, 1, precision=precision)[0])
    batch.close()
    for s in solvers:
        s.close()
