"""The streaming inner kernels (csrc/nh_stream.hip): launches of many columns. Every case is solved by them (no forced
tile height) and by the tiled kernels (tile_rows forced), which must agree bit for bit: both form the same products
and sum them in the same groups, and levels beyond a column's use hold zeros that add nothing. The operator and the
line solve alone are compared in the same way, on vectors that are not zero on land."""

import numpy as np
import pytest

from orctm_amd import abi, synth
from orctm_amd.nh import NHBatch, NHSolver, options

pytestmark = pytest.mark.gpu

# nx: an odd last column, a last tile column of its own (pairs stacked in y), a row of one pair; ny: remainders of the
# 4-row blocks; nz: 1, the ring of levels shorter than its depth, not a multiple of a batch, the most levels held.
GRIDS = {
    "one_level": synth.GridSpec(321, 260, 1, smooth=3.0, seed=synth.BASE_SEED + 201),
    "two_levels": synth.GridSpec(129, 1030, 2, smooth=3.0, seed=synth.BASE_SEED + 202),
    "odd": synth.GridSpec(201, 203, 13, smooth=3.0, seed=synth.BASE_SEED + 203),
    "deep": synth.GridSpec(191, 259, 64, smooth=3.0, seed=synth.BASE_SEED + 204),
    "cyclic": synth.GridSpec(193, 257, 7, cyclic_x=True, cyclic_y=True, smooth=3.0, seed=synth.BASE_SEED + 205),
    "cyclic_even": synth.GridSpec(256, 258, 9, cyclic_x=True, smooth=3.0, seed=synth.BASE_SEED + 206),
    "pairs": synth.GridSpec(519, 421, 5, smooth=3.0, seed=synth.BASE_SEED + 207),
    "pairs_cyclic": synth.GridSpec(577, 390, 6, cyclic_x=True, cyclic_y=True, smooth=3.0, seed=synth.BASE_SEED + 208),
}


def same(a, b):
    return np.array_equal(a, b, equal_nan=True)  # a zero's sign apart


def solved(g, divg, **kw):
    pnh = np.zeros((g.IE, g.JE, g.KE), order="F")
    with NHSolver(g, options(warm_start=False, maxit=400, **kw)) as s:
        dt = np.float32 if kw["precision"] == abi.MIXED else np.float64
        x = synth.normal(11, 3, g.cells).astype(dt)
        y = s.inner_apply(x)
        z, rho = s.inner_precond(x)
        st = s.solve(divg, pnh)
        # again, after vectors that filled every level
        p2 = np.zeros_like(pnh)
        s.solve(divg, p2)
    assert st["status"] == "OK", st
    assert same(pnh, p2)
    return y, z, rho, pnh, st


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
@pytest.mark.parametrize("table", [-1, 0])
@pytest.mark.parametrize("name", list(GRIDS))
def test_streaming_and_tiled_kernels_agree(name, table, precision):
    print(f"[stream] {name} table={table} precision={precision}", flush=True)
    g, divg = synth.build(GRIDS[name])
    a = solved(g, divg, precision=precision, zw_table=table)
    b = solved(g, divg, precision=precision, zw_table=table, tile_rows=4)
    assert a[4]["zw_table"] == (0 if table else 1) and a[4]["tile_rows"] == 4
    for u, v in zip(a[:4], b[:4]):
        assert same(np.asarray(u), np.asarray(v))
    assert a[4]["inner_iters"] == b[4]["inner_iters"] and a[4]["outer_iters"] == b[4]["outer_iters"]


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
def test_right_hand_side_and_guess_on_land(precision):
    """Dry cells with a right-hand side or a first guess of their own are solved too, and nothing of them stays for
    the next solve."""
    print(f"[stream land] precision={precision}", flush=True)
    g, divg = synth.build(synth.GridSpec(201, 203, 13, smooth=3.0, seed=synth.BASE_SEED + 211))
    rng = np.random.default_rng(5)
    land = np.asarray(g.weto) == 0.0
    odd = divg.copy(order="F")
    some = land & (rng.random(land.shape) < 0.01)
    odd[some] = np.abs(divg).max() * rng.standard_normal(int(some.sum()))
    guess = np.asfortranarray(np.where(land & (rng.random(land.shape) < 0.01), 1.0, 0.0))
    out = []
    for rows in (0, 4):
        with NHSolver(g, options(precision=precision, warm_start=True, maxit=400, tile_rows=rows)) as s:
            p1, p2, p3 = guess.copy(order="F"), np.zeros_like(guess), np.zeros_like(guess)
            s.solve(odd, p1)
            with_guess = s.solve(divg, p2)
        with NHSolver(g, options(precision=precision, warm_start=False, maxit=400, tile_rows=rows)) as s:
            s.solve(odd, p3)
            s.solve(divg, p3)
        out.append((p1, p2, p3, with_guess["inner_iters"]))
    assert np.any(out[0][0][some] != 0.0)
    for u, v in zip(out[0], out[1]):
        assert same(np.asarray(u), np.asarray(v))


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
def test_batch_matches_alone(precision):
    """Systems of different sizes and levels in one launch, one of them without the table."""
    print(f"[stream batch] precision={precision}", flush=True)
    tables = {"odd": 0, "cyclic": 0, "deep": -1}
    alone, solvers, grids = [], [], []
    for n, t in tables.items():
        g, divg = synth.build(GRIDS[n])
        alone.append(solved(g, divg, precision=precision, zw_table=t)[3])
        s = NHSolver(g, options(precision=precision, warm_start=False, maxit=400, zw_table=t))
        s.set_rhs(divg)
        solvers.append(s)
        grids.append(g)
    batch = NHBatch(solvers)
    rc, stats = batch.solve()
    assert rc == abi.OK, stats
    for g, s, p in zip(grids, solvers, alone):
        pnh = np.zeros_like(p)
        s.get_solution(pnh)
        assert same(g.interior(pnh), g.interior(p))
    batch.close()
    for s in solvers:
        s.close()
