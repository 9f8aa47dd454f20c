"""Either side of the lines between the three forms of the inner iteration (blocks of columns, streaming, tiled), which
follow from the rows of 64 columns, the levels, the precision, the ZW/ZP table and the addressing: the same solution
and iteration counts as the tiled kernels at a forced height."""
import numpy as np
import pytest

from orctm_amd import abi, synth
from orctm_amd.nh import NHBatch, NHSolver, options

pytestmark = pytest.mark.gpu

# nx, ny, nz, options: rows of 64 columns 256 | 257 and 512 | 513, few and more levels, in reach of the streaming kernels
# and not; without the table 775, 1200 | 1205, 4001 rows; one level 2000 | 2001, two 3100 | 3101, a channel 5000 | 5001
LINES = [(64, 256, 8, {}), (64, 257, 8, {}), (520, 57, 16, {}), (512, 64, 16, {}), (520, 57, 17, {}),
         (64, 256, 8, {"buffer_addressing": -1}), (64, 257, 8, {"buffer_addressing": -1}),
         (64, 257, 12, {"buffer_addressing": -1}), (64, 257, 13, {"buffer_addressing": -1}), (520, 57, 8, {"buffer_addressing": -1}),
         (260, 155, 16, {"zw_table": -1}), (260, 155, 17, {"zw_table": -1}), (300, 240, 9, {"zw_table": -1}),
         (300, 241, 9, {"zw_table": -1}), (300, 241, 8, {"zw_table": -1}), (50, 4001, 3, {"zw_table": -1}), (60, 2000, 1, {}), (60, 2001, 1, {}),
         (60, 3100, 2, {}), (60, 3101, 2, {}), (33, 5000, 3, {}), (33, 5001, 3, {}), (33, 5001, 10, {})]


def solve(g, divg, **kw):
    p = np.zeros((g.IE, g.JE, g.KE), order="F")
    with NHSolver(g, options(warm_start=False, maxit=400, **kw)) as s:
        st = s.solve(divg, p)
    assert st["status"] == "OK", st
    return p, st["inner_iters"], st["outer_iters"], st["rel_res"]


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
@pytest.mark.parametrize("case", LINES, ids=lambda c: f"{c[0]}x{c[1]}x{c[2]}" + "".join(f"-{k}" for k in c[3]))
def test_forms_agree_at_their_lines(case, precision):
    nx, ny, nz, kw = case
    print(f"[forms] {nx}x{ny}x{nz} {kw} precision={precision}", flush=True)
    g, divg = synth.build(synth.GridSpec(nx, ny, nz, smooth=3.0, seed=synth.BASE_SEED + 221))
    a = solve(g, divg, precision=precision, **kw)
    b = solve(g, divg, precision=precision, tile_rows=4, **kw)
    assert a[1:] == b[1:] and np.array_equal(a[0], b[0])


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
def test_batches_with_and_without_the_table(precision):
    """Most rows without the table, or few of them: the members' own results either way."""
    print(f"[forms batch] precision={precision}", flush=True)
    g, divg = synth.build(synth.GridSpec(200, 150, 20, smooth=3.0, seed=synth.BASE_SEED + 222))
    want = solve(g, divg, precision=precision, tile_rows=4)
    for tables in ((-1, -1, 0), (0, 0, -1)):
        solvers = [NHSolver(g, options(precision=precision, warm_start=False, maxit=400, zw_table=t)) for t in tables]
        for s in solvers:
            s.set_rhs(divg)
        batch = NHBatch(solvers)
        rc, stats = batch.solve()
        assert rc == abi.OK, stats
        for s, st in zip(solvers, stats):
            p = s.get_solution(np.zeros_like(want[0]))
            assert st["inner_iters"] == want[1] and np.array_equal(g.interior(p), g.interior(want[0]))
        batch.close()
        for s in solvers:
            s.close()
