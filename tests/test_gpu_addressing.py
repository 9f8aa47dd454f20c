"""The tiled matvec through buffer descriptors and through 64-bit pointers at sizes whose default is the kernels of
nh_small.hip, so a height is forced: the inner operator against the oracle, and the whole solve, with the ZW/ZP table and
without, in the chunked form of launches of few tiles and at every height."""
import numpy as np
import pytest

import oracle
from cases import build
from orctm_amd import abi, synth
from orctm_amd.nh import NHSolver, options

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    u = np.uint32 if a.dtype == np.float32 else np.uint64
    return np.array_equal(np.ascontiguousarray(a).view(u), np.ascontiguousarray(b).view(u))


@pytest.mark.parametrize("rows", [4, 8, 12])
@pytest.mark.parametrize("name", ["regional", "transect"])
@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
@pytest.mark.parametrize("zw_table", [-1, 1])
def test_addressing_agrees_on_tiles_of_few_columns(name, rows, precision, zw_table):
    print(f"[addressing] {name} rows={rows} precision={precision} zw_table={zw_table}", flush=True)
    g, divg = build(name)
    dt = np.float32 if precision == abi.MIXED else np.float64
    x = synth.normal(9, 3, g.cells).astype(dt)
    A, S = oracle.assemble(g)
    y_ref = oracle.matvec(g, oracle.inner_coef(A, S, dt, grid=g), x)
    out = []
    for addr in (0, -1):
        pnh = np.zeros((g.IE, g.JE, g.KE), order="F")
        with NHSolver(g, options(precision=precision, tile_rows=rows, zw_table=zw_table, buffer_addressing=addr,
                                 warm_start=False)) as s:
            y = s.inner_apply(x)
            st = s.solve(divg, pnh)
        assert st["status"] == "OK" and st["tile_rows"] == rows and st["buffer_addressing"] == (1 if addr == 0 else 0)
        assert bits_equal(y, y_ref)
        out.append((pnh, st["inner_iters"], st["outer_iters"]))
    assert bits_equal(out[0][0], out[1][0]) and out[0][1:] == out[1][1:]
