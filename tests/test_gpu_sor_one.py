"""The barotropic sweeps of a surface that one block holds (k_sor_one) at the edges of its range -- one, two and
three cells of a colour per thread, the largest surfaces it takes and the next ones, which run blocked,
two-cell and odd periods, one-cell-wide closed channels -- bit for bit against the oracle."""
import copy

import numpy as np
import pytest

import oracle
from orctm_amd import synth
from orctm_amd.nh import NHBarotropic

pytestmark = pytest.mark.gpu

# (nx, ny, periodic x, periodic y, runs in one launch)
SURFACES = [(1, 1, 0, 0, 1), (1, 9, 0, 1, 1), (2, 2, 1, 1, 1), (3, 2, 1, 1, 1), (2, 5, 0, 1, 1), (512, 4, 0, 1, 1),
            (512, 3, 0, 1, 1), (64, 32, 1, 0, 1), (65, 33, 1, 1, 1), (1024, 6, 0, 1, 1), (1024, 7, 0, 1, 0),
            (96, 64, 0, 0, 1), (97, 64, 0, 0, 0), (62, 96, 1, 1, 1), (5, 1000, 1, 0, 1)]


@pytest.mark.parametrize("surface", SURFACES, ids=lambda s: "x".join(map(str, s)))
def test_surface_in_one_block(surface):
    nx, ny, cx, cy, one = surface
    print(f"[sor one] {surface}", flush=True)
    g = synth.make_grid(synth.GridSpec(nx, ny, 2, smooth=1.5, cyclic_x=bool(cx), cyclic_y=bool(cy), open_w=not cx,
                                       open_n=not cy, seed=31))
    b = copy.copy(synth.make_barotropic(g))
    b.iterations = 40
    z_ref, b_ref = oracle.troneu(b, oracle.itprep(b), b1o=np.zeros((b.IE, b.JE), order="F"))
    with NHBarotropic(b) as s:
        assert (s.info()["launches"] == 1) == bool(one)
        for _ in range(2):
            z, b1 = np.full((b.IE, b.JE), 5.0, order="F"), np.full((b.IE, b.JE), -3.0, order="F")
            s.troneu(b.u1o, b.uzo, b.v1e, b.vze, b1, z)
            assert np.array_equal(z.view(np.uint64), z_ref.view(np.uint64))
            assert np.array_equal(b1.view(np.uint64), b_ref.view(np.uint64))
