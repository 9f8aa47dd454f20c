"""The transfers between the caller's arrays and the device (nh_xfer.cpp): what set_guess brings in,
get_solution brings back, bit for bit, on arrays below, at and above the sizes where a transfer takes
several chunks, worker threads (4 MiB) and the pinned path to the device (16 MiB), with rows that straddle
chunks, and from two threads at once; the halo of the caller's array stays as it was.
"""
import threading

import numpy as np
import pytest

from orctm_amd import synth
from orctm_amd.nh import NHSolver, options

pytestmark = pytest.mark.gpu

SIZES = [(3, 3, 1), (97, 41, 5), (128, 128, 32), (129, 127, 33), (131, 127, 31), (256, 256, 32), (257, 255, 33), (333, 301, 41)]


def _solver(nx, ny, nz):
    return NHSolver(synth.make_grid(synth.GridSpec(nx, ny, nz, bathy="flat", depth=900.0)), options(tile_rows=4))


def _round_trip(s, seed):
    rng = np.random.default_rng(seed)
    a = np.asfortranarray(rng.standard_normal(s.shape))
    b = np.asfortranarray(rng.standard_normal(s.shape))
    want = b.copy(order="F")
    want[1:-1, 1:-1, :] = a[1:-1, 1:-1, :]
    s.set_guess(a)
    s.get_solution(b)
    return np.array_equal(want.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_guess_comes_back(size):
    print(f"[transfer] {size}", flush=True)
    with _solver(*size) as s:
        assert _round_trip(s, 1) and _round_trip(s, 2)


def test_two_threads_at_once():
    solvers, ok = [_solver(*SIZES[-1]), _solver(*SIZES[3])], [None, None]

    def many(k):
        ok[k] = all(_round_trip(solvers[k], 10 * k + r) for r in range(5))

    threads = [threading.Thread(target=many, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in solvers:
        s.close()
    assert ok == [True, True]
    with _solver(*SIZES[1]) as s:  # after the last handle gave the pinned chunks back
        assert _round_trip(s, 7)
