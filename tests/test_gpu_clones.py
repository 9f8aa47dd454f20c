"""Handles that share an operator (orctm_nh_clone) and differ on dry cells: one with a right-hand side of 0, one with
a right-hand side on land, one with a first guess on land, and an ordinary one whose vectors hold an earlier solve.
Which levels of a column a solve works on follows its own residual, so each member gives the bits it gives as a solver
of its own, in one batch and on threads side by side, whichever kernels run: the streaming ones (203 rows of 4 tiles
each), the blocks of columns and the tiled ones."""
import threading

import numpy as np
import pytest

from orctm_amd import abi, synth
from orctm_amd.nh import NHBatch, NHSolver, options

pytestmark = pytest.mark.gpu

FORMS = {
    "streaming": ((201, 203, 13), {}),
    "columns": ((70, 40, 21), {"zw_table": 1}),
    "tiled": ((70, 40, 21), {"zw_table": 1, "tile_rows": 4}),
}
MEMBERS = ("ordinary", "rest", "rhs_on_land", "guess_on_land")


class Case:
    def __init__(self, form, precision):
        (nx, ny, nz), kw = FORMS[form]
        self.g, self.divg = synth.build(synth.GridSpec(nx, ny, nz, smooth=3.0, seed=synth.BASE_SEED + 221))
        self.opts = dict(precision=precision, warm_start=False, maxit=400, **kw)
        rng = np.random.default_rng(7)
        land = np.asarray(self.g.weto) == 0.0
        self.some = land & (rng.random(land.shape) < 0.01)
        self.odd = self.divg.copy(order="F")
        self.odd[self.some] = np.abs(self.divg).max() * rng.standard_normal(int(self.some.sum()))
        self.guess = np.asfortranarray(np.where(land & (rng.random(land.shape) < 0.01), 1.0, 0.0))

    def solver(self):
        return NHSolver(self.g, options(**self.opts))

    def load(self, s, member):
        rest = np.zeros_like(self.divg)
        s.set_rhs({"rest": rest, "rhs_on_land": self.odd}.get(member, self.divg))
        if member == "guess_on_land":
            s.set_guess(self.guess)

    def earlier(self, s):
        s.set_rhs(np.asfortranarray(-2.0 * self.odd))
        s.solve_resident()

    def solution(self, s):
        return self.g.interior(s.get_solution(np.zeros((self.g.IE, self.g.JE, self.g.KE), order="F"))).copy()

    def alone(self):
        out = {}
        for m in MEMBERS:
            with self.solver() as s:
                if m == "ordinary":
                    self.earlier(s)
                self.load(s, m)
                st = s.solve_resident()
                out[m] = (st["status"], st["inner_iters"], self.solution(s))
        return out

    def clones(self):
        model = self.solver()
        model.set_rhs(self.divg)
        states = {m: model.clone() for m in MEMBERS}
        self.earlier(states["ordinary"])
        return model, states


def check(got, want):
    for m in MEMBERS:
        assert got[m][:2] == want[m][:2], (m, got[m][:2], want[m][:2])
        assert np.array_equal(np.ascontiguousarray(got[m][2]).view(np.uint64),
                              np.ascontiguousarray(want[m][2]).view(np.uint64)), m


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
@pytest.mark.parametrize("form", list(FORMS))
def test_batch_of_clones_equals_each_alone(form, precision):
    print(f"[clones] batch {form} precision={precision}", flush=True)
    case = Case(form, precision)
    want = case.alone()
    assert want["ordinary"][0] == "OK" and not want["rest"][2].any()
    model, states = case.clones()
    for m, s in states.items():
        case.load(s, m)
    batch = NHBatch([states[m] for m in MEMBERS])
    _, stats = batch.solve()
    check({m: (st["status"], st["inner_iters"], case.solution(states[m])) for m, st in zip(MEMBERS, stats)}, want)
    batch.close()
    for s in states.values():
        s.close()
    model.close()


@pytest.mark.parametrize("precision", [abi.MIXED, abi.FP64])
@pytest.mark.parametrize("form", list(FORMS))
def test_clones_on_threads_equal_each_alone(form, precision):
    print(f"[clones] threads {form} precision={precision}", flush=True)
    case = Case(form, precision)
    want = case.alone()
    model, states = case.clones()
    got, failed = {}, []
    ready = threading.Barrier(len(MEMBERS) + 1, timeout=60)

    def run(m):
        try:
            ready.wait()
            for _ in range(4):
                case.load(states[m], m)
                st = states[m].solve_resident()
                got[m] = (st["status"], st["inner_iters"], case.solution(states[m]))
                check({**want, m: got[m]}, want)
        except Exception as e:
            failed.append((m, e))

    def operators():
        try:
            x = synth.normal(11, 3, case.g.cells).astype(np.float32 if precision == abi.MIXED else np.float64)
            ready.wait()
            for _ in range(6):
                model.inner_apply(x)
                model.inner_precond(x)
        except Exception as e:
            failed.append(("operators", e))

    threads = [threading.Thread(target=run, args=(m,)) for m in MEMBERS] + [threading.Thread(target=operators)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    check(got, want)
    for s in states.values():
        s.close()
    model.close()
