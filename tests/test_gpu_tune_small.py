"""Contexts on blocks of columns run no tile height: a batch of them (a serving cohort) times none and leaves the tuning
file alone; the members' own contexts keep one choice per size class."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCRIPT = f"""
import json, sys
sys.path.insert(0, {ROOT!r}); sys.path.insert(0, {os.path.join(ROOT, 'tests')!r})
from cases import build
from orctm_amd import abi
from orctm_amd.nh import NHBatch, NHSolver, options
solvers = []
for n in ("closed", "regional"):
    g, divg = build(n)
    s = NHSolver(g, options(precision=abi.MIXED))
    s.set_rhs(divg)
    solvers += [s, s.clone(), s.clone()]
rc, st = NHBatch(solvers).solve()
print(json.dumps([rc, [x["status"] for x in st], [x["tile_rows"] for x in st]]))
"""


def test_a_batch_on_blocks_of_columns_times_no_heights(tmp_path):
    print("[tune small]", flush=True)
    f = tmp_path / "tile_tuning.json"
    r = subprocess.run([sys.executable, "-c", SCRIPT], env=dict(os.environ, ORCTM_NH_TUNE_FILE=str(f)),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    rc, status, rows = json.loads(r.stdout.strip().splitlines()[-1])
    assert rc == 0 and status == ["OK"] * 6 and all(h in (4, 8, 12) for h in rows)
    assert all(e["mode"] < 100 and e["count_class"] == 0 for e in json.load(open(f))["entries"])
