"""Entries of the launch-shape file (PDMK_TUNE_CACHE) from before FP32 trees at p = 18 had matrix-core
transforms: there p2pw_bk and t3_div chose among the vector kernels, and the same values now ask
for a vector kernel in place of the matrix-core one.  Such an entry keeps its other knobs and
leaves these two at the built-in choice; entries written since, and those of other trees, are
taken whole.  The file is read once per process, so child processes load it."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import json, sys
sys.path.insert(0, sys.argv[1])
import periodicdmk_amd as P
from periodicdmk_amd import workloads as W
out = []
for n, precision in ((600, "float"), (2500, "float"), (600, "double")):
    s = P.PDMKSolver(W.cubic_cell(), W.uniform_positions(n, 1, W.cubic_cell()), n_digits=6, n_per_leaf=300, nz=4,
                     precision=precision)
    if sys.argv[2] == "tune":
        s.autotune(1)
    out.append(s.knobs())
    s.close()
print(json.dumps(out))
"""


def child(path, what):
    r = subprocess.run([sys.executable, "-c", CHILD, REPO, what], env=dict(os.environ, PDMK_TUNE_CACHE=str(path)),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout.splitlines()[-1])


def test_entries_of_the_vector_kernels(pdmk, cuda, tmp_path):
    path = tmp_path / "tune.txt"
    child(path, "tune")
    keys = [line.split()[0] for line in path.read_text().splitlines()]
    assert len(keys) == 3 and [k.endswith(":m4") for k in keys] == [True, True, False]
    # the first as an older file has it, the others as they are
    path.write_text("".join(f"{k} 16 1 32 64 2\n" for k in (keys[0][:-len(":m4")], keys[1], keys[2])))
    whole = {"near_wpb": 16, "near_late": 1, "p2pw_bk": 32, "pw2p_bk": 64, "t3_div": 2}
    assert child(path, "load") == [{**whole, "p2pw_bk": 0, "t3_div": 1}, whole, whole]
