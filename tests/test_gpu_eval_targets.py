"""Target evaluation on the matrix cores (k_eval_targets_mfma at p = 18, 28 and 38, FP32 and
FP64): the proxy / plane-wave stage against the oracle where its tiles end -- leaves of 1, 15,
16, 17, 31, 32, 33 and 65 targets (one or two 16-target tiles, stages of 32, pieces of 32) and a
few large leaves beside many small ones.  Single-box trees would have no far part, so every input
has points in all 64 level-0 boxes.

Tolerance as in the other stage tests: FP64 1e-12, FP32 1e-5 (relative L2)."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu


def points(per_box):
    """``per_box[i % len]`` points in each of the 4^3 boxes of side 1/4 of the unit cube."""
    out = []
    for b in range(64):
        k = per_box[b % len(per_box)]
        u = W.uniform01(100 + b, 3 * k).reshape(k, 3)
        out.append((u + np.array([b % 4, b // 4 % 4, b // 16])) / 4)
    return np.concatenate(out)


@pytest.mark.parametrize("per_box", [(1,), (15, 16, 17), (31, 32, 33), (65, 3), (400, 5, 5, 5)])
@pytest.mark.parametrize("precision,digits", [("float", 6), ("double", 6), ("double", 9), ("double", 12)])
def test_chain_stage(pdmk, oracle_mod, cuda, per_box, precision, digits):
    cell, pos = W.cubic_cell(), points(per_box)
    q = 2.0 * W.uniform01(5, pos.shape[0]) - 1.0
    o = oracle_mod.OracleTree(cell, pos, digits, 300, 4, precision="double")
    ref = o.evaluate(q, 1)
    o.close()
    s = pdmk.PDMKSolver(cell, pos, n_digits=digits, n_per_leaf=300, nz=4, precision=precision)
    got = s.run_stages(q, 1).astype(np.float64)
    s.close()
    assert np.linalg.norm(got - ref) <= (1e-12 if precision == "double" else 1e-5) * np.linalg.norm(ref)
