"""Target evaluation on the vector ALUs (k_eval_targets: p = 9, FP32 above 6 digits, FP32
quasi-periodic trees) where a workgroup's pass of 256 targets ends: the proxy / plane-wave stage
against the oracle with leaves of 255, 256, 257, 512 and 600 targets beside leaves of 3.

Tolerance as in the other stage tests: FP64 1e-12, FP32 1e-5 (relative L2)."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu

B = np.array([2.0, -1.0, 0.5])


def points(per_box):
    """``per_box[i % len]`` points in each of the 4^3 boxes of side 1/4 of the unit cube."""
    out = []
    for b in range(64):
        k = per_box[b % len(per_box)]
        u = W.uniform01(100 + b, 3 * k).reshape(k, 3)
        out.append((u + np.array([b % 4, b // 4 % 4, b // 16])) / 4)
    return np.concatenate(out)


@pytest.mark.parametrize("per_box", [(255, 3, 3), (256, 3, 3), (257, 3, 3), (512, 3, 3, 3), (600, 3, 3, 3)])
@pytest.mark.parametrize("precision,digits,bloch", [("float", 3, None), ("double", 3, None), ("float", 9, None),
                                                    ("float", 6, B), ("float", 3, B)])
def test_chain_stage(pdmk, oracle_mod, cuda, per_box, precision, digits, bloch):
    cell, pos = W.cubic_cell(), points(per_box)
    q = 2.0 * W.uniform01(5, pos.shape[0]) - 1.0
    o = oracle_mod.OracleTree(cell, pos, digits, 700, 4, precision="double")
    ref = o.evaluate(q, 1) if bloch is None else o.evaluate_complex(q, bloch, 1)
    o.close()
    s = pdmk.PDMKSolver(cell, pos, n_digits=digits, n_per_leaf=700, nz=4, precision=precision, bloch=bloch)
    got = s.run_stages(q, 1).astype(np.float64) if bloch is None else s.run_complex_stages(q, 1)
    s.close()
    assert np.linalg.norm(got - ref) <= (1e-12 if precision == "double" else 1e-5) * np.linalg.norm(ref)
