"""Charge -> proxy on 4-wide matrix-core blocks: the proxy / plane-wave stage against the oracle
where its tiles of sources end -- 1, 31, 32, 33, 59, 60, 61 and 121 points per level-0 box (tiles
of 60 in FP32 and 32 in FP64, groups of 3 and 5 sources per FP32 operand), boxes whose points lie
in many short leaves (a tile runs across them), every proxy order (9, 18, 28, 38) in both
precisions, and the workgroup shapes forced either way in FP64 (PDMK_C2P_WIDE), bit for bit.

Tolerance as in the other stage tests: FP64 1e-12; FP32 1e-5, for 9 and 12 digits as well (the
rounding of FP32 arithmetic does not depend on the order)."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu


def points(per_box):
    out = []
    for b in range(64):
        k = per_box[b % len(per_box)]
        u = W.uniform01(300 + b, 3 * k).reshape(k, 3)
        out.append((u + np.array([b % 4, b // 4 % 4, b // 16])) / 4)
    return np.concatenate(out)


@pytest.mark.parametrize("per_box,npl", [((1,), 300), ((31, 32, 33), 300), ((59, 60, 61), 300), ((121, 2), 300),
                                         ((40, 90), 6)])
@pytest.mark.parametrize("digits", [3, 6, 9, 12])
def test_chain_stage(pdmk, oracle_mod, cuda, monkeypatch, per_box, npl, digits):
    cell, pos = W.cubic_cell(), points(per_box)
    q = 2.0 * W.uniform01(6, pos.shape[0]) - 1.0
    o = oracle_mod.OracleTree(cell, pos, digits, npl, 4, precision="double")
    ref = o.evaluate(q, 1)
    o.close()
    for precision, tol in (("float", 1e-5), ("double", 1e-12)):
        out = []
        for mode in ("", "0", "1") if precision == "double" else ("",):
            if mode:
                monkeypatch.setenv("PDMK_C2P_WIDE", mode)
            s = pdmk.PDMKSolver(cell, pos, n_digits=digits, n_per_leaf=npl, nz=4, precision=precision)
            if mode:
                monkeypatch.delenv("PDMK_C2P_WIDE")
            out.append(s.run_stages(q, 1))
            s.close()
        assert np.linalg.norm(out[0] - ref) <= tol * np.linalg.norm(ref), precision
        for o2 in out[1:]:
            np.testing.assert_array_equal(o2, out[0])
