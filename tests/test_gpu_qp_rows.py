"""Quasi-periodic trees through the kernels that take both components at once.

* Near field: the row kernels (FP32: one residual for the two charges; FP64: the components
  along z) with 1, 4 and 8 waves per item (PDMK_NEAR_PARTS) against the wavefront-wide lists
  (PDMK_NEAR_ROWS=0), bit for bit: entries in the same order, the sums formed the same way.
  FP32 below 6 digits reads the entries' coefficients with their geometry.
* Stage by stage against the oracle at the digit counts and proxy orders that
  test_gpu_qp.py leaves out: FP32 at p = 9 (both components per chain launch), 28 and 38 (one
  after the other, each from its copy of the sources), FP64 at 3 and 12 digits.  Tolerances as
  there: FP64 1e-12, FP32 1e-5."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu

B = np.array([2.0, -1.0, 0.5])
TRI = W.triclinic_cell()
CASES = {
    "three_points": lambda: (W.cubic_cell(), W.uniform_positions(3, 2, W.cubic_cell()), 300),
    "sparse": lambda: (W.cubic_cell(), W.uniform_positions(700, 4, W.cubic_cell()), 7),
    "clustered": lambda: (TRI, W.gaussian_mixture(4000, 8, 0.02, 21, TRI), 30),
    "uniform": lambda: (TRI, W.uniform_positions(9001, 6, TRI), 300),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("precision,digits", [("float", 1), ("float", 3), ("float", 4), ("float", 5), ("float", 6),
                                              ("double", 6), ("double", 9), ("double", 12)])
def test_near_parts(pdmk, cuda, monkeypatch, name, precision, digits):
    cell, pos, npl = CASES[name]()
    q = 2.0 * W.uniform01(78, pos.shape[0]) - 1.0

    def near(**env):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        s = pdmk.PDMKSolver(cell, pos, n_digits=digits, n_per_leaf=npl, nz=4, precision=precision, bloch=B)
        for k in env:
            monkeypatch.delenv(k)
        out = s.run_complex_stages(q, 2)
        s.close()
        return out

    ref = near(PDMK_NEAR_ROWS="0")
    np.testing.assert_array_equal(near(), ref)
    for parts in ("1", "4", "8"):
        np.testing.assert_array_equal(near(PDMK_NEAR_PARTS=parts), ref, err_msg=parts)


@pytest.mark.parametrize("precision,digits", [("float", 1), ("float", 3), ("float", 4), ("float", 5), ("float", 9),
                                              ("float", 12), ("double", 3), ("double", 12)])
@pytest.mark.parametrize("name", ["sparse", "clustered"])
def test_stages(pdmk, oracle_mod, cuda, name, precision, digits):
    cell, pos, npl = CASES[name]()
    q = 2.0 * W.uniform01(78, pos.shape[0]) - 1.0
    s = pdmk.PDMKSolver(cell, pos, n_digits=digits, n_per_leaf=npl, nz=4, precision=precision, bloch=B)
    o = oracle_mod.OracleTree(cell, pos, digits, npl, 4, precision="double")
    tol = 1e-12 if precision == "double" else 1e-5
    for st in (1, 2, 4, 8, 15):
        g, r = s.run_complex_stages(q, st), o.evaluate_complex(q, B, st)
        assert np.linalg.norm(g - r) <= tol * np.linalg.norm(r), st
    s.close()
    o.close()
