"""The exact far field with 16 points per LDS tile: mode boxes with |i| + |j| + |k| past about 124,
whose tables for 32 points pass 64 KB (cubic at 12 digits and nz = 12: 54 per axis; a 1 x 1 x 16 cell
at 6 digits: 140 along the long axis), against the oracle's direct Fourier sum at point
counts around 16.

Tolerance: a phase is one sincos and at most 140 complex products (140 * 2 * 2^-53 = 3.1e-14, the
other axes less) in each direction, so the relative L2 difference stays below 1e-12; FP32 trees
return the same sums rounded (2^-23)."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33])
@pytest.mark.parametrize("cell,digits,nz", [(np.eye(3), 12, 12), (np.diag([1.0, 1.0, 16.0]), 6, 4)])
def test_far_stage(pdmk, oracle_mod, cuda, cell, digits, nz, n):
    pos = W.uniform_positions(n, 7 + n, cell)
    q = 2.0 * W.uniform01(9 + n, n) - 1.0
    o = oracle_mod.OracleTree(cell, pos, digits, 300, nz, precision="double")
    ref = o.evaluate(q, 8)
    o.close()
    for precision, tol in (("double", 1e-12), ("float", 2.0 ** -23)):
        s = pdmk.PDMKSolver(cell, pos, n_digits=digits, n_per_leaf=300, nz=nz, precision=precision)
        got = s.run_stages(q, 8).astype(np.float64)
        s.close()
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), (precision, np.linalg.norm(got - ref))
