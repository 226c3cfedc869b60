"""The exact far field (k_ff_structure, k_ff_reduce, k_ff_eval on the FP64 matrix cores) against
the oracle's direct Fourier sum, at the edges of its tiles: point counts around 16 and 32 (the
rows of a product and a workgroup's points) and past a workgroup column, mode boxes whose lines
need 1, 2 and 3 column tiles (nz 4 to 12, 3 to 12 digits), and unequal axes.

Tolerance: every phase comes from one sincos and at most 20 complex products (error below
20 * 2 * 2^-53 * 3 axes ~ 1.4e-14 per term) in both directions, so the relative L2 difference
stays below 1e-12, the bound of the other FP64 stage tests.  FP32 trees return the same sums
rounded to float (2^-24)."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu

CELLS = {"cubic": W.cubic_cell(), "triclinic": W.triclinic_cell(), "long": np.diag([0.5, 1.0, 2.3])}


@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 33, 1000])
@pytest.mark.parametrize("cell,digits,nz", [("cubic", 6, 4), ("triclinic", 3, 4), ("cubic", 6, 12), ("long", 9, 4),
                                            ("triclinic", 9, 8), ("cubic", 12, 4)])
def test_far_stage_edges(pdmk, oracle_mod, cuda, cell, digits, nz, n):
    c = CELLS[cell]
    pos = W.uniform_positions(n, 7 + n, c)
    q = 2.0 * W.uniform01(9 + n, n) - 1.0
    o = oracle_mod.OracleTree(c, pos, digits, 300, nz, precision="double")
    ref = o.evaluate(q, 8)
    o.close()
    for precision, tol in (("double", 1e-12), ("float", 2.0 ** -23)):
        s = pdmk.PDMKSolver(c, pos, n_digits=digits, n_per_leaf=300, nz=nz, precision=precision)
        got = s.run_stages(q, 8).astype(np.float64)
        s.close()
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), (precision, np.linalg.norm(got - ref))
