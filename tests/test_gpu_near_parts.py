"""The row near field with several waves per item (trees with few items: each wave walks the
lists of its share of an item's list1 entries) against the wavefront-wide lists
(PDMK_NEAR_ROWS=0): the entries' sums are added in entry order whatever the number of waves, so
the near-field potentials are bit-identical (tolerance 0).  Below 6 digits (FP32) the rows read
their entries' coefficients with the geometry.  4 and 8 waves (PDMK_NEAR_PARTS)
and the built-in choice; a single point, fewer targets than a row, partly filled items, more
parts than non-empty entries, uneven entries (clusters), 64 targets and one more."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu

TRI = W.triclinic_cell()
CASES = {
    "one_point": lambda: (W.cubic_cell(), W.uniform_positions(1, 1, W.cubic_cell()), 300),
    "three_points": lambda: (W.cubic_cell(), W.uniform_positions(3, 2, W.cubic_cell()), 300),
    "sparse": lambda: (W.cubic_cell(), W.uniform_positions(700, 4, W.cubic_cell()), 7),
    "items_of_65": lambda: (W.cubic_cell(), W.uniform_positions(65 * 64, 5, W.cubic_cell()), 300),
    "clustered": lambda: (TRI, W.gaussian_mixture(6000, 8, 0.02, 21, TRI), 30),
    "uniform": lambda: (TRI, W.uniform_positions(30_011, 6, TRI), 300),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("precision,digits", [("float", 1), ("float", 3), ("float", 4), ("float", 5), ("float", 6),
                                              ("double", 6), ("double", 9), ("double", 12)])
def test_parts_equal_wavefront_lists(pdmk, cuda, monkeypatch, name, precision, digits):
    cell, pos, npl = CASES[name]()
    q = 2.0 * W.uniform01(78, pos.shape[0]) - 1.0

    def near(**env):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        s = pdmk.PDMKSolver(cell, pos, n_digits=digits, n_per_leaf=npl, nz=4, precision=precision)
        for k in env:
            monkeypatch.delenv(k)
        out = s.run_stages(q, 2)
        s.close()
        return out

    ref = near(PDMK_NEAR_ROWS="0")
    np.testing.assert_array_equal(near(), ref)
    for parts in ("1", "4", "8"):
        np.testing.assert_array_equal(near(PDMK_NEAR_PARTS=parts), ref, err_msg=parts)
