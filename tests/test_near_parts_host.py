"""CPU test of the near field's part lists (several waves per item): the cuts of an item's list
entries, and the sizes past which an item keeps one wave.

Every row of a part is padded to the part's longest row.  When the longest row changes from part
to part, the parts together hold up to n_parts times the undivided list's steps, so the
undivided list's size says nothing of theirs.
"""
import ctypes as C

import numpy as np
import pytest

INT_MAX = 2 ** 31 - 1


def parts(pdmk, c, s):
    c = np.ascontiguousarray(c, dtype=np.int32)
    out = np.zeros((s, 3), dtype=np.int32)
    p = C.POINTER(C.c_int)
    assert pdmk.lib().pdmk_host_row_parts(c.ctypes.data_as(p), c.shape[0], s, out.ctypes.data_as(p)) == 0
    return out


@pytest.mark.parametrize("s", [4, 8])
@pytest.mark.parametrize("ne", [0, 1, 3, 27, 255])
def test_cuts_cover_the_entries(pdmk, s, ne):
    c = np.random.default_rng(ne + s).integers(0, 9, (ne, 16))
    out = parts(pdmk, c, s)
    assert out[0, 0] == 0 and out[-1, 1] == ne
    np.testing.assert_array_equal(out[1:, 0], out[:-1, 1])
    for b, e, k in out:
        longest = int(c[b:e].sum(axis=0).max()) if e > b else 0
        assert k == (longest + 3) // 4 * 4
    if ne >= 4 * s:  # even shares, to the largest entry's steps
        share = np.array([c[b:e].sum() for b, e, _ in out])
        assert np.abs(share - c.sum() / s).max() <= c.sum(axis=1).max()


@pytest.mark.parametrize("s", [4, 8])
def test_parts_that_outgrow_the_undivided_list(pdmk, s):
    # part p's steps all in row p: 50000 steps a row, 16 rows; 2560 items as in the largest tree cut
    c = np.zeros((s, 16), dtype=np.int32)
    c[np.arange(s), np.arange(s)] = 50_000
    out = parts(pdmk, c, s)
    items, whole = 2560, 16 * 50_000
    cut = 16 * int(out[:, 2].sum())
    assert cut == s * whole
    free = 288 << 30
    fit = pdmk.lib().pdmk_host_row_lists_fit
    assert items * whole <= INT_MAX and fit(items * whole, 0, free) == 1
    assert items * cut > INT_MAX and fit(items * cut, items * whole, free) == 0


def test_limits(pdmk):
    fit = pdmk.lib().pdmk_host_row_lists_fit
    big = 1 << 40
    assert fit(INT_MAX, 0, big) == 1 and fit(INT_MAX + 1, 0, big) == 0
    assert fit(1000, 24, 16 * 1024) == 1 and fit(1000, 25, 16 * 1024) == 0
