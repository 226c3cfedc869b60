"""FP32 tensor transforms at p = 18: the matrix-core blocks against the vector kernel, bit for bit.

A tensor-transform knob of 2 takes the vector kernel (k_tensor3); the default takes
k_tensor3_m4, whose outputs are the same chains of fused multiply-adds.  The trees have folded
and unfolded boxes, deep and shallow branches (expansions added to), child -> parent levels with
one item per child and fused per parent (PDMK_C2P_FUSE=1, inputs added in order), and two
vectors along z (quasi-periodic)."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell", ["cubic", "triclinic"])
@pytest.mark.parametrize("fuse", ["1", "1000000"])
@pytest.mark.parametrize("bloch", [None, (0.3, -0.2, 0.5)])
def test_same_bits_as_vector_kernel(pdmk, cuda, monkeypatch, cell, fuse, bloch):
    H = W.cubic_cell() if cell == "cubic" else W.triclinic_cell()
    n = 3001
    u = W.uniform01(17, 3 * n).reshape(n, 3)
    u[n // 2 :] = 0.05 + 0.1 * u[n // 2 :]  # half the points in one corner: several levels there
    q = 2.0 * W.uniform01(18, n) - 1.0
    q -= q.mean()
    monkeypatch.setenv("PDMK_C2P_FUSE", fuse)
    s = pdmk.PDMKSolver(H, u @ H.T, n_digits=6, n_per_leaf=20, nz=4, precision="float", bloch=bloch)
    assert s.stats()["n_levels"] >= 3
    got = []
    for div in (1, 2):
        s.knobs(**{s.KNOBS[4]: div})
        got.append(s.evaluate(q) if bloch is None else s.evaluate_complex(q))
    s.close()
    np.testing.assert_array_equal(got[0], got[1])
