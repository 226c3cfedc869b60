"""evaluate() with its stages on three streams, on one stream, and in a captured graph gives the
same potentials bit for bit, on both sides of the rules that choose: small trees on one
stream (FP64 3 digits up to 1400 points, 6 digits up to 1000, 5 digits none), and the near field
sent out before the chain (FP64 at 1 to 5 digits, 320 to 8192 items: N = 2e4 to 3e5), in
workgroups of 2 items where few boxes carry the chain (4 and 5 digits, cubic).
Three calls on changing charges, so that a call which ran ahead of the one before would show."""
import numpy as np
import pytest

from periodicdmk_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("digits,n", [(3, 1400), (3, 1401), (5, 500), (6, 1000), (6, 1001), (5, 10_000),
                                      (5, 20_000), (3, 60_000), (6, 60_000), (5, 150_000)])
def test_streams_agree(pdmk, cuda, digits, n):
    cell = W.cubic_cell() if n > 100_000 else W.triclinic_cell()
    s = pdmk.PDMKSolver(cell, W.uniform_positions(n, 100 + n, cell), n_digits=digits, n_per_leaf=300, nz=4,
                        precision="double")
    charges = [W.neutral_uniform_charges(n, 70 + i) for i in range(3)]
    dq, out = [pdmk.DeviceArray.from_numpy(q) for q in charges], [pdmk.DeviceArray(n, np.float64) for _ in charges]

    def run():
        for q, o in zip(dq, out):
            s.evaluate_device(q.ptr, o.ptr)
        pdmk.synchronize()
        return [o.numpy() for o in out]

    three = run()
    s.set_single_stream(True)
    one = run()
    s.set_single_stream(False)
    for o in out:
        o.upload(np.zeros(n))
    g = pdmk.BatchGraph([(s, q, o) for q, o in zip(dq, out)], n_branches=1)
    for _ in range(3):
        g.launch()
        pdmk.synchronize()
        for a, b, o in zip(three, one, out):
            np.testing.assert_array_equal(a, b)
            np.testing.assert_array_equal(a, o.numpy())
        run()
    g.close()
    s.close()
