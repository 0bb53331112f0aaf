"""Phonon linewidths when a batch of outer points needs several coupling launches
(their |g|^2 would exceed the builder's 2 GiB): the sums are the same bit for bit
as point by point."""
import numpy as np
import pytest

import phoebe_amd as P
from phoebe_amd import synth

pytestmark = pytest.mark.gpu


def test_groups_equal_single_points():
    prob = synth.make_problem(6, 16, 2, 2, 13, seed=77, window_ev=20.0)  # all 16 bands everywhere
    inter = P.InteractionElPhWan(None, prob.Re, prob.degE, prob.Rp, prob.degP, "fp64",
                                 synthetic=(prob.nw, prob.nm, prob.gw_decay, prob.gw_seed))
    ph = P.PhononElectronLinewidths(prob, inter, (13, 13, 13))
    k1 = np.arange(5, 37, dtype=np.int32)
    ph.set_timing(True)
    ph.run(k1)
    assert ph.kernel_times()["coupling_launches"] == 2
    ph.set_timing(False)
    a = ph.linewidths(average=False)
    ph.reset()
    for k in k1:
        ph.run(np.array([k], dtype=np.int32))
    b = ph.linewidths(average=False)
    assert np.any(a) and np.array_equal(a, b)
