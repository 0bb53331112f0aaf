"""Mesh-separable transform around its widest split panel (384 columns), where
the last stage changes kernels (k_sep_yx, then k_sep_y with k_sep_x) and at
default settings: against the direct transform."""
import numpy as np
import pytest

import phoebe_amd as P
from tests.helpers import rel_err, tiny_problem

pytestmark = pytest.mark.gpu


# 384 columns (the last split size), 405 and 480; 340 for 17 bands (never split)
@pytest.mark.parametrize("natoms,nw", [(8, 16), (9, 15), (10, 16), (6, 17)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 1e-6)])
@pytest.mark.parametrize("screen", [0.0, 6.0])
def test_separable_equals_direct(natoms, nw, precision, tol, screen):
    p = tiny_problem(natoms=natoms, nw=nw, rg_e=2, rg_p=2, mesh=(4, 5, 3), seed=19)
    gW = p.gw_host()
    ref = P.ElectronLinewidths(p, gW=gW, precision="fp64", transform="direct")
    ref.run()
    want = ref.linewidths(average=False)
    lw = P.ElectronLinewidths(p, gW=gW, precision=precision, transform="separable")
    lw.set_screen(screen)
    lw.set_timing(True)
    for _ in range(2):  # the second pass over buffers that hold the first one's stages
        lw.reset()
        lw.run()
        got = lw.linewidths(average=False)
        nz = want != 0
        assert nz.any() and np.array_equal(got != 0, nz)
        assert rel_err(got[nz], want[nz]).max() < tol
    lw.sync()
    assert (lw.split_times()["launches"] > 0) == (natoms * 3 * nw <= 384 and nw <= 16)
