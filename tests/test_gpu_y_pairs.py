"""y-stage of the mesh-separable transform, whose coordinates go in pairs jy,
my - jy, eight pairs per tile: y meshes of one point, without a self-paired
coordinate (odd) and with one (even), and on both sides of one and two tiles.
Against the direct transform, with the y-stage as a kernel of its own (fused
last stage) and inside the x-stage."""
import numpy as np
import pytest

import phoebe_amd as P
from tests.helpers import rel_err, tiny_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("my", [1, 2, 3, 15, 16, 17, 18, 32, 33, 34])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 1e-6)])
def test_y_meshes(my, precision, tol):
    p = tiny_problem(natoms=2, nw=4, rg_e=3, rg_p=4, mesh=(3, my, 2), seed=15)
    gW = p.gw_host()
    ref = P.ElectronLinewidths(p, gW=gW, precision="fp64", transform="direct")
    ref.run()
    want = ref.linewidths(average=False)
    assert (want != 0).any()
    for split in (0, 1):
        lw = P.ElectronLinewidths(p, gW=gW, precision=precision, transform="separable")
        lw.set_split_last_stage(split)
        lw.run()
        got = lw.linewidths(average=False)
        assert np.array_equal(got != 0, want != 0)
        nz = want != 0
        assert rel_err(got[nz], want[nz]).max() < tol
