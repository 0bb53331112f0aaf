"""Device memory of the split last stage: what it does without when the g3 rows,
or the second set of them that the epilogue overlap takes, find no room.  Chunks
of more panels than fit are asked for; every other buffer of the problem is
small (one mesh line of R_ph)."""
import numpy as np
import pytest
import torch

import phoebe_amd as P
from tests.helpers import tiny_problem

pytestmark = pytest.mark.gpu

MESH = (64, 16, 16)


def _handle(precision="fp32"):
    p = tiny_problem(natoms=1, nw=4, rg_e=3, rg_p=1, mesh=MESH, seed=3)
    return P.ElectronLinewidths(p, precision=precision, transform="separable", k1_batch=8)


def _chunk(share, precision="fp32"):
    """Panels whose g3 rows take this share of the card (complex, 12 columns, or g' of 8 bands)."""
    lw = _handle(precision)
    nb2 = int((lw.band_hi - lw.band_lo).max()) + 1
    per = np.prod(MESH) * max(12 * (8 if precision == "fp32" else 16), 2 * nb2 * 3 * 8)
    return int(share * torch.cuda.mem_get_info()[1] / per) + 1


def _run(chunk, overlap=False, precision="fp32"):
    lw = _handle(precision)
    lw.set_panel_chunk(chunk)
    lw.set_epilogue_overlap(overlap)
    lw.set_timing(True)
    lw.run(k1_list=np.arange(4, dtype=np.int32))
    lw.sync()
    return lw.linewidths(average=False), lw.split_times()["launches"]


@pytest.mark.parametrize("share,overlap,split", [(1.2, False, False), (0.55, True, True)])
def test_no_room(share, overlap, split):
    want, n = _run(0)
    assert n > 0 and want.any()
    got, n = _run(_chunk(share), overlap)
    assert (n > 0) == split
    assert np.array_equal(got != 0, want != 0)
    nz = want != 0
    assert np.abs(got[nz] / want[nz] - 1).max() < 1e-12
