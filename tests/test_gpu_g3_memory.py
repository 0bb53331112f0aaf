"""Device memory of the split last stage: no x-stage slabs (T2) beside the fused
y-stage, and what it does without when the g3 rows,
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


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_fused_y_stage_holds_no_slabs(precision):
    def used(fused, chunk):
        lw = _handle(precision)
        lw.set_panel_chunk(chunk)
        lw.set_fused_y_stage(fused)
        lw.sync()
        free = torch.cuda.mem_get_info()[0]
        lw.run(k1_list=np.arange(4, dtype=np.int32))
        lw.sync()
        return free - torch.cuda.mem_get_info()[0]

    # FP32: k_sep_xg's slabs; FP64: the fused last stage's, which has no g3 rows
    elem = 8 if precision == "fp32" else 16
    slabs, rows = 8000 * 16 * 16 * 12 * elem, 0 if precision == "fp32" else 8000 * int(np.prod(MESH)) * 12 * elem
    used(True, 4), used(False, 4)  # the runtime's own memory for these kernels
    a, b = used(True, 8000), used(False, 8000)
    assert abs((b - a) - (slabs - rows)) < 0.2 * slabs, (a, b, slabs, rows)
