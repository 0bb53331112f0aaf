"""Split last stage of the mesh-separable transform (k_sep_yx + k_sep_ep2) over
the sizes its kernels choose by: both precisions, mode counts on both sides of
each instance, y meshes around the 16-row tile, ragged column blocks, one to
four calculations, fixed and adaptive smearing.  Against the fused kernel (the
g3 are the same values, so to FP64 rounding) and against the oracle."""
import dataclasses

import numpy as np
import pytest

import phoebe_amd as P
from oracle import oracle as O
from phoebe_amd import synth
from tests.helpers import rel_err, tiny_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,natoms,nw,mesh,rg_p,nt,smearing", [
    ("fp64", 2, 6, (6, 17, 5), 3, 1, 0), ("fp64", 4, 16, (5, 4, 6), 3, 2, 0), ("fp64", 9, 5, (4, 3, 4), 2, 1, 0),
    ("fp64", 2, 7, (4, 16, 3), 3, 4, 1), ("fp64", 1, 9, (9, 5, 4), 4, 1, 0), ("fp32", 6, 10, (5, 6, 4), 3, 1, 0),
    ("fp32", 7, 8, (4, 5, 4), 2, 3, 0), ("fp32", 1, 9, (7, 16, 3), 3, 1, 0), ("fp32", 3, 16, (3, 33, 2), 4, 1, 1),
    ("fp32", 10, 3, (4, 4, 3), 2, 1, 0), ("fp32", 6, 16, (4, 5, 5), 4, 4, 1)])
def test_split_equals_fused_and_oracle(precision, natoms, nw, mesh, rg_p, nt, smearing):
    p = dataclasses.replace(tiny_problem(natoms=natoms, nw=nw, rg_e=3, rg_p=rg_p, mesh=mesh, seed=51))
    p.temperatures = p.temperatures[:1].repeat(nt) * np.arange(1, nt + 1)
    p.chem_pots = p.chem_pots[:1].repeat(nt)
    p.smearing = smearing
    gW = p.gw_host()
    out = []
    for split in (0, 1):
        lw = P.ElectronLinewidths(p, gW=gW, precision=precision, transform="separable")
        lw.set_split_last_stage(split)
        if not smearing:
            lw.set_screen(6.0)
        lw.set_timing(True)
        lw.run()
        lw.sync()
        assert (lw.split_times()["launches"] > 0) == bool(split)
        out.append(lw.linewidths(average=False))
    nz = out[0] != 0
    assert nz.any() and np.array_equal(out[1] != 0, nz)
    assert np.abs(out[1][nz] / out[0][nz] - 1).max() < 1e-12
    ref = O.Oracle(p, gW.reshape(-1)).linewidths()
    # adaptive widths: central differences summed in another order
    tol = 1e-6 if precision == "fp32" else 1e-7 if smearing else 1e-10
    assert rel_err(lw.linewidths(), ref).max() < tol


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("natoms,nw", [(1, 8), (2, 7), (3, 5), (4, 8), (5, 6), (8, 8)])
@pytest.mark.parametrize("nt,smearing", [(1, 1), (4, 1), (1, 0)])
def test_many_bands_per_point(precision, natoms, nw, nt, smearing):
    """Five to eight bands at every inner point: the epilogue's wide form, whose passes
    hold other numbers of rows (mesh lines of 13 points: whole passes and a remainder)."""
    p = synth.make_problem(natoms, nw, 3, 2, (13, 4, 3), seed=52, window_ev=30.0)
    p.temperatures = p.temperatures[:1] * np.arange(1, nt + 1)
    p.chem_pots = p.chem_pots[:1].repeat(nt)
    p.smearing = smearing
    out = []
    for split in (0, 1):
        lw = P.ElectronLinewidths(p, precision=precision, transform="separable")
        assert int((lw.band_hi - lw.band_lo).max()) + 1 == nw
        lw.set_split_last_stage(split)
        lw.set_timing(True)
        lw.run(k1_list=np.arange(0, lw.num_active, 11, dtype=np.int32))
        lw.sync()
        assert (lw.split_times()["launches"] > 0) == bool(split)
        out.append(lw.linewidths(average=False))
    nz = out[0] != 0
    assert nz.any() and np.array_equal(out[1] != 0, nz)
    assert np.abs(out[1][nz] / out[0][nz] - 1).max() < 1e-12
