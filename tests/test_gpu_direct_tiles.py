"""The direct coupling transform over its tilings: one, two and four column
waves, one and two row tiles per wave, panels in windows of modes, R_p counts
that are not whole quads, and point counts around the row tiles."""
import numpy as np
import pytest

import phoebe_amd as P
from phoebe_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nw,nm,nRp,nq", [(2, 3, 1, 1), (8, 6, 5, 65), (7, 9, 4, 33), (5, 15, 3, 16), (8, 18, 6, 31),
                                          (16, 12, 7, 33), (23, 15, 9, 17), (16, 24, 2, 15), (17, 24, 5, 18),
                                          (32, 12, 3, 2), (30, 27, 2, 16)])
def test_store_mode_against_direct_sum(nw, nm, nRp, nq, precision):
    rng = np.random.default_rng(7 * nw + nm)
    cx = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    gW = cx(2, nRp, nm, nw, nw)
    Re, Rp = rng.integers(-3, 4, (2, 3)) * 1.3, rng.integers(-3, 4, (nRp, 3)) * 1.3
    dE, dP = np.ones(2), rng.integers(1, 4, nRp).astype(float)
    U1 = np.linalg.qr(cx(nw, nw))[0][:, :2]
    U2 = [np.linalg.qr(cx(nw, nw))[0][:, :min(1 + i % 4, nw)] for i in range(nq)]
    e3 = [cx(nm, nm) for _ in range(nq)]
    k1, q3 = rng.standard_normal(3), rng.standard_normal((nq, 3))
    inter = P.InteractionElPhWan(gW, Re, dE, Rp, dP, precision)
    inter.cacheElPh(U1, k1)
    inter.calcCouplingSquared(U1, U2, e3, q3)
    g1 = np.einsum("e,epvab,ac->pvcb", np.exp(1j * Re @ k1) / dE, gW, U1)
    tol = 1e-12 if precision == "fp64" else 2e-6
    for i in range(nq):
        g3 = np.tensordot(np.exp(1j * Rp @ q3[i]) / dP, g1, axes=(0, 0))  # (nu, b1, w2)
        ref = np.abs(np.einsum("vcb,bd,vm->cdm", g3, U2[i].conj(), e3[i], optimize=True)) ** 2
        assert np.abs(inter.getCouplingSquared(i) - ref).max() <= tol * ref.max()


def _call(nw, nm, nb2, nq, precision, seed):
    rng = np.random.default_rng(seed)
    cx = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    gW = cx(1, 2, nm, nw, nw)
    U1, U2 = np.linalg.qr(cx(nw, nw))[0][:, :1], [np.linalg.qr(cx(nw, nw))[0][:, :nb2] for _ in range(nq)]
    e3, Rp, q3 = [cx(nm, nm) for _ in range(nq)], rng.integers(-3, 4, (2, 3)) * 1.3, rng.standard_normal((nq, 3))
    inter = P.InteractionElPhWan(gW, np.zeros((1, 3)), np.ones(1), Rp, np.ones(2), precision)
    inter.cacheElPh(U1, np.zeros(3))
    inter.calcCouplingSquared(U1, U2, e3, q3)
    g1 = np.einsum("epvab,ac->pvcb", gW, U1)
    for i in range(nq):
        g3 = np.tensordot(np.exp(1j * Rp @ q3[i]), g1, axes=(0, 0))
        ref = np.abs(np.einsum("vcb,bd,vm->cdm", g3, U2[i].conj(), e3[i], optimize=True)) ** 2
        assert np.abs(inter.getCouplingSquared(i) - ref).max() <= (1e-12 if precision == "fp64" else 2e-6) * ref.max()


@pytest.mark.parametrize("nw,nm,nb2,precision", [(31, 12, 31, "fp64"), (32, 36, 11, "fp64"), (31, 13, 31, "fp32"),
                                                 (29, 14, 29, "fp32")])
def test_windows_narrowed_by_many_bands(nw, nm, nb2, precision):
    """g' of the inner points' bands leaves LDS to a few modes per window."""
    _call(nw, nm, nb2, 2, precision, 5)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_too_many_bands_are_refused(precision):
    with pytest.raises(P.PhxError):
        _call(20, 24, 20, 1, precision, 6)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 2e-6)])
@pytest.mark.parametrize("natoms,nw", [(2, 8), (3, 8), (3, 12), (3, 16), (6, 16), (9, 17)])
def test_row_tiles_by_the_number_of_workgroups(natoms, nw, precision, tol):
    """A point alone takes 16 rows per workgroup, a batch of points 32 or 64, and runs
    of either may follow the other; the linewidths of the points are the same."""
    p = synth.make_problem(natoms, nw, 2, 3, (9, 8, 9), seed=23, window_ev=3.0)
    lw = P.ElectronLinewidths(p, precision=precision, transform="direct", k1_batch=32)
    k1 = np.arange(40, 72, dtype=np.int32)
    panels = int((lw.band_hi - lw.band_lo + 1)[k1].sum())
    assert -(-lw.num_active // 32) * panels > 256 >= -(-lw.num_active // 32) * int((lw.band_hi - lw.band_lo + 1).max())
    out = []
    for batch in (1, 32, 1, 32):
        lw.reset()
        lw.set_batching(k1_batch=batch)
        lw.run(k1_list=k1)
        out.append(lw.linewidths(average=False))
    nz = out[0] != 0
    assert nz.any()
    for o in out[1:]:
        assert np.array_equal(o != 0, nz) and np.abs(o[nz] / out[0][nz] - 1).max() <= tol
