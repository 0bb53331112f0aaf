"""cacheElPh over the column tilings of its kernel: Wannier counts on both sides
of every tile edge (several (Rp, nu) blocks per workgroup, one block on one,
two or four column waves, blocks in column passes), R_e counts that are not
whole quads, and batches of outer points on both sides of the 16-point tile."""
import numpy as np
import pytest

import phoebe_amd as P
from phoebe_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nw,nRe,nRp,nm", [(1, 1, 5, 3), (2, 3, 3, 6), (4, 9, 5, 3), (5, 7, 3, 3), (6, 5, 1, 3), (8, 13, 2, 3),
                                           (9, 6, 2, 3), (11, 11, 2, 3), (12, 4, 1, 6), (16, 10, 1, 3), (17, 5, 2, 3),
                                           (23, 6, 1, 3), (32, 7, 1, 3)])
def test_one_point_against_direct_sum(nw, nRe, nRp, nm, precision):
    rng = np.random.default_rng(100 * nw + nRe)
    cx = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    gW = cx(nRe, nRp, nm, nw, nw)
    Re, Rp = rng.integers(-3, 4, (nRe, 3)) * 1.7, rng.integers(-3, 4, (nRp, 3)) * 1.7
    dE, dP = rng.integers(1, 4, nRe).astype(float), rng.integers(1, 4, nRp).astype(float)
    nb1, nq = min(3, nw), 3
    U1 = np.linalg.qr(cx(nw, nw))[0][:, :nb1]
    U2 = [np.linalg.qr(cx(nw, nw))[0][:, :min(i + 1, nw)] for i in range(nq)]
    e3 = [cx(nm, nm) for _ in range(nq)]
    k1, q3 = rng.standard_normal(3), rng.standard_normal((nq, 3))
    inter = P.InteractionElPhWan(gW, Re, dE, Rp, dP, precision)
    inter.cacheElPh(U1, k1)
    inter.calcCouplingSquared(U1, U2, e3, q3)
    g1 = np.einsum("e,epvab,ac->pvcb", np.exp(1j * Re @ k1) / dE, gW, U1)
    # sums of nRe nw + nRp nw nm terms of order one, rounded per term
    tol = 1e-12 if precision == "fp64" else 2e-6
    for i in range(nq):
        g = np.einsum("p,pvcb,bd,vm->cdm", np.exp(1j * Rp @ q3[i]) / dP, g1, U2[i].conj(), e3[i])
        ref = np.abs(g) ** 2
        assert np.abs(inter.getCouplingSquared(i) - ref).max() <= tol * ref.max()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 2e-6)])
@pytest.mark.parametrize("nw,count", [(6, 15), (6, 16), (6, 17), (6, 32), (9, 31), (17, 20)])
def test_batches_equal_single_points(nw, count, precision, tol):
    prob = synth.make_problem(1, nw, 3, 3, (4, 3, 5), seed=60 + nw, window_ev=3.0)
    one = P.ElectronLinewidths(prob, precision=precision, k1_batch=1)
    k1 = np.arange(min(count, one.num_active), dtype=np.int32)
    assert len(k1) == count
    one.run(k1_list=k1)
    many = P.ElectronLinewidths(prob, precision=precision, k1_batch=32)
    many.run(k1_list=k1)
    a, b = one.linewidths(average=False), many.linewidths(average=False)
    m = a != 0
    assert m.any() and np.array_equal(m, b != 0)
    assert np.abs(b[m] / a[m] - 1).max() <= tol


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 2e-6)])
@pytest.mark.parametrize("mesh,nw", [((16, 2, 2), 9), ((17, 2, 2), 6), ((33, 2, 2), 6), ((52, 2, 1), 6), ((20, 2, 2), 17)])
def test_line_jobs_equal_gemm_batches(mesh, nw, precision, tol):
    """Mesh lines of 16 to 52 points: one, two or three tiles per job, several jobs per line."""
    prob = synth.make_problem(1, nw, 3, 3, mesh, seed=80 + nw, window_ev=3.0)
    gemm = P.ElectronLinewidths(prob, precision=precision, transform="separable" if nw < 17 else "direct")
    gemm.run()
    line = P.ElectronLinewidths(prob, precision=precision, transform="separable" if nw < 17 else "direct")
    line.set_line_batching(1)
    line.run()
    a, b = gemm.linewidths(average=False), line.linewidths(average=False)
    m = a != 0
    assert m.any() and np.array_equal(m, b != 0)
    assert np.abs(b[m] / a[m] - 1).max() <= tol
