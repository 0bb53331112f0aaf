"""Energy screen of the mesh-separable transform: the panels' closest approach
to resonance and the row masks of the last stage, over line lengths on both
sides of the lane counts a slot takes (16, 32, 64), one row and more rows than
a wave lists, and mode counts that are not powers of two.  The rows the last
stage computed, counted by their bands, against the rule restated here."""
import dataclasses

import numpy as np
import pytest

import phoebe_amd as P
from oracle import oracle as O
from tests.helpers import tiny_problem

pytestmark = pytest.mark.gpu


def kept_bands(p, n):
    """Band counts summed over the rows each panel keeps: certain, and undecided to rounding."""
    o = O.Oracle(p, p.gw_host().reshape(-1))
    w = o.phonons()[0]
    nb = o.band_hi - o.band_lo + 1
    e = np.split(o.energies, np.cumsum(nb)[:-1])
    m = np.array(p.mesh)
    xyz = np.stack(np.unravel_index(o.active, p.mesh, order="F"), 1)
    on = w >= O.phonon_cutoff()
    wlo = np.where(on, w, np.inf).min(1)
    whi = np.where(on, w, -np.inf).max(1)
    sure = unsure = 0
    for a in range(len(nb)):
        q = np.ravel_multi_index(tuple(((xyz - xyz[a]) % m).T), p.mesh, order="F")
        ok = on[q].any(1)
        for e1 in e[a]:
            best = np.inf
            for r in np.flatnonzero(ok):
                om = w[q[r]][on[q[r]]]
                for x in ((e1 - e[r][:, None] + om) / p.sigma, (e1 - e[r][:, None] - om) / p.sigma):
                    best = min(best, np.abs(x[x <= 6]).min(initial=np.inf))
            lim = (np.hypot(best, n) if np.isfinite(best) else n) * p.sigma
            for r in np.flatnonzero(ok):
                lo, hi = e1 - e[r][-1], e1 - e[r][0]
                ivs = ((lo + wlo[q[r]], hi + whi[q[r]]), (lo - whi[q[r]], hi - wlo[q[r]]))
                keep = [any(hi2 > -l and lo2 < l for lo2, hi2 in ivs) for l in (lim * (1 - 1e-7), lim * (1 + 1e-7))]
                sure += nb[r] * keep[0]
                unsure += nb[r] * (keep[1] and not keep[0])
    return sure, unsure


@pytest.mark.parametrize("mesh,natoms,width", [((1, 3, 2), 2, 4.), ((5, 3, 2), 1, 12.), ((16, 2, 2), 3, 6.),
                                               ((17, 2, 1), 2, 6.), ((32, 1, 2), 2, 20.), ((33, 2, 2), 2, 6.),
                                               ((64, 1, 1), 5, 6.)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_rows_of_the_last_stage(mesh, natoms, width, precision):
    p = tiny_problem(natoms=natoms, nw=4, rg_e=3, rg_p=2, mesh=mesh, seed=77)
    p = dataclasses.replace(p, sigma=p.sigma / width)  # narrow: the least screen is 6 sigma
    lw = P.ElectronLinewidths(p, gW=p.gw_host(), precision=precision, transform="separable")
    lw.set_screen(6.0)
    lw.set_timing(True)
    lw.run()
    lw.sync()
    got = lw.split_times()["bands"]
    sure, unsure = kept_bands(p, 6.0)
    assert sure <= got <= sure + unsure, (got, sure, unsure)
    assert got > 0
