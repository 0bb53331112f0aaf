"""The work a user of phoebe_amd has it do, as cases that can be timed.

A case is one pass through the package's public entry points: electron
linewidths of a batch of outer points in the forms that are used (plain FP64,
FP64 and FP32 mesh-separable, the builder's own choice, adaptive smearing, a
planned sweep replayed as a graph), phonon linewidths, one outer point through
the InteractionElPhWan calls, bands along a path and a batch of Hermitian
eigensolves on device buffers.  The systems are the package's synthetic ones
(phoebe_amd.synth), whose inputs come from the seed alone.
"""
from __future__ import annotations

import concurrent.futures
import math

import numpy as np
import torch

import phoebe_amd as P
from phoebe_amd import synth

CM1_RY = 1.0 / 109737.3156809956   # 1 cm^-1 in Ry
PHONON_CUTOFF = 5.0 * CM1_RY
LINE_FORMS = ("line32s6", "line64s6")


def _lw(name, form, natoms, nw, re, rp, mesh, lines=0, calcs=1, adaptive=False, graph=False):
    """Electron linewidths of whole mesh lines of outer points (lines = 0: every
    active point) against every active inner point."""
    c = dict(kind="lw", form=form, natoms=natoms, nw=nw, re=re, rp=rp, m0=mesh[0], m1=mesh[1], m2=mesh[2],
             lines=lines, calcs=calcs, adaptive=adaptive, graph=graph)
    return dict(c, name=name) if name else c


def listed():
    return [
        # electron bands along a path of a small crystal: the smallest call, host arrays in and out
        dict(name="bands_path", kind="bands", nk=101, nw=8, re=7),
        # eigensolves of H(k) on buffers that stay on the GPU (the step inside every band structure)
        dict(name="zheev_16", kind="zheev", n=16, count=32768),
        # one outer point through cacheElPh and calcCouplingSquared, as the reference's callers drive it
        dict(name="coupling_call", kind="couple", natoms=2, nw=8, re=7, rp=6, nq=1000, nb1=2, precision="fp64"),
        # a small crystal's whole sweep in the reference's own algorithm, FP64
        _lw("si_fp64", "fp64", 2, 8, 7, 6, (12, 12, 12)),
        # the same sweep in the fastest form
        _lw("si_chosen", "line32s6", 2, 8, 7, 6, (12, 12, 12)),
        # a planned sweep of a small odd system replayed as a graph, four (T, mu) pairs
        _lw("graph_calcs", "sep32s", 3, 9, 5, 5, (9, 8, 7), calcs=4, graph=True),
        # a crystal outside the narrow kernels (23 x 15 columns), ragged mesh, the builder picks the form
        _lw("odd_auto", "auto", 5, 23, 5, 4, (11, 13, 9), lines=24),
        # adaptive smearing on a metal-like grid
        _lw("adaptive", "line32s6", 3, 10, 6, 5, (20, 20, 20), lines=16, adaptive=True),
        # six atoms, 18 modes: the mesh-separable form beyond 192 columns
        _lw("six_atoms", "line32s6", 6, 16, 7, 6, (32, 32, 32), lines=4),
        # FP64 throughout with the exact algorithmic savings
        _lw("separable_fp64", "line64s6", 4, 16, 7, 7, (27, 28, 29), lines=6),
        # the package's headline system: 16 bands, 12 modes, 40^3 mesh, one stream of 16 mesh lines
        _lw("large_chosen", "line32s6", 4, 16, 10, 9, (40, 40, 40), lines=16),
        # phonon linewidths of every phonon of a mesh from a batch of outer electron points
        dict(name="phonon_lw", kind="phel", natoms=3, nw=12, re=6, rp=5, mesh=16, count=32, precision="fp64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("bands", "zheev", "couple", "lw", "lw", "lw", "lw", "lw", "phel"))
    if kind == "bands":
        return dict(kind=kind, nk=_log_int(rng, 30, 2000), nw=rng.randint(4, 24), re=rng.randint(4, 7))
    if kind == "zheev":
        n = rng.randint(4, 30)
        return dict(kind=kind, n=n, count=min(_log_int(rng, 64, 65536), 32768 * 4096 // n ** 3))
    if kind == "couple":
        return dict(kind=kind, natoms=rng.randint(1, 5), nw=rng.randint(4, 14), re=rng.randint(4, 6),
                    rp=rng.randint(3, 6), nq=_log_int(rng, 40, 3000), nb1=rng.randint(1, 4),
                    precision=rng.choice(("fp64", "fp32")))
    if kind == "phel":
        return dict(kind=kind, natoms=rng.randint(1, 4), nw=rng.randint(4, 12), re=rng.randint(3, 6),
                    rp=rng.randint(3, 5), mesh=rng.randint(6, 16), count=rng.randint(4, 32), precision="fp64")
    form = rng.choice(("fp64", "auto", "sep32s", "line64s6", "line32s6", "line32s6"))
    big = form in LINE_FORMS
    natoms = rng.randint(1, 6)
    nw = rng.randint(4, 16 if form != "auto" else 24)
    top = 32 if form == "line32s6" else 24 if form == "line64s6" else 14
    mesh = tuple(max(6, min(top, _log_int(rng, 6, top) + rng.randint(-1, 1))) for _ in range(3))
    return _lw("", form, natoms, nw, rng.randint(4, 7 if big else 6), rng.randint(4, 7 if big else 5), mesh,
               lines=rng.randint(2, 16), calcs=rng.choice((1, 1, 1, 2, 4)),
               adaptive=rng.random() < 0.2, graph=rng.random() < 0.25)


# ---------------------------------------------------------------- inputs
def _mesh(case):
    return (case["mesh"],) * 3 if case["kind"] == "phel" else (case["m0"], case["m1"], case["m2"])


def _problem(case, seed):
    """The electrons, and so the states of the window, come with the sizes; the seed
    draws the coupling and the atoms' masses."""
    prob = synth.make_problem(case["natoms"], case["nw"], case["re"], case["rp"], _mesh(case), seed=1000)
    rng = np.random.default_rng(seed)
    prob.gw_seed = int(rng.integers(1, 2 ** 62))
    prob.masses = prob.masses * np.repeat(rng.uniform(0.8, 1.2, case["natoms"]), 3)
    calcs = case.get("calcs", 1)
    prob.temperatures = prob.temperatures[0] * np.array([1.0 + 0.5 * i for i in range(calcs)])
    prob.chem_pots = prob.chem_pots[0] + 1.0e-3 * np.arange(calcs)
    prob.smearing = int(case.get("adaptive", False))
    return prob


def _pick_lines(active, m0, lines, seed):
    """Active indices of the outer points on `lines` mesh lines (0: None, all points)."""
    if not lines:
        return None
    line = np.asarray(active) // m0
    pick = np.random.default_rng(seed + 17).permutation(np.unique(line))[:lines]
    return np.concatenate([np.flatnonzero(line == x) for x in pick]).astype(np.int32)


def _pick_points(num_active, count, seed):
    return np.random.default_rng(seed + 29).permutation(num_active)[:count].astype(np.int32)


def _unitary_columns(rng, count, n, cols):
    a = rng.standard_normal((count, n, n)) + 1j * rng.standard_normal((count, n, n))
    return np.ascontiguousarray(np.linalg.qr(a)[0][:, :, :cols])


def _couple_inputs(case, seed):
    """Band and phonon eigenvectors of one outer point and its wavevectors."""
    prob = synth.make_problem(case["natoms"], case["nw"], case["re"], case["rp"], 4, seed=seed)
    rng = np.random.default_rng(seed + 41)
    nw, nm, nq = case["nw"], 3 * case["natoms"], case["nq"]
    U1 = _unitary_columns(rng, 1, nw, case["nb1"])[0]
    nb2 = np.random.default_rng(nq).integers(1, min(5, nw) + 1, nq)  # of the sizes, not of the seed
    u = _unitary_columns(rng, nq, nw, nw)
    U2 = [np.ascontiguousarray(u[i, :, :nb2[i]]) for i in range(nq)]
    e3 = list(_unitary_columns(rng, nq, nm, nm) / math.sqrt(prob.masses[0]))
    k1 = prob.recip @ rng.uniform(0, 1, 3)
    q3 = (prob.recip @ rng.uniform(0, 1, (3, nq))).T
    return prob, U1, U2, e3, k1, np.ascontiguousarray(q3)


def _hermitian(case, seed):
    """Hermitian matrices with the spread of H(k): (count, n, n) complex."""
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(case["count"], case["n"], case["n"], dtype=torch.complex128, generator=g)
    return 0.1 * (a + a.conj().transpose(1, 2))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "bands":
        f = synth.eig_family("el", case["nw"], seed=seed, rgrid=case["re"])
        return dict(kind=kind, k=_path(case, seed, f), **f)
    if kind == "zheev":
        n, m = case["n"], case["count"]
        return dict(kind=kind, A=_hermitian(case, seed).transpose(1, 2).contiguous().cuda(), n=n, count=m,
                    W=torch.empty(m, n, dtype=torch.float64, device="cuda"),
                    info=torch.empty(m, dtype=torch.int32, device="cuda"))
    if kind == "couple":
        prob, U1, U2, e3, k1, q3 = _couple_inputs(case, seed)
        inter = P.InteractionElPhWan(None, prob.Re, prob.degE, prob.Rp, prob.degP, case["precision"],
                                     synthetic=(prob.nw, prob.nm, prob.gw_decay, prob.gw_seed))
        return dict(kind=kind, inter=inter, U1=U1, U2=U2, e3=e3, k1=k1, q3=q3)
    prob = _problem(case, seed)
    if kind == "phel":
        inter = P.InteractionElPhWan(None, prob.Re, prob.degE, prob.Rp, prob.degP, case["precision"],
                                     synthetic=(prob.nw, prob.nm, prob.gw_decay, prob.gw_seed))
        ph = P.PhononElectronLinewidths(prob, inter, _mesh(case))
        return dict(kind=kind, ph=ph, k1=_pick_points(ph.num_active, case["count"], seed))
    if case["form"] == "auto":
        lw = P.linewidths_auto(prob)
    elif case["adaptive"]:  # the energy screen needs a fixed width: the form without it
        precision, transform, _, line_min = P.FORMS[case["form"]]
        lw = P.ElectronLinewidths(prob, precision=precision, transform=transform)
        lw.set_line_batching(line_min)
    else:
        lw = P.linewidths_form(prob, case["form"])
    k1 = _pick_lines(lw.active, case["m0"], case["lines"], seed)
    if case["graph"]:
        lw.plan(k1)
    return dict(kind=kind, lw=lw, k1=k1, graph=case["graph"])


def _path(case, seed, f):
    ends = np.random.default_rng(seed + 3).uniform(0, 1, (2, 3))
    t = np.linspace(0, 1, case["nk"])[:, None]
    return np.ascontiguousarray((f["recip"] @ ((1 - t) * ends[0] + t * ends[1]).T).T)


# ---------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "bands":
        E, U = P.el_bloch_diag(state["k"], state["R"], state["weight"], state["coef"])
        # eigenvectors are defined up to a phase: the first component real and positive
        ph = U[:, :1, :].conj()
        return {"E": E, "U": np.ascontiguousarray(U * (ph / np.abs(ph)))}
    if kind == "zheev":
        V = state["A"].clone()  # the call works in place
        rc = P.lib().phx_zheev_batched_dev(state["count"], state["n"], V.data_ptr(), state["W"].data_ptr(),
                                           state["info"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise P.PhxError(P.lib().phx_last_error().decode())
        return {"W": state["W"], "V": V * torch.sgn(V[:, :, :1].conj())}  # row j: eigenvector j, phase fixed as above
    if kind == "couple":
        inter = state["inter"]
        inter.cacheElPh(state["U1"], state["k1"])
        inter.calcCouplingSquared(state["U1"], state["U2"], state["e3"], state["q3"])
        return np.concatenate([inter.getCouplingSquared(i).reshape(-1, order="F") for i in range(len(state["U2"]))])
    if kind == "phel":
        ph = state["ph"]
        ph.reset()
        ph.run(state["k1"])
        return ph.linewidths()
    lw = state["lw"]
    lw.reset()
    if state["graph"]:
        lw.plan_run(graph=True)
    else:
        lw.run(k1_list=state["k1"])
    return lw.linewidths()


# ---------------------------------------------------------------- work and tolerance
_COUNTS = {}


def _vectors(grid):
    """Wigner-Seitz vectors of a grid^3 supercell, and the distinct (x, y) and x coordinates among them."""
    if grid not in _COUNTS:
        A = synth._fcc(10.26)
        R = synth.ws_vectors((grid,) * 3, A)[0]
        n = np.rint(np.linalg.solve(A, R.T).T).astype(int)
        _COUNTS[grid] = (len(R), len({tuple(x[:2]) for x in n}), len({x[0] for x in n}))
    return _COUNTS[grid]


def work(case):
    kind = case["kind"]
    if kind == "bands":
        n, nR = case["nw"], _vectors(case["re"])[0]
        return {"bytes": 16.0 * n * n * (nR + case["nk"]) + 8.0 * case["nk"] * (n + 3),
                "flops": case["nk"] * (8.0 * nR * n * n + 23.0 * n ** 3)}
    if kind == "zheev":
        n = case["n"]
        return {"bytes": case["count"] * (32.0 * n * n + 8.0 * n), "flops": 23.0 * n ** 3 * case["count"]}
    nw, nm = case["nw"], 3 * case["natoms"]
    nRe, linesE, grpE = _vectors(case["re"])
    nRp, linesP, grpP = _vectors(case["rp"])
    ncol = nm * nw
    gw = float(nRe) * nRp * nm * nw * nw
    if kind == "couple":
        nb2, nb1, elem = 0.5 * (1 + min(5, nw)), case["nb1"], 16.0 if case["precision"] == "fp64" else 8.0
        return {"bytes": elem * gw + case["nq"] * (16.0 * nw * nb2 + 16.0 * nm * nm + 8.0 * nb1 * nb2 * nm),
                "flops": 8.0 * gw + 8.0 * nRp * ncol * nw * nb1
                + case["nq"] * nb1 * 8.0 * (nRp * ncol + ncol * nb2 + nm * nm * nb2)}
    # about a tenth of the bands lie in the window
    m = _mesh(case)
    points, band = float(m[0] * m[1] * m[2]), 0.1 * nw
    active = points * min(1.0, 0.15 * nw)
    if kind == "phel":
        outer = case["count"] * max(1.0, band)
        return {"bytes": 16.0 * gw + points * (16.0 * nw * nw + 16.0 * nm * nm + 8.0 * nm),
                "flops": 8.0 * gw * case["count"]
                + outer * points * 8.0 * (nRp * ncol + ncol * nw + nm * nm * nw)}
    form = case["form"]
    fp64 = form in ("fp64", "line64s6")
    outer_points = case["lines"] * m[0] * min(1.0, 0.15 * nw) if case["lines"] else active
    lines = case["lines"] or m[1] * m[2]
    panels = outer_points * max(1.0, band / min(1.0, 0.15 * nw))
    direct = form == "fp64" or (form == "auto" and ncol > 192)
    keep = 0.45 if not direct and not case["adaptive"] else 1.0
    if direct:
        transform = active * 8.0 * nRp * ncol
    else:
        transform = 8.0 * ncol * (nRp * m[2] + linesP * m[1] * m[2] + grpP * keep * active)
    rows = keep * active * 8.0 * (ncol + nm * nm) * max(1.0, band)
    cache = 8.0 * (gw * lines + grpE * gw / nRe * outer_points)
    return {"bytes": (16.0 if fp64 else 8.0) * gw + points * (16.0 * nw * max(1.0, band) + 16.0 * nm * nm),
            "flops": cache + panels * (transform + rows)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("bands", "zheev"):
        return {"rel": 1e-12, "max": 1e-8}  # 1e-14 seen; eigenvectors of close levels move more
    fp32 = case.get("precision") == "fp32" or case.get("form") in ("auto", "sep32s", "line32s6")
    if fp32:
        return {"rel": 3e-7, "max": 1e-5}  # up to 7e-8 seen against 64 bits
    # adaptive widths come from central differences with a step of 1e-8
    return {"rel": 1e-7, "max": 1e-5} if case.get("adaptive") else {"rel": 1e-11, "max": 1e-9}  # 2e-13 seen


# ---------------------------------------------------------------- the same in 64 bits, plain torch and numpy
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _c(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.complex128, device=_device())


def _d(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_device())


def _eigh(H):
    """Eigen-decomposition of a stack on the host's cores."""
    H = H.cpu().numpy()
    with concurrent.futures.ThreadPoolExecutor(16) as ex:
        parts = list(ex.map(np.linalg.eigh, np.array_split(H, max(1, min(64, len(H) // 64)))))
    return np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts])


def _phases(k, R, sign=1.0):
    a = sign * (_d(k) @ _d(R).T)
    return torch.complex(torch.cos(a), torch.sin(a))


def _electrons(k, R, deg, h):
    n = h.shape[1]
    H = torch.cat([(_phases(kk, R) / _d(deg)) @ _c(h).reshape(len(R), n * n) for kk in np.array_split(k, len(k) // 8192 + 1)])
    return _eigh(H.reshape(-1, n, n))


def _phonons(q, prob):
    """omega (nq, nm) and e / sqrt(M) (nq, nm, nm)."""
    n = prob.nm
    D = torch.cat([(_phases(qq, prob.Rf, -1.0) * _d(prob.wf)) @ _c(prob.mat2R).reshape(len(prob.Rf), n * n)
                   for qq in np.array_split(q, len(q) // 8192 + 1)]).reshape(-1, n, n)
    D = 0.5 * (D + D.conj().transpose(1, 2)) / _d(np.sqrt(np.outer(prob.masses, prob.masses)))
    lam, e = _eigh(D)
    return np.sign(lam) * np.sqrt(np.abs(lam)), e / np.sqrt(prob.masses)[None, :, None]


def _mesh_points(prob):
    """Integer coordinates (x fastest) and Cartesian points of the mesh."""
    m = prob.mesh
    i = np.arange(m[0] * m[1] * m[2])
    n = np.stack([i % m[0], (i // m[0]) % m[1], i // (m[0] * m[1])], -1)
    return n, (prob.recip @ (n / np.array(m, dtype=float)).T).T


def _mix(x):
    for s, mul in ((30, 0xBF58476D1CE4E5B9), (27, 0x94D049BB133111EB)):
        x = (x ^ ((x >> s) & ((1 << (64 - s)) - 1))) * (mul - (1 << 64))
    return x ^ ((x >> 31) & ((1 << 33) - 1))


def _normal(seed, idx):
    """The synthetic coupling's normal deviate of a counter, in torch integers."""
    s = torch.zeros(idx.shape, dtype=torch.float64, device=idx.device)
    for j in range(4):
        h = _mix((idx * 4 + j) * (synth.GW_HASH_MUL - (1 << 64)) + seed)
        s = s + ((h >> 11) & ((1 << 53) - 1)).to(torch.float64) / 9007199254740992.0
    return (s - 2.0) * math.sqrt(3.0)


def _cache(prob, k, U):
    """sum_Re e^{ik.Re} gW / deg rotated by U1, per point: list of (nRp, nw (w2), nm, nb1) complex."""
    nw, nm, nRp, nRe = prob.nw, prob.nm, prob.nRp, prob.nRe
    per = nRp * nm * nw * nw
    ph = _phases(k, prob.Re) / _d(prob.degE)
    acc = torch.zeros(len(k), per, dtype=torch.complex128, device=_device())
    decay = _d(prob.gw_decay)
    step = max(1, int(6.0e7 // per))
    for r in range(0, nRe, step):
        n = min(step, nRe - r)
        f = torch.arange(r * per, (r + n) * per, dtype=torch.int64, device=_device())
        g = torch.complex(_normal(prob.gw_seed, 2 * f), _normal(prob.gw_seed, 2 * f + 1))
        g = (g.reshape(n, nRp, -1) * decay[r:r + n, :, None]).reshape(n, per)
        acc += ph[:, r:r + n] @ g
    out = []
    for i, u in enumerate(U):
        g = acc[i].reshape(nRp, nm, nw, nw)  # (Rp, nu, w1, w2)
        out.append(torch.tensordot(g, _c(u), dims=([2], [0])).permute(0, 2, 1, 3).contiguous())
    return out


def _coupling(g2, phase, U2, e3):
    """|g|^2 (rows, b2, nu, b1): phase (rows, nRp), U2 (rows, nw, nb2), e3 (rows, nm, nm)."""
    nRp, nw, nm, nb1 = g2.shape
    out = []
    for rows in torch.split(torch.arange(len(phase), device=phase.device), max(1, int(4.0e8 // (nw * nm * nb1 * U2.shape[2] * 16)))):
        g3 = (phase[rows] @ g2.reshape(nRp, -1)).reshape(len(rows), nw, nm * nb1)
        u = U2[rows].conj()
        g4 = torch.stack([(u[:, :, b, None] * g3).sum(1) for b in range(u.shape[2])], 1)
        g4 = g4.reshape(len(rows), -1, nm, nb1)
        e = e3[rows]
        g = torch.stack([(g4 * e[:, None, :, v, None]).sum(2) for v in range(nm)], 2)
        out.append(g.real ** 2 + g.imag ** 2)
    return torch.cat(out)


def _occupation(e, T, mu, bose):
    x = np.clip((e - mu) / T, -700, 700)
    with np.errstate(divide="ignore"):
        return np.maximum(1.0 / (np.exp(x) - 1.0), 0.0) if bose else 1.0 / (np.exp(x) + 1.0)


def _velocities(prob, k, U):
    """Group velocities (nk, nb, 3) of the bands in U (nk, nw, nb), zero at Gamma."""
    n = prob.nw
    out = np.zeros((len(k), U.shape[2], 3))
    for s in range(0, len(k), 4096):
        ph = _phases(k[s:s + 4096], prob.Rh) / _d(prob.degh)
        u = _c(U[s:s + 4096])
        for d in range(3):
            dH = ((1j * _d(prob.Rh[:, d])) * ph) @ _c(prob.h0R).reshape(-1, n * n)
            dU = torch.stack([(dH.reshape(-1, n, n) * u[:, None, :, b]).sum(2) for b in range(u.shape[2])], 2)
            out[s:s + 4096, :, d] = (u.conj() * dU).sum(1).real.cpu().numpy()
    out[np.linalg.norm(k, axis=1) < 1e-6] = 0.0
    return out


def _delta(prob, x, dv=None):
    """The one-sided Gaussian, or the adaptive one with velocity differences dv (..., 3)."""
    if dv is None:
        t = x / prob.sigma
        return torch.where(t > 6.0, torch.zeros_like(t), torch.exp(-t * t)) / (prob.sigma * math.sqrt(math.pi))
    q = prob.recip / np.array(prob.mesh, dtype=float)[:, None]
    w = torch.sqrt(((dv @ _d(q).T) ** 2).sum(-1) / 6.0).clamp_min(1e-4 / synth.ENERGY_RY_TO_EV)
    same = (dv == 0).all(-1)
    t = x / w
    g = torch.exp(-t * t) / (math.sqrt(math.pi) * w * 0.9953222650189527)
    g = torch.where(x.abs() > 2.0 * w, torch.zeros_like(g), g)
    return torch.where(same, (x == 0).to(g.dtype), g)


def _groups_distinct(E):
    return np.diff(E, axis=1).min() > 1.1e-6 if E.shape[1] > 1 else True


def _exact_lw(case, seed):
    prob = _problem(case, seed)
    n, k = _mesh_points(prob)
    E, U = _electrons(k, prob.Rh, prob.degh, prob.h0R)
    inside = (E > prob.win_min) & (E < prob.win_max)
    active = np.flatnonzero(inside.any(1))
    lo = inside[active].argmax(1)
    nb = E.shape[1] - inside[active][:, ::-1].argmax(1) - lo
    start = np.concatenate([[0], np.cumsum(nb)])
    k1 = _pick_lines(active, prob.mesh[0], case["lines"], seed)
    k1 = np.arange(len(active)) if k1 is None else np.sort(k1)
    om, e3 = _phonons(k, prob)
    if not (_groups_distinct(E) and _groups_distinct(om)):
        return None
    na, top = len(active), int(nb.max())
    U2 = np.zeros((na, prob.nw, top), dtype=complex)
    E2 = np.full((na, top), 1e3)
    for i, a in enumerate(active):
        U2[i, :, :nb[i]] = U[a][:, lo[i]:lo[i] + nb[i]]
        E2[i, :nb[i]] = E[a][lo[i]:lo[i] + nb[i]]
    V2 = _d(_velocities(prob, k[active], U2)) if case["adaptive"] else None
    calcs = list(zip(prob.temperatures, prob.chem_pots))
    f2 = [_d(np.clip(_occupation(E2, T, mu, False), 0, 1)) for T, mu in calcs]
    n3 = [_d(_occupation(om, T, 0.0, True)) for T, mu in calcs]
    U2, E2, e3, om = _c(U2), _d(E2), _c(e3), _d(om)
    m = np.array(prob.mesh)
    out = np.zeros((len(calcs), start[-1]))
    phase2 = _phases(k[active], prob.Rp)
    group = max(1, int(1.0e9 // (prob.nRp * prob.nm * prob.nw ** 2 * 16)) * 32)
    for s in range(0, len(k1), group):
        pts = k1[s:s + group]
        caches = _cache(prob, k[active[pts]], [U[active[a]][:, lo[a]:lo[a] + nb[a]] for a in pts])
        for i, a in enumerate(pts):
            d = (n[active] - n[active[a]]) % m
            q = torch.as_tensor(d[:, 0] + m[0] * (d[:, 1] + m[1] * d[:, 2]), device=_device())
            back = _phases(k[active[a]][None], prob.Rp, -1.0)[0] / _d(prob.degP)
            g = _coupling(caches[i] * back[:, None, None, None], phase2, U2, e3[q])
            w = om[q][:, None, :]
            for b in range(nb[a]):
                x = E2[a, b] - E2[:, :, None]
                dv = (V2[a, b] - V2)[:, :, None, :] if V2 is not None else None
                d1, d2 = _delta(prob, x + w, dv), _delta(prob, x - w, dv)
                base = g[..., b] / w * math.pi / float(m.prod())
                base = torch.where(w >= PHONON_CUTOFF, base, torch.zeros_like(base))
                for c in range(len(calcs)):
                    f, bn = f2[c][:, :, None], torch.nan_to_num(n3[c][q][:, None, :], posinf=0.0)
                    t = base * ((f + bn) * d1 + (1.0 - f + bn) * d2)
                    out[c, start[a] + b] = float(torch.where(E2[:, :, None] < 1e2, t, torch.zeros_like(t)).sum())
    return out


def _exact_phel(case, seed):
    prob = _problem(case, seed)
    n, k = _mesh_points(prob)
    E, U = _electrons(k, prob.Rh, prob.degh, prob.h0R)
    inside = (E > prob.win_min) & (E < prob.win_max)
    active = np.flatnonzero(inside.any(1))
    lo = inside[active].argmax(1)
    nb = E.shape[1] - inside[active][:, ::-1].argmax(1) - lo
    k1 = _pick_points(len(active), case["count"], seed)
    om, e3 = _phonons(k, prob)
    if not (_groups_distinct(E) and _groups_distinct(om)):
        return None
    m = np.array(prob.mesh)
    E2, U2, e3, w = _d(E), _c(U), _c(e3), _d(om)[:, None, :]
    phase = _phases(k, prob.Rp) / _d(prob.degP)
    T, mu = prob.temperatures[0], prob.chem_pots[0]
    out = torch.zeros(om.shape, dtype=torch.float64, device=_device())
    caches = _cache(prob, k[active[k1]], [U[active[a]][:, lo[a]:lo[a] + nb[a]] for a in k1])
    for i, a in enumerate(k1):
        d = (n + n[active[a]]) % m
        q2 = torch.as_tensor(d[:, 0] + m[0] * (d[:, 1] + m[1] * d[:, 2]), device=_device())
        g = _coupling(caches[i], phase, U2[q2], e3)
        for b in range(nb[a]):
            e1 = E[active[a], lo[a] + b]
            f = 0.25 / math.cosh((e1 - mu) / 2.0 / T) ** 2
            out += (g[..., b] * _delta(prob, e1 - E2[q2][:, :, None] + w)).sum(1) * f * math.pi / T / float(m.prod())
    out = torch.where(w[:, 0, :] >= PHONON_CUTOFF, out, torch.zeros_like(out))
    return out.cpu().numpy()[None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "bands":
        f = synth.eig_family("el", case["nw"], seed=seed, rgrid=case["re"])
        E, U = _electrons(_path(case, seed, f), f["R"], f["weight"], f["coef"])
        ph = U[:, :1, :].conj()
        return {"E": E, "U": np.ascontiguousarray(U * (ph / np.abs(ph)))}
    if kind == "zheev":
        W, V = _eigh(_hermitian(case, seed))
        V = np.ascontiguousarray(V.transpose(0, 2, 1))
        ph = V[:, :, :1].conj()
        return {"W": W, "V": V * (ph / np.abs(ph))}
    if kind == "couple":
        prob, U1, U2, e3, k1, q3 = _couple_inputs(case, seed)
        g2 = _cache(prob, k1[None], [U1])[0]
        top = max(u.shape[1] for u in U2)
        U2p = np.zeros((len(U2), prob.nw, top), dtype=complex)
        for i, u in enumerate(U2):
            U2p[i, :, :u.shape[1]] = u
        g = _coupling(g2, _phases(q3, prob.Rp) / _d(prob.degP), _c(U2p), _c(np.stack(e3))).cpu().numpy()
        # per q: (b1, b2, nu), first index fastest
        return np.concatenate([g[i, :u.shape[1]].transpose(2, 0, 1).reshape(-1, order="F") for i, u in enumerate(U2)])
    return _exact_phel(case, seed) if kind == "phel" else _exact_lw(case, seed)
