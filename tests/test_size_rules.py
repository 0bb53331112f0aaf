"""The rules that choose kernels by size, on the host: which kernels run the
mesh-separable last stage, over every combination of its limits; how the direct
transform cuts a panel, over every size."""
import itertools
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
FUSED, XG, ROT, YX = range(4)


@pytest.fixture(scope="session")
def rules(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "size_rules")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-o", exe, os.path.join(HERE, "cpp", "size_rules.cpp")],
                   check=True)

    def ask(kind, forms, timeout=60):
        text = "\n".join(kind + " " + " ".join(str(int(x)) for x in f) for f in forms) + "\n"
        r = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=timeout)
        return [tuple(int(x) for x in line.split()) for line in r.stdout.splitlines()]

    return ask


def test_last_stage(rules):
    sizes = [(3, 4), (12, 16), (15, 13), (16, 12), (16, 13), (18, 16), (24, 16), (25, 16), (27, 15), (27, 16), (30, 16),
             (32, 12), (32, 13), (32, 16), (12, 17), (6, 32)]
    forms = [(f64, bf, nm, nw, m0, my, nG0, nQ, ad, mode, fy, ls)
             for (nm, nw), f64, bf, (m0, my), (nG0, nQ), ad, mode, fy, ls in
             itertools.product(sizes, (0, 1), (0, 1), ((1, 1), (64, 64), (65, 5)), ((1, 1), (24, 100), (25, 100), (24, 4000)),
                               (0, 1), (0, 1, 2, 3), (0, 1), (0, 1)) if not (f64 and bf)]
    got = rules("stage", forms)
    assert len(got) == len(forms)
    for (f64, bf, nm, nw, m0, my, nG0, nQ, ad, mode, fy, ls), (g,) in zip(forms, got):
        if mode == 0 or bf or nw > 16 or m0 > 64 or nG0 > 24 or nm * nw > 384:
            want = FUSED
        elif fy and not ls and mode != 3 and nQ < 4000:  # 4000 quads: 144 KB of entries, beyond LDS with the rest
            want = YX
        elif f64 or nm > 16 or nm * nw > 192:
            want = FUSED
        else:
            want = ROT if mode == 3 and not ad else XG
        assert g == want, (f64, bf, nm, nw, m0, my, nG0, nQ, ad, mode, fy, ls)


# the instances of k_coupling, by precision
INSTANCES = {1: {(1, 1), (1, 2), (1, 3), (1, 4), (2, 3)},
             0: {(1, 1), (1, 2), (1, 3), (1, 4), (1, 5), (1, 6), (2, 3), (2, 4), (2, 5), (2, 6)}}


@pytest.mark.parametrize("f64", [1, 0])
def test_coupling_tiling(rules, f64):
    """Every size ends (some windows once never got smaller), the tiles cover the
    window's columns with an instance that exists, and a size is refused only when
    not even one mode at a time fits LDS."""
    forms = [(f64, nm, nw, nb, points, panels) for nm in range(1, 37) for nw in range(1, 33) for nb in range(1, nw + 1)
             for points, panels in ((8192, 1), (8193, 1), (33, 128), (33, 129), (0, 5), (64, 512), (65, 512), (1000000, 3))]
    got = rules("tiling", forms, timeout=120)
    assert len(got) == len(forms)
    elem, most = (16, 192) if f64 else (8, 384)
    seen = set()
    for (_, nm, nw, nb, points, panels), (mt, nt, wc, rows, modes, stage, lds) in zip(forms, got):
        at = (nm, nw, nb, points, panels)
        n64, n32, tiles = -(-points // 64) * panels, -(-points // 32) * panels, -(-modes * nw // 16)
        t64, t32 = 512 if n64 <= 512 else n64 + 154, 512 if n32 <= 512 else max(n32, 1024)
        tall = 8 * t64 <= 5 * t32 if tiles <= 5 else 7 * t64 <= 4 * t32
        if modes < nm or n32 <= 256:
            want = (1, 4)
        elif tiles > 8:
            want = (2, 4)
        elif not tall:
            want = (1, 2)
        else:
            want = (1, 1) if tiles <= (4 if f64 else 6) else (1, 2) if f64 else (2, 2)
        assert (mt, wc) == want, at
        scratch = 16 * nm * nb * 24
        up = lambda a, b: -(-a // b)
        whole = up(nm, up(nm, max(1, most // nw)))

        def fit(room):
            m = whole
            while m > 1 and max(16 * m * nw * elem + scratch, 1024) > room:
                m = min(m - 1, up(nm, up(nm, m) + 1))
            return m

        half = fit(80 * 1024)
        if up(points, 16) * panels <= 256 or 16 * half * nw * elem + scratch > 80 * 1024 or 4 * half < whole:
            half = fit(160 * 1024)
        assert modes == half, at
        assert 1 <= modes <= nm and (modes * nw <= most or modes == 1), at
        assert lds == max(16 * modes * nw * elem + scratch, 1024), at
        assert (lds <= 160 * 1024) == (16 * nw * elem + scratch <= 160 * 1024), at
        assert nt == -(-tiles // wc), at
        assert rows == (16 if modes < nm else 16 * mt * (4 // wc)), at
        assert stage == (16 * modes * nw * elem >= 16 * (nm + nb) * 8), at
        seen.add((mt, nt))
    assert seen == INSTANCES[f64]


def test_panel_chunk(rules):
    """At most 24 GiB of g3 rows, 16 to 128 panels."""
    G = 1 << 30
    forms = [(100 << 20, 100 * G), (100 << 20, 24 * G), (100 << 20, 10 * G), (100 << 20, G), (100 << 20, 0), (G, 100 * G),
             (4 * G, 100 * G), (1, 100 * G)]
    assert [c for c, in rules("chunk", forms)] == [128, 128, 102, 16, 16, 24, 16, 128]
