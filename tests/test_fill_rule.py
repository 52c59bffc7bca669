"""The rule that sends density chunks to the fast fill
(wgpu-voxel-engine_amd/csrc/vx_fill_rule.h) and the error bound its
comparisons rest on.  CPU only: the header is compiled on its own; the bound
is checked on f32 restatements of both evaluations."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "wgpu-voxel-engine_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include "vx_fill_rule.h"
int main() {
    int o, cx, cy, cz, e;
    float f, l, g;
    while (scanf("%d %f %f %f %d %d %d %d", &o, &f, &l, &g, &cx, &cy, &cz, &e) == 8) {
        const int v = vx::fast_variant(o, f, l, g, cx, cy, cz, e);
        printf("%d", v);
        for (int m = e; m <= 64; m *= 2) printf(" %d %d", v ? vx::fast_cols(e, m, v) : 0, vx::fast_tab(m));
        printf("\n");
    }
}
"""
F = np.float32


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("rule")
    (d / "drv.cpp").write_text(DRIVER)
    subprocess.run([cxx, "-std=c++17", "-O1", "-ffp-contract=off", "-I", CSRC, str(d / "drv.cpp"),
                    "-o", str(d / "drv")], check=True)

    def run(cases):
        text = "\n".join(" ".join(repr(float(v)) if isinstance(v, float) else str(v) for v in c)
                         for c in cases)
        out = subprocess.run([str(d / "drv")], input=text, capture_output=True, text=True, check=True)
        return [list(map(int, ln.split())) for ln in out.stdout.splitlines()]
    return run


def test_tables_fit(rule):
    """Whatever the rule accepts, one row's table entries (two y planes of
    every line's lattice points) fit a wave's share, at the f32 cells that the
    kernel computes, for any start of the chunk."""
    rng = np.random.default_rng(1)
    cases = []
    for _ in range(4000):
        edge = int(rng.choice([16, 32, 64]))
        f = float(F(np.exp(rng.uniform(np.log(1e-4), np.log(1.2)))))
        reach = int(np.exp(rng.uniform(0, np.log(2 ** 31 / edge - 2))))
        c = [int(v) for v in rng.integers(-reach, reach + 1, 3)]
        cases.append((int(rng.integers(1, 9)), f, float(F(rng.choice([0.5, 1.0, 1.9, 2.0, 2.5]))),
                      float(F(rng.choice([0.5, -0.7, 2.5, 1e30]))), *c, edge))
    taken = 0
    for case, got in zip(cases, rule(cases)):
        octaves, f, lac, gain, cx, cy, cz, edge = case
        v, rest = got[0], got[1:]
        if not v:
            continue
        taken += 1
        assert v >= octaves and v in (2, 3, 4, 6, 8)
        points, g, amp = 2 * (v - octaves), F(f), F(1)
        for _ in range(octaves):
            assert g <= F(0.75)
            for c in (cx, cy, cz):
                lo, hi = F(c * edge) * g, F(c * edge + edge - 1) * g
                assert abs(lo) < 2 ** 23 and abs(hi) < 2 ** 23
            span = int(np.floor(F(cx * edge + edge - 1) * g)) - int(np.floor(F(cx * edge) * g))
            points += span + 2
            assert np.isfinite(amp)
            g, amp = F(g * F(lac)), F(amp * F(gain))
        for cols, tab in zip(rest[::2], rest[1::2]):
            assert 2 * points * (64 // edge) * cols <= tab, case
    assert taken > 500


def test_known_terrains(rule):
    """The tuned terrains take their own octave count; fine or far ones go to
    a wider variant or to the general kernels."""
    got = [r[0] for r in rule([
        (4, 1 / 64, 2.0, 0.5, 5, 0, 9, 32),    # the benchmark's density
        (3, 0.09, 0.5, 2.5, -7, 0, 3, 32),     # the reference's parameters
        (6, 0.01, 2.0, 0.5, 0, 0, 0, 32),
        (4, 0.04, 2.0, 0.5, 0, 0, 0, 32),      # 28 points a line: half the columns
        (1, 0.75, 2.0, 0.5, 0, 0, 0, 16),
        (1, 0.7500001, 2.0, 0.5, 0, 0, 0, 16),
        (4, 1 / 64, 2.0, 0.5, 2 ** 20 - 2, 0, 0, 32),   # 2^25 / 8 = 2^22: the limit
        (4, 1 / 64, 2.0, 0.5, 2 ** 20, 0, 0, 32),
        (8, 1 / 64, 2.0, 1e30, 0, 0, 0, 32),
    ])]
    assert got == [4, 3, 6, 6, 2, 0, 4, 0, 0]


def fma(a, b, c):
    return (a.astype(np.float64) * b + c).astype(F)


def lerp(t, a, b):
    return a + t * (b - a)


def fade(t):
    return ((t * t) * t) * (t * (t * F(6) - F(15)) + F(10))


@pytest.mark.parametrize("octaves", [1, 2, 3, 4, 6, 8])
def test_error_bound(octaves):
    """|fast - oracle order| stays within eps = (48 + 8 O) 2^-24 sum|amp| over
    random gradients, fractions (cell corners and their neighbours among them)
    and amplitudes."""
    rng = np.random.default_rng(octaves)
    n = 200000
    grads = np.array([[1, 1, 0], [-1, 1, 0], [1, -1, 0], [-1, -1, 0], [1, 0, 1], [-1, 0, 1],
                      [1, 0, -1], [-1, 0, -1], [0, 1, 1], [0, -1, 1], [0, 1, -1], [0, -1, -1]], F)
    for gain in (F(0.5), F(2.5), F(-0.8), F(1.0)):
        exact = np.zeros(n, F)
        A0s, terms, mag, amp = np.zeros(n, F), [], F(0), F(1)
        for _ in range(octaves):
            x, y, z = (np.where(rng.random(n) < 0.1, rng.choice([0.0, 1e-7, 0.5, 1 - 2.0 ** -24, 1.0], n),
                                rng.random(n)).astype(F) for _ in range(3))
            x1, y1, z1 = x - F(1), y - F(1), z - F(1)
            u, v, w = fade(x), fade(y), fade(z)
            G = grads[rng.integers(0, 12, (8, n))]  # corner = x | row << 1 | col << 2

            def dot(k):
                g = G[k]
                xr, yr, zr = (x1 if k & 1 else x), (y1 if k & 2 else y), (z1 if k & 4 else z)
                p = [g[:, 0] * xr, g[:, 1] * yr, g[:, 2] * zr]
                s = [np.where(g[:, 0] == 0, p[1], p[0]),
                     np.where((g[:, 0] == 0) | (g[:, 1] == 0), p[2], p[1])]
                return s[0] + s[1]
            d = [dot(k) for k in range(8)]
            noise = lerp(w, lerp(v, lerp(u, d[0], d[1]), lerp(u, d[2], d[3])),
                         lerp(v, lerp(u, d[4], d[5]), lerp(u, d[6], d[7])))
            exact = exact + amp * noise

            def plane(row):  # table entries of both x corners, then the blend along x
                e = []
                for i in (0, 1):
                    g0, g1 = amp * G[i | row << 1], amp * G[i | row << 1 | 4]
                    q0, q1 = g0[:, 2] * z, g1[:, 2] * z1
                    e.append((fma(w, g1[:, 0] - g0[:, 0], g0[:, 0]), fma(w, q1 - q0, q0),
                              fma(w, g1[:, 1] - g0[:, 1], g0[:, 1])))
                l0, l1 = fma(e[0][0], x, e[0][1]), fma(e[1][0], x1, e[1][1])
                return fma(u, l1 - l0, l0), fma(u, e[1][2] - e[0][2], e[0][2])
            P0, P1 = plane(0)
            Q0, Q1 = plane(1)
            A0s = A0s + P0 if terms else P0
            terms.append((P1, (Q0 - Q1) - P0, Q1 - P1, y, v))
            mag, amp = mag + abs(amp), F(amp * gain)
        acc = A0s
        for A1, D0, D1, y, v in terms:
            acc = fma(A1, y, acc)
            acc = fma(v, fma(D1, y, D0), acc)
        eps = (48 + 8 * octaves) * 2.0 ** -24 * float(mag)
        err = np.abs(acc.astype(np.float64) - exact).max()
        assert err <= eps, (gain, err, eps)


PAYS = r"""
#include <cstdio>
#include "vx_fill_rule.h"
int main() {
    int o, z, e, m, n;
    float f, l;
    while (scanf("%d %f %f %d %d %d %d", &o, &f, &l, &z, &e, &m, &n) == 7)
        printf("%d\n", vx::fast_pays(o, f, l, z != 0, e, m, n));
}
"""


def test_batches_that_gain(tmp_path):
    """Where a batch's chunks leave the fast fill because the general kernels
    are faster: fine octaves, a zero threshold on lattice planes, small batches
    of 16^3; and the tuned terrains, which stay."""
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    (tmp_path / "p.cpp").write_text(PAYS)
    subprocess.run([cxx, "-std=c++17", "-O1", "-ffp-contract=off", "-I", CSRC, str(tmp_path / "p.cpp"),
                    "-o", str(tmp_path / "p")], check=True)
    cases = [  # octaves, frequency, lacunarity, zero threshold, edge, largest edge, chunks -> gains
        (4, 1 / 64, 2.0, 0, 32, 32, 4096, 1), (3, 0.09, 0.5, 1, 32, 32, 1640, 1), (4, 1 / 64, 2.0, 0, 64, 64, 323, 1),
        (6, 0.01, 2.0, 0, 32, 32, 1023, 1), (6, 1 / 64, 2.0, 1, 16, 16, 4, 1), (1, 0.09, 2.0, 1, 32, 32, 256, 1),
        # the finest octave
        (1, 0.32, 2.0, 0, 32, 32, 256, 1), (1, 0.33, 2.0, 0, 32, 32, 256, 0), (3, 0.125, 2.0, 0, 32, 32, 256, 0),
        (3, 0.09, 2.0, 0, 32, 32, 511, 0), (3, 0.09, 2.0, 0, 32, 32, 512, 1),
        (4, 0.055, 2.0, 0, 32, 32, 1023, 1), (4, 0.055, 2.0, 0, 32, 32, 1024, 0), (4, 0.0625, 2.0, 0, 32, 32, 256, 0),
        (4, 0.0625, 2.0, 0, 64, 64, 64, 0), (1, 0.45, 2.0, 0, 64, 64, 16, 1), (1, 0.45, 2.0, 0, 64, 64, 17, 0),
        (2, 0.225, 2.0, 0, 64, 64, 323, 1), (2, 0.25, 2.0, 0, 64, 64, 8, 0),
        (2, 0.2, 2.0, 0, 64, 64, 64, 1), (3, 0.6, 0.5, 0, 64, 64, 64, 0), (5, 1 / 32, 2.0, 0, 64, 64, 64, 1),
        # zero thresholds
        (1, 0.125, 2.0, 1, 32, 32, 1024, 0), (1, 1 / 64, 2.0, 1, 64, 64, 64, 0), (1, 1e-5, 2.0, 1, 32, 32, 256, 0),
        (2, 0.05, 2.0, 1, 32, 32, 256, 1), (2, 0.0625, 2.0, 1, 32, 32, 1023, 0), (2, 0.0625, 2.0, 1, 32, 32, 1024, 1),
        (2, 0.0625, 2.0, 1, 64, 64, 256, 1), (1, 0.35, 2.0, 1, 64, 64, 64, 0), (1, 0.3217, 2.0, 1, 64, 64, 64, 1),
        (6, 3e-7, 2.0, 1, 32, 32, 64, 0),
        (2, 0.0625, 1.9, 1, 32, 32, 256, 1), (3, 0.0625, 2.0, 1, 32, 32, 256, 1),
        # 16^3 chunks, alone and beside larger ones
        (3, 1 / 64, 2.0, 0, 16, 16, 383, 0), (3, 1 / 64, 2.0, 0, 16, 16, 384, 1), (3, 1 / 64, 2.0, 0, 16, 32, 64, 1),
        (1, 1 / 64, 2.0, 0, 16, 16, 4000, 0), (3, 1 / 64, 2.0, 1, 16, 16, 4000, 0), (3, 0.013, 1.9, 1, 16, 16, 512, 1),
        (4, 1 / 64, 2.0, 0, 16, 16, 8, 1), (4, 1 / 64, 2.0, 0, 16, 16, 9, 0), (4, 1 / 64, 2.0, 1, 16, 16, 1, 0),
        (3, 1 / 64, 2.0, 0, 16, 16, 1, 0), (4, 1 / 64, 2.0, 1, 16, 16, 1023, 0), (4, 1 / 64, 2.0, 1, 16, 16, 1024, 1),
    ]
    text = "\n".join(" ".join(repr(float(v)) if isinstance(v, float) else str(v) for v in c[:-1]) for c in cases)
    out = subprocess.run([str(tmp_path / "p")], input=text, capture_output=True, text=True, check=True)
    assert [int(v) for v in out.stdout.split()] == [c[-1] for c in cases]


TUNE = r"""
#include <cstdio>
#include "vx_fill_rule.h"
int main() {
    int n, m, general;
    while (scanf("%d %d %d", &n, &m, &general) == 3) {
        vx::FillMix mix;
        mix.fast = n - general;
        mix.general = general;
        int32_t hints[4];
        const int k = vx::tune_fill_hints(n, m, mix, hints);
        const vx::FillShape r = vx::fill_shape(n, m, mix, 0);
        printf("%d %d", r.fast, r.general);
        for (int i = 0; i < k; i++) {
            const vx::FillShape s = vx::fill_shape(n, m, mix, hints[i]);
            printf(" %d %d %d", hints[i], s.fast, s.general);
        }
        printf("\n");
    }
}
"""


def test_tuner_hints(tmp_path):
    """The fill shapes that the autotuner times: each another than the rule's
    and than each other's, half and twice what the kernels do take."""
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    (tmp_path / "t.cpp").write_text(TUNE)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", CSRC, str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")],
                   check=True)
    cases = [(n, m, g) for n in (1, 64, 127, 128, 300, 511, 512, 700, 1023, 1024, 4000) for m in (16, 32, 64)
             for g in sorted({0, 1, n // 2, n})]
    out = subprocess.run([str(tmp_path / "t")], input="\n".join("%d %d %d" % c for c in cases),
                         capture_output=True, text=True, check=True).stdout.splitlines()
    got = {}
    for case, line in zip(cases, out):
        v = list(map(int, line.split()))
        shapes = [tuple(v[:2])] + [tuple(v[i + 1:i + 3]) for i in range(2, len(v), 3)]
        hints = v[2::3]
        assert len(set(shapes)) == len(shapes), (case, v)
        assert set(hints) <= {1, 2, 4, 8} and (case[0] < 1024 or not hints), (case, v)
        assert (shapes[0][0] > 0) == (case[0] > case[2]) and (shapes[0][1] > 0) == (case[2] > 0), (case, v)
        got[case] = hints
    # 64^3 by the bounded fill: 16, 8 and 4 workgroups by the rule
    assert (got[64, 64, 0], got[300, 64, 0], got[700, 64, 0]) == ([8], [4], [4])
    assert got[300, 32, 0] == [2] and got[700, 32, 0] == [1, 4]   # as the general kernels
    assert got[300, 64, 300] == [2, 8] and got[64, 64, 64] == [4]
