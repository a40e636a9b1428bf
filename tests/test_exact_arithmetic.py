"""The device header's short forms of the islands (32 x 32 bit products where
the islands multiply in 128 bits) equal the oracle's islands bit for bit: the
activations over magnitudes on both sides of each form's bound, the softmax
exponential through orc_softmax_exact's two-element inputs, and the rounding of
scaled 64-bit sums against exact rationals.  The header is compiled for the host."""
import os
import shutil
import subprocess
from fractions import Fraction

import ctypes
import numpy as np
import pytest

import orc

HDR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "shannon-prime-system_amd", "csrc", "hip", "kvd_exact.h")
PRE = """#include <stdint.h>
#include <math.h>
#include <string.h>
#define __device__
#define __host__
#define __forceinline__ inline
static inline int64_t __double_as_longlong(double d) { int64_t r; memcpy(&r, &d, 8); return r; }
"""
POST = """
extern "C" void act(const float *x, int n, float *g, float *s) {
    for (int i = 0; i < n; i++) { g[i] = kvd::gelu_exact1(x[i]); s[i] = kvd::silu_exact1(x[i]); } }
extern "C" void expf30(const int64_t *d, int n, int64_t *o) { for (int i = 0; i < n; i++) o[i] = kvd::exp_fixed(d[i]); }
extern "C" void rne(const int64_t *v, const int *k, int n, float *o) { for (int i = 0; i < n; i++) o[i] = kvd::rne_i64_scaled(v[i], k[i]); }
"""


@pytest.fixture(scope="module")
def dev(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ is not installed")
    d = tmp_path_factory.mktemp("exact")
    body = "".join(line for line in open(HDR) if not line.startswith(("#include", "#pragma once")))
    (d / "e.cpp").write_text(PRE + body + POST)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-w",
                    str(d / "e.cpp"), "-o", str(d / "e.so")], check=True)
    return ctypes.CDLL(str(d / "e.so"))


def p(a):
    return ctypes.c_void_p(a.ctypes.data)


def test_activations_equal_the_islands(dev):
    rng = np.random.default_rng(1)
    x = np.concatenate([rng.standard_normal(200000) * s for s in (1e-3, 0.3, 3, 20, 300)] +
                       [np.arange(-70000, 70000) / 4096.0, [15.99999, 16.0, 16.00001, -16.0, 32767.9, 0.0, -0.0]]).astype(np.float32)
    g, s, og, os_ = (np.empty_like(x) for _ in range(4))
    dev.act(p(x), x.size, p(g), p(s))
    orc.lib().orc_gelu_exact(p(x), x.size, p(og))
    orc.lib().orc_silu_exact(p(x), x.size, p(os_))
    assert np.array_equal(g.view(np.uint32), og.view(np.uint32))
    assert np.array_equal(s.view(np.uint32), os_.view(np.uint32))


def test_exponential_equals_its_definition(dev):
    """2^-g with g = ceil(-d log2e) in Q30 and the island's polynomial, in Python integers."""
    FB, L = 30, 1549082005
    C = [1073741824, 744261118, 257941248, 59597083, 10327387, 1431680, 165394]
    rng = np.random.default_rng(2)
    d = -np.concatenate([np.arange(300), 1 << np.arange(36, dtype=np.int64), (1 << np.arange(1, 36, dtype=np.int64)) - 1,
                         rng.integers(0, 1 << 36, 20000), rng.integers(0, 1 << 31, 20000)]).astype(np.int64)
    o = np.empty_like(d)
    dev.expf30(p(d), d.size, p(o))
    for di, oi in zip(d.tolist(), o.tolist()):
        g = -((di * L) >> FB)
        n, r = g >> FB, g & ((1 << FB) - 1)
        want = 0
        if n < 32:
            acc, f = C[6], (1 << FB) - r
            for k in range(5, -1, -1):
                acc = ((acc * f) >> FB) + C[k]
            want = acc >> (n + 1) if r else (1 << FB) >> n
        assert oi == want, di


def test_scaled_rounding_is_nearest_even(dev):
    rng = np.random.default_rng(3)
    v = (rng.integers(-(1 << 62), 1 << 62, 30000) >> rng.integers(0, 60, 30000)).astype(np.int64)
    t = (np.int64(1) << rng.integers(24, 60, 3000)) + rng.integers(-3, 4, 3000) * (np.int64(1) << rng.integers(0, 36, 3000))
    v = np.concatenate([v, t, -t, [0]]).astype(np.int64)
    k = rng.integers(-200, 70, v.size).astype(np.int32)
    # around 2^-126, where 24 bits of a value below it are one more than a float
    # keeps: the midpoint to the largest subnormal (half), the one above it
    # (quarter) and their neighbours, for several widths of the sum
    for w in (26, 44, 61):
        one = 1 << w
        half, quarter = one >> 24, one >> 25
        b = [one + o + d for o in (0, -quarter, -half, -half - quarter, -2 * half, quarter, half) for d in (-2, -1, 0, 1, 2)]
        v = np.concatenate([v, b, -np.array(b)]).astype(np.int64)
        k = np.concatenate([k, np.full(2 * len(b), -126 - w)]).astype(np.int32)
    o = np.empty(v.size, np.float32)
    dev.rne(p(v), p(k), v.size, p(o))
    for vi, ki, oi in zip(v.tolist(), k.tolist(), o.tolist()):
        x = Fraction(vi) * Fraction(2) ** ki
        if abs(x) >= Fraction(2) ** 128 - Fraction(2) ** 103:
            assert np.isinf(oi) and (oi > 0) == (vi > 0)
            continue
        # neighbours of the result: none is nearer, ties have an even last bit
        b = np.float32(oi)
        e = abs(Fraction(float(b)) - x)
        for nb in (np.nextafter(b, np.float32(np.inf)), np.nextafter(b, np.float32(-np.inf))):
            if np.isfinite(nb):
                en = abs(Fraction(float(nb)) - x)
                assert e < en or (e == en and int(b.view(np.uint32)) % 2 == 0), (vi, ki)
