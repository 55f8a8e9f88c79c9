"""The coarsest solves' division by a known diagonal (csrc/quotient.hpp), compiled for the host,
against the division itself. An FP32 quotient is right or told as subnormal."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "maelstrom.jl_amd", "csrc")
SOURCE = r"""
#define __host__
#define __device__
#include "quotient.hpp"
#include <cstdint>
#include <cstring>
static bool told(float q) { return mael::subnormal_rank(q) < mael::SUBNORMALS; }
static bool told(double) { return false; }
template <class T, class B> static int64_t wrong(const T* a, const T* d, int64_t n) {
    int64_t w = 0;
    for (int64_t k = 0; k < n; ++k) {
        const T q = mael::quotient(a[k], d[k], 1.0 / (double)d[k]), e = a[k] / d[k];
        if (told(q)) continue;   // (FP32: the solve then divides)
        B x, y;
        std::memcpy(&x, &q, sizeof q);
        std::memcpy(&y, &e, sizeof e);
        w += x != y;
    }
    return w;
}
extern "C" int64_t wrong32(const float* a, const float* d, int64_t n) { return wrong<float, uint32_t>(a, d, n); }
extern "C" int64_t wrong64(const double* a, const double* d, int64_t n) { return wrong<double, uint64_t>(a, d, n); }
extern "C" int is_told(float q) { return told(q); }
// every FP32 numerator whose quotient by 1 .. 6 is subnormal or the smallest normal
extern "C" int64_t wrong_small() {
    int64_t w = 0;
    for (int d = 1; d <= 6; ++d)
        for (uint32_t b = 0;; ++b) {
            float a;
            std::memcpy(&a, &b, 4);
            const float q = mael::quotient(a, 0.0f, 1.0 / d), e = a / (float)d;
            w += std::memcmp(&q, &e, 4) != 0;
            if (e > 1.17549435e-38f) break;
        }
    return w;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("quotient") / "quotient.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, "-x", "c++", "-", "-o", so],
                   input=SOURCE, text=True, check=True)
    L = C.CDLL(so)
    for f, t in ((L.wrong32, C.c_float), (L.wrong64, C.c_double)):
        f.restype, f.argtypes = C.c_int64, [C.POINTER(t), C.POINTER(t), C.c_int64]
    L.wrong_small.restype = C.c_int64
    L.is_told.argtypes = [C.c_float]
    return L


def _wrong(fn, a, d):
    t = np.float32 if fn.argtypes[0] is C.POINTER(C.c_float) else np.float64
    a, d = np.ascontiguousarray(a, t), np.ascontiguousarray(d, t)
    return fn(a.ctypes.data_as(fn.argtypes[0]), d.ctypes.data_as(fn.argtypes[1]), a.size)


def test_fp32(lib):
    rng = np.random.default_rng(0)
    n = 2_000_000
    mant = lambda: np.ldexp(rng.integers(1 << 23, 1 << 24, n).astype(np.float64), -23)
    d = mant() * 2.0 ** rng.integers(-8, 12, n)
    assert _wrong(lib.wrong32, mant() * 2.0 ** rng.integers(-100, 100, n) * rng.choice([-1, 1], n), d) == 0
    # round the smallest normal quotient, and far below it
    assert _wrong(lib.wrong32, d * mant() * 2.0 ** rng.integers(-130, -124, n), d) == 0
    assert _wrong(lib.wrong32, d * mant() * 2.0 ** rng.integers(-150, -130, n), d) == 0
    # quotients in the middle between two subnormal numbers: (2 m + 1) 2^-150
    u, m = 2 * rng.integers(1, 1 << 12, n) + 1, 2 * rng.integers(0, 1 << 10, n) + 1
    s = rng.integers(2, 14, n)
    assert _wrong(lib.wrong32, u * m * 2.0 ** (s - 150), u * 2.0 ** s) == 0
    assert _wrong(lib.wrong32, [0.0, -0.0, np.inf, -np.inf], [3.0] * 4) == 0


def test_subnormal_is_told(lib):
    q = np.array([0, -0.0, 2.0 ** -149, -2.0 ** -149, 2.0 ** -126 - 2.0 ** -149, 2.0 ** -126, -1, np.inf, np.nan], np.float32)
    assert [bool(lib.is_told(float(x))) for x in q] == [False, False, True, True, True, False, False, False, False]


def test_fp32_small_diagonals(lib):
    """A count of neighbours as the diagonal: right whatever the quotient."""
    assert lib.wrong_small() == 0


def test_fp64(lib):
    rng = np.random.default_rng(1)
    n = 2_000_000
    for spread in (1, 40):
        a = rng.uniform(1, 2, n) * 2.0 ** rng.integers(-spread, spread + 1, n) * rng.choice([-1, 1], n)
        d = rng.uniform(1, 2, n) * 2.0 ** rng.integers(-8, 12, n)
        assert _wrong(lib.wrong64, a, d) == 0
    # quotients next to the middle between two numbers: a is a multiple of d plus half a unit, rounded
    d = (2 * rng.integers(1 << 30, 1 << 31, n) + 1).astype(np.float64)
    q = (2 * rng.integers(1 << 20, 1 << 21, n) + 1).astype(np.float64)
    assert _wrong(lib.wrong64, np.nextafter(d * q, np.inf), d) == 0
    # a coarse diagonal is a sum of FP32 couplings
    d = rng.integers(1, 1 << 24, n) / 2.0 ** 18
    assert _wrong(lib.wrong64, rng.normal(0, 1, n), d) == 0
