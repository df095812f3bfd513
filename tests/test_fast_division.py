"""The divisions half_kernel replaces (kh_div.hpp), on the CPU.

Index division by a magic number is exact, and the quotient from two residual
corrections is the IEEE quotient.  The first two tests restate the steps in
numpy (float32, sigma up to 3.2, fused multiply-adds formed in extended
precision: the products are exact there, the sums round once more far below one
ulp).  The others compile the header itself for the host and compare it with
the compiler's own division, in both precisions: sigma from 0 to 2^20, the
largest the kernel is used with, values at and around the guard for tiny ones,
powers of two and their neighbours, the largest and the smallest numbers,
zeros, infinities and NaN.
"""
import ctypes
import subprocess

import numpy as np
import pytest


def test_division_by_multiplication():
    rng = np.random.default_rng(0)
    for d in [1, 2, 3, 5, 7, 40, 64, 65, 127, 192, 641, 4095, 65537, (1 << 30) - 1]:
        length = max(0, (d - 1).bit_length())
        m = ((1 << (31 + length)) + d - 1) // d
        assert m < 1 << 32
        for c in [0, 1, d - 1, d, d + 1, (1 << 31) - 1, *rng.integers(0, 1 << 31, 200).tolist()]:
            assert (c * m) >> (31 + length) == c // d


def test_quotient_by_residual_corrections_is_the_ieee_quotient():
    f, wide = np.float32, np.longdouble
    rng = np.random.default_rng(1)

    def fma(a, b, c):
        return (a.astype(wide) * b.astype(wide) + c.astype(wide)).astype(f)

    for s in np.concatenate([rng.uniform(0, 2, 100), 10 ** rng.uniform(-8, 0.5, 100)]).astype(f):
        b = np.full(20000, f(1) + s, f)
        r = (f(1) / b).astype(f)
        a = (rng.standard_normal(20000) * 10.0 ** rng.uniform(-29, 6, 20000)).astype(f)
        a = a[(np.abs(a) >= 2.0 ** -100)]
        b, r = b[:a.size], r[:a.size]
        q = (a * r).astype(f)
        q = fma(fma(-b, q, a), r, q)
        q = fma(fma(-b, q, a), r, q)
        assert np.array_equal(q, a / b)


SOURCE = r"""
#define __host__
#define __device__
#define __forceinline__ inline
#include "kh_div.hpp"
extern "C" {
void index_div(uint32_t d, const uint32_t *c, uint32_t *q, long n) {
    const kh::FastDiv f = kh::div_magic(d);
    for (long i = 0; i < n; ++i) q[i] = kh::fdiv(c[i], f);
}
#define QUOTIENT(T) \
    void quotient_##T(const T *a, const T *s, T *got, T *want, long n) { \
        for (long i = 0; i < n; ++i) { \
            const T b = T(1) + s[i], b1 = T(1) + s[n - 1 - i]; \
            T other; \
            kh::div_by(a[i], a[n - 1 - i], b, b1, T(1) / b, T(1) / b1, got[i], other); \
            want[i] = a[i] / b; \
        } \
    }
QUOTIENT(float)
QUOTIENT(double)
double sigma_max() { return kh::DIV_SIGMA_MAX; }
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    import os
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "khronos.jl_amd", "csrc")
    d = tmp_path_factory.mktemp("div")
    (d / "div.cpp").write_text(SOURCE)
    out = str(d / "libdiv.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", csrc, str(d / "div.cpp"),
                    "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.sigma_max.restype = ctypes.c_double
    return lib


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_header_index_division(host):
    rng = np.random.default_rng(2)
    for d in [1, 2, 3, 5, 7, 40, 64, 65, 127, 192, 641, 4095, 65537, (1 << 30) - 1, (1 << 31) - 1]:
        c = np.concatenate([[0, 1, d - 1, d, min(d + 1, (1 << 31) - 1), (1 << 31) - 1],
                            rng.integers(0, 1 << 31, 2000)]).astype(np.uint32)
        q = np.zeros_like(c)
        host.index_div(ctypes.c_uint32(d), _p(c), _p(q), ctypes.c_long(c.size))
        assert np.array_equal(q, c // np.uint32(d))


@pytest.mark.parametrize("name,dtype,guard", [("float", np.float32, -100), ("double", np.float64, -960)])
def test_header_quotient(host, name, dtype, guard):
    rng = np.random.default_rng(3)
    top = dtype(host.sigma_max())
    info = np.finfo(dtype)
    assert top == 2.0 ** 20
    two = np.array([2.0 ** k for k in range(-20, 21)], dtype)
    sig = np.concatenate([[0.0], two, np.nextafter(two, dtype(0)), np.nextafter(two[:-1], top), rng.uniform(0, 3, 200),
                          10.0 ** rng.uniform(-9, 6, 200), [top]]).astype(dtype)
    lim = dtype(2.0) ** dtype(guard)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, info.max, -info.max, info.tiny, info.smallest_subnormal, 1.0,
                        lim, np.nextafter(lim, dtype(0)), np.nextafter(lim, dtype(1))], dtype)
    n = 4000
    for s in sig:
        near = (lim * rng.uniform(0.5, 4, n)).astype(dtype)
        wide = rng.standard_normal(n).astype(dtype) * (dtype(10) ** rng.uniform(np.log10(float(lim)), 30, n)).astype(dtype)
        ties = (dtype(1) + s) * rng.integers(1, 1 << 12, n).astype(dtype) * lim  # quotients that end early
        a = np.concatenate([special, near, wide, ties]).astype(dtype)
        got, want = np.zeros_like(a), np.zeros_like(a)
        getattr(host, f"quotient_{name}")(_p(a), _p(np.full_like(a, s)), _p(got), _p(want), ctypes.c_long(a.size))
        same = (got == want) & (np.signbit(got) == np.signbit(want)) | (np.isnan(got) & np.isnan(want))
        assert same.all(), (s, a[~same][:3], got[~same][:3], want[~same][:3])


def test_header_quotient_has_a_range(host):
    """Outside 0 <= sigma <= 2^20 the quotient is not the IEEE one, which is why
    the kernel is not used there."""
    # a / b = (2k + 1) 2^-150, half way between two subnormal numbers
    a = np.array([3 * (2 * k + 1) * 2.0 ** -120 for k in range(1 << 19, (1 << 19) + 64)] + [3e38], np.float32)
    s = np.array([3 * 2.0 ** 30] * 64 + [-0.5], np.float32)
    got, want = np.zeros_like(a), np.zeros_like(a)
    host.quotient_float(_p(a), _p(s), _p(got), _p(want), ctypes.c_long(a.size))
    assert np.isinf(want[-1]) and np.isnan(got[-1])
    assert (got[:-1] != want[:-1]).any()
