"""The divisions kh_half.hpp replaces, on the CPU with the same operations.

Index division by a magic number is exact; the quotient from two residual
corrections is the IEEE quotient for every sigma a profile can hold and every
value its guard lets through (fused multiply-adds formed in extended precision:
the products are exact there, the sums round once more far below one ulp).
"""
import numpy as np


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
