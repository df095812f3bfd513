// kh_div.hpp -- the divisions of half_kernel: an index by a constant, and a
// quotient by a number whose reciprocal is known.  Plain C++ but for two
// builtins, so that a test can run the same code on the host.
#pragma once

#include <cmath>
#include <cstdint>

namespace kh {

// c / d for c < 2^31 by a multiplication, with d's magic number from
// div_magic() (Granlund and Montgomery, Division by invariant integers using
// multiplication, 1994).
struct FastDiv {
    uint32_t m, s;
};

inline FastDiv div_magic(uint32_t d) {
    uint32_t l = 0;
    while (l < 31 && (1u << l) < d) ++l;  // 2^l >= d
    return FastDiv{(uint32_t)((((uint64_t)1 << (31 + l)) + d - 1) / d), l};
}

__host__ __device__ __forceinline__ uint32_t fdiv(uint32_t c, const FastDiv &f) {
    return (uint32_t)(((uint64_t)c * f.m) >> (31 + f.s));
}

__host__ __device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__host__ __device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }

// q as the quotient a / b, with the sign and the special values (zeros,
// infinities, NaN) that a and b give it
#if defined(__AMDGCN__)
__device__ __forceinline__ float fixup_(float q, float b, float a) { return __builtin_amdgcn_div_fixupf(q, b, a); }
__device__ __forceinline__ double fixup_(double q, double b, double a) { return __builtin_amdgcn_div_fixup(q, b, a); }
__device__ __forceinline__ bool any_(bool v) { return __any(v); }
#else
template <typename T>
inline T fixup_(T q, T b, T a) {
    const bool special = a == 0 || b == 0 || !std::isfinite(a) || !std::isfinite(b);
    return special ? a / b : std::copysign(q, std::copysign(T(1), a) * std::copysign(T(1), b));
}
inline bool any_(bool v) { return v; }
#endif

// 0 < |a| < 2^-100 (2^-960): the residuals of div_by could underflow
__host__ __device__ __forceinline__ bool tiny_(float a) {
    return (__builtin_bit_cast(uint32_t, a) & 0x7fffffffu) - 1u < (27u << 23) - 1u;
}
__host__ __device__ __forceinline__ bool tiny_(double a) {
    return ((uint32_t)(__builtin_bit_cast(uint64_t, a) >> 32) & 0x7fffffffu) < (63u << 20) && a != 0.0;
}

// (a0 / b0, a1 / b1) as IEEE division rounds them, r = 1 / b rounded to
// nearest, 1 <= b <= 1 + DIV_SIGMA_MAX: two residual corrections of a r
// (Markstein's division), half the instructions of a general division.  Below 1
// a large quotient overflows on the way, past 2^26 a quotient of the smallest a
// that is not tiny_ is subnormal, where a r can lie half way between two values.  A wave that holds a tiny value (the
// front of a wave that is still building up) divides.  (A product with 1 / b
// in double rounds right for float as well, in fewer instructions, but the
// conversions are slow: 64^3 12.3 us a step against 11.3.)
constexpr double DIV_SIGMA_MAX = 1048576.0;  // 2^20

template <typename T>
__host__ __device__ __forceinline__ void div_by(T a0, T a1, T b0, T b1, T r0, T r1, T &q0, T &q1) {
    T p = a0 * r0, q = a1 * r1;
    p = fma_(fma_(-b0, p, a0), r0, p);
    q = fma_(fma_(-b1, q, a1), r1, q);
    p = fma_(fma_(-b0, p, a0), r0, p);
    q = fma_(fma_(-b1, q, a1), r1, q);
    q0 = fixup_(p, b0, a0);  // infinities and NaN
    q1 = fixup_(q, b1, a1);
    if (any_(tiny_(a0) || tiny_(a1))) {
        q0 = a0 / b0;
        q1 = a1 / b1;
    }
}

}  // namespace kh
