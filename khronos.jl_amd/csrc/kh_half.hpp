// kh_half.hpp -- the FAST half step (H or E) on the whole grid where the
// last-level cache holds most of what a step touches (Ctx::choose_form has the
// line), without conductivity: the update of the pml_* kernels with the same
// operations on the same values (bit for bit).
//
// Up to about 64^3 float cells (two waves a SIMD) a launch is one round of waves
// and its time is that of one wave: 5.4 us with 16.5 MB past the L2, 3.0 TB/s.
// From about 80^3 double or 100^3 float cells on it is what the caches give
// back: 131 x 117 x 101 float 12 waves a SIMD, 91 MB (H) and 97 MB (E) past the
// L2 in 17-18 us, 5.4 TB/s, the address units half busy.  So
//   * a pair's (x, y, z) comes from two multiplications (FastDiv), its
//     accesses from a scalar base and one 32-bit offset;
//   * which stages exist is decided by index (outside the longest run of zero
//     sigma of an axis), not by loading sigma first, so the stages, the sigma
//     samples and the fields are all one round of loads;
//   * three straight-line forms of the code, chosen per wave: no sigma at all,
//     sigma along x only (the ends of every row), anything;
//   * 1 / (1 + sigma) comes from a table, the quotient from div_by instead of
//     a division's dozen instructions;
//   * x + 1 / x - 1 across lanes by a wave shift, loaded only by end lanes;
//   * the material table in LDS, a copy per wave: waves of one block take
//     different forms of the code, so nothing makes them meet;
//   * accesses keep their lines (the pml_* kernels stream with nontemporal
//     hints), and each XCD takes one contiguous eighth of the grid, so that
//     what an XCD wrote in one half step is in its L2 or the last-level cache
//     in the next.
// One step (two half steps), against the pml_* kernels: 64^3 float 13.8 ->
// 11.3 us, 131 x 117 x 101 float 46.3 -> 41.3, 160 x 145 x 120 float with
// per-voxel arrays 61.2 -> 54.7, 80^3 double 28.1 -> 20.4.  The launch shape
// and the code gave 12.3 / 44.5 / 59.5 / 25.2 of that, the last item the rest.
// Of 64^3's 11.3 us two dependent launches that copy its six arrays explain 6.0
// (two empty ones 3.6).
#pragma once

#include "kh_div.hpp"
#include "kh_kernels.hpp"

namespace kh {

// the value of the lane before (AFTER: after); the end lane keeps its own
template <bool AFTER>
__device__ __forceinline__ int lane_beside(int i) {
    return __builtin_amdgcn_update_dpp(i, i, AFTER ? 0x130 : 0x138, 0xf, 0xf, false);
}
template <bool AFTER>
__device__ __forceinline__ float lane_beside(float v) {
    return __builtin_bit_cast(float, lane_beside<AFTER>(__builtin_bit_cast(int, v)));
}
template <bool AFTER>
__device__ __forceinline__ double lane_beside(double v) {
    const uint64_t q = __builtin_bit_cast(uint64_t, v);
    const uint32_t a = (uint32_t)lane_beside<AFTER>((int)(uint32_t)q);
    const uint32_t b = (uint32_t)lane_beside<AFTER>((int)(uint32_t)(q >> 32));
    return __builtin_bit_cast(double, ((uint64_t)b << 32) | a);
}

// sigma of a cell along one axis and 1 / (1 + sigma)
template <typename T>
struct Sig {
    T s, r;
};

// A pair of cells of one component: pml_update's arithmetic.  PO/PN/PP: some
// lane of the wave has a non-zero own/next/prev sigma (elsewhere the division
// by 1 and the multiplication by 1 - 0 are exact and left out).
template <bool PO, bool PN, bool PP, typename V, typename T>
__device__ __forceinline__ V half_value(V ao, V &u, V &w, V m, T K0, T K1, const Sig<T> &so0, const Sig<T> &so1,
                                        const Sig<T> &sn0, const Sig<T> &sn1, const Sig<T> &sp0, const Sig<T> &sp1) {
    T in0 = K0, in1 = K1;
    if constexpr (PN) {
        T un0, un1;
        div_by((T(1) - sn0.s) * u.x + in0, (T(1) - sn1.s) * u.y + in1, T(1) + sn0.s, T(1) + sn1.s, sn0.r, sn1.r, un0,
               un1);
        in0 = sn0.s != T(0) ? un0 - u.x : in0;
        in1 = sn1.s != T(0) ? un1 - u.y : in1;
        u.x = sn0.s != T(0) ? un0 : u.x;
        u.y = sn1.s != T(0) ? un1 : u.y;
    }
    const bool w0 = PO && so0.s != T(0), w1 = PO && so1.s != T(0);
    const T b0 = w0 ? w.x : ao.x, b1 = w1 ? w.y : ao.y;
    V t;
    if constexpr (PP) {
        div_by((T(1) - sp0.s) * b0 + m.x * in0, (T(1) - sp1.s) * b1 + m.y * in1, T(1) + sp0.s, T(1) + sp1.s, sp0.r,
               sp1.r, t.x, t.y);
    } else {
        t.x = b0 + m.x * in0;
        t.y = b1 + m.y * in1;
    }
    if constexpr (PO) {
        const T a0 = (ao.x + (T(1) + so0.s) * t.x) - (T(1) - so0.s) * w.x;
        const T a1 = (ao.y + (T(1) + so1.s) * t.y) - (T(1) - so1.s) * w.y;
        w.x = w0 ? t.x : w.x;
        w.y = w1 ? t.y : w.y;
        t.x = w0 ? a0 : t.x;
        t.y = w1 ? a1 : t.y;
    }
    return t;
}

constexpr int LUT_SIZE = 256;  // a byte indexes the table; four entries a lane of a wave

template <typename T>
struct HalfArgs {
    uint32_t sy, sz;       // element strides
    uint32_t npair, ncell; // pairs per row, in all
    FastDiv dpair, dy;
    int n[3];
    int zr[3][2];          // per axis, the longest run of zero sigma, inclusive
    const T *sigp[3];      // (sigma, 1 / (1 + sigma)) per index
    // the arrays, materials (minv, mid, lut), XCD mapping, sources, snapshots
    // and DFT monitors as the pml_* kernels take them
    PmlArgs<T> q;
};

template <typename T, bool ELEC, int EPS, int NP, bool PRE, bool SNAP, bool DFTE>
struct HalfLane {
    using V = typename V2<T>::t;
    static constexpr uint32_t S = sizeof(T);
    typedef T E2 __attribute__((ext_vector_type(2)));
    const HalfArgs<T> &p;
    typedef T E4 __attribute__((ext_vector_type(4)));
    T *lut;      // the wave's copy of the material table
    E4 lut_mine; // its entries 4 lane .. 4 lane + 3
    uint32_t o, sy, sz;
    int x, y, z;
    bool live, v1, bx, by, bz;
    Sig<T> sx0, sx1, sgy, sgz;
    V m[3];
    uint32_t mq[3];

    __device__ __forceinline__ explicit HalfLane(const HalfArgs<T> &a) : p(a) {}

    template <typename P>
    static __device__ __forceinline__ __attribute__((address_space(1))) P *at(const void *b, uint32_t off) {
        typedef __attribute__((address_space(1))) char G;
        return (__attribute__((address_space(1))) P *)((G *)(uintptr_t)b + off);
    }
    static __device__ __forceinline__ V ld(const T *b, uint32_t off) {
        const E2 r = *at<E2>(b, off);
        V v;
        v.x = r[0];
        v.y = r[1];
        return v;
    }
    static __device__ __forceinline__ T ld1(const T *b, uint32_t off) { return *at<T>(b, off); }
    static __device__ __forceinline__ void st(T *b, uint32_t off, V v) {
        const E2 r = {v.x, v.y};
        *at<E2>(b, off) = r;
    }

    __device__ __forceinline__ Sig<T> sig(int axis, int i) const {
        const V v = ld(p.sigp[axis], 2 * S * (uint32_t)i);
        return Sig<T>{v.x, v.y};
    }

    // update and store component a of part f; u, w: its old stages
    template <bool PO, bool PN, bool PP>
    __device__ __forceinline__ void update(const PmlPart<T> &f, int a, V ao, V u, V w, bool bo, bool bn, T K0, T K1,
                                           const Sig<T> &so0, const Sig<T> &so1, const Sig<T> &sn0, const Sig<T> &sn1,
                                           const Sig<T> &sp0, const Sig<T> &sp1, T dw0, T dw1, bool h0, bool h1, V &kept,
                                           V &stored) const {
        V an = half_value<PO, PN, PP>(ao, u, w, m[a], K0, K1, so0, so1, sn0, sn1, sp0, sp1);
        if (PRE && h0) {
            if (so0.s == T(0)) {
                an.x = an.x + dw0;
            } else {
                w.x = w.x + dw0;
                an.x = an.x + (T(1) + so0.s) * dw0;
            }
        }
        if (PRE && h1) {
            if (so1.s == T(0)) {
                an.y = an.y + dw1;
            } else {
                w.y = w.y + dw1;
                an.y = an.y + (T(1) + so1.s) * dw1;
            }
        }
        if (!v1) {
            // the pair's second element is the ghost: written back unchanged
            // (its stages are zero and stay so)
            an.y = ao.y;
            u.y = w.y = T(0);
        }
        if (live) {
            if (PN && bn) st(f.U[a], o, u);
            if (PO && bo) st(f.W[a], o, w);
            st(f.A[a], o, an);
        }
        if (SNAP) {
            kept.x = so0.s != T(0) ? w.x : an.x;
            kept.y = so1.s != T(0) ? w.y : an.y;
        }
        if (DFTE) stored = an;
    }

    template <bool PX, bool PY, bool PZ>
    __device__ __forceinline__ void part(int q, T dw0, T dw1, bool h0, bool h1) {
        const PmlPart<T> &f = p.q.f[q];
        const T *F0 = f.F[0], *F1 = f.F[1], *F2 = f.F[2];
        const bool edge = ELEC ? (x == 1 || (threadIdx.x & 63) == 0) : (x + 2 > p.n[0] || (threadIdx.x & 63) == 63);
        // the differentiated field: own cells, one row and one plane on (H) or
        // back (E), and the elements beside the pair of components 1 and 2
        const V a0 = ld(F0, o);
        V a1 = ld(F1, o), a2 = ld(F2, o);
        const uint32_t oz = ELEC ? o - sz : o + sz, oy = ELEC ? o - sy : o + sy;
        const V z0 = ld(F0, oz), z1 = ld(F1, oz), y2 = ld(F2, oy), y0 = ld(F0, oy);
        T e1 = 0, e2 = 0;
        if (edge) {
            e1 = ld1(F1, ELEC ? o - S : o + 2 * S);
            e2 = ld1(F2, ELEC ? o - S : o + 2 * S);
        }
        const V ao0 = ld(f.A[0], o), ao1 = ld(f.A[1], o), ao2 = ld(f.A[2], o);
        // (U, W) of component 0: next y, own x; 1: next z, own y; 2: next x, own z
        V u0{}, u1{}, u2{}, w0{}, w1{}, w2{};
        if (PX && bx) {
            u2 = ld(f.U[2], o);
            w0 = ld(f.W[0], o);
        }
        if (PY && by) {
            u0 = ld(f.U[0], o);
            w1 = ld(f.W[1], o);
        }
        if (PZ && bz) {
            u1 = ld(f.U[1], o);
            w2 = ld(f.W[2], o);
        }
        if (q == 0) {
            sx0 = sx1 = sgy = sgz = Sig<T>{T(0), T(1)};
            if (PX && bx) {
                sx0 = sig(0, x);
                sx1 = sig(0, x + 1);
            }
            if (PY && by) sgy = sig(1, y);
            if (PZ && bz) sgz = sig(2, z);
            if constexpr (EPS == 2) {
                // the table is the oldest load in flight, all the others are
                // behind it; only this wave's lanes read what it writes
                *(E4 *)(lut + 4 * (threadIdx.x & 63)) = lut_mine;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                for (int a = 0; a < 3; ++a) {
                    m[a].x = lut[mq[a] & 0xff];
                    m[a].y = lut[mq[a] >> 8];
                }
            }
        }
        // beside the pair: from the next (H) or the previous (E) lane
        T b1 = lane_beside<!ELEC>(ELEC ? a1.y : a1.x), b2 = lane_beside<!ELEC>(ELEC ? a2.y : a2.x);
        if (edge) {
            b1 = e1;
            b2 = e2;
        }
        if (p.q.perx) {
            // H reads E at x = N + 1 as E at x = 1 times the Bloch phase, E reads H
            // at x = 0 as H at x = N times the reverse phase
            const size_t i = (size_t)(o / S);
            if (ELEC) {
                if (x == 1) {
                    b2 = xwrap_val(f, 2, i - 1 + (size_t)p.q.nxg);
                    b1 = xwrap_val(f, 1, i - 1 + (size_t)p.q.nxg);
                }
            } else if (x + 1 == p.q.nxg) {
                b2 = xwrap_val(f, 2, i + 2 - (size_t)p.q.nxg);
                b1 = xwrap_val(f, 1, i + 2 - (size_t)p.q.nxg);
            } else if (x == p.q.nxg) {
                a2.y = xwrap_val(f, 2, i + 1 - (size_t)p.q.nxg);
                a1.y = xwrap_val(f, 1, i + 1 - (size_t)p.q.nxg);
            }
        }
        const T dt = p.q.dt, ix = p.q.inv[0], iy = p.q.inv[1], iz = p.q.inv[2];
        // d(.) = inv * (neighbour - own) for both directions of the difference
        const T Kx0 = dt * (iz * (z1.x - a1.x) - iy * (y2.x - a2.x));
        const T Kx1 = dt * (iz * (z1.y - a1.y) - iy * (y2.y - a2.y));
        const T Ky0 = dt * (ix * ((ELEC ? b2 : a2.y) - a2.x) - iz * (z0.x - a0.x));
        const T Ky1 = dt * (ix * ((ELEC ? a2.x : b2) - a2.y) - iz * (z0.y - a0.y));
        const T Kz0 = dt * (iy * (y0.x - a0.x) - ix * ((ELEC ? b1 : a1.y) - a1.x));
        const T Kz1 = dt * (iy * (y0.y - a0.y) - ix * ((ELEC ? a1.x : b1) - a1.y));
        const int pc = p.q.pre_comp;
        V kept[3], stored[3];
        update<PX, PY, PZ>(f, 0, ao0, u0, w0, bx, by, Kx0, Kx1, sx0, sx1, sgy, sgy, sgz, sgz, dw0, dw1, h0 && pc == 0,
                           h1 && pc == 0, kept[0], stored[0]);
        update<PY, PZ, PX>(f, 1, ao1, u1, w1, by, bz, Ky0, Ky1, sgy, sgy, sgz, sgz, sx0, sx1, dw0, dw1, h0 && pc == 1,
                           h1 && pc == 1, kept[1], stored[1]);
        update<PZ, PX, PY>(f, 2, ao2, u2, w2, bz, bx, Kz0, Kz1, sgz, sgz, sx0, sx1, sgy, sgy, dw0, dw1, h0 && pc == 2,
                           h1 && pc == 2, kept[2], stored[2]);
        if (live) {
            if (SNAP)
                for (int a = 0; a < 3; ++a) pml_snap(p.q, a, x, y, z, true, v1, kept[a]);
            if (DFTE)
                for (int a = 0; a < 3; ++a) pml_dft(p.q, a, x, y, z, true, v1, stored[a]);
        }
    }

    template <bool PX, bool PY, bool PZ>
    __device__ __forceinline__ void run() {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if constexpr (EPS == 2) {
                mq[a] = *at<unsigned short>(p.q.mid[a], o / S);
            } else if constexpr (EPS == 1) {
                m[a] = ld(p.q.minv[a], o);
            } else {
                m[a].x = m[a].y = p.q.minv_s;
            }
        }
        T dw0 = T(0), dw1 = T(0);
        bool h0 = false, h1 = false;
        if (PRE) pml_pre_load(p.q, x, y, z, true, v1, dw0, dw1, h0, h1);
        part<PX, PY, PZ>(0, dw0, dw1, h0, h1);
        if (NP == 2) part<PX, PY, PZ>(1, T(0), T(0), false, false);
        if (live && p.q.nsrc > 0) pml_sources(p.q, (size_t)(o / S), x, y, z, true, v1);
    }
};

// EPS: 0 scalar material, 1 per-voxel arrays, 2 byte per cell into a table.
// NP: parts (2: complex fields).  PRE, SNAP, DFTE: as the pml_* kernels.
template <typename T, bool ELEC, int EPS, int NP = 1, bool PRE = false, bool SNAP = false, bool DFTE = false>
__global__ __launch_bounds__(CBLK) void half_kernel(HalfArgs<T> args) {
    // the arguments where they lie (they start the argument segment): read as
    // needed; indexing the parameter itself makes the compiler copy all of it
    // to scratch memory in the larger variants
    const HalfArgs<T> &p = *(const HalfArgs<T> *)__builtin_amdgcn_kernarg_segment_ptr();
    __shared__ __attribute__((aligned(32))) T lut[EPS == 2 ? CBLK / 64 * LUT_SIZE : 1];
    HalfLane<T, ELEC, EPS, NP, PRE, SNAP, DFTE> k(p);
    k.lut = lut + (EPS == 2 ? threadIdx.x / 64 * LUT_SIZE : 0);
    if constexpr (EPS == 2) k.lut_mine = ((const typename decltype(k)::E4 *)p.q.lut)[threadIdx.x & 63];
    // physical block b runs on XCD b % 8: block j of XCD x is logical block
    // x * per_xcd + j
    const int j = (int)(blockIdx.x / NXCD), L = (int)(blockIdx.x % NXCD) * p.q.per_xcd + j;
    if (L >= p.q.nblock) return;
    const uint32_t t = (uint32_t)L * CBLK + threadIdx.x;
    k.live = t < p.ncell;
    const uint32_t c = k.live ? t : p.ncell - 1;  // lanes past the end repeat the last pair
    const uint32_t row = fdiv(c, p.dpair), zr = fdiv(row, p.dy);
    k.x = 1 + 2 * (int)(c - row * p.npair);
    k.y = 1 + (int)(row - zr * (uint32_t)p.n[1]);
    k.z = 1 + (int)zr;
    k.v1 = k.x + 1 <= p.n[0];
    constexpr uint32_t S = sizeof(T);
    k.sy = p.sy * S;
    k.sz = p.sz * S;
    k.o = ((uint32_t)k.x + (uint32_t)k.y * p.sy + (uint32_t)k.z * p.sz) * S;
    k.bx = k.x < p.zr[0][0] || k.x + 1 > p.zr[0][1];
    k.by = k.y < p.zr[1][0] || k.y > p.zr[1][1];
    k.bz = k.z < p.zr[2][0] || k.z > p.zr[2][1];
    if (__any(k.by || k.bz)) k.template run<true, true, true>();
    else if (__any(k.bx)) k.template run<true, false, false>();
    else k.template run<false, false, false>();
}

}  // namespace kh
