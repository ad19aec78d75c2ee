// Device code shared by the kernels of the LC2 engine: samplers, the least-squares fit,
// reductions and window sums. Included by the .hip files only.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <initializer_list>
#include <type_traits>

#include "lc2e_kernels.hpp"

namespace lc2e {

namespace {

constexpr double kZeroThreshold = 1e-6;  // cu_lc2_helper.cuh:5
constexpr double kTauConst = 1e-10;      // centred energy below this fraction of raw -> constant
constexpr double kTauColl = 1e-10;       // Gram determinant below this fraction -> collinear

// Compile-time loop: calls f(integral_constant<int, K>) for K = B .. E-1.
template <int B, int E>
struct Unroll {
    template <class F>
    __device__ __forceinline__ static void run(F&& f) {
        f(std::integral_constant<int, B>{});
        Unroll<B + 1, E>::run(f);
    }
};
template <int E>
struct Unroll<E, E> {
    template <class F>
    __device__ __forceinline__ static void run(F&&) {}
};

template <typename T>
__device__ __forceinline__ float ld1(const T* p, int i) {
    if constexpr (sizeof(T) == 2) return __half2float(p[i]);
    else return p[i];
}

// The voxels at x0 and x0 + 1 of one row in a single load. Volumes are allocated with a
// zeroed tail, so x0 + 1 is readable even for the last voxel; when the sample lies on
// the integer x0 the reference reads x0 twice (ceil == floor), which is restored here.
template <typename T>
__device__ __forceinline__ void ld2(const T* p, int i, bool same, float& a, float& b) {
    if constexpr (sizeof(T) == 2) {
        __half2 h;
        __builtin_memcpy(&h, p + i, sizeof(h));
        a = __low2float(h);
        b = __high2float(h);
    } else {
        float2 f;
        __builtin_memcpy(&f, p + i, sizeof(f));
        a = f.x;
        b = f.y;
    }
    if (same) b = a;
}

// Voxel coordinates of a position in mm: (p - origin) / spacing with one rounding, as the
// reference's ToPxl computes it (spatialMappers.cuh:143-169). The fused kernels are
// instantiated per form, so their samplers carry no branch for it: P2 (every spacing a
// power of two) multiplies by the exact 1/s; otherwise the IEEE division. (A division by a
// constant as fmaf(a, RN(1/s), RN(a * zl)), exact for a checked spacing, took more time
// on the CT workload than the division it replaced, once its guard for tiny numerators was
// in: 12.05 vs 11.20 ms per launch, measured. The product with RN(1/s) and one correction by the
// remainder, exact for every divisor, left k_warp_grad3 at 640 us for 8 poses of that CT: its
// gathers bound it, not the division.)
template <bool P2>
__device__ __forceinline__ float to_voxel1(float p, float o, float sp, float rs) {
    if (P2) return (p - o) * rs;
    return (p - o) / sp;
}

template <bool P2>
__device__ __forceinline__ void to_voxel2(const SGeom& s, float px, float py, float& vx,
                                          float& vy) {
    vx = to_voxel1<P2>(px, s.ox, s.sx, s.rsx);
    vy = to_voxel1<P2>(py, s.oy, s.sy, s.rsy);
}

template <bool P2>
__device__ __forceinline__ void to_voxel(const SGeom& s, float px, float py, float pz, float& vx,
                                         float& vy, float& vz) {
    to_voxel2<P2>(s, px, py, vx, vy);
    vz = to_voxel1<P2>(pz, s.oz, s.sz, s.rsz);
}

// The same with the form chosen at run time (the one-off samplers).
__device__ __forceinline__ void to_voxel_rt(const SGeom& s, float px, float py, float pz,
                                            float& vx, float& vy, float& vz) {
    if (s.pow2) to_voxel<true>(s, px, py, pz, vx, vy, vz);
    else to_voxel<false>(s, px, py, pz, vx, vy, vz);
}
__device__ __forceinline__ void to_voxel2_rt(const SGeom& s, float px, float py, float& vx,
                                             float& vy) {
    if (s.pow2) to_voxel2<true>(s, px, py, vx, vy);
    else to_voxel2<false>(s, px, py, vx, vy);
}

// round(b - a) in f32 for the low / high halves of two half2 words: v_fma_mix_f32 with
// f16 sources b and -a and the f32 constant 1.0, i.e. fma(b, 1, -a) with one rounding.
__device__ __forceinline__ float hsub_lo(unsigned b, unsigned a) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,1]" : "=v"(r) : "v"(b), "v"(a));
    return r;
}
__device__ __forceinline__ float hsub_hi(unsigned b, unsigned a) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]"
        : "=v"(r) : "v"(b), "v"(a));
    return r;
}
__device__ __forceinline__ float hlo(unsigned w) {
    __half2 h;
    __builtin_memcpy(&h, &w, sizeof(h));
    return __low2float(h);
}
__device__ __forceinline__ float hhi(unsigned w) {
    __half2 h;
    __builtin_memcpy(&h, &w, sizeof(h));
    return __high2float(h);
}

// Interpolate_3Dkernel sample (interpolator.cu:76-174): L -> M*L -> voxel -> trilinear
// z, y, x with floor/ceil corners; 0 outside [0, dim-1].
template <typename T>
__device__ __forceinline__ float sample3(const T* __restrict__ src, const SGeom& s, const float* m,
                                         float lx, float ly, float lz) {
    const float px = fmaf(m[2], lz, fmaf(m[1], ly, m[0] * lx)) + m[3];
    const float py = fmaf(m[6], lz, fmaf(m[5], ly, m[4] * lx)) + m[7];
    const float pz = fmaf(m[10], lz, fmaf(m[9], ly, m[8] * lx)) + m[11];
    float vx, vy, vz;
    to_voxel_rt(s, px, py, pz, vx, vy, vz);
    if (!(vx >= 0.0f && vx <= (float)(s.X - 1) && vy >= 0.0f && vy <= (float)(s.Y - 1) &&
          vz >= 0.0f && vz <= (float)(s.Z - 1)))
        return 0.0f;
    const float fx = floorf(vx), fy = floorf(vy), fz = floorf(vz);
    const int x0 = (int)fx, y0 = (int)fy, z0 = (int)fz;
    const int y1 = (int)ceilf(vy), z1 = (int)ceilf(vz);
    const bool xs = (fx == vx);
    const float rx = vx - fx, ry = vy - fy, rz = vz - fz;
    const int sxy = s.X * s.Y;
    const int r00 = y0 * s.X + z0 * sxy, r01 = y0 * s.X + z1 * sxy;
    const int r10 = y1 * s.X + z0 * sxy, r11 = y1 * s.X + z1 * sxy;
    if constexpr (sizeof(T) == 2) {
        // half2 words of the two x neighbours; on an integer x (xs) rx == 0 selects x0
        const char* base = reinterpret_cast<const char*>(src);
        unsigned wa, wb, wc, wd;
        __builtin_memcpy(&wa, base + (size_t)(x0 + r00) * 2, 4);
        __builtin_memcpy(&wb, base + (size_t)(x0 + r01) * 2, 4);
        __builtin_memcpy(&wc, base + (size_t)(x0 + r10) * 2, 4);
        __builtin_memcpy(&wd, base + (size_t)(x0 + r11) * 2, 4);
        const float lu = fmaf(rz, hsub_lo(wb, wa), hlo(wa));
        const float ru = fmaf(rz, hsub_hi(wb, wa), hhi(wa));
        const float lb = fmaf(rz, hsub_lo(wd, wc), hlo(wc));
        const float rb = fmaf(rz, hsub_hi(wd, wc), hhi(wc));
        const float yl = fmaf(ry, lb - lu, lu);
        const float yr = fmaf(ry, rb - ru, ru);
        return fmaf(rx, yr - yl, yl);
    }
    float a0, a1, b0, b1;
    ld2(src, x0 + r00, xs, a0, a1);  // (x0, y0, z0), (x1, y0, z0)
    ld2(src, x0 + r01, xs, b0, b1);  // (x0, y0, z1), (x1, y0, z1)
    const float lu = fmaf(rz, b0 - a0, a0);
    const float ru = fmaf(rz, b1 - a1, a1);
    ld2(src, x0 + r10, xs, a0, a1);  // (x0, y1, z0), (x1, y1, z0)
    ld2(src, x0 + r11, xs, b0, b1);  // (x0, y1, z1), (x1, y1, z1)
    const float lb = fmaf(rz, b0 - a0, a0);
    const float rb = fmaf(rz, b1 - a1, a1);
    const float yl = fmaf(ry, lb - lu, lu);
    const float yr = fmaf(ry, rb - ru, ru);
    return fmaf(rx, yr - yl, yl);
}

// The same trilinear sample split in two for software pipelining: issue3() computes the
// voxel coordinates and starts the four paired loads, finish3() does the lerps once the
// data has arrived, so a whole z-step of work can run in between. Nothing but the loaded
// values and the fractions is carried across the step (no per-lane flags):
//  * a sample outside the source, or a position outside the grid (inside == false),
//    loads from the volume's zeroed tail, so its lerps give exactly 0;
//  * on an integer x the reference reads x0 twice (ceil == floor); here rx == 0 then, and
//    fmaf(0, yr - yl, yl) == yl for the finite values a resident volume holds (f16
//    storage rejects values beyond its range), up to the sign of a zero.
// Inside the volume the clamps change nothing: the result is the reference's.
// f32 sources keep the eight corner values; half sources keep the four loaded half2 words
// as they are, and the lerps read them through mixed-precision FMAs (exactly the f32
// arithmetic on the converted values, without separate conversions).
template <typename T>
struct Pending3 {
    float a0, a1, b0, b1, c0, c1, d0, d1;
    float rx, ry, rz;
};
template <>
struct Pending3<__half> {
    unsigned a, b, c, d;  // half2: x0 in the low half, x0 + 1 in the high half
    float rx, ry, rz;
};
// Half sources of even X: each pair within the two aligned words that hold it (a load at an odd
// element takes longer than one of 8 aligned bytes), shifted into place when it is used. All four
// pairs of a sample are at offsets of the same parity then. The last word read is 2 elements past
// what the zeroed tail must hold, of its 64 to spare.
struct Pending3W {
    uint2 a, b, c, d;
    unsigned sh;  // bits, in the low 5
    float rx, ry, rz;
};
template <typename T, bool WORDS>
struct PendSel {
    using type = Pending3<T>;
};
template <>
struct PendSel<__half, true> {
    using type = Pending3W;
};


template <typename T>
__device__ __forceinline__ void ld2_off(const T* __restrict__ base, unsigned idx, float& a,
                                        float& b) {
    // 32-bit element offset from a uniform base: one saddr + voffset load, no 64-bit math
    const char* p = reinterpret_cast<const char*>(base) + idx * (unsigned)sizeof(T);
    if constexpr (sizeof(T) == 2) {
        __half2 h;
        __builtin_memcpy(&h, p, sizeof(h));
        a = __low2float(h);
        b = __high2float(h);
    } else {
        float2 f;
        __builtin_memcpy(&f, p, sizeof(f));
        a = f.x;
        b = f.y;
    }
}

template <bool P2, typename T, typename PEND>
__device__ __forceinline__ void issue3v(const T* __restrict__ src, const SGeom& s, float px,
                                        float py, float pz, bool inside, PEND& p);

template <bool P2, typename T>
__device__ __forceinline__ void issue3(const T* __restrict__ src, const SGeom& s, const float* m,
                                       float lx, float ly, float lz, bool inside, Pending3<T>& p) {
    const float px = fmaf(m[2], lz, fmaf(m[1], ly, m[0] * lx)) + m[3];
    const float py = fmaf(m[6], lz, fmaf(m[5], ly, m[4] * lx)) + m[7];
    const float pz = fmaf(m[10], lz, fmaf(m[9], ly, m[8] * lx)) + m[11];
    issue3v<P2>(src, s, px, py, pz, inside, p);
}

// v clamped to [0, hi] in one instruction (fminf / fmaxf cost four: IEEE mode makes each
// quieten its inputs first). The coordinates here come from arithmetic, so a NaN is quiet,
// and v_med3_f32 then returns the minimum of the other two operands, 0.
__device__ __forceinline__ float clamp_med3(float v, float hi) {
    return __builtin_amdgcn_fmed3f(v, 0.0f, hi);
}

// The paired loads of the pipelined samplers always take the rows y0 + 1 and planes
// z0 + 1, where the reference takes ceil(v) (equal to v on an integer coordinate). On an
// integer coordinate the fraction is exactly 0 there, so fmaf(0, b - a, a) == a for the
// finite values a resident volume holds (uploads reject non-finite voxels), up to the sign
// of a zero: the reference's value. One row / plane past the last one lands in the zeroed
// tail (volume_pad_elems), as do all four corners of a sample outside the source. So a
// sample needs one 32-bit element offset: the four corners are two byte offsets (plane z0
// and z0 + 1) from two uniform bases (rows y0 and y0 + 1), with no per-corner arithmetic.
template <typename T>
__device__ __forceinline__ void corners_off(const T* __restrict__ src, const SGeom& s, unsigned e0,
                                            unsigned plane, unsigned& o0, unsigned& o1,
                                            const char*& b0, const char*& b1) {
    o0 = e0 * (unsigned)sizeof(T);
    o1 = o0 + plane * (unsigned)sizeof(T);
    b0 = reinterpret_cast<const char*>(src);
    b1 = b0 + (size_t)s.X * sizeof(T);
}

// issue3 from the source position (px, py, pz) in mm.
template <bool P2, typename T, typename PEND>
__device__ __forceinline__ void issue3v(const T* __restrict__ src, const SGeom& s, float px,
                                        float py, float pz, bool inside, PEND& p) {
    float vx, vy, vz;
    to_voxel<P2>(s, px, py, pz, vx, vy, vz);
    const float xm = (float)(s.X - 1), ym = (float)(s.Y - 1), zm = (float)(s.Z - 1);
    // clamped coordinates (one v_med3_f32 each; with a quiet-NaN input it returns the
    // smaller bound, 0); a coordinate lies in [0, dim - 1] exactly when the clamp leaves it
    // unchanged, which NaN never is
    const float cx = clamp_med3(vx, xm), cy = clamp_med3(vy, ym), cz = clamp_med3(vz, zm);
    const bool ok = inside && cx == vx && cy == vy && cz == vz;
    // on c >= 0: conversion truncates to floor(c), and v_fract_f32 gives c - floor(c) exactly
    p.rx = __builtin_amdgcn_fractf(cx);
    p.ry = __builtin_amdgcn_fractf(cy);
    p.rz = __builtin_amdgcn_fractf(cz);
    const unsigned X = (unsigned)s.X, sxy = (unsigned)(s.X * s.Y);
    const unsigned tail = sxy * (unsigned)s.Z;  // first element of the zeroed tail
    unsigned e0 = tail;
    if (ok) {
        const unsigned x0 = (unsigned)cx, y0 = (unsigned)cy, z0 = (unsigned)cz;
        // 24-bit multiply-adds (full rate; a 32-bit multiply is quarter rate): dimensions
        // are below 2^24, and so is X*Y for every source the fused kernels sample (pairs
        // with larger slices take the separable path)
        e0 = __umul24(z0, sxy) + (__umul24(y0, X) + x0);
    }
    unsigned o0, o1;
    const char *b0, *b1;
    corners_off(src, s, e0, sxy, o0, o1, b0, b1);
    if constexpr (std::is_same<PEND, Pending3W>::value) {
        p.sh = o0 << 3;
        const unsigned q0 = o0 & ~3u, q1 = o1 & ~3u;
        __builtin_memcpy(&p.a, __builtin_assume_aligned(b0 + q0, 4), 8);
        __builtin_memcpy(&p.b, __builtin_assume_aligned(b0 + q1, 4), 8);
        __builtin_memcpy(&p.c, __builtin_assume_aligned(b1 + q0, 4), 8);
        __builtin_memcpy(&p.d, __builtin_assume_aligned(b1 + q1, 4), 8);
    } else if constexpr (sizeof(T) == 2) {
        __builtin_memcpy(&p.a, b0 + o0, 4);  // (y0, z0)
        __builtin_memcpy(&p.b, b0 + o1, 4);  // (y0, z0 + 1)
        __builtin_memcpy(&p.c, b1 + o0, 4);  // (y0 + 1, z0)
        __builtin_memcpy(&p.d, b1 + o1, 4);  // (y0 + 1, z0 + 1)
    } else {
        float2 f;
        __builtin_memcpy(&f, b0 + o0, 8);
        p.a0 = f.x, p.a1 = f.y;
        __builtin_memcpy(&f, b0 + o1, 8);
        p.b0 = f.x, p.b1 = f.y;
        __builtin_memcpy(&f, b1 + o0, 8);
        p.c0 = f.x, p.c1 = f.y;
        __builtin_memcpy(&f, b1 + o1, 8);
        p.d0 = f.x, p.d1 = f.y;
    }
}

// issue3 with the in-plane part of the source coordinates given: c = m*(lx, ly, 0) as
// issue3 forms it, so px = fmaf(m[2], lz, c[0]) + m[3] is issue3's px bit for bit.
template <bool P2, typename T, typename PEND>
__device__ __forceinline__ void issue3c(const T* __restrict__ src, const SGeom& s, const float* m,
                                        const float* c, float lz, bool inside, PEND& p) {
    const float px = fmaf(m[2], lz, c[0]) + m[3];
    const float py = fmaf(m[6], lz, c[1]) + m[7];
    const float pz = fmaf(m[10], lz, c[2]) + m[11];
    issue3v<P2>(src, s, px, py, pz, inside, p);
}

template <typename T>
__device__ __forceinline__ float finish3(const Pending3<T>& p) {
    float lu, ru, lb, rb;
    if constexpr (sizeof(T) == 2) {
        lu = fmaf(p.rz, hsub_lo(p.b, p.a), hlo(p.a));
        ru = fmaf(p.rz, hsub_hi(p.b, p.a), hhi(p.a));
        lb = fmaf(p.rz, hsub_lo(p.d, p.c), hlo(p.c));
        rb = fmaf(p.rz, hsub_hi(p.d, p.c), hhi(p.c));
    } else {
        lu = fmaf(p.rz, p.b0 - p.a0, p.a0);
        ru = fmaf(p.rz, p.b1 - p.a1, p.a1);
        lb = fmaf(p.rz, p.d0 - p.c0, p.c0);
        rb = fmaf(p.rz, p.d1 - p.c1, p.c1);
    }
    const float yl = fmaf(p.ry, lb - lu, lu);
    const float yr = fmaf(p.ry, rb - ru, ru);
    return fmaf(p.rx, yr - yl, yl);
}
__device__ __forceinline__ float finish3(const Pending3W& p) {
    Pending3<__half> q;
    q.a = __builtin_amdgcn_alignbit(p.a.y, p.a.x, p.sh);
    q.b = __builtin_amdgcn_alignbit(p.b.y, p.b.x, p.sh);
    q.c = __builtin_amdgcn_alignbit(p.c.y, p.c.x, p.sh);
    q.d = __builtin_amdgcn_alignbit(p.d.y, p.d.x, p.sh);
    q.rx = p.rx;
    q.ry = p.ry;
    q.rz = p.rz;
    return finish3(q);
}

// Interpolate_2Dkernel sample (interpolator.cu:186-230): bilinear, y then x. The 2x3
// matrix sits in the 3x4 layout as m[0], m[1], m[3] / m[4], m[5], m[7].
template <typename T>
__device__ __forceinline__ float sample2(const T* __restrict__ src, const SGeom& s, const float* m,
                                         float lx, float ly) {
    const float px = fmaf(m[1], ly, m[0] * lx) + m[3];
    const float py = fmaf(m[5], ly, m[4] * lx) + m[7];
    float vx, vy;
    to_voxel2_rt(s, px, py, vx, vy);
    if (!(vx >= 0.0f && vx <= (float)(s.X - 1) && vy >= 0.0f && vy <= (float)(s.Y - 1)))
        return 0.0f;
    const float fx = floorf(vx), fy = floorf(vy);
    const int x0 = (int)fx, y0 = (int)fy, y1 = (int)ceilf(vy);
    const bool xs = (fx == vx);
    const float ry = vy - fy;
    if constexpr (sizeof(T) == 2) {
        const char* base = reinterpret_cast<const char*>(src);
        unsigned wa, wb;
        __builtin_memcpy(&wa, base + (size_t)(x0 + y0 * s.X) * 2, 4);
        __builtin_memcpy(&wb, base + (size_t)(x0 + y1 * s.X) * 2, 4);
        const float xl = fmaf(ry, hsub_lo(wb, wa), hlo(wa));
        const float xr = fmaf(ry, hsub_hi(wb, wa), hhi(wa));
        return fmaf(vx - fx, xr - xl, xl);  // 0 * (xr - xl) on an integer x
    }
    float a0, a1, b0, b1;
    ld2(src, x0 + y0 * s.X, xs, a0, a1);
    ld2(src, x0 + y1 * s.X, xs, b0, b1);
    const float xl = fmaf(ry, b0 - a0, a0);
    const float xr = fmaf(ry, b1 - a1, a1);
    const float rx = vx - fx;
    return fmaf(rx, xr - xl, xl);
}

// sample2 split like issue3 / finish3: coordinates and the two paired loads now, the
// lerps later. Same flag-free rules: outside the source (or inside == false) the loads
// read the zeroed tail; on an integer x, rx == 0 selects x0.
template <typename T>
struct Pending2 {
    float a0, a1, b0, b1;
    float rx, ry;
};
template <>
struct Pending2<__half> {
    unsigned a, b;  // half2 words at (x0, y0) and (x0, y1)
    float rx, ry;
};

template <bool P2, typename T>
__device__ __forceinline__ void issue2(const T* __restrict__ src, const SGeom& s, const float* m,
                                       float lx, float ly, bool inside, Pending2<T>& p) {
    const float px = fmaf(m[1], ly, m[0] * lx) + m[3];
    const float py = fmaf(m[5], ly, m[4] * lx) + m[7];
    float vx, vy;
    to_voxel2<P2>(s, px, py, vx, vy);
    const float xm = (float)(s.X - 1), ym = (float)(s.Y - 1);
    const float cx = clamp_med3(vx, xm), cy = clamp_med3(vy, ym);
    const bool ok = inside && cx == vx && cy == vy;
    p.rx = __builtin_amdgcn_fractf(cx);  // as in issue3v
    p.ry = __builtin_amdgcn_fractf(cy);
    const unsigned X = (unsigned)s.X;
    const unsigned tail = X * (unsigned)s.Y * (unsigned)s.Z;  // first element of the zeroed tail
    // rows y0 and y0 + 1 (see corners_off): one offset from two uniform bases
    const unsigned o =
        (ok ? __umul24((unsigned)cy, X) + (unsigned)cx : tail) * (unsigned)sizeof(T);
    const char* b0 = reinterpret_cast<const char*>(src);
    const char* b1 = b0 + (size_t)s.X * sizeof(T);
    if constexpr (sizeof(T) == 2) {
        __builtin_memcpy(&p.a, b0 + o, 4);
        __builtin_memcpy(&p.b, b1 + o, 4);
    } else {
        float2 f;
        __builtin_memcpy(&f, b0 + o, 8);
        p.a0 = f.x, p.a1 = f.y;
        __builtin_memcpy(&f, b1 + o, 8);
        p.b0 = f.x, p.b1 = f.y;
    }
}

template <typename T>
__device__ __forceinline__ float finish2(const Pending2<T>& p) {
    float xl, xr;
    if constexpr (sizeof(T) == 2) {
        xl = fmaf(p.ry, hsub_lo(p.b, p.a), hlo(p.a));
        xr = fmaf(p.ry, hsub_hi(p.b, p.a), hhi(p.a));
    } else {
        xl = fmaf(p.ry, p.b0 - p.a0, p.a0);
        xr = fmaf(p.ry, p.b1 - p.a1, p.a1);
    }
    return fmaf(p.rx, xr - xl, xl);
}

// FP64 reciprocal and reciprocal square root: hardware estimate + two Newton steps
// (relative error a few ulp), instead of the long IEEE division / sqrt sequences.
__device__ __forceinline__ double rcp64(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    r = fma(r, fma(-x, r, 1.0), r);
    return r;
}

__device__ __forceinline__ double rsq64(double x) {
    double r = __builtin_amdgcn_rsq(x);
    r = r * fma(-0.5 * x * r, r, 1.5);
    r = r * fma(-0.5 * x * r, r, 1.5);
    return r;
}

// s^T C^+ s for the two-column centred fit. Rank rule: a column whose centred energy is
// at most kTauConst of its raw energy is dropped; two columns with det <= kTauColl*a*b
// are collinear and U is projected on the leading singular direction of the centred,
// unit-normalised columns, I' + sign(rho) G' (of squared norm 2 + 2|rho|): least squares
// by truncated SVD with the cutoff sigma_min/sigma_max <= sqrt(kTauColl)/2. The full-rank
// case is computed without a branch (most patches; independent voxels of a thread can then
// overlap), the others replace it.
__device__ __forceinline__ double explained_var(double a, double b, double c, double p, double q,
                                                double rawa, double rawb) {
    const bool ikeep = a > kTauConst * rawa;
    const bool gkeep = b > kTauConst * rawb;
    const double ab = a * b, det = fma(-c, c, ab), cq = c * q;
    double e = fma(fma(-2.0, cq, b * p), p, (a * q) * q) * rcp64(det);
    if (!(ikeep && gkeep && det > kTauColl * ab)) {
        if (ikeep && gkeep) {
            // reciprocal square roots through the refined hardware estimates (a few ulp)
            const double ra = rsq64(a), rb = rsq64(b);
            const double t = p * ra + (c < 0.0 ? -1.0 : 1.0) * q * rb;
            e = (t * t) * rcp64(2.0 + 2.0 * fabs(c) * ra * rb);
        } else {
            e = ikeep ? p * p * rcp64(a) : gkeep ? q * q * rcp64(b) : 0.0;
        }
    }
    return e;
}

// Weight and measure from the centred energy of U (cyy) and the explained part e
// (cu_lc2_3d.cu:258-284 weight, :596-611 measure): w = sqrt(cyy/(N-1)),
// measure = w - var_res / w with var_res = (cyy - e)/(N-1); 0 if not > 0.
__device__ __forceinline__ void weight_measure(double cyy, double e, double inv_n1, double& w,
                                               double& meas) {
    const double var_u = cyy * inv_n1;
    const double rw = rsq64(var_u);  // 1 / w
    w = var_u * rw;
    // w - ((cyy - e) * inv_n1) / w, with w * w = cyy * inv_n1
    e = fmin(fmax(e, 0.0), cyy);
    meas = (e * inv_n1) * rw;
    if (!(meas > 0.0) || isinf(meas)) meas = 0.0;
}

// Channels I, G, U, II, GG, IG, UU, UI, UG and the count of U > 1e-6. false where w = 0.
__device__ __forceinline__ bool combine(const double* S, int cnt, int N, double& w_out,
                                        double& m_out) {
    if (cnt != N) return false;
    const double inv_n = 1.0 / (double)N, inv_n1 = 1.0 / (double)(N - 1);
    const double sy = S[2];
    const double my = sy * inv_n;
    const double cyy = fma(-my, sy, S[6]);
    if (!(cyy * inv_n1 > kZeroThreshold)) return false;
    const double si = S[0], sg = S[1];
    const double mi = si * inv_n, mg = sg * inv_n;
    const double cii = fma(-mi, si, S[3]);
    const double cgg = fma(-mg, sg, S[4]);
    const double cig = fma(-mi, sg, S[5]);
    const double cyi = fma(-my, si, S[7]);
    const double cyg = fma(-my, sg, S[8]);
    const double e = explained_var(cii, cgg, cig, cyi, cyg, S[3], S[4]);
    weight_measure(cyy, e, inv_n1, w_out, m_out);
    return true;
}

// Static ultrasound: channels I, G, II, GG, IG, UI, UG; mu = patch mean of U,
// cyy = its centred energy (< 0 where w = 0).
__device__ __forceinline__ void combine_static_u_any(const double* S, double mu, double cyy, int N,
                                                     double& w_out, double& m_out) {
    const double inv_n = 1.0 / (double)N, inv_n1 = 1.0 / (double)(N - 1);
    const double si = S[0], sg = S[1];
    const double mi = si * inv_n, mg = sg * inv_n;
    const double cii = fma(-mi, si, S[2]);
    const double cgg = fma(-mg, sg, S[3]);
    const double cig = fma(-mi, sg, S[4]);
    const double cyi = fma(-mu, si, S[5]);
    const double cyg = fma(-mu, sg, S[6]);
    const double e = explained_var(cii, cgg, cig, cyi, cyg, S[2], S[3]);
    weight_measure(cyy, e, inv_n1, w_out, m_out);
}

// The same where the ultrasound has a weight; false elsewhere.
__device__ __forceinline__ bool combine_static_u(const double* S, double mu, double cyy, int N,
                                                 double& w_out, double& m_out) {
    if (!(cyy >= 0.0)) return false;
    combine_static_u_any(S, mu, cyy, N, w_out, m_out);
    return true;
}

// The part of the fit that a static high-resolution image decides, from its channels I, G, II,
// GG, IG: patch means and the coefficients of e = A p^2 + B p q + C q^2, the explained part of
// an ultrasound with the centred products p = C_UI, q = C_UG (explained_var with its rank rule).
// A is 0 exactly where the column I is dropped, C where G is.
__device__ __forceinline__ void store_image_stats(const double* S, int N, double* out, long long stride) {
    const double inv_n = 1.0 / (double)N;
    const double si = S[0], sg = S[1], mi = si * inv_n, mg = sg * inv_n;
    const double a = fma(-mi, si, S[2]), b = fma(-mg, sg, S[3]), c = fma(-mi, sg, S[4]);
    const bool ikeep = a > kTauConst * S[2], gkeep = b > kTauConst * S[3];
    const double ab = a * b, det = fma(-c, c, ab);
    double A = 0.0, B = 0.0, C = 0.0;
    if (ikeep && gkeep) {
        if (det > kTauColl * ab) {
            const double d = rcp64(det);
            A = b * d;
            B = -2.0 * c * d;
            C = a * d;
        } else {
            const double ra = rsq64(a), rb = rsq64(b);
            const double k = rcp64(2.0 + 2.0 * fabs(c) * ra * rb);
            A = ra * ra * k;
            B = (c < 0.0 ? -2.0 : 2.0) * ra * rb * k;
            C = rb * rb * k;
        }
    } else if (ikeep) {
        A = rcp64(a);
    } else if (gkeep) {
        C = rcp64(b);
    }
    out[0] = mi;
    out[stride] = mg;
    out[2 * stride] = A;
    out[3 * stride] = B;
    out[4 * stride] = C;
}

// Static high-resolution image: channels U, UU, UI, UG (NaN where a pixel of the patch is not
// above the threshold) and the image's statistics st[k * stride]. false where w = 0.
struct ImageStats {
    double mi, mg, A, B, C;
};
__device__ __forceinline__ ImageStats load_image_stats(const double* st, long long stride) {
    return {st[0], st[stride], st[2 * stride], st[3 * stride], st[4 * stride]};
}
__device__ __forceinline__ bool combine_static_image(const double* S, const ImageStats& t, int N,
                                                     double& w_out, double& m_out) {
    const double inv_n = 1.0 / (double)N, inv_n1 = 1.0 / (double)(N - 1);
    const double su = S[0], my = su * inv_n;
    const double cyy = fma(-my, su, S[1]);
    const bool ok = cyy * inv_n1 > kZeroThreshold;
    // a column left out of the fit may hold infinities (|Sobel| past single precision's range),
    // which its zero coefficient would turn into NaN
    const double p = t.A == 0.0 ? 0.0 : fma(-t.mi, su, S[2]), q = t.C == 0.0 ? 0.0 : fma(-t.mg, su, S[3]);
    const double e = fma(fma(t.B, q, t.A * p), p, (t.C * q) * q);
    weight_measure(ok ? cyy : 1.0, e, inv_n1, w_out, m_out);
    return ok;
}

// Patch statistics of a static ultrasound from its channels U, UU: mean and centred energy, or
// 0 and -1 where w = 0.
__device__ __forceinline__ void store_us_stats(const double* S, int N, double* mean, double* cyy) {
    const double inv_n = 1.0 / (double)N, m = S[0] * inv_n, c = fma(-m, S[0], S[1]);
    const bool ok = c * (1.0 / (double)(N - 1)) > kZeroThreshold;
    *mean = ok ? m : 0.0;
    *cyy = ok ? c : -1.0;
}

// Channels of a role and the products of one position added to their sums.
// kRoleMovingImage: I, G, II, GG, IG, UI, UG; kRoleStaticImage: U, UU, UI, UG, followed in
// kRoleStaticImageFull by I, G, II, GG, IG; kRoleImageStats: those five; kRoleUsStats: U, UU.
template <int ROLE>
struct Role {
    static constexpr int NC = ROLE == kRoleMovingImage ? 7 : ROLE == kRoleStaticImage ? 4
                            : ROLE == kRoleStaticImageFull ? 9 : ROLE == kRoleImageStats ? 5 : 2;
    static constexpr bool HAS_I = ROLE != kRoleUsStats, HAS_U = ROLE != kRoleImageStats;
    static constexpr bool SUMS = ROLE == kRoleMovingImage || ROLE == kRoleStaticImage || ROLE == kRoleStaticImageFull;
    __device__ __forceinline__ static void add(double (&t)[NC], double I, double G, double U) {
        constexpr bool STAT = ROLE == kRoleStaticImage || ROLE == kRoleStaticImageFull;
        constexpr int c = ROLE == kRoleStaticImageFull ? 4 : 0;
        if constexpr (STAT || ROLE == kRoleUsStats) {
            t[0] += U;
            t[1] = fma(U, U, t[1]);  // products of two floats are exact in FP64
            if constexpr (STAT) {
                t[2] = fma(U, I, t[2]);
                t[3] = fma(U, G, t[3]);
            }
        }
        if constexpr (HAS_I && ROLE != kRoleStaticImage) {
            t[c] += I;
            t[c + 1] += G;
            t[c + 2] = fma(I, I, t[c + 2]);
            t[c + 3] = fma(G, G, t[c + 3]);
            t[c + 4] = fma(I, G, t[c + 4]);
        }
        if constexpr (ROLE == kRoleMovingImage) {
            t[5] = fma(U, I, t[5]);
            t[6] = fma(U, G, t[6]);
        }
    }
};

// A uniform base plus a 32-bit byte offset per lane (one saddr + voffset access). The empty
// asm keeps the sum out of the loop optimiser's sight: it would carry a 64-bit pointer per
// lane for every unrolled step.
__device__ __forceinline__ const char* at_bytes(const void* base, unsigned ofs) {
    asm volatile("" : "+v"(ofs));
    return static_cast<const char*>(base) + ofs;
}
template <typename V>
__device__ __forceinline__ V load_at(const V* base, unsigned ofs) {
    V v;
    __builtin_memcpy(&v, at_bytes(base, ofs), sizeof(V));
    return v;
}

// Matrix i of the launch: from memory, or from the kernel's arguments, which spares small
// launches a round trip to the host's memory.
__device__ __forceinline__ void load_matrix(const FusedArgs& a, size_t i, float (&m)[12]) {
    if (a.inline_mat) {
#pragma unroll
        for (int k = 0; k < 12; ++k) m[k] = a.m0[i * 12 + k];
    } else {
        const float* mp = a.mats + i * 12;
#pragma unroll
        for (int k = 0; k < 12; ++k) m[k] = mp[k];
    }
}

// Work-group -> (tile, pose) on a 1D grid of roundup(tiles, 8) x npose work-groups.
// Work-groups go to the 8 XCDs round-robin by linear id; this mapping keeps all poses of
// one tile on the same XCD and adjacent in time (32 poses fill that XCD's 32 CUs), so the
// tile's static data (ultrasound statistics, fixed image) and the overlapping source
// footprint are fetched into that XCD's L2 once and shared by every pose. Returns false
// for the padding work-groups (tile >= tiles), which exit at once.
__device__ __forceinline__ bool map_block(int tiles, int npose, int& tile, int& pose) {
    const int w = blockIdx.x;
    const int xcd = w % kXcds, slot = w / kXcds;
    pose = slot % npose;
    tile = (slot / npose) * kXcds + xcd;
    return tile < tiles;
}

// Raises the dynamic LDS limit of a kernel, once per device: the attribute belongs to the function
// on the current device.
struct LdsLimit {
    std::atomic<unsigned long long> done{0};  // bit d: device d
    hipError_t raise(std::initializer_list<const void*> kernels, size_t bytes) {
        int d = 0;
        hipError_t err = hipGetDevice(&d);
        const unsigned long long bit = 1ULL << (d & 63);
        if (err != hipSuccess || (done.load() & bit)) return err;
        for (const void* k : kernels)
            if ((err = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes)) != hipSuccess)
                return err;
        done |= bit;
        return hipSuccess;
    }
};

template <int NTHR>
__device__ __forceinline__ void block_reduce_store(double am, double aw, double* s_red,
                                                   double* dst) {
    for (int off = 32; off > 0; off >>= 1) {
        am += __shfl_down(am, off, 64);
        aw += __shfl_down(aw, off, 64);
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        s_red[2 * wid] = am;
        s_red[2 * wid + 1] = aw;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = 0.0, w = 0.0;
        for (int i = 0; i < NTHR / 64; ++i) {
            m += s_red[2 * i];
            w += s_red[2 * i + 1];
        }
        dst[0] = m;
        dst[1] = w;
    }
}

// Sums am and aw over the 64 lanes of a wave; lane 0 writes them to dst[0], dst[1].
__device__ __forceinline__ void wave_reduce_store(double am, double aw, double* dst) {
    for (int off = 32; off > 0; off >>= 1) {
        am += __shfl_down(am, off, 64);
        aw += __shfl_down(aw, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        dst[0] = am;
        dst[1] = aw;
    }
}

// LDS row strides of the products planes and of the x-pass output: 2 (mod 4) doubles.
// The x pass reads and writes each lane's row two doubles at a time (ds_read_b128 /
// ds_write2_b64), 8 lanes per LDS cycle; with a stride of 4k + 2 doubles the 8 lanes that
// walk down consecutive rows cover 8 distinct groups of 4 banks. (Odd strides suit
// single-double accesses and left 33% more conflict cycles here.)
__host__ __device__ constexpr int lds_stride(int n) { return n + ((6 - n % 4) % 4); }
// Products of one position into the channel planes of the LDS buffer (plane size np,
// position i). NC = 9 (+count): I, G, U, II, GG, IG, UU, UI, UG.
// NC = 7: I, G, II, GG, IG, UI, UG.
template <int NC>
__device__ __forceinline__ void store_products(double* s_prod, int* s_cnt, int np, int i, float I,
                                               float G, float U) {
    const double di = I, dg = G, du = U;
    if (NC == 9) {
        s_prod[0 * np + i] = di;
        s_prod[1 * np + i] = dg;
        s_prod[2 * np + i] = du;
        s_prod[3 * np + i] = di * di;
        s_prod[4 * np + i] = dg * dg;
        s_prod[5 * np + i] = di * dg;
        s_prod[6 * np + i] = du * du;
        s_prod[7 * np + i] = du * di;
        s_prod[8 * np + i] = du * dg;
        s_cnt[i] = (du > kZeroThreshold) ? 1 : 0;
    } else {
        s_prod[0 * np + i] = di;
        s_prod[1 * np + i] = dg;
        s_prod[2 * np + i] = di * di;
        s_prod[3 * np + i] = dg * dg;
        s_prod[4 * np + i] = di * dg;
        s_prod[5 * np + i] = du * di;
        s_prod[6 * np + i] = du * dg;
    }
}

// Window sums of width W over a run of NO outputs: out[o] = in[o] + ... + in[o + W - 1],
// o = 0..NO-1, inputs in[0 .. NO + W - 2] (elements `stride` apart). van Herk / Gil-Werman
// form: the run is cut into blocks of W inputs and a window is the suffix of its block
// plus the prefix of the next one, so a partial sum never holds a value from outside the
// window. (A sliding sum that adds the entering and subtracts the leaving value keeps the
// rounding residue of every large value that passed through it, which swamps windows of
// small variance further along the run.) Each input is read once.
template <int W, typename V, int NO = 16>
__device__ __forceinline__ void window_run(const V* in, int stride, V* out, int ostride) {
    constexpr int NB = (NO + W - 1) / W;  // blocks that hold outputs
    constexpr int NIN = NO - 1 + W;       // inputs of the run
    V raw[W];
#pragma unroll
    for (int j = 0; j < W; ++j) raw[j] = in[j * stride];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        V suf[W];  // suffix sums of block b
        suf[W - 1] = raw[W - 1];
#pragma unroll
        for (int j = W - 2; j >= 0; --j) suf[j] = raw[j] + suf[j + 1];
        V pre = 0;  // prefix of block b + 1: elements 0 .. j - 1 at output b * W + j
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const int o = b * W + j;
            if (o < NO) out[o * ostride] = j == 0 ? suf[0] : suf[j] + pre;
            const int t = (b + 1) * W + j;
            if (t < NIN) {
                raw[j] = in[t * stride];
                pre = j == 0 ? raw[j] : pre + raw[j];
            }
        }
    }
}

}  // namespace

}  // namespace lc2e
