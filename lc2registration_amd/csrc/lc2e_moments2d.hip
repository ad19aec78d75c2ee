// 2D LC2 (single images and frame stacks) without tile halos along x: k_moments2d forms the patch
// moments of strips of columns and combines them. It warps the moving image in place, or, where
// that is the high-resolution one and the launch is large, reads it and its |Sobel| from the
// grid, written by k_warp2.
#include "lc2e_device.hpp"

namespace lc2e {

namespace {

constexpr int kWarpX = 32, kWarpY = 16;  // output tile of k_warp2

template <bool P2, bool SRC3D, typename T, typename Pend>
__device__ __forceinline__ void issue_any(const T* src, const SGeom& s, const float* m, float lx, float ly,
                                          float lz, bool inside, Pend& p) {
    if constexpr (SRC3D) issue3<P2>(src, s, m, lx, ly, lz, inside, p);
    else issue2<P2>(src, s, m, lx, ly, inside, p);
}
template <bool SRC3D, typename Pend>
__device__ __forceinline__ float finish_any(const Pend& p) {
    if constexpr (SRC3D) return finish3(p);
    else return finish2(p);
}

// The warped image and its in-plane |Sobel| per pixel, frame and pose as float2, bit for bit as
// k_fused2d forms them: a 32x16 tile over a run of frames, the next frame's gathers in flight
// during this one's Sobel. Bound by VALU issue (98 instructions per pixel, 70% of the slots):
// 480 us for 5 poses of 128 frames 512x384.
template <bool SRC3D, typename T, bool P2>
__global__ __launch_bounds__(256) void k_warp2(FusedArgs a, int ntx, int nty, int frun, int tiles, int npose) {
    constexpr int IXE = kWarpX + 2, IYE = kWarpY + 2, NI = IXE * IYE;
    constexpr int SPT = (NI + 255) / 256;
    __shared__ float s_in[2][NI];
    int tile, pose;
    if (!map_block(tiles, npose, tile, pose)) return;
    const int tid = threadIdx.x;
    const int tcol = tile % (ntx * nty), run = tile / (ntx * nty);
    const int x0 = (tcol % ntx) * kWarpX, y0 = (tcol / ntx) * kWarpY;
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z;
    const int f0 = run * frun, f1 = min(f0 + frun, Z);
    const T* __restrict__ src = static_cast<const T*>(a.src);
    const int wbase = __builtin_amdgcn_readfirstlane(tid & ~63);
    auto has = [&](int j) { return (j + 1) * 256 <= NI || j * 256 + wbase < NI; };
    float gLx[SPT], gLy[SPT];
    unsigned in_xy = 0;
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
        const int i = tid + j * 256;
        const int gx = x0 - 1 + i % IXE, gy = y0 - 1 + i / IXE;
        if (i < NI && gx >= 0 && gx < X && gy >= 0 && gy < Y) in_xy |= 1u << j;
        gLx[j] = fmaf((float)gx, a.v.sx, a.v.ox);
        gLy[j] = fmaf((float)gy, a.v.sy, a.v.oy);
    }
    using Pend = typename std::conditional<SRC3D, Pending3<T>, Pending2<T>>::type;
    Pend pend[SPT];
    auto issue = [&](int f) {
        float m[12];
        load_matrix(a, (size_t)pose * a.mats_per_pose + (a.mats_per_pose > 1 ? f : 0), m);
#pragma unroll
        for (int j = 0; j < SPT; ++j)
            if (has(j)) issue_any<P2, SRC3D>(src, a.s, m, gLx[j], gLy[j], a.v.oz, (in_xy >> j) & 1u, pend[j]);
    };
    issue(f0);
    const int lx = tid % kWarpX, ly = 2 * (tid / kWarpX);
    const int gx = x0 + lx, gy = y0 + ly;
    const bool ok0 = gx < X && gy < Y, ok1 = gx < X && gy + 1 < Y;
    for (int f = f0, buf = 0; f < f1; ++f, buf ^= 1) {
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            if (!has(j)) continue;
            const int i = tid + j * 256;
            const float v = finish_any<SRC3D>(pend[j]);
            if (i < NI) s_in[buf][i] = v;
        }
        __syncthreads();
        if (f + 1 < f1) issue(f + 1);
        const float* row = s_in[buf] + ly * IXE + lx;
        float sm[4], df[4], cm[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float l = row[r * IXE], c = row[r * IXE + 1], rr = row[r * IXE + 2];
            sm[r] = fmaf(2.0f, c, l) + rr;  // (l + 2c) + r: 2c is exact
            df[r] = rr - l;
            cm[r] = c;
        }
        float2* out = a.warp2 + ((size_t)pose * Z + f) * X * Y + (size_t)gy * X + gx;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float gxv = fmaf(2.0f, df[e + 1], df[e]) + df[e + 2];
            const float gyv = sm[e + 2] - sm[e];
            const float G = sqrtf(fmaf(gyv, gyv, gxv * gxv));
            if (e ? ok1 : ok0) out[e * X] = make_float2(cm[e + 1], G);
        }
    }
}

// ---------------------------------------------------------------------------
// Patch moments and combine. A wave owns 64 columns (64 - 2R outputs per row; 62 - 2R with the
// Sobel in place) and 8 output rows: each lane forms the y window sums of its column for the 8
// rows in registers, then per channel the x window sums through 5 KB of LDS that no other wave uses
// (wave fences, no barrier), and combines the 8 pixels of its column. Four waves of a work-group take
// four groups of rows and share one partial sum per run of frames. Warping in place takes barriers
// around the shared rows: per frame one before and one after the warp, and one after the Sobel.
// OUT = 4 (below) has eight waves of four rows. A tile has no halo along y but the rows' own (2R + 8 for 8) and
// a short one along x, where 16x16 tiles form the products of (16 + 2R)^2 positions for 256
// outputs: 4.5 times each at R = 9.
// With a static high-resolution image its sums do not depend on the pose (kRoleImageStats, at
// pair creation): 4 channels instead of 9 and a count. Two to three waves per SIMD (130 to 230
// VGPRs); bound by the latency of the three LDS trips per channel and of the FP64 chains (VALU a
// quarter busy). Measured, static image: 256x256, R = 3, 64 poses 104 -> 38 us; 261x261, R = 9,
// 13 poses 100 -> 20 us; moving image: 336x205 slice in a CT, R = 9, 13 poses 60 -> 25 us after
// 11 us of k_warp2. In place the waves share the warped rows (32 + 2R for 32, where each warped
// 8 + 2R of its own): per call 256x256, R = 3, 64 poses 62 -> 55 us, one pose 27.7 -> 26.9 (OUT = 4:
// 25.2); R = 9, 13 poses 45 -> 40 (OUT = 4: 36.5).
// ---------------------------------------------------------------------------
// LDS column x of a wave's row: 2 doubles of padding after every 8, and rows 80 doubles apart,
// spread the 16-byte reads of the x pass (8 runs of 8 columns, 8 rows) over all banks.
__device__ __forceinline__ constexpr int lds_col(int x) { return x + 2 * (x / 8); }
constexpr int kRowS = 80, kWaveS = 8 * kRowS + 32;  // one wave's LDS in doubles

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Output columns of a wave: with the moving image as the high-resolution one the outermost
// lanes only feed the Sobel of the variant that warps in place.
constexpr int strip2(int r, int role) { return (role == kRoleMovingImage ? 62 : 64) - 2 * r; }

// Rows of the warped image a work-group keeps in LDS when it warps in place, 64 floats each: its 32
// output rows' with their halo, each warped once for the four waves.
template <int R, int ROLE>
struct InPlace {
    static constexpr int H = ROLE == kRoleMovingImage ? 1 : 0;  // halo of the Sobel
    static constexpr int ROWS = 32 + 2 * R + 2 * H, FLOATS = ROWS * 64 * (1 + H);
};

// The moving image at column gx (this lane's) of rows gy0 .. gy0 + rows - 1 of frame's matrix m,
// 0 outside the grid, into dst (rows 64 floats apart): this wave's share of the work-group's NW
// waves', every NWth group of four rows, whose gathers are in flight at once.
template <int NW, bool P2, bool SRC3D, typename T>
__device__ __forceinline__ void warp_rows(const FusedArgs& a, const float* m, int gx, int gy0, int rows,
                                          float* dst, int wave) {
    const T* __restrict__ src = static_cast<const T*>(a.src);
    using Pend = typename std::conditional<SRC3D, Pending3<T>, Pending2<T>>::type;
    const float lx = fmaf((float)gx, a.v.sx, a.v.ox);
    const bool inx = gx >= 0 && gx < a.v.X;
    for (int j0 = 4 * wave; j0 < rows; j0 += 4 * NW) {
        Pend p[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int gy = gy0 + j0 + k;
            issue_any<P2, SRC3D>(src, a.s, m, lx, fmaf((float)gy, a.v.sy, a.v.oy), a.v.oz,
                                 inx && gy >= 0 && gy < a.v.Y, p[k]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float v = finish_any<SRC3D>(p[k]);
            if (j0 + k < rows) dst[(j0 + k) * 64] = v;
        }
    }
}
template <int NW>
__device__ __forceinline__ void warp_rows_any(const FusedArgs& a, int src3, const float* m, int gx, int gy0,
                                              int rows, float* dst, int wave) {
    const int form = (src3 ? 4 : 0) + (a.s.pow2 ? 2 : 0) + (a.src_f16 ? 1 : 0);  // uniform
    switch (form) {
        case 7: return warp_rows<NW, true, true, __half>(a, m, gx, gy0, rows, dst, wave);
        case 6: return warp_rows<NW, true, true, float>(a, m, gx, gy0, rows, dst, wave);
        case 5: return warp_rows<NW, false, true, __half>(a, m, gx, gy0, rows, dst, wave);
        case 4: return warp_rows<NW, false, true, float>(a, m, gx, gy0, rows, dst, wave);
        case 3: return warp_rows<NW, true, false, __half>(a, m, gx, gy0, rows, dst, wave);
        case 2: return warp_rows<NW, true, false, float>(a, m, gx, gy0, rows, dst, wave);
        case 1: return warp_rows<NW, false, false, __half>(a, m, gx, gy0, rows, dst, wave);
        default: return warp_rows<NW, false, false, float>(a, m, gx, gy0, rows, dst, wave);
    }
}

// OUT = 8: as above. OUT = 4, for launches that leave the chip idle: two waves share a block of eight
// rows and take four outputs each, summed over the same suffixes and prefixes, so every pixel's
// sums keep their bits; the x pass takes two channels at a time (all lanes busy, half the trips), and
// a wave's chain is about half as long. Measures and weights are added up per lane over the four
// rows of each half block, the two halves, the lanes, and then the blocks, in either form.
template <int R, int ROLE, bool INPLACE, int OUT>
__global__ __launch_bounds__(64 * 32 / OUT) __attribute__((amdgpu_waves_per_eu(
    ROLE == kRoleStaticImage || ROLE == kRoleUsStats ? 3 : 2)))
void k_moments2d(FusedArgs a) {
    using Ro = Role<ROLE>;
    using IP = InPlace<R, ROLE>;
    constexpr int NC = Ro::NC, W = 2 * R + 1, TX = strip2(R, ROLE), N = W * W;
    constexpr int H = INPLACE ? IP::H : 0;  // lane of the first column
    constexpr int NW = 32 / OUT, CP = 8 / OUT;  // waves; channels per trip of the x pass
    __shared__ __align__(16) double s_all[NW * kWaveS];
    __shared__ double s_red[8];
    extern __shared__ float s_rows[];  // INPLACE: IP::FLOATS

    int tile, pose;
    if constexpr (OUT == 4) {
        // A part of a small launch's time is its reads of the arguments, which lie in the host's
        // memory: one request for every line of them, where the compiler would read and wait seven
        // times (1.9 -> 1.4 us), and a pose that does not depend on them.
        asm volatile("" ::"s"(a.v.X), "s"(a.s.oz), "s"(a.src), "s"(a.stat_img), "s"(a.stat_grad), "s"(a.mats),
                     "s"(a.inline_mat), "s"(a.ntx), "s"(a.tiles), "s"(a.istat), "s"(a.src3));
        tile = blockIdx.x;
        pose = blockIdx.y;
        if (tile >= a.tiles) return;
    } else {
        if (!map_block(a.tiles, a.npose, tile, pose)) return;  // whole work-group
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int cols = a.ntx * a.nty;
    const int tcol = tile % cols, run = tile / cols;
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z, XY = X * Y;
    const int x0 = R + (tcol % a.ntx) * TX, y0 = R + (tcol / a.ntx) * 32 + wave * OUT;
    const int col = lane - H;  // column of the strip
    const bool has_rows = y0 < Y - R;  // the wave has output rows
    const int f0 = run * a.zchunk, f1 = INPLACE || has_rows ? min(f0 + a.zchunk, Z) : f0;
    double acc_m[OUT / 4] = {}, acc_w[OUT / 4] = {};

    {
        double* const s = s_all + wave * kWaveS;
        // this lane's column; rows and columns past the grid repeat its edge and only reach
        // outputs that are not valid
        const unsigned gx4 = (unsigned)min(max(x0 - R + col, 0), X - 1) * 4u;
        const int ox = x0 + col;
        const bool okx = col >= 0 && col < TX && ox < X - R;
        const int s_col = lds_col(min(max(col, 0), 63));
        const bool has_col = col >= 0;
        float* const rows = s_rows + (INPLACE ? wave * OUT * 64 + lane : 0);
        const int run_x = lane % 8, run_y = lane / 8;
        double* const xp = s + run_y * kRowS + run_x * 10;
        for (int f = f0; f < f1; ++f) {
            const size_t plane = (size_t)f * XY, pz = (size_t)pose * Z * XY + plane;
            if constexpr (INPLACE) {
                float m[12];
                load_matrix(a, (size_t)pose * a.mats_per_pose + (a.mats_per_pose > 1 ? f : 0), m);
                const int top = y0 - wave * OUT - R - H;  // grid row of the first one
                const int nrows = min(IP::ROWS, Y + H - top);  // none past the grid's but the Sobel's
                if (f > f0) __syncthreads();  // the last frame's are read
                warp_rows_any<NW>(a, a.src3, m, x0 - R + col, top, nrows, s_rows + lane, wave);
                __syncthreads();
                if constexpr (ROLE == kRoleMovingImage) {
                    // |Sobel| of the rows between, a part per wave; the outermost lanes' is not used
                    constexpr int Q = (IP::ROWS - 2 + NW - 1) / NW;
                    const float* const in = s_rows + lane;
                    float* const g = s_rows + IP::ROWS * 64 + lane;
                    const int left = lane > 0 ? -1 : 0, right = lane < 63 ? 1 : 0;
                    const int j0 = wave * Q, j1 = min(j0 + Q + 2, nrows);
                    float sm[3], df[3];
                    auto line = [&](int j, int k) {
                        const float l = in[j * 64 + left], c = in[j * 64], r = in[j * 64 + right];
                        sm[k] = fmaf(2.0f, c, l) + r;
                        df[k] = r - l;
                    };
                    auto store = [&](int j, int k) {  // of lines k, k + 1, k + 2
                        const float gxv = fmaf(2.0f, df[k + 1], df[k]) + df[k + 2], gyv = sm[k + 2] - sm[k];
                        g[(j + 1) * 64] = sqrtf(fmaf(gyv, gyv, gxv * gxv));
                    };
                    if (j0 + 2 < j1) {
                        line(j0, 0);
                        line(j0 + 1, 1);
                    }
                    for (int j = j0 + 2; j < j1; ++j) {
                        line(j, 2);
                        store(j - 2, 0);
                        sm[0] = sm[1], sm[1] = sm[2], df[0] = df[1], df[1] = df[2];
                    }
                    __syncthreads();
                }
                if (!has_rows) continue;
            }
            // row y0 - R + j at this lane's column
            auto input = [&](int j, double& I, double& G, double& U) {
                const size_t row = (size_t)min(y0 - R + j, Y - 1) * X;  // wave-uniform
                I = G = U = 0.0;
                if constexpr (INPLACE && ROLE == kRoleMovingImage) {
                    I = rows[(j + 1) * 64];
                    G = rows[(IP::ROWS + j + 1) * 64];
                    U = load_at(a.stat_img + plane + row, gx4);
                } else if constexpr (ROLE == kRoleMovingImage) {
                    const float2 v = load_at(a.warp2 + pz + row, gx4 * 2u);
                    I = v.x;
                    G = v.y;
                    U = load_at(a.stat_img + plane + row, gx4);
                } else {
                    if constexpr (Ro::HAS_I) {
                        I = load_at(a.stat_img + plane + row, gx4);
                        G = load_at(a.stat_grad + plane + row, gx4);
                    }
                    if constexpr (INPLACE) {
                        const float u = rows[j * 64];
                        U = (double)u > kZeroThreshold ? u : NAN;
                    }
                    if constexpr (ROLE == kRoleUsStats) {
                        const float u = load_at(a.stat_img + plane + row, gx4);
                        U = (double)u > kZeroThreshold ? u : NAN;
                    }
                }
            };
            // 1. y window sums of the wave's rows. Of a block of eight: the rows all eight windows
            // share, the suffixes before them and the prefixes after them (A: the wave's first row
            // of its block)
            double S[OUT][NC];
            if constexpr (W >= 7 && OUT == 8 && (ROLE != kRoleMovingImage || (!INPLACE && R == 6))) {
                // (As the lambda below, with A = 0, these take 2 to 11% longer, and the others 2 to 18%
                // less: the compiler orders the loads differently. 512x400, moving image, 32 poses,
                // in line and lambda: R = 6 99 and 110 us, R = 7 114 and 110, R = 9 141 and 116.)
                double t[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) t[c] = 0.0;
#pragma unroll
                for (int j = 6; j >= 0; --j) {
                    double I, G, U;
                    input(j, I, G, U);
                    Ro::add(t, I, G, U);
#pragma unroll
                    for (int c = 0; c < NC; ++c) S[j][c] = t[c];
                }
                __builtin_amdgcn_sched_barrier(0);  // bounds the loads in flight
#pragma unroll
                for (int c = 0; c < NC; ++c) t[c] = 0.0;
#pragma unroll
                for (int j = 7; j < W; ++j) {
                    double I, G, U;
                    input(j, I, G, U);
                    Ro::add(t, I, G, U);
                    if (j % 8 == 7) __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (W > 7)
#pragma unroll
                    for (int o = 0; o < 7; ++o)
#pragma unroll
                        for (int c = 0; c < NC; ++c) S[o][c] += t[c];
#pragma unroll
                for (int c = 0; c < NC; ++c) S[OUT - 1][c] = t[c], t[c] = 0.0;
#pragma unroll
                for (int o = 1; o < 8; ++o) {
                    double I, G, U;
                    input(W - 1 + o, I, G, U);
                    Ro::add(t, I, G, U);
#pragma unroll
                    for (int c = 0; c < NC; ++c) S[o][c] += t[c];
                }
            } else if constexpr (W >= 7) {
                auto y_sums = [&](auto first) {
                    constexpr int A = decltype(first)::value, B = A + OUT;
                    double t[NC];
#pragma unroll
                    for (int c = 0; c < NC; ++c) t[c] = 0.0;
#pragma unroll
                    for (int j = 6; j >= A; --j) {
                        double I, G, U;
                        input(j - A, I, G, U);
                        Ro::add(t, I, G, U);
                        if (j < B)
#pragma unroll
                            for (int c = 0; c < NC; ++c) S[j - A][c] = t[c];
                    }
                    __builtin_amdgcn_sched_barrier(0);  // bounds the loads in flight
#pragma unroll
                    for (int c = 0; c < NC; ++c) t[c] = 0.0;
#pragma unroll
                    for (int j = 7; j < W; ++j) {
                        double I, G, U;
                        input(j - A, I, G, U);
                        Ro::add(t, I, G, U);
                        if (j % 8 == 7) __builtin_amdgcn_sched_barrier(0);
                    }
                    if constexpr (W > 7)
#pragma unroll
                        for (int o = A; o < B && o < 7; ++o)
#pragma unroll
                            for (int c = 0; c < NC; ++c) S[o - A][c] += t[c];
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        if (B == 8) S[OUT - 1][c] = t[c];
                        t[c] = 0.0;
                    }
#pragma unroll
                    for (int o = 1; o < B; ++o) {
                        double I, G, U;
                        input(W - 1 + o - A, I, G, U);
                        Ro::add(t, I, G, U);
                        if (o >= A)
#pragma unroll
                            for (int c = 0; c < NC; ++c) S[o - A][c] += t[c];
                    }
                };
                if (OUT == 8 || wave % 2 == 0) y_sums(std::integral_constant<int, 0>{});
                else if constexpr (OUT == 4) y_sums(std::integral_constant<int, 4>{});
            } else {
#pragma unroll
                for (int o = 0; o < OUT; ++o)
#pragma unroll
                    for (int c = 0; c < NC; ++c) S[o][c] = 0.0;
#pragma unroll
                for (int j = 0; j < W + OUT - 1; ++j) {
                    double I, G, U;
                    input(j, I, G, U);
#pragma unroll
                    for (int o = 0; o < OUT; ++o)
                        if (j >= o && j < o + W) Ro::add(S[o], I, G, U);
                }
            }
            // 2. x window sums, CP channels at a time (the pins and scheduling barriers keep the
            // compiler from running phases into each other, which costs a wave per SIMD)
            auto pin = [&]() {
#pragma unroll
                for (int o = 0; o < OUT; ++o)
#pragma unroll
                    for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(S[o][c]));
                __builtin_amdgcn_sched_barrier(0);
            };
            pin();
            // the pixels' statistics, requested before the last channels' LDS work
            const unsigned vx = (unsigned)(okx ? ox : R) * 8u;
            double mu[OUT], cyy[OUT];
            ImageStats ist[OUT];
            auto stats = [&](int o0, int o1) {
#pragma unroll
                for (int o = o0; o < o1; ++o) {
                    const size_t row = plane + (size_t)min(y0 + o, Y - R - 1) * X;
                    if constexpr (ROLE == kRoleMovingImage) {
                        mu[o] = load_at(a.ustat_mean + row, vx);
                        cyy[o] = load_at(a.ustat_cyy + row, vx);
                    }
                    if constexpr (ROLE == kRoleStaticImage) {
                        const double* st = a.istat + row;
                        ist[o] = {load_at(st, vx), load_at(st + a.istat_stride, vx),
                                  load_at(st + 2 * a.istat_stride, vx), load_at(st + 3 * a.istat_stride, vx),
                                  load_at(st + 4 * a.istat_stride, vx)};
                    }
                }
            };
            constexpr bool EARLY = ROLE == kRoleMovingImage || (ROLE == kRoleStaticImage && OUT == 4);
#pragma unroll
            for (int c = 0; c < NC; c += CP) {
                if (EARLY && c + CP >= NC) stats(0, OUT);
#pragma unroll
                for (int k = 0; k < CP && c + k < NC; ++k)
#pragma unroll
                    for (int o = 0; o < OUT; ++o)
                        if (has_col) s[(k * OUT + o) * kRowS + s_col] = S[o][c + k];
                wave_fence();
                if (run_x * 8 < TX) {
                    double in[W + 8], out[8];
#pragma unroll
                    for (int j = 0; j < W + 7; j += 2) {  // 16 bytes at a time
                        const double* p = static_cast<const double*>(
                            __builtin_assume_aligned(xp + lds_col(j), 16));
                        in[j] = p[0];
                        in[j + 1] = p[1];
                    }
                    if constexpr (W >= 7) {
                        double t = in[6];
                        out[6] = t;
#pragma unroll
                        for (int j = 5; j >= 0; --j) t = in[j] + t, out[j] = t;
                        if constexpr (W > 7) {
                            t = in[7];
#pragma unroll
                            for (int j = 8; j < W; ++j) t += in[j];
#pragma unroll
                            for (int o = 0; o < 7; ++o) out[o] += t;
                            out[7] = t;
                        }
                        t = in[W];
                        out[1] += t;
#pragma unroll
                        for (int o = 2; o < 7; ++o) t += in[W - 1 + o], out[o] += t;
                        t += in[W + 6];
                        out[7] = W > 7 ? out[7] + t : t;
                    } else {
#pragma unroll
                        for (int o = 0; o < 8; ++o) {
                            out[o] = in[o];
#pragma unroll
                            for (int j = 1; j < W; ++j) out[o] += in[o + j];
                        }
                    }
                    // other lanes read what is overwritten now: no store before the last read
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    double* p = static_cast<double*>(__builtin_assume_aligned(xp, 16));
#pragma unroll
                    for (int o = 0; o < 8; ++o) p[o] = out[o];
                }
                wave_fence();
#pragma unroll
                for (int k = 0; k < CP && c + k < NC; ++k)
#pragma unroll
                    for (int o = 0; o < OUT; ++o) {
                        S[o][c + k] = s[(k * OUT + o) * kRowS + s_col];
                        asm volatile("" : "+v"(S[o][c + k]));
                    }
                wave_fence();
                __builtin_amdgcn_sched_barrier(0);
            }
            pin();
            // 3. combine
#pragma unroll
            for (int o = 0; o < OUT; ++o) {
                const int oy = y0 + o;
                if (o % 2 == 0) __builtin_amdgcn_sched_barrier(0);
                const bool ok_row = oy < Y - R;  // wave-uniform
                const size_t vz = plane + (size_t)min(oy, Y - R - 1) * X + (okx ? ox : R);
                double w = 0.0, meas = 0.0;
                bool ok = okx && ok_row;
                if (ROLE == kRoleStaticImage && !EARLY && o % 2 == 0) stats(o, o + 2);
                if constexpr (ROLE == kRoleMovingImage) {
                    ok = ok && cyy[o] >= 0.0;
                    combine_static_u_any(S[o], mu[o], ok ? cyy[o] : 1.0, N, w, meas);
                } else if constexpr (ROLE == kRoleStaticImage) {
                    ok = combine_static_image(S[o], ist[o], N, w, meas) && ok;
                } else if constexpr (ROLE == kRoleStaticImageFull) {
                    double t[kImageStats];
                    store_image_stats(S[o] + 4, N, t, 1);
                    ok = combine_static_image(S[o], load_image_stats(t, 1), N, w, meas) && ok;
                } else if constexpr (ROLE == kRoleImageStats) {
                    if (ok) store_image_stats(S[o], N, a.istat_out + vz, a.istat_stride);
                } else {
                    if (ok) store_us_stats(S[o], N, a.ustat_mean_out + vz, a.ustat_cyy_out + vz);
                }
                if constexpr (Ro::SUMS) {
                    acc_m[o / 4] += ok ? meas : 0.0;
                    acc_w[o / 4] += ok ? w : 0.0;
                    if (a.wmap && ok) {
                        a.wmap[vz] = w;
                        a.mmap[vz] = meas;
                    }
                }
            }
        }
    }
    if constexpr (Ro::SUMS) {
        double am = acc_m[0], aw = acc_w[0];
        if constexpr (OUT == 4) {  // the odd wave's lanes join the even one's
            double* const mine = s_all + wave * kWaveS + 2 * lane;
            if (wave % 2) mine[0] = am, mine[1] = aw;
            __syncthreads();
            if (wave % 2 == 0) am += mine[kWaveS], aw += mine[kWaveS + 1];
        } else {
            am += acc_m[1];
            aw += acc_w[1];
        }
        if (OUT == 8 || wave % 2 == 0) wave_reduce_store(am, aw, s_red + 2 * (wave / (8 / OUT)));
        __syncthreads();
        if (threadIdx.x == 0) {
            double m = 0.0, w = 0.0;
            for (int k = 0; k < 4; ++k) m += s_red[2 * k], w += s_red[2 * k + 1];
            double* dst = a.partials + ((size_t)pose * a.blocks_per_pose + tile) * 2;
            dst[0] = m;
            dst[1] = w;
        }
    }
}

template <bool SRC3D, typename T, bool P2>
void warp2(const FusedArgs& a, int n, hipStream_t st) {
    const int ntx = (a.v.X + kWarpX - 1) / kWarpX, nty = (a.v.Y + kWarpY - 1) / kWarpY;
    // runs of frames: about 4096 work-groups, at most 16 frames each (the next frame's gathers
    // are in flight during this one's work, from two frames on)
    const long long per = (long long)ntx * nty * n;
    const int frun = (int)std::max(1LL, std::min(16LL, per * a.v.Z / 4096));
    const int tiles = ntx * nty * ((a.v.Z + frun - 1) / frun);
    const int tiles8 = (tiles + kXcds - 1) / kXcds * kXcds;
    hipLaunchKernelGGL((k_warp2<SRC3D, T, P2>), dim3((unsigned)((long long)tiles8 * n)), dim3(256), 0, st,
                       a, ntx, nty, frun, tiles, n);
}
template <bool SRC3D>
void warp2t(const FusedArgs& a, int n, hipStream_t st) {
    if (a.s.pow2) {
        if (a.src_f16) warp2<SRC3D, __half, true>(a, n, st);
        else warp2<SRC3D, float, true>(a, n, st);
    } else {
        if (a.src_f16) warp2<SRC3D, __half, false>(a, n, st);
        else warp2<SRC3D, float, false>(a, n, st);
    }
}

template <int R, int ROLE, bool INPLACE, int OUT>
hipError_t moments2k(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    const size_t lds = INPLACE ? InPlace<R, ROLE>::FLOATS * sizeof(float) : 0;
    constexpr int NT = 64 * 32 / OUT;
    if constexpr (INPLACE) {
        static LdsLimit limit;
        const hipError_t err =
            limit.raise({reinterpret_cast<const void*>(&k_moments2d<R, ROLE, INPLACE, OUT>)}, lds);
        if (err != hipSuccess) return err;
    }
    if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, k_moments2d<R, ROLE, INPLACE, OUT>, NT, lds);
    hipLaunchKernelGGL((k_moments2d<R, ROLE, INPLACE, OUT>), grid, dim3(NT), lds, st, a);
    return hipGetLastError();
}
template <int ROLE, bool INPLACE, int OUT, int R = ROLE == kRoleMovingImage ? kMaxRFused2 + 1 : 1>
hipError_t moments2r(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    if (a.r == R) return moments2k<R, ROLE, INPLACE, OUT>(a, grid, st, occ);
    if constexpr (R < kMaxR2) return moments2r<ROLE, INPLACE, OUT, R + 1>(a, grid, st, occ);
    return hipErrorInvalidValue;
}
// In place: four rows per wave up to one work-group per CU. Kernel, 256x256, four rows and eight:
// moving, R = 4, 40 to 160 work-groups 12.2 and 16.2 us, 320 20.9 and 19.8; R = 9, 192 14.9 and 18.4,
// 384 25.0 and 22.2; static, R = 3, 40 10.2 and 12.8, 640 18.6 and 18.6; R = 9, 192 12.4 and 15.2,
// 384 20.5 and 17.7 (with events; radii up to 3 of a static image would gain up to 600).
constexpr long long kSplitGroups = 256;
template <int ROLE>
hipError_t moments2i(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    if (!occ && (long long)a.tiles * a.npose <= kSplitGroups) return moments2r<ROLE, true, 4>(a, dim3((unsigned)((a.tiles + kXcds - 1) / kXcds * kXcds), (unsigned)a.npose), st, occ);
    return moments2r<ROLE, true, 8>(a, grid, st, occ);
}

}  // namespace

hipError_t launch_warp2(const FusedArgs& a, int src_ndim, int n, hipStream_t st) {
    if (src_ndim == 3) warp2t<true>(a, n, st);
    else warp2t<false>(a, n, st);
    return hipGetLastError();
}

int strip_width_2d(int r, int role) { return strip2(r, role); }

hipError_t moments2(const FusedArgs& a, int role, int n, hipStream_t st, int* occ) {
    const long long tiles8 = (a.tiles + kXcds - 1) / kXcds * (long long)kXcds;
    if (tiles8 * n > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(tiles8 * n));
    switch (role) {
        case kRoleMovingImage:
            return a.in_place ? moments2i<kRoleMovingImage>(a, grid, st, occ)
                              : moments2r<kRoleMovingImage, false, 8>(a, grid, st, occ);
        case kRoleStaticImage: return moments2i<kRoleStaticImage>(a, grid, st, occ);
        case kRoleStaticImageFull: return moments2i<kRoleStaticImageFull>(a, grid, st, occ);
        case kRoleImageStats: return moments2r<kRoleImageStats, false, 8>(a, grid, st, occ);
        default: return moments2r<kRoleUsStats, false, 8>(a, grid, st, occ);
    }
}

}  // namespace lc2e
