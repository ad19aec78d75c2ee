// Device code of the LC2 engine for gfx950 (MI355X).
//
// One fused kernel per pose batch computes, for every patch centre of the
// virtual grid, the reference's LC2 measure and weight
// (cu_lc2_3d.cu:181-618 / cu_lc2_2d.cu:88-480) and reduces them per work-group:
//   warp of the moving image (interpolator.cu:69-232) -> |Sobel| (cu_lc2_3d.cu:100-179)
//   -> FP64 patch moments -> closed-form least-squares projection -> measure, w.
// The reference's per-voxel FP32 conjugate gradient (cu_lc2_3d.cu:289-524) is
// replaced by the projection it converges to, computed from centred moments:
//   var_res * (N-1) = C_yy - s^T C^+ s,  s = (C_yI, C_yG),  C = [[C_II, C_IG], [C_IG, C_GG]].
//
// Numerics: the FP32 stages (coordinates, trilinear/bilinear lerps, Sobel) are
// written with explicit fmaf and the file is compiled with -ffp-contract=off, so
// they reproduce the oracle bit for bit. Patch moments are FP64 (products of two
// FP32 values are exact in FP64), which removes the cancellation an FP32
// sliding-window sum would suffer on intensities with small local variance.
//
// Pairs are evaluated by k_moments3d / k_moments2d (their files say how), by k_fused2d (2D, moving
// high-resolution image, small patches), by k_fused3d (3D under an HBM budget: it needs no
// workspace) or by the separable path (the remaining radii).
//
// 3D structure (k_fused3d): a 256-thread work-group (two per CU) owns a 16x16 column
// of output voxels over `zchunk` planes and marches along z. Per input plane:
// warp the plane (+ Sobel halo) into LDS, separable Sobel of each 3x3 neighbourhood
// with a 3-plane register ring along z, FP64 products into LDS, x then y window sums in
// LDS (van Herk / Gil-Werman: no partial sum holds a value from outside its window), and
// a (2R+1)-slot register ring of plane sums and pair sums of planes gives the z window
// sum; complete patch sums are combined in FP64 and accumulated per thread. No
// intermediate volume touches HBM.
#include <algorithm>
#include <map>
#include <mutex>

#include "lc2e_device.hpp"

namespace lc2e {

namespace {

// Box sums of width W along x then y, for NC FP64 channels and (CNT) one integer count
// channel, over a region of py rows (row stride ps >= TX + W - 1) into TX x TY outputs:
//   s_prod[c][py][ps] -> s_xp[c][py][TX + 1] -> s_out[c][TY][TX]   (s_out may alias s_prod).
// Rows (x pass) are cut into runs of 16 outputs and columns (y pass) into runs of 8, one
// task each (runs of 8 put twice as many threads to work in the y pass); neighbouring
// lanes take neighbouring rows (x pass) or columns (y pass).
// PRIO_X / PRIO_Y: run the x / y pass at raised wave priority. With several work-groups
// per CU out of phase, the LDS passes gain from going first (2D +3.2%, 3D +1.3% with
// three barriers per z-step, measured). The 3D kernel's half-step overlap keeps only the
// y pass raised (x pass raised too: 0.5% slower, measured).
// x pass of box_xy: s_prod[c][py][ps] -> s_xp[c][py][XS] (TX outputs per row).
template <int NC, bool CNT, int TX, int NTHR, int W, int XS, bool PRIO = false>
__device__ __forceinline__ void box_x(const double* s_prod, const int* s_cnt, double* s_xp,
                                      int* s_xcnt, int ps, int py, int tid) {
    static_assert(TX % 16 == 0, "tile edges are multiples of 16");
    static_assert(XS > TX, "x-pass rows hold TX outputs");
    constexpr int NT = NC + (CNT ? 1 : 0);
    constexpr int SX = TX / 16;
    const int np = ps * py;
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(2);
    for (int t = tid; t < NT * py * SX; t += NTHR) {
        const int row = t % py, rest = t / py;
        const int seg = rest % SX, c = rest / SX;
        if (c < NC)
            window_run<W>(s_prod + c * np + row * ps + seg * 16, 1,
                        s_xp + (c * py + row) * XS + seg * 16, 1);
        else
            window_run<W>(s_cnt + row * ps + seg * 16, 1, s_xcnt + row * XS + seg * 16, 1);
    }
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
}

// y pass of box_xy: s_xp[c][py][XS] -> s_out[c][TY][TX].
template <int NC, bool CNT, int TX, int TY, int NTHR, int W, int XS, bool PRIO = false>
__device__ __forceinline__ void box_y(const double* s_xp, const int* s_xcnt, double* s_out,
                                      int* s_ocnt, int py, int tid) {
    static_assert(TY % 16 == 0, "tile edges are multiples of 16");
    constexpr int NT = NC + (CNT ? 1 : 0);
    constexpr int SY8 = TY / 8;  // y runs of 8 outputs
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(2);
    for (int t = tid; t < NT * TX * SY8; t += NTHR) {
        const int col = t % TX, rest = t / TX;
        const int seg = rest % SY8, c = rest / SY8;
        if (c < NC)
            window_run<W, double, 8>(s_xp + (c * py + seg * 8) * XS + col, XS,
                                   s_out + c * TX * TY + seg * 8 * TX + col, TX);
        else
            window_run<W, int, 8>(s_xcnt + seg * 8 * XS + col, XS, s_ocnt + seg * 8 * TX + col, TX);
    }
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
}

template <int NC, bool CNT, int TX, int TY, int NTHR, int W, int XS, bool PRIO_X = false,
          bool PRIO_Y = false>
__device__ __forceinline__ void box_xy(const double* s_prod, const int* s_cnt, double* s_xp,
                                       int* s_xcnt, double* s_out, int* s_ocnt, int ps, int py,
                                       int tid) {
    box_x<NC, CNT, TX, NTHR, W, XS, PRIO_X>(s_prod, s_cnt, s_xp, s_xcnt, ps, py, tid);
    __syncthreads();
    box_y<NC, CNT, TX, TY, NTHR, W, XS, PRIO_Y>(s_xp, s_xcnt, s_out, s_ocnt, py, tid);
    __syncthreads();
}

// ---------------------------------------------------------------------------
// 3D fused kernel: a TX x TY column of output voxels over `zchunk` planes of one pose.
// MOVI: the moving image is the high-resolution I (warped + Sobel here), the fixed
// ultrasound U is static with precomputed patch statistics (7 channels). Otherwise U is
// warped here and I, |grad I| are static (9 channels + count).
// Global loads are software-pipelined one z-step ahead: the gathers of the next warped
// plane, the static image values of the next products plane and the statistics of the
// next output plane are issued early in a step and consumed in the following one.
// ---------------------------------------------------------------------------
template <int R, bool MOVI, typename T, int TX, int TY, bool P2>
__global__ __launch_bounds__(TX * TY, 1) void k_fused3d(FusedArgs a) {
    constexpr int NTHR = TX * TY;
    constexpr int W = 2 * R + 1;
    constexpr int PX = TX + 2 * R, PY = TY + 2 * R;  // patch-support region
    constexpr int NP = PX * PY;
    constexpr int PS = lds_stride(PX);               // LDS row stride of the products planes
    constexpr int XS = lds_stride(TX + 1);           // LDS row stride of the x-pass output
    constexpr int IXE = PX + 2, IYE = PY + 2;        // Sobel input region
    constexpr int NI = MOVI ? IXE * IYE : NP;        // warped positions per plane
    constexpr int SPT = (NI + NTHR - 1) / NTHR;      // warped samples per thread
    constexpr int PPT = (NP + NTHR - 1) / NTHR;      // products positions per thread
    constexpr int N3 = W * W * W;
    constexpr int LAG = MOVI ? 2 : 0;
    constexpr int NC = MOVI ? 7 : 9;
    constexpr bool CNT = !MOVI;
    // PIPE: steps overlap by half a step (two barriers per z-step instead of four; the
    // loop below says how). The plane sums then need their own LDS (s_sum) instead of
    // reusing s_prod, which the next step's products overwrite while the ring still
    // reads; that fits two work-groups per CU with 7 channels, not with 9. Not at R = 1,
    // where the longer-lived gather registers cost a wave per SIMD (2.64 -> 3.44 ms with
    // the gathers finished a phase early, measured).
    constexpr bool PIPE = MOVI && R >= 2;
    // PAIR: with the moving image warped here and two products slots per thread, a thread
    // takes two vertically adjacent positions of one column (rows ly0 and ly0 + 1, ly0
    // even) instead of positions tid and tid + NTHR: their 3x3 neighbourhoods share two
    // rows, so 4 rows of the warped plane are read and smoothed instead of 6, with the
    // same operations per position. The warped plane's LDS rows are then SIS = 32 + PX/2
    // floats apart: the PX lanes of a pair row read one row of it, the next PX lanes the
    // row two below (2 SIS = 64 + PX words on), so the groups of a wave fall into
    // distinct banks (32 or 64 banks).
    constexpr int NPAIR = PX * (PY / 2);
    constexpr bool PAIR = MOVI && PY % 2 == 0 && (NPAIR + NTHR - 1) / NTHR * 2 == PPT;
    constexpr int SIS = PAIR ? 32 + PX / 2 : IXE;  // row stride of the warped plane in LDS
    static_assert(SIS >= IXE, "warped rows fit their stride");

    __shared__ float s_in[PAIR ? IYE * SIS : NI];
    __shared__ double s_prod[NC * PY * PS];
    __shared__ int s_cnt[CNT ? PY * PS : 1];
    __shared__ double s_xp[NC * PY * XS];
    __shared__ int s_xcnt[CNT ? PY * XS : 1];
    __shared__ double s_sum[PIPE ? NC * TX * TY : 1];
    double* const s_out = PIPE ? s_sum : s_prod;

    int tile, pose;
    if (!map_block(a.tiles, a.npose, tile, pose)) return;  // whole work-group
    const int tid = threadIdx.x;
    const int tcol = tile % (a.ntx * a.nty), zc = tile / (a.ntx * a.nty);
    const int tx = tcol % a.ntx, ty = tcol / a.ntx;
    const int x0 = R + tx * TX, y0 = R + ty * TY;
    const int z0 = R + zc * a.zchunk;
    const int zend = min(z0 + a.zchunk, a.v.Z - R);
    const int nout = zend - z0;
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z;
    const T* __restrict__ src = static_cast<const T*>(a.src);
    float m[12];
    {
        load_matrix(a, (size_t)pose * a.mats_per_pose, m);
    }
    // warped plane of step s: MOVI -> zi = z0-R-1+s (Sobel input), else zp = z0-R+s
    const int zw0 = MOVI ? z0 - R - 1 : z0 - R;
    const int wex = MOVI ? IXE : PX;     // warped region edge along x
    const int wofs = MOVI ? R + 1 : R;   // warped region starts at x0 - wofs, y0 - wofs
    const int nsteps = nout + 2 * R + LAG;

    Pending3<T> pend[SPT];
    // A wave whose 64 positions of slot j all lie past the region skips that slot (its
    // gathers and lerps, or its Sobel and products). The test is wave-uniform (scalar
    // branch).
    const int wbase = __builtin_amdgcn_readfirstlane(tid & ~63);
    auto wave_has = [&](int j, int n) { return (j + 1) * NTHR <= n || j * NTHR + wbase < n; };
    // The partial last gather slot goes to the last waves instead of the first (with 576
    // positions on 256 threads the third slot belongs to wave 3 alone): those are the
    // waves the x pass leaves idle (its 7 x PY row tasks fill the first waves).
    constexpr int GREM = NI - (SPT - 1) * NTHR;           // positions in the last slot
    constexpr int GSKIP = NTHR - (GREM + 63) / 64 * 64;   // threads before its first wave
    auto gpos = [&](int j) { return j < SPT - 1 ? tid + j * NTHR : j * NTHR + tid - GSKIP; };
    auto gwave_has = [&](int j) { return j < SPT - 1 || wbase >= GSKIP; };
    // the in-plane part of each warped position's source coordinates, m*(Lx, Ly, 0), is the
    // same for every plane: computed once, in the order issue3 uses
    float cxy[SPT][3];
    int sin_ofs[SPT];  // LDS offset of warped position gpos(j) in s_in
    unsigned in_xy = 0;
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
        const int i = gpos(j);
        const int lx = i % wex, ly = i / wex;
        sin_ofs[j] = PAIR ? ly * SIS + lx : i;
        const int gx = x0 - wofs + lx, gy = y0 - wofs + ly;
        if (i >= j * NTHR && i < NI && gx >= 0 && gx < X && gy >= 0 && gy < Y) in_xy |= 1u << j;
        const float Lx = fmaf((float)gx, a.v.sx, a.v.ox), Ly = fmaf((float)gy, a.v.sy, a.v.oy);
        cxy[j][0] = fmaf(m[1], Ly, m[0] * Lx);
        cxy[j][1] = fmaf(m[5], Ly, m[4] * Lx);
        cxy[j][2] = fmaf(m[9], Ly, m[8] * Lx);
    }
    auto issue_plane = [&](int zi) {
        const bool zin = zi >= 0 && zi < Z;
        const float lz = fmaf((float)zi, a.v.sz, a.v.oz);
#pragma unroll
        for (int j = 0; j < SPT; ++j)
            if (gwave_has(j)) issue3c<P2>(src, a.s, m, cxy[j], lz, zin && ((in_xy >> j) & 1u), pend[j]);
    };
    // finish the gathers of the plane in flight into s_in. The finishing wave runs at
    // raised priority so that every wave reaches the next barrier sooner (+0.3%, measured).
    auto finish_plane = [&]() {
        __builtin_amdgcn_s_setprio(2);
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            if (!gwave_has(j)) continue;
            const int i = gpos(j);
            const float v = finish3(pend[j]);
            if (i >= j * NTHR && i < NI) s_in[sin_ofs[j]] = v;
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // static image values (U if MOVI, else I and |grad I|) of the products positions
    float pre0[PPT], pre1[PPT];
    // products position (lx, ly) of slot j; false past the region
    auto ppos = [&](int j, int& lx, int& ly) {
        if (PAIR) {
            const int t = tid + (j >> 1) * NTHR;
            lx = t % PX;
            ly = 2 * (t / PX) + (j & 1);
            return t < NPAIR;
        }
        const int i = tid + j * NTHR;
        lx = i % PX;
        ly = i / PX;
        return i < NP;
    };
    auto issue_static = [&](int zp) {
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            int lx, ly;
            const bool pin = ppos(j, lx, ly);
            const int gx = x0 - R + lx, gy = y0 - R + ly;
            const bool in = pin && gx < X && gy < Y && zp >= 0 && zp < Z;
            const int vidx = (zp * Y + gy) * X + gx;
            pre0[j] = in ? a.stat_img[vidx] : 0.0f;
            if (!MOVI) pre1[j] = in ? a.stat_grad[vidx] : 0.0f;
        }
    };
    // static ultrasound statistics of this thread's output voxel
    const int ox = tid % TX, oy = tid / TX;
    const bool col_valid = (x0 + ox < X - R) && (y0 + oy < Y - R);
    double mu_pre = 0.0, cyy_pre = -1.0;
    auto issue_stats = [&](int zo) {
        if (MOVI) {
            const int vo = (zo * Y + (y0 + oy)) * X + (x0 + ox);
            const bool ok = col_valid && zo >= z0 && zo < zend;
            mu_pre = ok ? a.ustat_mean[vo] : 0.0;
            cyy_pre = ok ? a.ustat_cyy[vo] : -1.0;
        }
    };

    float tA[PPT][3], tBx[PPT][3], tBy[PPT][3], Iprev[PPT], Icur[PPT];
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
#pragma unroll
        for (int k = 0; k < 3; ++k) { tA[j][k] = 0.f; tBx[j][k] = 0.f; tBy[j][k] = 0.f; }
        Iprev[j] = 0.f;
        Icur[j] = 0.f;
        pre0[j] = 0.f;
        pre1[j] = 0.f;
    }
    double ring[W][NC];
    int ringc[W];
    int SC = 0;
#pragma unroll
    for (int k = 0; k < W; ++k) {
        ringc[k] = 0;
#pragma unroll
        for (int c = 0; c < NC; ++c) ring[k][c] = 0.0;
    }
    double acc_m = 0.0, acc_w = 0.0;
    const int cols = a.ntx * a.nty;

    issue_plane(zw0);
    issue_static(z0 - R);      // products plane of the first products step
    issue_stats(z0);           // first output plane
    if (PIPE) {
        finish_plane();
        __syncthreads();
    }

    // 2. in-plane Sobel of the 3x3 neighbourhood of the warped plane in s_in (rows: smooth
    // s = (l + 2c) + r and difference d = r - l along x; then A, Bx, By down the rows), a
    // 3-plane ring in registers along z, |grad| and, for q >= 0, the products of plane
    // z0 - R + q into s_prod
    auto sobel_products = [&](int q, const float* cur0, const float* cur1) {
        if constexpr (PAIR) {
#pragma unroll
            for (int jp = 0; jp < PPT / 2; ++jp) {
                if (!wave_has(jp, NPAIR)) continue;
                const int t = tid + jp * NTHR;
                if (t < NPAIR) {
                    const int lx = t % PX, ly0 = 2 * (t / PX);
                    // rows ly0 .. ly0 + 3: smooth s = (l + 2c) + r, difference d = r - l
                    const float* row = s_in + ly0 * SIS + lx;
                    float sm[4], df[4], cm[4];
#pragma unroll
                    for (int rr = 0; rr < 4; ++rr) {
                        const float l = row[rr * SIS], c = row[rr * SIS + 1], r = row[rr * SIS + 2];
                        sm[rr] = (l + 2.0f * c) + r;
                        df[rr] = r - l;
                        cm[rr] = c;
                    }
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int j = 2 * jp + e;
                        // A = (s0 + 2 s1) + s2, Bx = (d0 + 2 d1) + d2, By = s2 - s0 over the
                        // position's rows ly0 + e .. ly0 + e + 2
                        tA[j][0] = tA[j][1]; tA[j][1] = tA[j][2];
                        tBx[j][0] = tBx[j][1]; tBx[j][1] = tBx[j][2];
                        tBy[j][0] = tBy[j][1]; tBy[j][1] = tBy[j][2];
                        tA[j][2] = (sm[e] + 2.0f * sm[e + 1]) + sm[e + 2];
                        tBx[j][2] = (df[e] + 2.0f * df[e + 1]) + df[e + 2];
                        tBy[j][2] = sm[e + 2] - sm[e];
                        Iprev[j] = Icur[j];
                        Icur[j] = cm[e + 1];
                        if (q >= 0) {
                            const float gxv = (tBx[j][0] + 2.0f * tBx[j][1]) + tBx[j][2];
                            const float gyv = (tBy[j][0] + 2.0f * tBy[j][1]) + tBy[j][2];
                            const float gzv = tA[j][2] - tA[j][0];
                            const float G = sqrtf(fmaf(gzv, gzv, fmaf(gyv, gyv, gxv * gxv)));
                            store_products<NC>(s_prod, s_cnt, PY * PS, (ly0 + e) * PS + lx,
                                               Iprev[j], G, cur0[j]);
                        }
                    }
                }
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            if (!wave_has(j, NP)) continue;
            const int i = tid + j * NTHR;
            if (i < NP) {
                const int lx = i % PX, ly = i / PX;
                if (MOVI) {
                    // rows in order, accumulating A = (s0 + 2 s1) + s2,
                    // Bx = (d0 + 2 d1) + d2 and By = s2 - s0 as they arrive
                    const float* row = s_in + ly * IXE + lx;
                    float l = row[0], c = row[1], r = row[2];
                    const float s0 = (l + 2.0f * c) + r;
                    float a = s0, bx = r - l;
                    row += IXE;
                    l = row[0], c = row[1], r = row[2];
                    a = a + 2.0f * ((l + 2.0f * c) + r);
                    bx = bx + 2.0f * (r - l);
                    const float cc = c;
                    row += IXE;
                    l = row[0], c = row[1], r = row[2];
                    const float s2 = (l + 2.0f * c) + r;
                    tA[j][0] = tA[j][1]; tA[j][1] = tA[j][2];
                    tBx[j][0] = tBx[j][1]; tBx[j][1] = tBx[j][2];
                    tBy[j][0] = tBy[j][1]; tBy[j][1] = tBy[j][2];
                    tA[j][2] = a + s2;
                    tBx[j][2] = bx + (r - l);
                    tBy[j][2] = s2 - s0;
                    Iprev[j] = Icur[j];
                    Icur[j] = cc;
                }
                if (q >= 0) {
                    float I, G, U;
                    if (MOVI) {
                        const float gxv = (tBx[j][0] + 2.0f * tBx[j][1]) + tBx[j][2];
                        const float gyv = (tBy[j][0] + 2.0f * tBy[j][1]) + tBy[j][2];
                        const float gzv = tA[j][2] - tA[j][0];
                        G = sqrtf(fmaf(gzv, gzv, fmaf(gyv, gyv, gxv * gxv)));
                        I = Iprev[j];
                        U = cur0[j];
                    } else {
                        U = s_in[i];
                        I = cur0[j];
                        G = cur1[j];
                    }
                    store_products<NC>(s_prod, s_cnt, PY * PS, ly * PS + lx, I, G, U);
                }
            }
        }
    };
    // 4. z ring of plane sums and combine, for the step of products plane q (q >= 0) whose
    // plane sums are in s_out, ring slot SLOT. The patch sums add the W plane sums in z
    // order (no running sum), so a voxel's value does not depend on where its work-group's
    // z-chunk starts; integer counts can run.
    auto ring_combine = [&](auto slot_c, int q) {
        constexpr int slot = decltype(slot_c)::value;
        const int zp = z0 - R + q;
        if (CNT) {
            const int cc = s_cnt[tid];
            SC += cc - ringc[slot];
            ringc[slot] = cc;
        }
        // pair sums: slot (q-1) turns from plane q-1 into Q(q-1) = P(q-1) + P(q), slot q
        // takes P(q); a window of W = 2R+1 planes ending at q is then the R pair sums
        // Q(q-2R), Q(q-2R+2), ..., Q(q-2) plus P(q): R+1 adds per channel, not 2R
        constexpr int prev = (slot + W - 1) % W;
        double Pn[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            Pn[c] = s_out[c * TX * TY + tid];
            ring[prev][c] = ring[prev][c] + Pn[c];
            ring[slot][c] = Pn[c];
        }
        if (q >= 2 * R) {
            const double mu = mu_pre, cyy = cyy_pre;
            if (q + 1 < nout + 2 * R) issue_stats(zp - R + 1);
            double S[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                double t = ring[(slot + 1) % W][c];  // Q(q-2R)
#pragma unroll
                for (int j = 1; j < R; ++j) t += ring[(slot + 1 + 2 * j) % W][c];
                S[c] = t + Pn[c];
            }
            if (col_valid) {
                double w, meas;
                bool ok;
                if (MOVI) ok = combine_static_u(S, mu, cyy, N3, w, meas);
                else ok = combine(S, SC, N3, w, meas);
                if (ok) {
                    acc_m += meas;
                    acc_w += w;
                    if (a.wmap) {
                        const int vo = ((zp - R) * Y + (y0 + oy)) * X + (x0 + ox);
                        a.wmap[vo] = w;
                        a.mmap[vo] = meas;
                    }
                }
            }
            // Partial sums per block of kZBlock output planes, tile column and wave, at
            // fixed positions in z: every z-chunk (a multiple of kZBlock) and every batch
            // size then adds the same numbers in the same order. One partial per wave needs
            // no barrier (a work-group sum would take one every kZBlock steps).
            const int zo = zp - R;  // this step's output plane (block-uniform)
            if ((zo - R + 1) % kZBlock == 0 || zo + 1 == zend) {
                constexpr int NW = NTHR / 64;
                double* dst = a.partials + (((size_t)pose * a.blocks_per_pose +
                                             ((size_t)((zo - R) / kZBlock) * cols + tcol) * NW +
                                             (tid >> 6)) * 2);
                wave_reduce_store(acc_m, acc_w, dst);
                acc_m = 0.0;
                acc_w = 0.0;
            }
        }
    };

    if constexpr (PIPE) {
        // Two barriers per z-step: step s's Sobel and products share a phase with step
        // s - 1's y pass, and step s's x pass with step s - 1's ring and combine and the
        // finishing of plane s + 1's gathers. Each phase writes only LDS that the other
        // phase reads, so one barrier closes it: phase 1 writes s_prod and s_sum and reads
        // s_in and s_xp, phase 2 writes s_xp and s_in and reads s_prod and s_sum.
        for (int s0 = 0; s0 <= nsteps; s0 += W) {
            // W consecutive steps with compile-time ring slots, so the z ring stays in VGPRs.
            Unroll<0, W>::run([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const int s = s0 + k;
                if (s > nsteps) return;  // block-uniform; step nsteps only drains s - 1
                const int q = s - LAG;
                const bool here = s < nsteps;
                const bool more = s + 1 < nsteps;
                const bool prev = s >= 1 && q >= 1;  // step s - 1 made products
                // phase 1
                if (here) {
                    float cur0[PPT], cur1[PPT];
#pragma unroll
                    for (int j = 0; j < PPT; ++j) {
                        cur0[j] = pre0[j];
                        cur1[j] = pre1[j];
                    }
                    if (q >= 0 && q + 1 < nout + 2 * R) issue_static(z0 - R + q + 1);
                    sobel_products(q, cur0, cur1);
                    // the next plane's gathers fly during the y pass, the barrier and the
                    // x pass
                    if (more) issue_plane(zw0 + s + 1);
                }
                if (prev) box_y<NC, CNT, TX, TY, NTHR, W, XS, true>(s_xp, s_xcnt, s_out, s_cnt, PY, tid);
                __syncthreads();
                // phase 2
                if (here && q >= 0)
                    box_x<NC, CNT, TX, NTHR, W, XS, false>(s_prod, s_cnt, s_xp, s_xcnt, PS, PY, tid);
                if (more) finish_plane();
                // the ring and combine at raised priority: 0.7% faster (measured); the x pass
                // stays at normal priority
                __builtin_amdgcn_s_setprio(1);
                if (prev) ring_combine(std::integral_constant<int, (k - 1 - LAG + 2 * W) % W>{}, q - 1);
                __builtin_amdgcn_s_setprio(0);
                __syncthreads();
            });
        }
        return;
    }

    for (int s0 = 0; s0 < nsteps; s0 += W) {
        // W consecutive steps with compile-time ring slots (k), so the z ring stays in VGPRs.
        Unroll<0, W>::run([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            const int s = s0 + k;
            if (s >= nsteps) return;  // block-uniform
            const int q = s - LAG;
            const int zp = z0 - R + q;
            // 1. finish the plane issued last step
            finish_plane();
            float cur0[PPT], cur1[PPT];
#pragma unroll
            for (int j = 0; j < PPT; ++j) {
                cur0[j] = pre0[j];
                cur1[j] = pre1[j];
            }
            if (q >= 0 && q + 1 < nout + 2 * R) issue_static(zp + 1);
            __syncthreads();
            sobel_products(q, cur0, cur1);
            __syncthreads();  // s_in reads done; products visible
            // the next plane's gathers fly during the box sums and the combine
            if (s + 1 < nsteps) issue_plane(zw0 + s + 1);
            if (q < 0) return;  // block-uniform: Sobel ring warm-up only
            // 3. in-plane box sums
            box_xy<NC, CNT, TX, TY, NTHR, W, XS, true, true>(s_prod, s_cnt, s_xp, s_xcnt, s_out,
                                                            s_cnt, PS, PY, tid);
            ring_combine(std::integral_constant<int, (k - LAG + W) % W>{}, q);
        });
    }
}

// ---------------------------------------------------------------------------
// Separable path for patch radii beyond the other kernels (3D r > kMaxRMom3, 2D r > kMaxR2):
// the reference switches to a global-memory kernel there (cu_lc2_3d.cu:769-827, chosen at
// :1133-1177). Here, per pose: the moving image is warped (and, if it is the high-resolution
// one, its |Sobel| taken) into two f32 grids, then the patch sums of every moment channel are
// box sums along z (3D) and y through two f64 buffers, each a van Herk / Gil-Werman pass
// (exact in the sense of the fused kernels: no partial sum holds a value from outside its
// window), and a last kernel sums along x, combines per voxel and reduces per work-group.
// Channels: moving high-resolution image (7): I, G, II, GG, IG, UI, UG; moving ultrasound
// (10): I, G, U, II, GG, IG, UU, UI, UG and the count of U > 1e-6 (exact as a double); static
// ultrasound's statistics (3): U, UU, count.
// ---------------------------------------------------------------------------
enum { kSepMovingImage, kSepMovingUs, kSepUsStats };
template <int KIND>
constexpr int kSepNC = KIND == kSepMovingImage ? 7 : KIND == kSepMovingUs ? 10 : 3;

// One box pass: window sums of width W along lines of n elements, `stride` apart, to `dst` at
// the index of the window start; buffers are [channel][V]. Line l of a channel starts at
// (l / X) * outer + l % X, a lane per line, so loads and stores are whole rows. KIND >= 0: the
// inputs are the products of the I, G, U grids; -1: `src`. A work-group (one wave) takes the
// outputs [s, s + seg) of its lines, seg a multiple of W. A block's inputs lie in LDS, where they
// become its suffix sums; the sum of output j is suffix j plus the running prefix of the next
// block, so each input is read and each output written once. Channels of the same lines run on one
// XCD one after the other (they read the same grids). Bound by memory: a pose of 161x150x131, r = 7,
// 7 channels: z 53 us, y 110, then 76 for the last kernel; 2D, 260x260, r = 16, 10 channels: 22 and 15.
// With the suffix sums in `dst` and a pass along x with a lane per line (strided loads) the
// three passes took 240 to 1500 us each, the 2D ones 160 and over 360.
template <int KIND>
__global__ __launch_bounds__(64) void k_sep_pass(const float* __restrict__ I, const float* __restrict__ G,
                                                 const float* __restrict__ U, const double* __restrict__ src,
                                                 double* __restrict__ dst, long long V, int X, long long lines,
                                                 long long outer, int stride, int n, int W, int seg, int nc) {
    extern __shared__ double s_sep[];
    double* suf = s_sep + threadIdx.x;
    const int xcd = blockIdx.x % kXcds, k = blockIdx.x / kXcds;
    const int c = k % nc;
    const long long l = ((long long)(k / nc) * kXcds + xcd) * 64 + threadIdx.x;
    if (l >= lines) return;  // (no barriers: a lane only touches its own LDS column)
    const long long base = (l / X) * outer + l % X;
    const int s0 = blockIdx.y * seg, s1 = min(s0 + seg, n - W + 1);
    double* o = dst + (size_t)c * V + base;
    // channel c is p * q of the grids, p alone, or the count
    const float *p = nullptr, *q = nullptr;
    bool count = false;
    if constexpr (KIND == kSepMovingImage) {
        p = c == 0 || c == 2 || c == 4 ? I : c == 1 || c == 3 ? G : U;
        q = c < 2 ? nullptr : c == 2 || c == 5 ? I : G;
    } else if constexpr (KIND == kSepMovingUs) {
        p = c == 0 || c == 3 || c == 5 ? I : c == 1 || c == 4 ? G : U;
        q = c < 3 || c == 9 ? nullptr : c == 3 || c == 7 ? I : c == 6 ? U : G;
        count = c == 9;
    } else if constexpr (KIND == kSepUsStats) {
        p = U;
        q = c == 1 ? U : nullptr;
        count = c == 2;
    }
    constexpr int B = 8;  // inputs in flight
    // inputs i .. i + B - 1, none past `last`
    auto load = [&](int i, int last, double (&x)[B]) {
        if constexpr (KIND >= 0) {
            float f[B], g[B];
#pragma unroll
            for (int e = 0; e < B; ++e) f[e] = p[base + (long long)min(i + e, last) * stride];
            if (q) {
#pragma unroll
                for (int e = 0; e < B; ++e) g[e] = q[base + (long long)min(i + e, last) * stride];
            }
#pragma unroll
            for (int e = 0; e < B; ++e) {
                x[e] = q ? (double)f[e] * (double)g[e] : (double)f[e];
                if (count) x[e] = x[e] > kZeroThreshold ? 1.0 : 0.0;
            }
        } else {
            const double* in = src + (size_t)c * V + base;
#pragma unroll
            for (int e = 0; e < B; ++e) x[e] = in[(long long)min(i + e, last) * stride];
        }
    };
    for (int j0 = 0; j0 < W; j0 += B) {
        double x[B];
        load(s0 + j0, s0 + W - 1, x);
#pragma unroll
        for (int e = 0; e < B; ++e)
            if (j0 + e < W) suf[(j0 + e) * 64] = x[e];
    }
    for (int b = s0;; b += W) {
        double acc = 0.0;
#pragma unroll 8
        for (int j = W - 1; j >= 0; --j) {
            acc += suf[j * 64];
            suf[j * 64] = acc;
        }
        o[(long long)b * stride] = acc;
        const bool more = b + W < s1;
        const int m = min(W, s1 - b);           // outputs of this block
        const int cnt = more ? W : m - 1;       // inputs of the next one that are needed
        double pre = 0.0;
        for (int j0 = 0; j0 < cnt; j0 += B) {
            double x[B];
            load(b + W + j0, b + W + cnt - 1, x);
#pragma unroll
            for (int e = 0; e < B; ++e) {
                const int j = j0 + e;
                if (j < cnt) {
                    pre += x[e];
                    if (j + 1 < m) o[(long long)(b + j + 1) * stride] = suf[(j + 1) * 64] + pre;
                    suf[j * 64] = x[e];
                }
            }
        }
        if (!more) return;
    }
}

// Orders a wave's LDS writes and reads across its lanes (the hardware keeps them in order).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Sums along x and combine: a wave takes 64 outputs of a row, with the row's 64 + 2r sums of every
// channel in its part of the LDS; wave i of the grid takes the strips i, i + waves, ... Per
// output voxel: weight and measure; per work-group sums into the pose's partials (fixed
// positions, fixed order). kSepUsStats writes the statistics instead.
template <int KIND>
__global__ __launch_bounds__(256) void k_sep_combine(const double* __restrict__ S, double* __restrict__ ustat_mean,
                                                     double* __restrict__ ustat_cyy, VGeom v, int r, int grid3,
                                                     double* partials, double* wmap, double* mmap) {
    extern __shared__ double s_rows[];
    __shared__ double s_red[8];
    constexpr int NC = kSepNC<KIND>;
    const long long V = (long long)v.X * v.Y * v.Z;
    const int W = 2 * r + 1, L = 64 + 2 * r;
    const int ex = v.X - 2 * r, ey = v.Y - 2 * r, ez = grid3 ? v.Z - 2 * r : v.Z;
    const int N = grid3 ? W * W * W : W * W;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double* row = s_rows + (size_t)wave * NC * L;
    const int per_row = (ex + 63) / 64;
    const long long strips = (long long)per_row * ey * ez;
    double am = 0.0, aw = 0.0;
    for (long long s = (long long)blockIdx.x * 4 + wave; s < strips; s += (long long)gridDim.x * 4) {
        const int x0 = (int)(s % per_row) * 64;
        const long long yz = s / per_row;
        const int sy = (int)(yz % ey), sz = (int)(yz / ey);
        const long long line = ((long long)sz * v.Y + sy) * v.X;
        for (int i = lane; i < L; i += 64)
#pragma unroll
            for (int c = 0; c < NC; ++c) row[c * L + i] = x0 + i < v.X ? S[(size_t)c * V + line + x0 + i] : 0.0;
        wave_lds_sync();
        double Sc[NC] = {};
#pragma unroll 2
        for (int j = 0; j < W; ++j)
#pragma unroll
            for (int c = 0; c < NC; ++c) Sc[c] += row[c * L + lane + j];
        wave_lds_sync();
        if (x0 + lane < ex) {
            const long long vo = ((long long)(sz + (grid3 ? r : 0)) * v.Y + (sy + r)) * v.X + (x0 + lane + r);
            if constexpr (KIND == kSepUsStats) {
                const double cc = Sc[1] - Sc[0] * Sc[0] * (1.0 / (double)N);
                const bool ok = Sc[2] == (double)N && cc * (1.0 / (double)(N - 1)) > kZeroThreshold;
                ustat_mean[vo] = ok ? Sc[0] * (1.0 / (double)N) : 0.0;
                ustat_cyy[vo] = ok ? cc : -1.0;
            } else {
                double w, meas;
                bool ok;
                if constexpr (KIND == kSepMovingImage) ok = combine_static_u(Sc, ustat_mean[vo], ustat_cyy[vo], N, w, meas);
                else ok = combine(Sc, (int)Sc[9], N, w, meas);
                if (ok) {
                    am += meas;
                    aw += w;
                    if (wmap) {
                        wmap[vo] = w;
                        mmap[vo] = meas;
                    }
                }
            }
        }
    }
    if constexpr (KIND != kSepUsStats) block_reduce_store<256>(am, aw, s_red, partials + (size_t)blockIdx.x * 2);
}

// Per-pose fixed-order reduction of the work-group partials -> (sum m, sum w, LC2)
// (GetSimilarityMetric, cu_lc2_3d.cu:1181-1191; sums in FP64, NaN/Inf -> 0).
__global__ __launch_bounds__(256) void k_reduce(const double* __restrict__ partials, int nb,
                                                double* __restrict__ out) {
    __shared__ double sm[256], sw[256];
    const int pose = blockIdx.x;
    const double2* p = reinterpret_cast<const double2*>(partials) + (size_t)pose * nb;
    double m = 0.0, w = 0.0;
    // each thread adds partials tid, tid + 256, ... in that order; four loads are in
    // flight at a time (the order of the additions, and so the result, is unchanged)
    int i = threadIdx.x;
    for (; i + 3 * 256 < nb; i += 4 * 256) {
        const double2 a0 = p[i], a1 = p[i + 256], a2 = p[i + 512], a3 = p[i + 768];
        m += a0.x; w += a0.y;
        m += a1.x; w += a1.y;
        m += a2.x; w += a2.y;
        m += a3.x; w += a3.y;
    }
    for (; i < nb; i += 256) {
        const double2 a = p[i];
        m += a.x;
        w += a.y;
    }
    sm[threadIdx.x] = m;
    sw[threadIdx.x] = w;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            sm[threadIdx.x] += sm[threadIdx.x + h];
            sw[threadIdx.x] += sw[threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double M = sm[0], Wt = sw[0];
        double l = M / Wt;
        if (isnan(l) || isinf(l)) l = 0.0;
        out[pose * 3 + 0] = M;
        out[pose * 3 + 1] = Wt;
        out[pose * 3 + 2] = l;
    }
}

template <typename T>
__global__ void k_warp_static(const T* fixed, SGeom fg, VGeom v, int mode, float* out) {
    // mode 0: 3D grid, trilinear; 1: 2D grid, bilinear per frame (frames = v.Z)
    const long long n = (long long)v.X * v.Y * v.Z;
    const float ident[12] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0};
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(i % v.X), y = (int)((i / v.X) % v.Y), z = (int)(i / ((long long)v.X * v.Y));
        const float lx = fmaf((float)x, v.sx, v.ox), ly = fmaf((float)y, v.sy, v.oy);
        float val;
        if (mode == 0)
            val = sample3(fixed, fg, ident, lx, ly, fmaf((float)z, v.sz, v.oz));
        else
            val = sample2(fixed + (size_t)z * fg.X * fg.Y, fg, ident, lx, ly);
        out[i] = val;
    }
}

template <typename T>
__global__ void k_warp_moving(FusedArgs a, int grid3, int src3, float* out) {
    const VGeom v = a.v;
    const T* src = static_cast<const T*>(a.src);
    const long long n = (long long)v.X * v.Y * v.Z;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(i % v.X), y = (int)((i / v.X) % v.Y), z = (int)(i / ((long long)v.X * v.Y));
        float m[12];
        load_matrix(a, grid3 ? 0 : (a.mats_per_pose > 1 ? z : 0), m);
        const float lx = fmaf((float)x, v.sx, v.ox), ly = fmaf((float)y, v.sy, v.oy);
        const float lz = grid3 ? fmaf((float)z, v.sz, v.oz) : v.oz;
        out[i] = src3 ? sample3(src, a.s, m, lx, ly, lz) : sample2(src, a.s, m, lx, ly);
    }
}

// Static ultrasound patch statistics (weight half of cu_lc2_3d.cu:181-287 /
// cu_lc2_2d.cu:88-180) per voxel in FP64: count of U > 1e-6, sum, sum of squares in a
// fixed x-fastest order; mean and centred energy, or -1 where w = 0. For grids of large planes
// only: the others have the moments kernels' or the box passes' statistics.
__global__ void k_ustats(const float* img, VGeom v, int grid3, int r, double* mean, double* cyy) {
    const long long n = (long long)v.X * v.Y * v.Z;
    const int w = 2 * r + 1;
    const int N = grid3 ? w * w * w : w * w;
    const int rz = grid3 ? r : 0;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(i % v.X), y = (int)((i / v.X) % v.Y), z = (int)(i / ((long long)v.X * v.Y));
        double m = 0.0, c = -1.0;
        const bool inside = x >= r && y >= r && x + r < v.X && y + r < v.Y &&
                            (!grid3 || (z >= r && z + r < v.Z));
        if (inside) {
            int cnt = 0;
            double s1 = 0.0, s2 = 0.0;
            for (int dz = -rz; dz <= rz; ++dz)
                for (int dy = -r; dy <= r; ++dy) {
                    const float* row = img + ((long long)(z + dz) * v.Y + (y + dy)) * v.X + x;
                    for (int dx = -r; dx <= r; ++dx) {
                        const double u = row[dx];
                        cnt += (u > kZeroThreshold) ? 1 : 0;
                        s1 += u;
                        s2 += u * u;
                    }
                }
            if (cnt == N) {
                const double cc = s2 - s1 * s1 * (1.0 / (double)N);
                if (cc * (1.0 / (double)(N - 1)) > kZeroThreshold) {
                    m = s1 * (1.0 / (double)N);
                    c = cc;
                }
            }
        }
        mean[i] = m;
        cyy[i] = c;
    }
}

__global__ void k_ustats_none(long long n, double* mean, double* cyy) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        mean[i] = 0.0;
        cyy[i] = -1.0;
    }
}

__device__ __forceinline__ float at_img(const float* img, const VGeom& v, int x, int y, int z) {
    if (x < 0 || y < 0 || x >= v.X || y >= v.Y) return 0.0f;
    return img[(z * v.Y + y) * v.X + x];
}

// Separable Sobel triplet (A, Bx, By) of plane z at (x, y), zero padding.
__device__ __forceinline__ void sobel_triplet(const float* img, const VGeom& v, int x, int y,
                                              int z, float& A, float& Bx, float& By) {
    float s[3], d[3];
    for (int k = 0; k < 3; ++k) {
        const int yy = y + k - 1;
        const float l = at_img(img, v, x - 1, yy, z), c = at_img(img, v, x, yy, z),
                    r = at_img(img, v, x + 1, yy, z);
        d[k] = r - l;
        s[k] = (l + 2.0f * c) + r;
    }
    A = (s[0] + 2.0f * s[1]) + s[2];
    Bx = (d[0] + 2.0f * d[1]) + d[2];
    By = s[2] - s[0];
}

__global__ void k_sobel(const float* img, VGeom v, int grid3, float* out) {
    const long long n = (long long)v.X * v.Y * v.Z;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(i % v.X), y = (int)((i / v.X) % v.Y), z = (int)(i / ((long long)v.X * v.Y));
        float A, Bx, By;
        sobel_triplet(img, v, x, y, z, A, Bx, By);
        float gx, gy, gz;
        if (grid3) {
            float Am = 0.f, Bxm = 0.f, Bym = 0.f, Ap = 0.f, Bxp = 0.f, Byp = 0.f;
            if (z > 0) sobel_triplet(img, v, x, y, z - 1, Am, Bxm, Bym);
            if (z + 1 < v.Z) sobel_triplet(img, v, x, y, z + 1, Ap, Bxp, Byp);
            gx = (Bxm + 2.0f * Bx) + Bxp;
            gy = (Bym + 2.0f * By) + Byp;
            gz = Ap - Am;
        } else {
            gx = Bx;
            gy = By;
            gz = 0.0f;
        }
        out[i] = sqrtf(fmaf(gz, gz, fmaf(gy, gy, gx * gx)));
    }
}

__device__ __forceinline__ float raw_value(const void* in, int dtype, long long i) {
    switch (dtype) {
        case 0: return (float)static_cast<const unsigned char*>(in)[i];
        case 1: return (float)static_cast<const short*>(in)[i];
        case 2: return __half2float(static_cast<const __half*>(in)[i]);
        default: return static_cast<const float*>(in)[i];
    }
}

// 16 bytes of input per thread and step (blocks from hipMalloc are aligned to that); the last
// elements one by one. Both kernels below read at the memory's rate: k_check 50 MB in 14 us.
template <typename F>
__device__ __forceinline__ void for_vectors(long long n, int per, F&& f) {
    const long long nv = (n + per - 1) / per;
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < nv; v += (long long)gridDim.x * 256) f(v * per, min((long long)per, n - v * per));
}

__global__ __launch_bounds__(256) void k_check(const void* in, int in_dtype, long long n, float lim, int* flag) {
    bool bad = false, large = false;
    const int per = in_dtype == 3 ? 4 : 8;
    for_vectors(n, per, [&](long long i0, long long m) {
        if (m == per) {
            uint4 w = static_cast<const uint4*>(in)[i0 / per];
            if (in_dtype == 3) {
                float x[4];
                __builtin_memcpy(x, &w, 16);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    bad |= !(fabsf(x[k]) <= lim);
                    large |= fabsf(x[k]) > kHalfRange;
                }
            } else {
                short x[8];
                __builtin_memcpy(x, &w, 16);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    __half h;
                    __builtin_memcpy(&h, &x[k], 2);
                    bad |= !(fabsf(in_dtype == 1 ? (float)x[k] : __half2float(h)) <= lim);
                }
            }
        } else {
            for (long long i = i0; i < i0 + m; ++i) {
                const float x = fabsf(raw_value(in, in_dtype, i));
                bad |= !(x <= lim);
                large |= x > kHalfRange;
            }
        }
    });
    if (__any(bad) && (threadIdx.x & 63) == 0) flag[0] = 1;
    if (__any(large) && (threadIdx.x & 63) == 0) flag[1] = 1;
}

__global__ void k_convert(const void* in, int in_dtype, void* out, int out_f16, long long n) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const float v = raw_value(in, in_dtype, i);
        if (out_f16) static_cast<__half*>(out)[i] = __float2half_rn(v);
        else static_cast<float*>(out)[i] = v;
    }
}

// The launch helpers below either launch (occ == nullptr) or report, in *occ, how many
// work-groups of the kernel they would launch fit on one CU at once.
template <int R, typename T, bool P2>
hipError_t launch3(const FusedArgs& a, bool movi, dim3 grid, hipStream_t st, int* occ) {
    constexpr int nt = kTile3X * kTile3Y;
    if (occ) {
        return movi ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                          occ, k_fused3d<R, true, T, kTile3X, kTile3Y, P2>, nt, 0)
                    : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                          occ, k_fused3d<R, false, T, kTile3X, kTile3Y, P2>, nt, 0);
    }
    if (movi) hipLaunchKernelGGL((k_fused3d<R, true, T, kTile3X, kTile3Y, P2>), grid, dim3(nt), 0, st, a);
    else hipLaunchKernelGGL((k_fused3d<R, false, T, kTile3X, kTile3Y, P2>), grid, dim3(nt), 0, st, a);
    return hipGetLastError();
}

template <typename T, bool P2>
hipError_t launch3r(const FusedArgs& a, bool movi, dim3 grid, hipStream_t st, int* occ) {
    switch (a.r) {
        case 1: return launch3<1, T, P2>(a, movi, grid, st, occ);
        case 2: return launch3<2, T, P2>(a, movi, grid, st, occ);
        case 3: return launch3<3, T, P2>(a, movi, grid, st, occ);
        case 4: return launch3<4, T, P2>(a, movi, grid, st, occ);
        default: return hipErrorInvalidValue;
    }
}

// The fused kernel for the moving image's storage type and spacing form (SGeom::pow2).
hipError_t launch3d(const FusedArgs& a, bool movi, dim3 grid, hipStream_t st, int* occ) {
    if (a.s.pow2)
        return a.src_f16 ? launch3r<__half, true>(a, movi, grid, st, occ)
                         : launch3r<float, true>(a, movi, grid, st, occ);
    return a.src_f16 ? launch3r<__half, false>(a, movi, grid, st, occ)
                     : launch3r<float, false>(a, movi, grid, st, occ);
}

}  // namespace

int fused_blocks_3d(const VGeom& v, int r, int zchunk, int* ntx, int* nty, int* nzc) {
    const int ex = v.X - 2 * r, ey = v.Y - 2 * r, ez = v.Z - 2 * r;
    if (ex <= 0 || ey <= 0 || ez <= 0 || zchunk <= 0) { *ntx = *nty = *nzc = 0; return 0; }
    *ntx = (ex + kTile3X - 1) / kTile3X;
    *nty = (ey + kTile3Y - 1) / kTile3Y;
    *nzc = (ez + zchunk - 1) / zchunk;
    return *ntx * *nty * *nzc;
}

int fused_partials_3d(const VGeom& v, int r) {
    int ntx, nty, nzc;
    if (fused_blocks_3d(v, r, kZBlock, &ntx, &nty, &nzc) <= 0) return 0;
    return ntx * nty * nzc * (kTile3X * kTile3Y / 64);  // one per wave
}

hipError_t launch_fused(const FusedArgs& a, int movi, int n_poses, hipStream_t st) {
    if (a.tiles == 0 || n_poses <= 0) return hipSuccess;
    if (a.zchunk <= 0 || a.zchunk % kZBlock != 0) return hipErrorInvalidValue;
    FusedArgs b = a;
    b.npose = n_poses;
    const long long tiles8 = (a.tiles + kXcds - 1) / kXcds * (long long)kXcds;
    if (tiles8 * n_poses > 0x7fffffffLL) return hipErrorInvalidValue;
    return launch3d(b, movi, dim3((unsigned)(tiles8 * n_poses)), st, nullptr);
}

hipError_t fused_resident_per_cu(const FusedArgs& a, int movi, int* per_cu) {
    *per_cu = 0;
    return launch3d(a, movi, dim3(1), nullptr, per_cu);
}

static dim3 grid_for(long long n) {
    long long b = (n + 255) / 256;
    if (b > 65535LL * 16) b = 65535LL * 16;
    if (b < 1) b = 1;
    return dim3((unsigned)b);
}

int sep_blocks(const VGeom& v, int r, int grid_ndim) {
    const long long ex = v.X - 2 * r, ey = v.Y - 2 * r, ez = grid_ndim == 3 ? v.Z - 2 * r : v.Z;
    if (ex <= 0 || ey <= 0 || ez <= 0) return 0;
    return (int)((ex * ey * ez + 255) / 256);
}

namespace {

// The box passes over the grids, and the last kernel on nb work-groups.
template <int KIND>
hipError_t sep_sums(const float* I, const float* G, const float* U, double* sum_a, double* sum_b, const VGeom& v,
                    int r, int grid_ndim, int nb, double* mean, double* cyy, double* partials, double* wmap,
                    double* mmap, hipStream_t st) {
    constexpr int NC = kSepNC<KIND>;
    const long long V = (long long)v.X * v.Y * v.Z;
    const int W = 2 * r + 1;
    // 66 KB at the largest radius, 61 KB for the rows
    static LdsLimit pass_limit, rows_limit;
    hipError_t err = pass_limit.raise({reinterpret_cast<const void*>(&k_sep_pass<KIND>),
                                       reinterpret_cast<const void*>(&k_sep_pass<-1>)},
                                      (2 * kMaxRSep + 1) * 64 * sizeof(double));
    if (err == hipSuccess)
        err = rows_limit.raise({reinterpret_cast<const void*>(&k_sep_combine<KIND>)},
                               4 * NC * (64 + 2 * kMaxRSep) * sizeof(double));
    if (err != hipSuccess) return err;
    bool first = true;
    auto pass = [&](long long lines, long long outer, int stride, int n, const double* src, double* dst) {
        const long long tiles8 = ((lines + 63) / 64 + kXcds - 1) / kXcds * kXcds;
        // 16 waves per CU where that leaves each at least two blocks (the first one's inputs
        // are read twice)
        const int blocks = (n - W + 1 + W - 1) / W;
        const int segs = (int)std::max(1LL, std::min<long long>(4096 / (tiles8 * NC), blocks / 2));
        const int seg = (blocks + segs - 1) / segs * W;
        const dim3 grid((unsigned)(tiles8 * NC), (unsigned)((n - W + seg) / seg));
        const size_t lds = (size_t)W * 64 * sizeof(double);
        if (first)
            hipLaunchKernelGGL(k_sep_pass<KIND>, grid, dim3(64), lds, st, I, G, U, src, dst, V, v.X, lines, outer,
                               stride, n, W, seg, NC);
        else
            hipLaunchKernelGGL(k_sep_pass<-1>, grid, dim3(64), lds, st, I, G, U, src, dst, V, v.X, lines, outer,
                               stride, n, W, seg, NC);
        first = false;
    };
    const int XY = v.X * v.Y;
    const double* S = sum_a;
    if (grid_ndim == 3) {
        pass(XY, v.X, XY, v.Z, nullptr, sum_a);
        pass((long long)v.X * (v.Z - W + 1), XY, v.X, v.Y, sum_a, sum_b);
        S = sum_b;
    } else {
        pass((long long)v.X * v.Z, XY, v.X, v.Y, nullptr, sum_a);
    }
    hipLaunchKernelGGL(k_sep_combine<KIND>, dim3(nb), dim3(256), 4 * NC * (size_t)(64 + 2 * r) * sizeof(double), st, S,
                       mean, cyy, v, r, grid_ndim == 3 ? 1 : 0, partials, wmap, mmap);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_sep(const FusedArgs& a, int grid_ndim, int src_ndim, int movi, int n_poses,
                      hipStream_t st) {
    const VGeom& v = a.v;
    const int nb = sep_blocks(v, a.r, grid_ndim);
    if (nb == 0 || n_poses <= 0) return hipSuccess;
    for (int pose = 0; pose < n_poses; ++pose) {
        FusedArgs b = a;
        b.mats = a.mats + (size_t)pose * a.mats_per_pose * 12;
        b.inline_mat = 0;
        // the moving image on the grid; its |Sobel| when it is the high-resolution image
        hipError_t e = launch_warp_moving(b, grid_ndim, src_ndim, a.sep_img, st);
        if (e != hipSuccess) return e;
        if (movi && (e = launch_sobel(a.sep_img, v, grid_ndim, a.sep_grad, st)) != hipSuccess) return e;
        double* part = a.partials + (size_t)pose * a.blocks_per_pose * 2;
        double *mean = const_cast<double*>(a.ustat_mean), *cyy = const_cast<double*>(a.ustat_cyy);  // read only
        e = movi ? sep_sums<kSepMovingImage>(a.sep_img, a.sep_grad, a.stat_img, a.sep_a, a.sep_b, v, a.r, grid_ndim,
                                             nb, mean, cyy, part, a.wmap, a.mmap, st)
                 : sep_sums<kSepMovingUs>(a.stat_img, a.stat_grad, a.sep_img, a.sep_a, a.sep_b, v, a.r, grid_ndim,
                                          nb, mean, cyy, part, a.wmap, a.mmap, st);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_warp_grid(const FusedArgs& a, int grid_ndim, int src_ndim, int movi, int n, hipStream_t st) {
    return grid_ndim == 3 ? launch_warp3(a, movi, n, st) : launch_warp2(a, src_ndim, n, st);
}

hipError_t launch_moments(const FusedArgs& a, int grid_ndim, int role, int n, hipStream_t st) {
    if (a.tiles == 0 || n <= 0) return hipSuccess;
    FusedArgs b = a;
    b.npose = n;
    return grid_ndim == 3 ? moments3(b, role, n, st, nullptr) : moments2(b, role, n, st, nullptr);
}

void moments_tiling(FusedArgs* a, int grid_ndim, int role) {
    const VGeom& v = a->v;
    if (grid_ndim == 3) {
        int tx, ty, blocks;
        a->tiles = fused_blocks_3d(v, a->r, a->zchunk, &a->ntx, &a->nty, &a->nzc);
        (void)fused_blocks_3d(v, a->r, kZBlock, &tx, &ty, &blocks);
        a->blocks_per_pose = tx * ty * blocks * moments3_waves(a->r, role);
        return;
    }
    // k_moments2d: a strip of columns and 32 rows per work-group, over a run of frames that depends
    // on the grid alone: about kStripGroups work-groups for one pose, and no more partial sums than
    // a 16x16 tile over kFrameRun frames each would give. One pose of 40 frames 256x200 with a matrix
    // each, r = 4: 152 us in runs of 16, 74 in runs of 3 (moving image), 119 and 64 (static); 128
    // frames 512x384, 5 poses: 2.15 ms for 512 to 2048 groups, 2.27 for 4096 (moving).
    constexpr long long kStripGroups = 2048;
    const int ex = v.X - 2 * a->r, ey = v.Y - 2 * a->r, w = strip_width_2d(a->r, role);
    a->ntx = ex > 0 && ey > 0 ? (ex + w - 1) / w : 0;
    a->nty = ex > 0 && ey > 0 ? (ey + 31) / 32 : 0;
    int tx, ty;
    (void)fused_blocks_2d(v, a->r, &tx, &ty);
    const long long per = std::max(1, a->ntx * a->nty);
    const long long most = (long long)tx * ty * ((v.Z + kFrameRun - 1) / kFrameRun);
    int run = (int)std::max(1LL, std::min<long long>(kFrameRun, per * v.Z / kStripGroups));
    while (run < kFrameRun && per * ((v.Z + run - 1) / run) > most) ++run;
    a->zchunk = std::min(v.Z, run);
    a->nzc = (v.Z + a->zchunk - 1) / a->zchunk;
    a->tiles = a->blocks_per_pose = a->ntx * a->nty * a->nzc;
}

hipError_t moments_resident_per_cu(const FusedArgs& a, int grid_ndim, int role, int* per_cu) {
    *per_cu = 0;
    return grid_ndim == 3 ? moments3(a, role, 1, nullptr, per_cu) : moments2(a, role, 1, nullptr, per_cu);
}

hipError_t launch_reduce(const double* partials, int blocks_per_pose, int n_poses, double* out,
                         hipStream_t st) {
    hipLaunchKernelGGL(k_reduce, dim3(n_poses), dim3(256), 0, st, partials, blocks_per_pose, out);
    return hipGetLastError();
}


hipError_t launch_warp_static(const void* fixed, int fixed_f16, const SGeom& fg, const VGeom& v,
                              int grid_ndim, int src_ndim, float* out, hipStream_t st) {
    const long long n = (long long)v.X * v.Y * v.Z;
    // A 2D grid over a 3D fixed "volume" of one slice (2D->3D) samples trilinearly with
    // Z = 1, which equals the bilinear per-frame path bit for bit.
    const int mode = (grid_ndim == 3) ? 0 : 1;
    (void)src_ndim;
    if (fixed_f16)
        hipLaunchKernelGGL(k_warp_static<__half>, grid_for(n), dim3(256), 0, st,
                           static_cast<const __half*>(fixed), fg, v, mode, out);
    else
        hipLaunchKernelGGL(k_warp_static<float>, grid_for(n), dim3(256), 0, st,
                           static_cast<const float*>(fixed), fg, v, mode, out);
    return hipGetLastError();
}

hipError_t launch_warp_moving(const FusedArgs& a, int grid_ndim, int src_ndim, float* out,
                              hipStream_t st) {
    const long long n = (long long)a.v.X * a.v.Y * a.v.Z;
    if (a.src_f16)
        hipLaunchKernelGGL(k_warp_moving<__half>, grid_for(n), dim3(256), 0, st, a,
                           grid_ndim == 3 ? 1 : 0, src_ndim == 3 ? 1 : 0, out);
    else
        hipLaunchKernelGGL(k_warp_moving<float>, grid_for(n), dim3(256), 0, st, a,
                           grid_ndim == 3 ? 1 : 0, src_ndim == 3 ? 1 : 0, out);
    return hipGetLastError();
}

hipError_t launch_ustats(const float* img, const VGeom& v, int grid_ndim, int r, double* mean,
                         double* cyy, double* sum_a, double* sum_b, hipStream_t st) {
    const long long n = (long long)v.X * v.Y * v.Z;
    const int nb = sep_blocks(v, r, grid_ndim);
    if (sum_a) {
        hipLaunchKernelGGL(k_ustats_none, grid_for(n), dim3(256), 0, st, n, mean, cyy);
        if (nb > 0)
            return sep_sums<kSepUsStats>(nullptr, nullptr, img, sum_a, sum_b, v, r, grid_ndim, nb, mean, cyy, nullptr,
                                         nullptr, nullptr, st);
    } else {
        hipLaunchKernelGGL(k_ustats, grid_for(n), dim3(256), 0, st, img, v, grid_ndim == 3 ? 1 : 0, r, mean, cyy);
    }
    return hipGetLastError();
}

hipError_t launch_sobel(const float* img, const VGeom& v, int grid_ndim, float* out,
                        hipStream_t st) {
    const long long n = (long long)v.X * v.Y * v.Z;
    hipLaunchKernelGGL(k_sobel, grid_for(n), dim3(256), 0, st, img, v, grid_ndim == 3 ? 1 : 0,
                       out);
    return hipGetLastError();
}

// The scratch array of lc2e_eval_batch_noalloc. In host code its name is only a stand-in
// for the symbol: kernels get the device address that scratch_address() looks up.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

hipError_t scratch_address(int device, void** out) {
    static std::mutex mu;
    static std::map<int, void*> addr;  // device -> address of its copy of the array
    std::lock_guard<std::mutex> lk(mu);
    auto it = addr.find(device);
    if (it != addr.end()) {
        *out = it->second;
        return hipSuccess;
    }
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return e;
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (cur != device) (void)hipSetDevice(cur);
    if (e != hipSuccess) return e;
    if (!ptr) return hipErrorInvalidSymbol;
    addr[device] = ptr;
    *out = ptr;
    return hipSuccess;
}

hipError_t launch_check(const void* d_in, int in_dtype, long long n, float lim, int* flag, hipStream_t st) {
    if (in_dtype == 0) return hipSuccess;  // bytes are always in range
    const long long blocks = std::min<long long>((n / 4 + 255) / 256 + 1, 2048);
    hipLaunchKernelGGL(k_check, dim3((unsigned)blocks), dim3(256), 0, st, d_in, in_dtype, n, lim, flag);
    return hipGetLastError();
}

hipError_t launch_convert(const void* d_in, int in_dtype, void* d_out, int out_f16, long long n,
                          hipStream_t st) {
    hipLaunchKernelGGL(k_convert, grid_for(n), dim3(256), 0, st, d_in, in_dtype, d_out, out_f16, n);
    return hipGetLastError();
}

}  // namespace lc2e
