// The fused 2D kernel of small patches with the moving image as the high-resolution one.
#include <algorithm>
#include <mutex>

#include "lc2e_device.hpp"

namespace lc2e {

namespace {

constexpr int kTile2X = 16;    // output tile: kTile2X x kTile2Y, one thread per output
constexpr int kTile2Y = 16;
constexpr int kThreads = kTile2X * kTile2Y;

// The 2D kernel's 16-wide tiles: odd strides. Its x pass has one run of 16 per row, and
// there odd strides give 1.5% more throughput than 2 (mod 4), by measurement.
__host__ __device__ constexpr int lds_stride_2d(int n) { return n | 1; }

// Row of output oy of the in-place box sums (box_xy_inplace) in the products planes.
__host__ __device__ constexpr int box_row(int oy, int w) { return oy < 8 ? oy : oy + w - 1; }

// Box sums in place (the 2D kernel), for 16x16 outputs: the x pass writes each row's 16
// outputs over the start of that row of s_prod, and the y pass writes each column run's 8
// outputs over rows that no other run reads: run 0 over rows 0..7, run 1 over rows
// W+7 .. W+14 (the last 8 of its own input rows). A task reads each of its inputs before it
// overwrites it, so output (ox, oy) of channel c ends up at
// s_prod[c * ps * py + box_row(oy, W) * ps + ox] with no second buffer: the LDS of the x
// pass's output and of the sums is saved, which lets more work-groups share a CU.
template <int NC, int NTHR, int W>
__device__ __forceinline__ void box_xy_inplace(double* s_prod, int ps, int py, int tid) {
    const int np = ps * py;
    __builtin_amdgcn_s_setprio(2);
    for (int t = tid; t < NC * py; t += NTHR) {
        const int row = t % py, c = t / py;
        double* r = s_prod + c * np + row * ps;
        window_run<W>(r, 1, r, 1);
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
    __builtin_amdgcn_s_setprio(2);
    for (int t = tid; t < NC * 16 * 2; t += NTHR) {
        const int col = t % 16, rest = t / 16;
        const int seg = rest % 2, c = rest / 2;
        const int in_ofs = seg * 8 * ps + col, out_ofs = box_row(seg * 8, W) * ps + col;
        window_run<W, double, 8>(s_prod + c * np + in_ofs, ps, s_prod + c * np + out_ofs, ps);
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
}

// box_xy_inplace for a patch radius known only at run time, 1 <= r <= RMAX.
template <int NC, int NTHR, int RMAX, int RR = 1>
__device__ __forceinline__ void box_xy_inplace_r(int r, double* s_prod, int tid) {
    if (r == RR)
        box_xy_inplace<NC, NTHR, 2 * RR + 1>(s_prod, lds_stride_2d(16 + 2 * RR), 16 + 2 * RR, tid);
    else if constexpr (RR < RMAX)
        box_xy_inplace_r<NC, NTHR, RMAX, RR + 1>(r, s_prod, tid);
}

// ---------------------------------------------------------------------------
// 2D fused kernel for a moving high-resolution image at small radii (r <= kMaxRFused2; from r = 4
// on its 16x16 tiles' halos make k_moments2d the faster one: 128 frames 512x384, 3 poses, r = 4
// 2.02 -> 1.68 ms, r = 6 2.28 -> 1.59 ms; at r = 3 this kernel takes 4.45 ms for 13 poses, that
// one 4.9 in place and 6.4 through the grid): one 16x16 output tile of a run of `zchunk`
// (kFrameRun) consecutive frames of one pose (a single image is one frame). Dynamic LDS sized for
// the runtime patch radius. Frame f + 1's gathers (and its static image values and ultrasound statistics)
// are issued while frame f's box sums and combine run, as in the 3D kernel's z-steps. Each
// thread adds its pixel's measure and weight over the run's frames in frame order, and the
// work-group reduces them once into the partial of (run, tile). The run length does not
// depend on the batch, so neither do the results.
// ---------------------------------------------------------------------------
template <bool SRC3D, typename T, bool P2>
// at most 128 VGPRs, four work-groups per CU (the f32-source variant would take 129 and drop
// to three)
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_fused2d(FusedArgs a) {
    extern __shared__ double s_dyn[];
    static_assert(kTile2X == 16 && kTile2Y == 16, "box_xy_inplace sums 16x16 tiles");
    constexpr int NC = 7, RMAX = kMaxRFused2;
    // per-thread gathers / products positions at the largest radius of this variant
    // (r <= RMAX): the pipelined gathers are held in registers
    constexpr int SPT = ((kTile2X + 2 * RMAX + 2) * (kTile2Y + 2 * RMAX + 2) + kThreads - 1) / kThreads;
    constexpr int PPT = ((kTile2X + 2 * RMAX) * (kTile2Y + 2 * RMAX) + kThreads - 1) / kThreads;
    const int R = a.r, W = 2 * R + 1, PX = kTile2X + 2 * R, PY = kTile2Y + 2 * R;
    const int IXE = PX + 2, IYE = PY + 2;
    // warped rows 32 + PX/2 floats apart in LDS, so the paired Sobel reads of a wave
    // (PX lanes per row group, groups two rows apart) fall into distinct banks
    const int SIS = 32 + PX / 2;
    const int PS = lds_stride_2d(PX);                         // products row stride
    const int wex = IXE;                         // warped region edge
    const int wofs = R + 1;                       // it starts at x0 - wofs
    const int NI = IXE * IYE;
    // The box sums run in place in the products planes (box_xy_inplace).
    double* s_prod = s_dyn;                                   // NC*PY*PS
    double* s_red = s_prod + NC * PY * PS;                    // 8
    float* s_in = reinterpret_cast<float*>(s_red + 8);        // NI

    // A work-group takes one tile of either a run of frames of one pose (frame stacks, 3D
    // sources) or, with a.prun > 1 (single images of a 2D source), a run of a.prun poses:
    // their gathers pipeline like a run's frames, and the tile's static values are loaded
    // once. Each pose still gets one partial per tile, so the results do not depend on the
    // run length. (With a 3D source prun is the constant 1: the frame stacks' code is not
    // touched by the pose runs.)
    const int prun = (!SRC3D && a.prun > 1) ? a.prun : 1;
    int tile, prun_idx;
    if (!map_block(a.tiles, (a.npose + prun - 1) / prun, tile, prun_idx)) return;  // whole work-group
    const int p0 = prun_idx * prun, p1 = min(p0 + prun, a.npose);
    const int tid = threadIdx.x;
    const int cols = a.ntx * a.nty;
    const int tcol = tile % cols, run = tile / cols;
    const int f0 = run * a.zchunk, f1 = min(f0 + a.zchunk, a.v.Z);
    const int nit = prun > 1 ? p1 - p0 : f1 - f0;  // iterations: poses or frames
    const int tx = tcol % a.ntx, ty = tcol / a.ntx;
    const int x0 = R + tx * kTile2X, y0 = R + ty * kTile2Y;
    const int X = a.v.X, Y = a.v.Y;
    const float lz = a.v.oz;
    const T* __restrict__ src = static_cast<const T*>(a.src);

    // Per-thread positions, the same for every frame (the radius is a run-time value, so
    // the divisions are done once here, not per frame): virtual-grid coordinates of the
    // warped positions, and the LDS / image offsets of the products positions.
    float gLx[SPT], gLy[SPT];
    int g_sin[SPT];     // LDS offset of warped position j in s_in
    unsigned g_in = 0;  // bit j: warped position j lies in the grid
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
        const int i = tid + j * kThreads;
        const int lx = i % wex, ly = i / wex;
        g_sin[j] = ly * SIS + lx;
        const int gx = x0 - wofs + lx, gy = y0 - wofs + ly;
        if (i < NI && gx >= 0 && gx < X && gy >= 0 && gy < Y) g_in |= 1u << j;
        gLx[j] = fmaf((float)gx, a.v.sx, a.v.ox);
        gLy[j] = fmaf((float)gy, a.v.sy, a.v.oy);
    }
    // Slots 2k and 2k + 1 are the vertically adjacent products positions (lx, ly0)
    // and (lx, ly0 + 1), ly0 even, of pair t = tid + k * kThreads: their 3x3 Sobel
    // neighbourhoods share two rows, so 4 rows are read and smoothed instead of 6, with the
    // same operations per position. (PPT is even at every RMAX; PY = 16 + 2R is even.)
    static_assert(PPT % 2 == 0, "products slots come in pairs");
    const int NPAIR = PX * (PY / 2);
    int p_in_ofs[PPT], p_prod_ofs[PPT], p_img_ofs[PPT];  // s_in, s_prod, image (frame 0)
    unsigned p_in = 0;  // bit j: products position j holds an image value
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        const int t = tid + (j >> 1) * kThreads;
        
        const int lx = t % PX;
        const int ly = 2 * (t / PX) + (j & 1);
        const int gx = x0 - R + lx, gy = y0 - R + ly;
        if (t < NPAIR && gx < X && gy < Y) p_in |= 1u << j;
        p_in_ofs[j] = ly * SIS + lx;
        p_prod_ofs[j] = ly * PS + lx;
        p_img_ofs[j] = gy * X + gx;
    }

    using Pend = typename std::conditional<SRC3D, Pending3<T>, Pending2<T>>::type;
    Pend pend[SPT];
    // (No wave-uniform skip of empty slots here, unlike the 3D kernel: in this kernel it
    // cost 6% on the tracked sweep, 29.09 -> 30.93 ms per launch, measured.)
    // the matrix of iteration it: pose p0 + it (pose runs) or frame f0 + it of pose p0
    auto issue_frame = [&](int it) {
        float m[12];
        const float* mp = prun > 1 ? a.mats + (size_t)(p0 + it) * a.mats_per_pose * 12
                                   : a.mats + ((size_t)p0 * a.mats_per_pose +
                                               (a.mats_per_pose > 1 ? f0 + it : 0)) * 12;
#pragma unroll
        for (int k = 0; k < 12; ++k) m[k] = mp[k];
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            if (j * kThreads >= NI) break;  // uniform
            const bool inside = (g_in >> j) & 1u;
            if constexpr (SRC3D) issue3<P2>(src, a.s, m, gLx[j], gLy[j], lz, inside, pend[j]);
            else issue2<P2>(src, a.s, m, gLx[j], gLy[j], inside, pend[j]);
        }
    };
    // ultrasound of the products positions
    float pre0[PPT];
    auto issue_static = [&](int frame) {
        const int plane = frame * X * Y;
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            // uniform: slot j holds pair j / 2
            if ((j >> 1) * kThreads >= NPAIR) break;
            const bool in = (p_in >> j) & 1u;
            const int vidx = plane + p_img_ofs[j];
            pre0[j] = in ? a.stat_img[vidx] : 0.0f;
        }
    };
    // static ultrasound statistics of this thread's output pixel
    const int ox = tid % kTile2X, oy = tid / kTile2X;
    const bool out_ok = (x0 + ox < X - R) && (y0 + oy < Y - R);
    double mu_pre = 0.0, cyy_pre = -1.0;
    auto issue_stats = [&](int frame) {
        if (out_ok) {
            const int vo = frame * X * Y + (y0 + oy) * X + (x0 + ox);
            mu_pre = a.ustat_mean[vo];
            cyy_pre = a.ustat_cyy[vo];
        }
    };

    double acc_m = 0.0, acc_w = 0.0;
    issue_frame(0);
    issue_static(f0);
    issue_stats(f0);
    for (int it = 0; it < nit; ++it) {
        const int f = prun > 1 ? f0 : f0 + it;  // frame of this iteration
        // 1. the warped tile of iteration it (raised wave priority, as in the 3D kernel)
        __builtin_amdgcn_s_setprio(2);
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            if (j * kThreads >= NI) break;  // uniform
            const int i = tid + j * kThreads;
            float v;
            if constexpr (SRC3D) v = finish3(pend[j]);
            else v = finish2(pend[j]);
            if (i < NI) s_in[g_sin[j]] = v;
        }
        __builtin_amdgcn_s_setprio(0);
        float cur0[PPT];
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            cur0[j] = pre0[j];
        }
        const double mu = mu_pre, cyy = cyy_pre;
        if (prun == 1 && f + 1 < f1) {  // the next frame's static values (pose runs: the same)
            issue_static(f + 1);
            issue_stats(f + 1);
        }
        __syncthreads();
        // 2. |Sobel| and the products
#pragma unroll
        for (int jp = 0; jp < PPT / 2; ++jp) {
            if (jp * kThreads >= NPAIR) break;  // uniform
            if (tid + jp * kThreads < NPAIR) {
                // 3x3 Sobel read from the warped tile: rows ly0 .. ly0 + 3, smooth
                // s = (l + 2c) + r and difference d = r - l along x
                float sv[4], dv[4], cv[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float* row = s_in + p_in_ofs[2 * jp] + k * SIS;
                    const float l = row[0], c = row[1], r = row[2];
                    dv[k] = r - l;
                    sv[k] = (l + 2.0f * c) + r;
                    cv[k] = c;
                }
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float gxv = (dv[e] + 2.0f * dv[e + 1]) + dv[e + 2];
                    const float gyv = sv[e + 2] - sv[e];
                    const float G = sqrtf(fmaf(gyv, gyv, gxv * gxv));
                    store_products<NC>(s_prod, nullptr, PY * PS, p_prod_ofs[2 * jp + e],
                                       cv[e + 1], G, cur0[2 * jp + e]);
                }
            }
        }
        __syncthreads();  // s_in reads done; products visible
        // the next iteration's gathers fly during the box sums and the combine
        if (it + 1 < nit) issue_frame(it + 1);
        // 3. box sums
        box_xy_inplace_r<NC, kThreads, RMAX>(R, s_prod, tid);
        // 4. combine; each thread adds its pixel's values over the run's frames in order
        if (out_ok) {
            const int so = box_row(oy, W) * PS + ox;  // this pixel's sums
            double S[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) S[c] = s_prod[c * PY * PS + so];
            double w, meas;
            const bool ok = combine_static_u(S, mu, cyy, W * W, w, meas);
            if (ok) {
                acc_m += meas;
                acc_w += w;
                if (a.wmap) {
                    const int vo = f * X * Y + (y0 + oy) * X + (x0 + ox);
                    a.wmap[vo] = w;
                    a.mmap[vo] = meas;
                }
            }
        }
        if (prun > 1) {  // block-uniform: this pose's partial of the tile
            double* dst = a.partials + ((size_t)(p0 + it) * a.blocks_per_pose + (size_t)run * cols + tcol) * 2;
            block_reduce_store<kThreads>(acc_m, acc_w, s_red, dst);
            acc_m = 0.0;
            acc_w = 0.0;
        }
    }
    if (prun == 1) {
        double* dst = a.partials + ((size_t)p0 * a.blocks_per_pose + (size_t)run * cols + tcol) * 2;
        block_reduce_store<kThreads>(acc_m, acc_w, s_red, dst);
    }
}

// The dynamic LDS layout of k_fused2d: 7 FP64 products planes, the reduction scratch and the
// warped tile.
constexpr size_t lds_bytes_2d(int r) {
    const size_t PX = kTile2X + 2 * r, PY = kTile2Y + 2 * r, IYE = PY + 2, PS = lds_stride_2d((int)PX);
    return sizeof(double) * (7 * PY * PS + 8) + sizeof(float) * (32 + PX / 2) * IYE;
}
static_assert(lds_bytes_2d(kMaxRFused2) <= 160 * 1024, "2D fused kernel exceeds the 160 KiB of LDS");

template <bool SRC3D, typename T, bool P2>
hipError_t launch2(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    const size_t lds = lds_bytes_2d(a.r);
    if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, k_fused2d<SRC3D, T, P2>, kThreads, lds);
    hipLaunchKernelGGL((k_fused2d<SRC3D, T, P2>), grid, dim3(kThreads), lds, st, a);
    return hipGetLastError();
}
template <typename T, bool P2>
hipError_t launch2t(const FusedArgs& a, int src_ndim, dim3 grid, hipStream_t st, int* occ) {
    return src_ndim == 3 ? launch2<true, T, P2>(a, grid, st, occ) : launch2<false, T, P2>(a, grid, st, occ);
}
hipError_t launch2d(const FusedArgs& a, int src_ndim, dim3 grid, hipStream_t st, int* occ) {
    if (a.s.pow2)
        return a.src_f16 ? launch2t<__half, true>(a, src_ndim, grid, st, occ)
                         : launch2t<float, true>(a, src_ndim, grid, st, occ);
    return a.src_f16 ? launch2t<__half, false>(a, src_ndim, grid, st, occ)
                     : launch2t<float, false>(a, src_ndim, grid, st, occ);
}

}  // namespace

int fused_blocks_2d(const VGeom& v, int r, int* ntx, int* nty) {
    const int ex = v.X - 2 * r, ey = v.Y - 2 * r;
    if (ex <= 0 || ey <= 0) { *ntx = *nty = 0; return 0; }
    *ntx = (ex + kTile2X - 1) / kTile2X;
    *nty = (ey + kTile2Y - 1) / kTile2Y;
    return *ntx * *nty * v.Z;
}

int pose_run(const VGeom& v, int src_ndim, int mats_per_pose, int tiles, int n_poses) {
    // runs of poses per work-group while at least about two work-groups per CU slot remain
    constexpr int kMaxPoseRun = 8;
    constexpr long long kPoseRunWGs = 2048;
    if (src_ndim != 2 || v.Z != 1 || mats_per_pose != 1) return 1;
    const long long tiles8 = (tiles + kXcds - 1) / kXcds * (long long)kXcds;
    return (int)std::max(1LL, std::min<long long>(kMaxPoseRun, tiles8 * n_poses / kPoseRunWGs));
}

hipError_t launch_fused2(const FusedArgs& a, int src_ndim, int n_poses, hipStream_t st) {
    if (a.tiles == 0 || n_poses <= 0) return hipSuccess;
    if (a.zchunk <= 0 || a.r < 1 || a.r > kMaxRFused2) return hipErrorInvalidValue;
    FusedArgs b = a;
    b.npose = n_poses;
    const long long tiles8 = (a.tiles + kXcds - 1) / kXcds * (long long)kXcds;
    b.prun = pose_run(a.v, src_ndim, a.mats_per_pose, a.tiles, n_poses);
    const long long runs = (n_poses + b.prun - 1) / b.prun;
    if (tiles8 * runs > 0x7fffffffLL) return hipErrorInvalidValue;
    return launch2d(b, src_ndim, dim3((unsigned)(tiles8 * runs)), st, nullptr);
}

hipError_t fused2_resident_per_cu(const FusedArgs& a, int src_ndim, int* per_cu) {
    *per_cu = 0;
    return launch2d(a, src_ndim, dim3(1), nullptr, per_cu);
}

}  // namespace lc2e
