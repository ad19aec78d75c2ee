// Normalized mutual information (the patchSize 0 metric).
#include <algorithm>

#include "lc2e_device.hpp"

namespace lc2e {

namespace {

// ---------------------------------------------------------------------------
// Normalized mutual information, the reference's patchSize == 0 metric
// (GetMutualInformationSimilarityMetric, cu_lc2_3d.cu:1196-1301; histogram kernels
// :868-923): NMI = (H_U + H_I) / H_joint over the whole virtual grid, with bins spread
// between each image's minimum and maximum.
// ---------------------------------------------------------------------------

// Floats as ints whose signed order is the float order (for atomic min / max).
__device__ __forceinline__ int ford(float f) {
    const int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ float fdec(int i) { return __int_as_float(i >= 0 ? i : i ^ 0x7fffffff); }

// The moving image warped at virtual voxel i of pose `pose` (as k_warp_moving).
template <typename T>
__device__ __forceinline__ float warped_at(const FusedArgs& a, int grid3, int src3, int pose,
                                           long long i) {
    const VGeom& v = a.v;
    const int x = (int)(i % v.X), y = (int)((i / v.X) % v.Y), z = (int)(i / ((long long)v.X * v.Y));
    const float* mp = a.mats + ((size_t)pose * a.mats_per_pose +
                                (grid3 ? 0 : (a.mats_per_pose > 1 ? z : 0))) * 12;
    float m[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) m[k] = mp[k];
    const float lx = fmaf((float)x, v.sx, v.ox), ly = fmaf((float)y, v.sy, v.oy);
    const float lz = grid3 ? fmaf((float)z, v.sz, v.oz) : v.oz;
    const T* src = static_cast<const T*>(a.src);
    if (src3) return sample3(src, a.s, m, lx, ly, lz);
    return sample2(src, a.s, m, lx, ly);
}

template <int NTHR>
__device__ __forceinline__ void block_minmax(float mn, float mx, int* s_red, int* dst) {
    for (int off = 32; off > 0; off >>= 1) {
        mn = fminf(mn, __shfl_down(mn, off, 64));
        mx = fmaxf(mx, __shfl_down(mx, off, 64));
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        s_red[2 * wid] = ford(mn);
        s_red[2 * wid + 1] = ford(mx);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int a = s_red[0], b = s_red[1];
        for (int w = 1; w < NTHR / 64; ++w) {
            a = min(a, s_red[2 * w]);
            b = max(b, s_red[2 * w + 1]);
        }
        atomicMin(&dst[0], a);
        atomicMax(&dst[1], b);
    }
}

// Extremes of the warped moving image per pose (blockIdx.y): ext[pose] = {min, max}.
template <typename T>
__global__ __launch_bounds__(256) void k_mi_extrema(FusedArgs a, int grid3, int src3, int* ext) {
    __shared__ int s_red[8];
    const int pose = blockIdx.y;
    const long long n = (long long)a.v.X * a.v.Y * a.v.Z;
    float mn = INFINITY, mx = -INFINITY;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const float v = warped_at<T>(a, grid3, src3, pose, i);
        mn = fminf(mn, v);
        mx = fmaxf(mx, v);
    }
    block_minmax<256>(mn, mx, s_red, ext + 2 * pose);
}

// Extremes of a resident image.
__global__ __launch_bounds__(256) void k_mi_extrema_img(const float* img, long long n, int* ext) {
    __shared__ int s_red[8];
    float mn = INFINITY, mx = -INFINITY;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        mn = fminf(mn, img[i]);
        mx = fmaxf(mx, img[i]);
    }
    block_minmax<256>(mn, mx, s_red, ext);
}

__global__ void k_mi_init(int* ext, int n_pairs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_pairs) {
        ext[2 * i] = 0x7fffffff;
        ext[2 * i + 1] = (int)0x80000000;
    }
}

// The moving image warped onto a 3D grid (a.warp1, a float per voxel and pose) and its extremes
// per pose. A thread marches along z with the next planes' gathers in flight; bound by VALU
// issue and the gathers' addresses like k_warp_us3. 8 poses of 192x192x160: 130 us, where the
// extremes alone took 255 us with one sample at a time and the histogram warped everything again.
template <typename T, bool P2>
__global__ __launch_bounds__(256) void k_mi_warp3(FusedArgs a, int ntx, int nty, int zc, int tiles, int npose,
                                                  int* ext) {
    __shared__ int s_red[8];
    int tile, pose;
    if (!map_block(tiles, npose, tile, pose)) return;  // whole work-group
    const int tcol = tile % (ntx * nty), zci = tile / (ntx * nty);
    const int gx = (tcol % ntx) * 64 + (threadIdx.x & 63), gy = (tcol / ntx) * 4 + (threadIdx.x >> 6);
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z;
    const int z0 = zci * zc, z1 = min(z0 + zc, Z);
    float mn = INFINITY, mx = -INFINITY;
    if (gx < X && gy < Y) {
        const T* __restrict__ src = static_cast<const T*>(a.src);
        float m[12];
        load_matrix(a, pose, m);
        const float Lx = fmaf((float)gx, a.v.sx, a.v.ox), Ly = fmaf((float)gy, a.v.sy, a.v.oy);
        const float c[3] = {fmaf(m[1], Ly, m[0] * Lx), fmaf(m[5], Ly, m[4] * Lx), fmaf(m[9], Ly, m[8] * Lx)};
        float* out = a.warp1 + (size_t)pose * X * Y * Z + (size_t)gy * X + gx;
        Pending3<T> p[2];
        auto issue = [&](int z, Pending3<T>& q) { issue3c<P2>(src, a.s, m, c, fmaf((float)z, a.v.sz, a.v.oz), true, q); };
        issue(z0, p[0]);
        issue(min(z0 + 1, z1 - 1), p[1]);
        for (int z = z0; z < z1; z += 2) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float v = finish3(p[e]);  // past the chunk: its last plane again
                mn = fminf(mn, v);
                mx = fmaxf(mx, v);
                if (z + e < z1) out[(size_t)(z + e) * X * Y] = v;
                issue(min(z + e + 2, z1 - 1), p[e]);
            }
        }
    }
    block_minmax<256>(mn, mx, s_red, ext + 2 * pose);
}

// cu_lc2_3d.cu:882-887: bin of v; the scaling is formed in double as there, roundf() rounds its
// float conversion. The single-precision quotient is off by less than 5e-5 (bins <= 256), so
// where it is further than 1e-4 from a half it has the same bin; the others (and quotients
// out of the range where that holds) go through the double arithmetic.
struct MiBin {
    float mn, k;  // k: bins per grey value, NaN where only the double arithmetic will do
    double scale, d;
    int bins;
    __device__ MiBin(float lo, float hi, int n) : mn(lo), scale(n - 1.0), d((double)(hi - lo)), bins(n) {
        k = (float)(scale / d);
        if (!(k > 1e-30f && k < 1e30f)) k = NAN;
    }
    // the bin; 0 without a quotient (a constant image), -1 beyond the histogram
    __device__ __forceinline__ int operator()(float v) const {
        const float h = fmaf(v - mn, k, 0.5f);
        const float fr = __builtin_amdgcn_fractf(h);
        if (fr > 1e-4f && fr < 1.0f - 1e-4f) return (int)h;
        const float f = (float)((double)(v - mn) * scale / d);
        const int b = f == f ? (int)roundf(f) : 0;
        return b >= 0 && b < bins ? b : -1;
    }
};

// Joint histogram [pose][bin_i][bin_u] of (U, I) over a chunk of voxels per work-group:
// privatised in LDS as 16-bit counters packed two to a word (128 KiB for 256 x 256 bins), then
// the non-zero bins are added to the pose's histogram. Every kMiSweep voxels the counters of
// 32768 and above are emptied, so a chunk may be as long as the chip's share of the work. A
// wave whose voxels all fall into one bin (the background) adds them at once.
// Bound by the LDS atomics and VALU issue (a voxel took 20 FP64 operations; its 2 loads take 80 us
// of 8 poses of 192x192x160 at the copy rate). Measured there: 699 us while it warped each
// voxel again, 190 with chunks of 65535 voxels and FP64 bins, now 129.
// U: voxels per thread and step, the next step's in flight. WAVES: per SIMD.
constexpr int kMiVox = 4096;  // of four voxels per thread
constexpr int kMiSweep = 7 * kMiVox;  // + 32767 < 65536
template <typename T, int U, int WAVES>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(WAVES)))
void k_mi_joint(FusedArgs a, int grid3, int src3, const float* stat,
                                                   int stat_is_u, const int* ext_mov, const int* ext_stat,
                                                   int bins_u, int bins_i, long long chunk, int stride,
                                                   unsigned* hist) {
    extern __shared__ unsigned s_h[];
    const int pose = blockIdx.y;
    const int nb = bins_u * bins_i, nw = (nb + 1) / 2;
    for (int w = threadIdx.x; w < nw; w += 1024) s_h[w] = 0u;
    const float mnm = fdec(ext_mov[2 * pose]), mxm = fdec(ext_mov[2 * pose + 1]);
    const float mns = fdec(ext_stat[0]), mxs = fdec(ext_stat[1]);
    const MiBin bin_m(mnm, mxm, stat_is_u ? bins_i : bins_u), bin_s(mns, mxs, stat_is_u ? bins_u : bins_i);
    const int step_m = stat_is_u ? bins_u : 1, step_s = stat_is_u ? 1 : bins_u;
    unsigned* h = hist + (size_t)pose * stride;
    __syncthreads();
    const long long n = (long long)a.v.X * a.v.Y * a.v.Z;
    const long long i0 = (long long)blockIdx.x * chunk;
    const long long len = min(chunk, n - i0);
    const float* wm = a.warp1 ? a.warp1 + (size_t)pose * n + i0 : nullptr;
    const float* ws = stat + i0;
    constexpr int VOX = U * 1024;  // per step
    float vm[U], vs[U];
    auto load = [&](long long k0) {
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const long long i = min(k0 + threadIdx.x + k * 1024, len - 1);
            vm[k] = wm ? wm[i] : warped_at<T>(a, grid3, src3, pose, i0 + i);
            vs[k] = ws[i];
        }
    };
    load(0);
    int since = 0;
    for (long long k0 = 0; k0 < len; k0 += VOX) {
        float cm[U], cs[U];
#pragma unroll
        for (int k = 0; k < U; ++k) cm[k] = vm[k], cs[k] = vs[k];
        if (k0 + VOX < len) load(k0 + VOX);
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int bm = bin_m(cm[k]), bs = bin_s(cs[k]);
            const bool in = k0 + threadIdx.x + k * 1024 < len && bm >= 0 && bs >= 0;
            const int j = in ? step_m * bm + step_s * bs : -1;
            const int j0 = __builtin_amdgcn_readfirstlane(j);
            if (__all(j == j0)) {
                if (j0 >= 0 && (threadIdx.x & 63) == 0) atomicAdd(&s_h[j0 >> 1], 64u << ((j0 & 1) * 16));
            } else if (j >= 0) {
                atomicAdd(&s_h[j >> 1], (j & 1) ? 65536u : 1u);
            }
        }
        since += VOX;
        if (since == kMiSweep) {  // work-group uniform
            since = 0;
            __syncthreads();
            for (int w = threadIdx.x; w < nw; w += 1024) {
                const unsigned c = s_h[w];
                if (c & 0x80008000u) {
                    if (c & 0x8000u) atomicAdd(&h[2 * w], c & 0xffffu);
                    if (c >> 31) atomicAdd(&h[2 * w + 1], c >> 16);
                    s_h[w] = ((c & 0x8000u) ? 0u : c & 0xffffu) | ((c >> 31) ? 0u : c & 0xffff0000u);
                }
            }
            __syncthreads();
        }
    }
    __syncthreads();
    for (int w = threadIdx.x; w < nw; w += 1024) {
        const unsigned c = s_h[w];
        if (c & 0xffffu) atomicAdd(&h[2 * w], c & 0xffffu);
        if ((c >> 16) && 2 * w + 1 < nb) atomicAdd(&h[2 * w + 1], c >> 16);
    }
}

__device__ __forceinline__ double neg_plogp(unsigned long long c, double n) {
    if (!c) return 0.0;
    const double p = c / n;
    return -(p * log(p));
}

// Entropies in FP64 from the joint histogram (its marginals are the single-image histograms:
// every finite value falls into a bin). First kernel, blockIdx = (group of 4 bins of I, the last
// group with the remainder; pose): the group's part of the joint and of the I entropy and its
// marginal counts of U, left in place of the group's counts: bins_u counts, then two doubles.
// Second, one work-group per pose: their sums in a fixed order and NMI; 0 when an image is
// constant. (One work-group per pose for everything took 181 us, mostly in the column sums.)
constexpr int kMiRows = 4;
__device__ __forceinline__ int mi_groups(int bins_i) { return max(1, bins_i / kMiRows); }

__global__ __launch_bounds__(256) void k_mi_entropy_part(unsigned* hist, int stride, int bins_u, int bins_i, double n) {
    __shared__ double s_j[4];
    __shared__ unsigned s_r[2 * kMiRows][4];
    const int g = blockIdx.x, u = threadIdx.x, lane = u & 63, wave = u >> 6;
    unsigned* h = hist + (size_t)blockIdx.y * stride + g * kMiRows * bins_u;
    const int rows = g + 1 == mi_groups(bins_i) ? bins_i - g * kMiRows : kMiRows;  // < 2 kMiRows
    double hj = 0.0;
    unsigned col = 0;
    for (int k = 0; k < rows; ++k) {
        unsigned c = u < bins_u ? h[u + bins_u * k] : 0u;
        hj += neg_plogp(c, n);
        col += c;
        for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
        if (lane == 0) s_r[k][wave] = c;
    }
    for (int o = 32; o > 0; o >>= 1) hj += __shfl_down(hj, o, 64);
    if (lane == 0) s_j[wave] = hj;
    __syncthreads();
    if (u < bins_u) h[u] = col;
    if (u == 0) {
        double hi = 0.0;
        for (int k = 0; k < rows; ++k)
            hi += neg_plogp((unsigned long long)s_r[k][0] + s_r[k][1] + s_r[k][2] + s_r[k][3], n);
        hj = ((s_j[0] + s_j[1]) + s_j[2]) + s_j[3];
        h[bins_u] = __double2loint(hj);
        h[bins_u + 1] = __double2hiint(hj);
        h[bins_u + 2] = __double2loint(hi);
        h[bins_u + 3] = __double2hiint(hi);
    }
}

__global__ __launch_bounds__(1024) void k_mi_entropy(const unsigned* hist, int stride, const int* ext_mov,
                                                     const int* ext_stat, int bins_u, int bins_i, double n,
                                                     double* out) {
    __shared__ unsigned long long s_c[1024];
    __shared__ double s_red[3][256];
    const int pose = blockIdx.x, t = threadIdx.x, u = t & 255, groups = mi_groups(bins_i);
    const unsigned* h = hist + (size_t)pose * stride;
    unsigned long long c = 0;
    if (u < bins_u)
#pragma unroll
        for (int k = 0; k < kMiMaxBins / kMiRows / 4; ++k) {  // all in flight
            const int g = (t >> 8) + 4 * k;
            c += g < groups ? h[g * kMiRows * bins_u + u] : 0u;
        }
    s_c[t] = c;
    double hj = 0.0, hi = 0.0;
    if (t < groups) {
        const unsigned* q = h + t * kMiRows * bins_u + bins_u;
        hj = __hiloint2double(q[1], q[0]);
        hi = __hiloint2double(q[3], q[2]);
    }
    __syncthreads();
    if (t < 256) {
        s_red[0][t] = hj;
        s_red[1][t] = neg_plogp((s_c[t] + s_c[t + 256]) + (s_c[t + 512] + s_c[t + 768]), n);
        s_red[2][t] = hi;
    }
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (t < k)
            for (int q = 0; q < 3; ++q) s_red[q][t] += s_red[q][t + k];
        __syncthreads();
    }
    if (t == 0) {
        const bool flat = !(fdec(ext_mov[2 * pose + 1]) > fdec(ext_mov[2 * pose])) ||
                          !(fdec(ext_stat[1]) > fdec(ext_stat[0]));
        const double HJ = s_red[0][0], HU = s_red[1][0], HI = s_red[2][0];
        out[pose] = (flat || !(HJ > 0.0)) ? 0.0 : (HU + HI) / HJ;
    }
}

template <typename T, bool P2>
void mi_warp3(const FusedArgs& a, int n, int* ext, hipStream_t st) {
    const int ntx = (a.v.X + 63) / 64, nty = (a.v.Y + 3) / 4;
    const int want = (int)std::max(1LL, 2048LL / ((long long)ntx * nty * n));  // as launch_warp3
    const int zc = std::max(8, (a.v.Z + want - 1) / want);
    const int tiles = ntx * nty * ((a.v.Z + zc - 1) / zc);
    const int tiles8 = (tiles + kXcds - 1) / kXcds * kXcds;
    hipLaunchKernelGGL((k_mi_warp3<T, P2>), dim3((unsigned)tiles8 * n), dim3(256), 0, st, a, ntx, nty, zc, tiles, n,
                       ext);
}

}  // namespace

hipError_t launch_mi(const FusedArgs& a, int grid_ndim, int src_ndim, int movi, int n_poses,
                     int bins_u, int bins_i, const float* stat, int* ext_stat, int stat_ready,
                     int* ext_mov, unsigned* hist, double* out, hipStream_t st) {
    if (bins_u < 2 || bins_i < 2 || bins_u > kMiMaxBins || bins_i > kMiMaxBins || n_poses <= 0)
        return hipErrorInvalidValue;
    const long long n = (long long)a.v.X * a.v.Y * a.v.Z;
    const int g3 = grid_ndim == 3 ? 1 : 0, s3 = src_ndim == 3 ? 1 : 0;
    const int nb = bins_u * bins_i, stride = mi_hist_size(bins_u, bins_i);
    hipLaunchKernelGGL(k_mi_init, dim3((n_poses + 1 + 255) / 256), dim3(256), 0, st, ext_mov,
                       n_poses);
    // 4 work-groups per CU and pose for the extremes: each ends with two atomics on one address
    const unsigned ge = (unsigned)std::min<long long>((n + 255) / 256, 1024);
    if (!stat_ready) {
        hipLaunchKernelGGL(k_mi_init, dim3(1), dim3(256), 0, st, ext_stat, 1);
        hipLaunchKernelGGL(k_mi_extrema_img, dim3(ge), dim3(256), 0, st, stat, n, ext_stat);
    }
    if (a.warp1) {
        if (a.s.pow2) {
            if (a.src_f16) mi_warp3<__half, true>(a, n_poses, ext_mov, st);
            else mi_warp3<float, true>(a, n_poses, ext_mov, st);
        } else {
            if (a.src_f16) mi_warp3<__half, false>(a, n_poses, ext_mov, st);
            else mi_warp3<float, false>(a, n_poses, ext_mov, st);
        }
    } else if (a.src_f16) {
        hipLaunchKernelGGL(k_mi_extrema<__half>, dim3(ge, (unsigned)n_poses), dim3(256), 0, st, a, g3, s3, ext_mov);
    } else {
        hipLaunchKernelGGL(k_mi_extrema<float>, dim3(ge, (unsigned)n_poses), dim3(256), 0, st, a, g3, s3, ext_mov);
    }
    hipError_t e = hipMemsetAsync(hist, 0, (size_t)n_poses * stride * sizeof(unsigned), st);
    if (e != hipSuccess) return e;
    // One round of the 256 CUs (one work-group each, by its LDS) for all poses; at least 4096
    // voxels per work-group, or the final additions dominate. Where each voxel is warped again, a
    // chain of gathers, and the histograms leave room for two work-groups per CU, large launches
    // take eight rounds of two voxels per thread, twice the wavefronts: 40 poses of 200x180x160, 32
    // bins, 2.61 -> 2.25 ms; 5 poses of 128^3 (10 million voxels) 254 -> 258 us, 13 poses 508 -> 466.
    const size_t lds = (size_t)((nb + 1) / 2) * sizeof(unsigned);
    const bool many = !a.warp1 && lds <= 80 * 1024 && n * n_poses >= 1LL << 24;
    const long long per_pose = std::max(1LL, std::min<long long>(std::max(1, (many ? 2048 : 256) / n_poses), n / kMiVox));
    const long long chunk = (n + per_pose - 1) / per_pose;
    const dim3 gj((unsigned)((n + chunk - 1) / chunk), (unsigned)n_poses);
    const int stat_is_u = movi ? 1 : 0;
    auto joint = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, gj, dim3(1024), lds, st, a, g3, s3, stat, stat_is_u, ext_mov, ext_stat, bins_u,
                           bins_i, chunk, stride, hist);
    };
    if (many) {
        if (a.src_f16) joint(k_mi_joint<__half, 2, 8>);
        else joint(k_mi_joint<float, 2, 8>);
    } else {
        static LdsLimit limit;
        e = limit.raise({reinterpret_cast<const void*>(&k_mi_joint<float, 4, 4>),
                         reinterpret_cast<const void*>(&k_mi_joint<__half, 4, 4>)},
                        (kMiMaxBins * kMiMaxBins / 2) * sizeof(unsigned));
        if (e != hipSuccess) return e;
        if (a.src_f16) joint(k_mi_joint<__half, 4, 4>);
        else joint(k_mi_joint<float, 4, 4>);
    }
    const int groups = std::max(1, bins_i / kMiRows);
    hipLaunchKernelGGL(k_mi_entropy_part, dim3((unsigned)groups, (unsigned)n_poses), dim3(256), 0, st, hist, stride,
                       bins_u, bins_i, (double)n);
    hipLaunchKernelGGL(k_mi_entropy, dim3(n_poses), dim3(1024), 0, st, hist, stride, ext_mov, ext_stat, bins_u,
                       bins_i, (double)n, out);
    return hipGetLastError();
}

}  // namespace lc2e
