// 3D LC2 in two kernels. The first writes the warped moving image of every voxel of the grid and
// pose: k_warp_grad3 a high-resolution one and its |Sobel| (8 bytes), k_warp_us3 an ultrasound
// (4 bytes). k_moments3d forms the patch moments from those grids and combines them.
//
// The fused kernel (k_fused3d) computes both per 16x16 tile, so it warps 2.25 and takes the
// Sobel of 1.89 positions per output voxel, and its 238 VGPRs hold two waves per SIMD. Apart,
// the first kernel's tile has 1.2 warped positions per voxel, and the second needs 84 VGPRs.
// The grids cost 8 bytes written and about 10 read per voxel and pose, at 1 TB/s far from the
// memory's rate. Per call, 192x192x160 grid, 7^3 patch, moving image high-resolution, 32 poses:
// 3.40 -> 2.65 ms; static, 16 poses: the ultrasound's 4 channels, the other sums once per pair
// (kRoleImageStats), 226 us of warp and 848 of moments.
#include "lc2e_device.hpp"

namespace lc2e {

namespace {

constexpr int kGradX = 32, kGradY = 16;  // output tile of k_warp_grad3

// The moving high-resolution image I and its |Sobel| G at every grid voxel of a pose, as
// float2, bit for bit as k_fused3d forms them. A work-group marches along z over a 32x16
// column; the gathers of the next plane are in flight during the Sobel of this one, and the
// two LDS planes take one barrier per step. Bound by VALU issue (102 instructions per voxel,
// 73% of the issue slots): 352 us for 16 poses of 192x192x160, 2.1 TB/s written.
template <typename T, bool P2, bool WORDS>
__global__ __launch_bounds__(256) void k_warp_grad3(FusedArgs a, int ntx, int nty, int zc, int tiles,
                                                    int npose) {
    constexpr int IXE = kGradX + 2, IYE = kGradY + 2, NI = IXE * IYE;
    constexpr int SPT = (NI + 255) / 256;
    __shared__ float s_in[2][NI];
    int tile, pose;
    if (!map_block(tiles, npose, tile, pose)) return;
    const int tid = threadIdx.x;
    const int tcol = tile % (ntx * nty), zci = tile / (ntx * nty);
    const int x0 = (tcol % ntx) * kGradX, y0 = (tcol / ntx) * kGradY;
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z;
    const int z0 = zci * zc, z1 = min(z0 + zc, Z);
    const T* __restrict__ src = static_cast<const T*>(a.src);
    float m[12];
    {
        load_matrix(a, pose, m);
    }
    const int wbase = __builtin_amdgcn_readfirstlane(tid & ~63);
    float cxy[SPT][3];
    unsigned in_xy = 0;
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
        const int i = tid + j * 256;
        const int lx = i % IXE, ly = i / IXE;
        const int gx = x0 - 1 + lx, gy = y0 - 1 + ly;
        if (i < NI && gx >= 0 && gx < X && gy >= 0 && gy < Y) in_xy |= 1u << j;
        const float Lx = fmaf((float)gx, a.v.sx, a.v.ox), Ly = fmaf((float)gy, a.v.sy, a.v.oy);
        cxy[j][0] = fmaf(m[1], Ly, m[0] * Lx);
        cxy[j][1] = fmaf(m[5], Ly, m[4] * Lx);
        cxy[j][2] = fmaf(m[9], Ly, m[8] * Lx);
    }
    typename PendSel<T, WORDS>::type pend[SPT];
    auto has = [&](int j) { return (j + 1) * 256 <= NI || j * 256 + wbase < NI; };
    auto issue = [&](int z) {
        const bool zin = z >= 0 && z < Z;
        const float lz = fmaf((float)z, a.v.sz, a.v.oz);
#pragma unroll
        for (int j = 0; j < SPT; ++j)
            if (has(j)) issue3c<P2>(src, a.s, m, cxy[j], lz, zin && ((in_xy >> j) & 1u), pend[j]);
    };
    auto finish = [&](float* dst) {
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            if (!has(j)) continue;
            const int i = tid + j * 256;
            const float v = finish3(pend[j]);
            if (i < NI) dst[i] = v;
        }
    };
    const int lx = tid % kGradX, ly = 2 * (tid / kGradX);
    const int gx = x0 + lx, gy = y0 + ly;
    const bool ok0 = gx < X && gy < Y, ok1 = gx < X && gy + 1 < Y;
    float2* __restrict__ out = a.warp2 + (size_t)pose * X * Y * Z;
    const unsigned o0 = (unsigned)(gy * X + gx);
    float tA[2][3], tBx[2][3], tBy[2][3], Ip[2], Ic[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int k = 0; k < 3; ++k) tA[e][k] = tBx[e][k] = tBy[e][k] = 0.f;
        Ip[e] = Ic[e] = 0.f;
    }
    issue(z0 - 1);
    int buf = 0;
    for (int z = z0 - 1; z <= z1; ++z, buf ^= 1) {
        finish(s_in[buf]);
        __syncthreads();
        if (z < z1) issue(z + 1);
        const float* row = s_in[buf] + ly * IXE + lx;
        float sm[4], df[4], cm[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float l = row[r * IXE], c = row[r * IXE + 1], rr = row[r * IXE + 2];
            sm[r] = fmaf(2.0f, c, l) + rr;  // (l + 2c) + r: 2c is exact
            df[r] = rr - l;
            cm[r] = c;
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            tA[e][0] = tA[e][1]; tA[e][1] = tA[e][2];
            tBx[e][0] = tBx[e][1]; tBx[e][1] = tBx[e][2];
            tBy[e][0] = tBy[e][1]; tBy[e][1] = tBy[e][2];
            tA[e][2] = fmaf(2.0f, sm[e + 1], sm[e]) + sm[e + 2];
            tBx[e][2] = fmaf(2.0f, df[e + 1], df[e]) + df[e + 2];
            tBy[e][2] = sm[e + 2] - sm[e];
            Ip[e] = Ic[e];
            Ic[e] = cm[e + 1];
        }
        if (z > z0) {
            float2* o = out + (size_t)(z - 1) * X * Y;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float gxv = fmaf(2.0f, tBx[e][1], tBx[e][0]) + tBx[e][2];
                const float gyv = fmaf(2.0f, tBy[e][1], tBy[e][0]) + tBy[e][2];
                const float gzv = tA[e][2] - tA[e][0];
                const float G = sqrtf(fmaf(gzv, gzv, fmaf(gyv, gyv, gxv * gxv)));
                if (e ? ok1 : ok0) o[o0 + (e ? X : 0)] = make_float2(Ip[e], G);
            }
        }
    }
}

// The moving ultrasound at every grid voxel of a pose, NaN where it is not above the weight's
// threshold: every sum that holds such a voxel is NaN then, and its patch has no weight (no
// count of the voxels above the threshold is needed). A thread marches along z with the next
// plane's gathers in flight.
template <typename T, bool P2>
__global__ __launch_bounds__(256) void k_warp_us3(FusedArgs a, int ntx, int nty, int zc, int tiles, int npose) {
    int tile, pose;
    if (!map_block(tiles, npose, tile, pose)) return;
    const int tcol = tile % (ntx * nty), zci = tile / (ntx * nty);
    const int gx = (tcol % ntx) * 64 + (threadIdx.x & 63), gy = (tcol / ntx) * 4 + (threadIdx.x >> 6);
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z;
    if (gx >= X || gy >= Y) return;
    const int z0 = zci * zc, z1 = min(z0 + zc, Z);
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
            const float v = finish3(p[e]);
            if (z + e < z1) out[(size_t)(z + e) * X * Y] = (double)v > kZeroThreshold ? v : NAN;
            issue(min(z + e + 2, z1 - 1), p[e]);
        }
    }
}

// ---------------------------------------------------------------------------
// Patch moments and combine on the grids: a 16x16 column of output voxels over `zchunk`
// planes of one pose, one work-group per CU, its waves in three roles that work on three LDS
// buffers at once, with one barrier per step:
//   z waves: z window sums of the 7 products channels of step s, two planes at a time (they
//     share W - 1 planes; the ring of input planes is 3 floats per plane, where a ring of
//     plane sums would be 14 VGPRs per plane), written to buffer s;
//   x waves: x window sums of step s - 1 in place, a row of 16 outputs per lane;
//   y waves: y window sums of two pixels per lane of step s - 2, and their combine.
// The LDS and the VALU are both about two thirds busy at R = 3. LDS writes are what costs:
// per wave a ds_write_b64 takes 6.2 cycles, a ds_write_b128 13, a ds_read_b64 2.2, a
// ds_read_b128 4.1, but a ds_read2_b64 of two rows 8.0 (measured), so the y sums stay in
// registers up to the combine (no second write) and are read row by row.
// Measured at 192x192x160, R = 3, 16 poses: 0.95 ms. Before its last change of layout (1.03 ms): every phase on all waves, a
// barrier between phases 1.13 ms (512 threads, 80 VGPRs), with the z sums last in a VGPR ring
// 1.13 ms (256 threads, 158 VGPRs); one plane per step, two work-groups per CU: 1.62 ms.
// Raised priorities for the x or the y waves: 1 to 8% slower.
// ---------------------------------------------------------------------------
// Planes a pipeline step carries: two where three buffers of them fit the LDS.
template <int R, int ROLE>
struct Mom {
    static constexpr int NC = Role<ROLE>::NC;
    static constexpr int W = 2 * R + 1, PX = kTile3X + 2 * R, PY = kTile3Y + 2 * R, NP = PX * PY;
    static constexpr int PS = lds_stride(PX), PL = PY * PS;  // LDS row stride, plane size
    static constexpr int KP = 3 * 2 * NC * PL * 8 <= 160 * 1024 ? 2 : 1;
    static constexpr int BUF = KP * NC * PL;                 // doubles per buffer
    // waves per role; a z wave takes ZP positions per lane
    static constexpr int ZP = 2;
    static constexpr int ZW = (NP + ZP * 64 - 1) / (ZP * 64), YW = 2 * KP, XW = (KP * NC * PY + 63) / 64;
    static constexpr int NW = ZW + YW + XW, NTHR = NW * 64;
    static constexpr size_t lds = 3 * BUF * sizeof(double);
    static_assert(NW <= 16 && lds <= 160 * 1024, "roles and buffers fit a CU");
};

// Two window sums of width W of in[0 .. W].
template <int W>
__device__ __forceinline__ void window2(const double (&in)[W + 1], double& o0, double& o1) {
    double mid = in[1];
#pragma unroll
    for (int j = 2; j < W; ++j) mid += in[j];
    o0 = in[0] + mid;
    o1 = mid + in[W];
}

template <int R, int ROLE>
__global__ __launch_bounds__((Mom<R, ROLE>::NTHR)) void k_moments3d(FusedArgs a) {
    using M = Mom<R, ROLE>;
    using Ro = Role<ROLE>;
    constexpr int NC = M::NC;
    constexpr int TX = kTile3X, TY = kTile3Y, W = M::W, PX = M::PX, PY = M::PY, NP = M::NP, PS = M::PS,
                  PL = M::PL, KP = M::KP, BUF = M::BUF, N3 = W * W * W;
    extern __shared__ __align__(16) double s_buf[];

    int tile, pose;
    if (!map_block(a.tiles, a.npose, tile, pose)) return;  // whole work-group
    const int rank = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int cols = a.ntx * a.nty;
    const int tcol = tile % cols, zc = tile / cols;
    const int x0 = R + (tcol % a.ntx) * TX, y0 = R + (tcol / a.ntx) * TY;
    const int z0 = R + zc * a.zchunk;
    const int zend = min(z0 + a.zchunk, a.v.Z - R);
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z, XY = X * Y;
    const int nout = zend - z0;
    const int n = (nout + KP - 1) / KP;  // steps with products

    if (rank >= M::YW && rank < M::YW + M::ZW) {
        // z window sums of ZP positions per lane, two planes at a time
        constexpr int ZP = M::ZP, K = W + 1;
        const int i0 = (rank - M::YW) * 64 + lane;
        int d_ofs[ZP];
        unsigned g_ofs[ZP];  // bytes of one float per voxel
#pragma unroll
        for (int e = 0; e < ZP; ++e) {
            const int i = min(i0 + e * M::ZW * 64, NP - 1);
            const int lx = i % PX, ly = i / PX;
            d_ofs[e] = ly * PS + lx;
            g_ofs[e] = (unsigned)(min(y0 - R + ly, Y - 1) * X + min(x0 - R + lx, X - 1)) * 4u;
        }
        const float2* __restrict__ ig = a.warp2 + (size_t)pose * Z * XY;
        const float* __restrict__ wu = a.warp1 + (size_t)pose * Z * XY;
        float vi[K][ZP], vg[K][ZP], vu[K][ZP];  // the inputs the role has
        auto load = [&](auto slot_c, int z) {
            constexpr int k = decltype(slot_c)::value;
            const size_t zo = (size_t)min(z, Z - 1) * XY;
#pragma unroll
            for (int e = 0; e < ZP; ++e) {
                if constexpr (ROLE == kRoleMovingImage) {
                    const float2 v = load_at(ig + zo, g_ofs[e] * 2u);
                    vi[k][e] = v.x;
                    vg[k][e] = v.y;
                    vu[k][e] = load_at(a.stat_img + zo, g_ofs[e]);
                } else {
                    if constexpr (Ro::HAS_I) {
                        vi[k][e] = load_at(a.stat_img + zo, g_ofs[e]);
                        vg[k][e] = load_at(a.stat_grad + zo, g_ofs[e]);
                    }
                    if constexpr (ROLE == kRoleStaticImage) vu[k][e] = load_at(wu + zo, g_ofs[e]);
                    if constexpr (ROLE == kRoleUsStats) vu[k][e] = load_at(a.stat_img + zo, g_ofs[e]);
                }
            }
        };
        Unroll<0, K>::run([&](auto kc) { load(kc, z0 - R + decltype(kc)::value); });
        int buf = 0;
        for (int p0 = 0; p0 < nout; p0 += 2 * (R + 1)) {
            Unroll<0, R + 1>::run([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const int p = p0 + 2 * k;
                if (p >= nout) return;  // block-uniform
                double s[ZP][NC];
#pragma unroll
                for (int e = 0; e < ZP; ++e) {
                    auto add = [&](double (&t)[NC], int j) {
                        const int i = (2 * k + j) % K;
                        float I = 0.f, G = 0.f, U = 0.f;
                        if constexpr (Ro::HAS_I) I = vi[i][e], G = vg[i][e];
                        if constexpr (Ro::HAS_U) U = vu[i][e];
                        if constexpr (ROLE == kRoleUsStats) U = (double)U > kZeroThreshold ? U : NAN;
                        Ro::add(t, I, G, U);
                    };
                    // the ring stays in floats: without this the compiler keeps each plane's
                    // FP64 values from step to step as well, and spills
#pragma unroll
                    for (int j = 0; j < K; ++j) {
                        if constexpr (Ro::HAS_I) asm volatile("" : "+v"(vi[j][e]), "+v"(vg[j][e]));
                        if constexpr (Ro::HAS_U) asm volatile("" : "+v"(vu[j][e]));
                    }
#pragma unroll
                    for (int c = 0; c < NC; ++c) s[e][c] = 0.0;
#pragma unroll
                    for (int j = 1; j < W; ++j) add(s[e], j);
                    double t[NC];
#pragma unroll
                    for (int c = 0; c < NC; ++c) t[c] = s[e][c];
                    add(t, 0);
                    add(s[e], W);
                    // the positions past the region repeat the last one, with its values
                    double* d = s_buf + buf * BUF + d_ofs[e];
#pragma unroll
                    for (int c = 0; c < NC; ++c) d[c * PL] = t[c];
                    if (KP == 2)
#pragma unroll
                        for (int c = 0; c < NC; ++c) d[(NC + c) * PL] = s[e][c];
                }
                // the two oldest planes make room for the next two
                load(std::integral_constant<int, (2 * k) % K>{}, z0 - R + p + W + 1);
                load(std::integral_constant<int, (2 * k + 1) % K>{}, z0 - R + p + W + 2);
                __syncthreads();
                buf = buf == 2 ? 0 : buf + 1;
                if (KP == 1 && p + 1 < nout) {
#pragma unroll
                    for (int e = 0; e < ZP; ++e)
#pragma unroll
                        for (int c = 0; c < NC; ++c) s_buf[buf * BUF + d_ofs[e] + c * PL] = s[e][c];
                    __syncthreads();
                    buf = buf == 2 ? 0 : buf + 1;
                }
            });
        }
        __syncthreads();
        return;
    }
    if (rank >= M::YW + M::ZW) {
        // x window sums in place
        const int t0 = (rank - M::YW - M::ZW) * 64 + lane;
        __syncthreads();
        int buf = 0;
        for (int s = 0; s < n; ++s) {
            for (int t = t0; t < KP * NC * PY; t += M::XW * 64) {  // one round
                double* r = s_buf + buf * BUF + (t / PY) * PL + (t % PY) * PS;
                r = static_cast<double*>(__builtin_assume_aligned(r, 16));
                window_run<W>(r, 1, r, 1);
            }
            buf = buf == 2 ? 0 : buf + 1;
            __syncthreads();
        }
        return;
    }
    // y window sums of two pixels of a column and their combine. Lanes 16 apart take rows 8
    // apart: their LDS reads then fall into distinct halves of the banks.
    const int plane = rank >> 1;
    const int ox = lane % TX, oy = 8 * (lane / TX & 1) + 2 * (lane / (2 * TX)) + 4 * (rank & 1);
    const bool ok0 = x0 + ox < X - R && y0 + oy < Y - R, ok1 = ok0 && y0 + oy + 1 < Y - R;
    const unsigned vo0 = ok0 ? (unsigned)((y0 + oy) * X + (x0 + ox)) * 8u : 0u;
    const unsigned vo1 = ok1 ? vo0 + (unsigned)X * 8u : 0u;
    double mu[2], cyy[2];
    ImageStats ist[2];
    auto stats = [&](int zo) {
        const size_t zp = (size_t)min(zo, zend - 1) * XY;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const unsigned vo = j ? vo1 : vo0;
            if constexpr (ROLE == kRoleMovingImage) {
                mu[j] = load_at(a.ustat_mean + zp, vo);
                cyy[j] = load_at(a.ustat_cyy + zp, vo);
            }
            if constexpr (ROLE == kRoleStaticImage) {
                const double* st = a.istat + zp;
                ist[j] = {load_at(st, vo), load_at(st + a.istat_stride, vo), load_at(st + 2 * a.istat_stride, vo),
                          load_at(st + 3 * a.istat_stride, vo), load_at(st + 4 * a.istat_stride, vo)};
            }
        }
    };
    double acc_m = 0.0, acc_w = 0.0;
    __syncthreads();
    if constexpr (Ro::SUMS) stats(z0 + plane);
    __syncthreads();
    int buf = 0;
    for (int s = 0; s < n; ++s) {
        const int zo = z0 + s * KP + plane;
        const bool zok = zo < zend;
        // one address per row, of unknown relation to the others: the compiler would pair two
        // rows in a ds_read2_b64, which takes 8 cycles where two ds_read_b64 take 4.4 (measured)
        const double* row[W + 1];
#pragma unroll
        for (int j = 0; j < W + 1; ++j) {
            unsigned ofs = (unsigned)(buf * BUF + plane * NC * PL + (oy + j) * PS + ox);
            asm volatile("" : "+v"(ofs));
            row[j] = s_buf + ofs;
        }
        double S[2][NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            double in[W + 1];
#pragma unroll
            for (int j = 0; j < W + 1; ++j) in[j] = row[j][c * PL];
            window2<W>(in, S[0][c], S[1][c]);
            // at most two channels in flight: all reads first would take 112 VGPRs
            asm volatile("" : "+v"(S[0][c]), "+v"(S[1][c]));
            if (c % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        double m0[2], c0[2];
        ImageStats i0[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (ROLE == kRoleMovingImage) m0[j] = mu[j], c0[j] = cyy[j];
            if constexpr (ROLE == kRoleStaticImage) i0[j] = ist[j];
        }
        if constexpr (Ro::SUMS) stats(zo + KP);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const bool in = (j ? ok1 : ok0) && zok;
            const size_t vo = (size_t)zo * XY + (size_t)(y0 + oy + j) * X + (x0 + ox);
            if constexpr (Ro::SUMS) {
                double w, meas;
                bool ok;
                if constexpr (ROLE == kRoleMovingImage) {
                    ok = in && c0[j] >= 0.0;
                    combine_static_u_any(S[j], m0[j], ok ? c0[j] : 1.0, N3, w, meas);
                } else {
                    ok = combine_static_image(S[j], i0[j], N3, w, meas) && in;
                }
                acc_m += ok ? meas : 0.0;
                acc_w += ok ? w : 0.0;
                if (a.wmap && ok) {
                    a.wmap[vo] = w;
                    a.mmap[vo] = meas;
                }
            } else if (in) {
                if constexpr (ROLE == kRoleImageStats) store_image_stats(S[j], N3, a.istat_out + vo, a.istat_stride);
                else store_us_stats(S[j], N3, a.ustat_mean_out + vo, a.ustat_cyy_out + vo);
            }
        }
        // partials per block of kZBlock output planes, tile column and combining wave, at
        // fixed positions in z
        const int ze = z0 + (s + 1) * KP;
        if (Ro::SUMS && ((ze - R) % kZBlock == 0 || ze >= zend)) {
            wave_reduce_store(acc_m, acc_w,
                              a.partials + (((size_t)pose * a.blocks_per_pose +
                                             ((size_t)((ze - 1 - R) / kZBlock) * cols + tcol) * M::YW + rank) * 2));
            acc_m = 0.0;
            acc_w = 0.0;
        }
        buf = buf == 2 ? 0 : buf + 1;
        if (s + 1 < n) __syncthreads();
    }
}

template <typename T, bool P2, bool WORDS = false>
void warp_grad3(const FusedArgs& a, int ntx, int nty, int zc, int tiles, int n, hipStream_t st) {
    const int tiles8 = (tiles + kXcds - 1) / kXcds * kXcds;
    hipLaunchKernelGGL((k_warp_grad3<T, P2, WORDS>), dim3((unsigned)tiles8 * n), dim3(256), 0, st, a, ntx, nty,
                       zc, tiles, n);
}

template <typename T, bool P2>
void warp_us3(const FusedArgs& a, int ntx, int nty, int zc, int tiles, int n, hipStream_t st) {
    const int tiles8 = (tiles + kXcds - 1) / kXcds * kXcds;
    hipLaunchKernelGGL((k_warp_us3<T, P2>), dim3((unsigned)tiles8 * n), dim3(256), 0, st, a, ntx, nty, zc, tiles, n);
}

template <int R, int ROLE>
hipError_t moments3k(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    using M = Mom<R, ROLE>;
    static LdsLimit limit;
    const hipError_t err = limit.raise({reinterpret_cast<const void*>(&k_moments3d<R, ROLE>)}, M::lds);
    if (err != hipSuccess) return err;
    if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, k_moments3d<R, ROLE>, M::NTHR, M::lds);
    hipLaunchKernelGGL((k_moments3d<R, ROLE>), grid, dim3(M::NTHR), M::lds, st, a);
    return hipGetLastError();
}

template <int ROLE, int R = 1>
hipError_t moments3r(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    if (a.r == R) return moments3k<R, ROLE>(a, grid, st, occ);
    if constexpr (R < kMaxRMom3) return moments3r<ROLE, R + 1>(a, grid, st, occ);
    return hipErrorInvalidValue;
}
template <int ROLE, int R = 1>
int waves3r(int r) {
    if (r == R) return Mom<R, ROLE>::YW;
    if constexpr (R < kMaxRMom3) return waves3r<ROLE, R + 1>(r);
    return 0;
}

}  // namespace

hipError_t launch_warp3(const FusedArgs& a, int movi, int n, hipStream_t st) {
    const int tx = movi ? kGradX : 64, ty = movi ? kGradY : 4;
    const int ntx = (a.v.X + tx - 1) / tx, nty = (a.v.Y + ty - 1) / ty;
    // z-chunks: about 2048 work-groups (the CUs hold about that many), at least 8 planes each
    // (with the Sobel, two more are warped per chunk), or 4 where that still leaves most of the
    // chip idle: a call of 4 poses 64x64x64, r = 1, 47.7 -> 44.5 us, up to 1 pose of 96^3 2 to 4 us less
    const int want = (int)std::max(1LL, 2048LL / ((long long)ntx * nty * n));
    int zc = std::max(8, (a.v.Z + want - 1) / want);
    if ((long long)ntx * nty * n * ((a.v.Z + zc - 1) / zc) <= 512) zc = std::min(zc, 4);
    const int tiles = ntx * nty * ((a.v.Z + zc - 1) / zc);
    const int form = (movi ? 4 : 0) + (a.s.pow2 ? 2 : 0) + (a.src_f16 ? 1 : 0);
    // half sources of even X in aligned words: 8 poses of the CT 660 -> 610 us
    const bool words = movi && a.src_f16 && a.s.X % 2 == 0;
    if (words) {
        if (a.s.pow2) warp_grad3<__half, true, true>(a, ntx, nty, zc, tiles, n, st);
        else warp_grad3<__half, false, true>(a, ntx, nty, zc, tiles, n, st);
        return hipGetLastError();
    }
    switch (form) {
        case 7: warp_grad3<__half, true>(a, ntx, nty, zc, tiles, n, st); break;
        case 6: warp_grad3<float, true>(a, ntx, nty, zc, tiles, n, st); break;
        case 5: warp_grad3<__half, false>(a, ntx, nty, zc, tiles, n, st); break;
        case 4: warp_grad3<float, false>(a, ntx, nty, zc, tiles, n, st); break;
        case 3: warp_us3<__half, true>(a, ntx, nty, zc, tiles, n, st); break;
        case 2: warp_us3<float, true>(a, ntx, nty, zc, tiles, n, st); break;
        case 1: warp_us3<__half, false>(a, ntx, nty, zc, tiles, n, st); break;
        default: warp_us3<float, false>(a, ntx, nty, zc, tiles, n, st); break;
    }
    return hipGetLastError();
}

hipError_t moments3(const FusedArgs& a, int role, int n, hipStream_t st, int* occ) {
    if (!occ && (a.zchunk <= 0 || a.zchunk % kZBlock != 0)) return hipErrorInvalidValue;
    const long long tiles8 = (a.tiles + kXcds - 1) / kXcds * (long long)kXcds;
    if (tiles8 * n > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(tiles8 * n));
    switch (role) {
        case kRoleMovingImage: return moments3r<kRoleMovingImage>(a, grid, st, occ);
        case kRoleStaticImage: return moments3r<kRoleStaticImage>(a, grid, st, occ);
        case kRoleImageStats: return moments3r<kRoleImageStats>(a, grid, st, occ);
        default: return moments3r<kRoleUsStats>(a, grid, st, occ);
    }
}

int moments3_waves(int r, int role) {
    return role == kRoleMovingImage ? waves3r<kRoleMovingImage>(r) : waves3r<kRoleStaticImage>(r);
}

}  // namespace lc2e
