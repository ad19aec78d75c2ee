// 3D LC2 in two kernels: the moving image is warped (with its |Sobel| where it is the
// high-resolution one) onto the virtual grid, a float2 or float per voxel and pose, and a
// second kernel forms the patch moments from those grids and combines them.
#include "lc2e_device.hpp"

namespace lc2e {

namespace {

constexpr int kGradX = 32, kGradY = 16;  // output tile of k_warp_grad3

// The moving high-resolution image I and its |Sobel| G at every grid voxel of a pose, as
// float2, bit for bit as k_fused3d forms them.
template <typename T, bool P2>
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
        const float* mp = a.mats + (size_t)pose * 12;
#pragma unroll
        for (int k = 0; k < 12; ++k) m[k] = mp[k];
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
    Pending3<T> pend[SPT];
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

// A uniform base plus a 32-bit byte offset per lane (one saddr + voffset access). The empty
// asm keeps the sum out of the loop optimiser's sight: it would carry a 64-bit pointer per
// lane for every unrolled step (46 spilled VGPRs at R = 3).
__device__ __forceinline__ const char* at_bytes(const void* base, unsigned ofs) {
    asm volatile("" : "+v"(ofs));
    return static_cast<const char*>(base) + ofs;
}

// ---------------------------------------------------------------------------
// Patch moments and combine on the grids: a 16x16 column of output voxels over `zchunk`
// planes of one pose.
// ---------------------------------------------------------------------------
// LDS row strides (bytes) that are odd multiples of 16: eight lanes that read 16 bytes each
// from consecutive rows then cover the 128 bytes of a cycle.
constexpr int odd16(int bytes) { return (bytes + 15) / 16 * 16 + ((bytes + 15) / 16 % 2 ? 0 : 16); }

// Products of channel c at a position.
template <int C>
__device__ __forceinline__ double product7(float I, float G, float U) {
    const double di = I, dg = G, du = U;
    return C == 0 ? di : C == 1 ? dg : C == 2 ? di * di : C == 3 ? dg * dg : C == 4 ? di * dg : C == 5 ? du * di : du * dg;
}

#ifndef XO
#define XO 4
#endif
// XO window sums of width W of in[0 .. XO + W - 2].
template <int W>
__device__ __forceinline__ void window_xo(const double* in, double* out) {
#if XO == 8
    window_run<W, double, 8>(in, 1, out, 1);
#else
    double mid = in[3];
#pragma unroll
    for (int j = 4; j < W; ++j) mid += in[j];
    const double l1 = in[1] + in[2], l0 = in[0] + l1;
    const double p1 = in[W] + in[W + 1], p2 = p1 + in[W + 2];
    if (W == 3) {
        out[0] = l0; out[1] = l1 + in[W]; out[2] = in[2] + p1; out[3] = p2;
    } else {
        out[0] = l0 + mid; out[1] = (l1 + mid) + in[W]; out[2] = (in[2] + mid) + p1; out[3] = mid + p2;
    }
#endif
}

template <int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(R <= 3 ? 3 : 2)))
void k_moments3d(FusedArgs a) {
    constexpr int TX = kTile3X, TY = kTile3Y, NTHR = TX * TY;
    constexpr int W = 2 * R + 1, PX = TX + 2 * R, PY = TY + 2 * R, NP = PX * PY;
    constexpr int XS = lds_stride(TX + 1);
    constexpr int PPT = (NP + NTHR - 1) / NTHR;
    constexpr int N3 = W * W * W;
    constexpr int NC = 7;
    constexpr int SIG = odd16(PX * 8), SU = odd16(PX * 4);  // row strides of the input planes
    constexpr int SEGS = TX / XO, NX = PY * SEGS, XN = XO + W - 1;
    __shared__ __align__(16) unsigned char s_ig[2][PY * SIG];
    __shared__ __align__(16) unsigned char s_u[2][PY * SU];
    __shared__ double s_xp[NC * PY * XS];
    __shared__ double s_sum[NC * TX * TY];

    int tile, pose;
    if (!map_block(a.tiles, a.npose, tile, pose)) return;  // whole work-group
    const int tid = threadIdx.x;
    const int cols = a.ntx * a.nty;
    const int tcol = tile % cols, zc = tile / cols;
    const int x0 = R + (tcol % a.ntx) * TX, y0 = R + (tcol / a.ntx) * TY;
    const int z0 = R + zc * a.zchunk;
    const int zend = min(z0 + a.zchunk, a.v.Z - R);
    const int nout = zend - z0;
    const int X = a.v.X, Y = a.v.Y, Z = a.v.Z, XY = X * Y;
    const int nq = nout + 2 * R;

    // products positions: LDS offset and in-plane grid offset (clamped into the grid; what
    // lies past it only reaches outputs that are not valid)
    int ig_ofs[PPT], u_ofs[PPT];
    unsigned g_ofs[PPT];  // bytes of one float per voxel
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        const int i = min(tid + j * NTHR, NP - 1);
        const int lx = i % PX, ly = i / PX;
        ig_ofs[j] = ly * SIG + lx * 8;
        u_ofs[j] = ly * SU + lx * 4;
        g_ofs[j] = (unsigned)(min(y0 - R + ly, Y - 1) * X + min(x0 - R + lx, X - 1)) * 4u;
    }
    const int wbase = __builtin_amdgcn_readfirstlane(tid & ~63);
    auto wave_has = [&](int j) { return (j + 1) * NTHR <= NP || j * NTHR + wbase < NP; };
    const float2* __restrict__ ig = a.warp2 + ((size_t)pose * Z + (z0 - R)) * XY;
    const float* __restrict__ ug = a.stat_img + (size_t)(z0 - R) * XY;
    float2 ci[PPT];
    float cu[PPT];
    auto issue = [&](int q) {
        const float2* p = ig + (size_t)q * XY;
        const float* u = ug + (size_t)q * XY;
#pragma unroll
        for (int j = 0; j < PPT; ++j)
            if (wave_has(j)) {
                __builtin_memcpy(&ci[j], at_bytes(p, g_ofs[j] * 2u), 8);
                __builtin_memcpy(&cu[j], at_bytes(u, g_ofs[j]), 4);
            }
    };
    auto stage = [&](int b) {
#pragma unroll
        for (int j = 0; j < PPT; ++j)
            if (wave_has(j)) {  // the last positions are written more than once, with one value
                __builtin_memcpy(__builtin_assume_aligned(s_ig[b] + ig_ofs[j], 8), &ci[j], 8);
                __builtin_memcpy(__builtin_assume_aligned(s_u[b] + u_ofs[j], 4), &cu[j], 4);
            }
    };
    const int ox = tid % TX, oy = tid / TX;
    const bool col_valid = (x0 + ox < X - R) && (y0 + oy < Y - R);
    const unsigned vo = col_valid ? (unsigned)((y0 + oy) * X + (x0 + ox)) : 0u;
    double mu_pre = 0.0, cyy_pre = -1.0;
    auto issue_stats = [&](int zo) {
        __builtin_memcpy(&mu_pre, at_bytes(a.ustat_mean + (size_t)zo * XY, vo * 8u), 8);
        __builtin_memcpy(&cyy_pre, at_bytes(a.ustat_cyy + (size_t)zo * XY, vo * 8u), 8);
    };

    double ring[W][NC];
#pragma unroll
    for (int k = 0; k < W; ++k)
#pragma unroll
        for (int c = 0; c < NC; ++c) ring[k][c] = 0.0;
    double acc_m = 0.0, acc_w = 0.0;

    // x window sums of plane q's products: a task per row and run of XO outputs, products
    // formed on the fly. The waves that take them change from plane to plane.
    auto x_pass = [&](int q) {
        const int t = (tid + 64 * (q & 3)) & (NTHR - 1);
        if (t < NX) {
            const int row = t % PY, seg = t / PY;
            float vi[XN], vg[XN], vu[XN];
            const unsigned char* pi = s_ig[q & 1] + row * SIG + seg * XO * 8;
            const unsigned char* pu = s_u[q & 1] + row * SU + seg * XO * 4;
#pragma unroll
            for (int i = 0; i < XN; i += 2) {
                float t4[4] = {0.f, 0.f, 0.f, 0.f};
                __builtin_memcpy(t4, __builtin_assume_aligned(pi + i * 8, 16), i + 1 < XN ? 16 : 8);
                vi[i] = t4[0];
                vg[i] = t4[1];
                if (i + 1 < XN) vi[i + 1] = t4[2], vg[i + 1] = t4[3];
            }
#pragma unroll
            for (int i = 0; i < XN; i += 4) {
                constexpr int all = XN;
                float t4[4] = {0.f, 0.f, 0.f, 0.f};
                __builtin_memcpy(t4, __builtin_assume_aligned(pu + i * 4, 16), (all - i >= 4 ? 4 : all - i) * 4);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (i + k < XN) vu[i + k] = t4[k];
            }
            double* o = s_xp + row * XS + seg * XO;
            Unroll<0, NC>::run([&](auto cc) {
                constexpr int c = decltype(cc)::value;
                double in[XN], out[XO];
#pragma unroll
                for (int i = 0; i < XN; ++i) in[i] = product7<c>(vi[i], vg[i], vu[i]);
                window_xo<W>(in, out);
#pragma unroll
                for (int i = 0; i < XO; ++i) o[c * PY * XS + i] = out[i];
            });
        }
    };
    auto y_pass = [&]() {
        const int col = tid % TX, seg = (tid / TX) % 2, c = tid / (2 * TX);
        if (c < NC)
            window_run<W, double, 8>(s_xp + c * PY * XS + seg * 8 * XS + col, XS,
                                     s_sum + c * TX * TY + seg * 8 * TX + col, TX);
    };
    auto ring_combine = [&](auto slot_c, int q) {
        constexpr int k = decltype(slot_c)::value;
        constexpr int prev = (k + W - 1) % W;
        double S[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const double Pn = s_sum[c * TX * TY + tid];
            ring[prev][c] = ring[prev][c] + Pn;
            ring[k][c] = Pn;
            S[c] = Pn;
        }
        if (q < 2 * R) return;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            double t = ring[(k + 1) % W][c];
#pragma unroll
            for (int j = 1; j < R; ++j) t += ring[(k + 1 + 2 * j) % W][c];
            S[c] = t + S[c];
        }
        const int zo = z0 + q - 2 * R;
        const double mu = mu_pre, cyy = cyy_pre;
        if (q + 1 < nq) issue_stats(zo + 1);
        double w, meas;
        if (col_valid && combine_static_u(S, mu, cyy, N3, w, meas)) {
            acc_m += meas;
            acc_w += w;
            if (a.wmap) {
                a.wmap[(size_t)zo * XY + vo] = w;
                a.mmap[(size_t)zo * XY + vo] = meas;
            }
        }
        if ((zo - R + 1) % kZBlock == 0 || zo + 1 == zend) {
            constexpr int NW = NTHR / 64;
            double* dst = a.partials + (((size_t)pose * a.blocks_per_pose +
                                         ((size_t)((zo - R) / kZBlock) * cols + tcol) * NW +
                                         (tid >> 6)) * 2);
            wave_reduce_store(acc_m, acc_w, dst);
            acc_m = 0.0;
            acc_w = 0.0;
        }
    };

    issue(0);
    issue_stats(z0);
    stage(0);
    issue(1);  // nq >= 2R + 1 >= 3
    __syncthreads();
    for (int q0 = 0; q0 <= nq; q0 += W) {
        // W consecutive steps with compile-time ring slots, so the z ring stays in VGPRs.
        Unroll<0, W>::run([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            const int q = q0 + k;
            if (q > nq) return;  // block-uniform; step nq only drains step nq - 1
            if (q < nq) x_pass(q);
            if (q > 0) ring_combine(std::integral_constant<int, (k - 1 + W) % W>{}, q - 1);
            if (q == nq) return;
            __syncthreads();
            y_pass();
            if (q + 1 < nq) stage((q + 1) & 1);
            if (q + 2 < nq) issue(q + 2);
            __syncthreads();
        });
    }
}

template <typename T, bool P2>
void warp_grad3(const FusedArgs& a, int ntx, int nty, int zc, int tiles, int n, hipStream_t st) {
    const int tiles8 = (tiles + kXcds - 1) / kXcds * kXcds;
    hipLaunchKernelGGL((k_warp_grad3<T, P2>), dim3((unsigned)tiles8 * n), dim3(256), 0, st, a, ntx, nty,
                       zc, tiles, n);
}

template <int R>
hipError_t moments3(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    if (occ) return hipOccupancyMaxActiveBlocksPerMultiprocessor(occ, k_moments3d<R>, 256, 0);
    hipLaunchKernelGGL((k_moments3d<R>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t moments3r(const FusedArgs& a, dim3 grid, hipStream_t st, int* occ) {
    switch (a.r) {
        case 1: return moments3<1>(a, grid, st, occ);
        case 2: return moments3<2>(a, grid, st, occ);
        case 3: return moments3<3>(a, grid, st, occ);
        case 4: return moments3<4>(a, grid, st, occ);
        case 5: return moments3<5>(a, grid, st, occ);
        case 6: return moments3<6>(a, grid, st, occ);
        case 7: return moments3<7>(a, grid, st, occ);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_warp_grad3(const FusedArgs& a, int n, hipStream_t st) {
    const int ntx = (a.v.X + kGradX - 1) / kGradX, nty = (a.v.Y + kGradY - 1) / kGradY;
    // z-chunks: about 2048 work-groups, at least 8 planes each (two more are warped)
    const int want = (int)std::max(1LL, 2048LL / ((long long)ntx * nty * n));
    const int zc = std::max(8, (a.v.Z + want - 1) / want);
    const int tiles = ntx * nty * ((a.v.Z + zc - 1) / zc);
    if (a.s.pow2) {
        if (a.src_f16) warp_grad3<__half, true>(a, ntx, nty, zc, tiles, n, st);
        else warp_grad3<float, true>(a, ntx, nty, zc, tiles, n, st);
    } else {
        if (a.src_f16) warp_grad3<__half, false>(a, ntx, nty, zc, tiles, n, st);
        else warp_grad3<float, false>(a, ntx, nty, zc, tiles, n, st);
    }
    return hipGetLastError();
}

hipError_t launch_moments3(const FusedArgs& a, int n, hipStream_t st) {
    if (a.tiles == 0 || n <= 0) return hipSuccess;
    if (a.zchunk <= 0 || a.zchunk % kZBlock != 0) return hipErrorInvalidValue;
    FusedArgs b = a;
    b.npose = n;
    const long long tiles8 = (a.tiles + kXcds - 1) / kXcds * (long long)kXcds;
    if (tiles8 * n > 0x7fffffffLL) return hipErrorInvalidValue;
    return moments3r(b, dim3((unsigned)(tiles8 * n)), st, nullptr);
}

hipError_t moments_resident_per_cu(const FusedArgs& a, int* per_cu) {
    *per_cu = 0;
    return moments3r(a, dim3(1), nullptr, per_cu);
}

}  // namespace lc2e
