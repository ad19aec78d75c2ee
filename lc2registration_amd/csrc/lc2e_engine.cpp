// C ABI of the LC2 engine (include/lc2e.h): resident volumes, pairs, batched
// evaluation on one HIP stream, HBM budget accounting, optional HIP-graph replay.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include "lc2e.h"
#include "lc2e_geometry.hpp"
#include "lc2e_kernels.hpp"

namespace {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

#define HIP_TRY(expr)                                                                      \
    do {                                                                                   \
        hipError_t _e = (expr);                                                            \
        if (_e != hipSuccess)                                                              \
            return fail(LC2E_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), \
                        __FILE__, __LINE__);                                               \
    } while (0)

int dtype_size(int dt) {
    switch (dt) {
        case LC2E_U8: return 1;
        case LC2E_I16: return 2;
        case LC2E_F16: return 2;
        case LC2E_F32: return 4;
        default: return 0;
    }
}

// Gives memory of the device back that its owners can do without, a piece at a time; false if
// there is no more (defined below).
bool reclaim(int device);

}  // namespace

struct lc2e_engine {
    int device = 0;
    int cus = 0;  // compute units of the device
    hipStream_t stream = nullptr;
    // the device's scratch array for lc2e_eval_batch_noalloc (null if its lookup failed,
    // then scratch_error says why)
    void* scratch = nullptr;
    std::string scratch_error;
    // workspace of lc2e_eval_batch_noalloc for the pairs that need one (na_pairs of them); its
    // calls on a device run one at a time, so one serves them all (guarded by noalloc_lock)
    void* na = nullptr;
    size_t na_bytes = 0;
    int na_pairs = 0;
    size_t budget = 0;  // 0 = unlimited
    size_t used = 0;
    std::mutex mu;      // guards `used`: a serving loop allocates from its own thread

    // Freed device and pinned host blocks kept for the next allocation of about their size,
    // by an engine without a budget: a hipMalloc or hipFree of a volume takes 0.1 to 0.5 ms. At
    // most kKeepDevice and kKeepHost bytes; given back when an allocation fails and with the
    // engine. A block is kept only once the device is idle (as hipFree waits for it).
    struct Block {
        void* p;
        size_t bytes;
    };
    static constexpr size_t kKeepDevice = size_t(1) << 30, kKeepHost = size_t(16) << 20;
    std::vector<Block> kept_device, kept_host;  // guarded by mu

    void* take(std::vector<Block>& kept, size_t bytes) {
        if (budget) return nullptr;
        std::lock_guard<std::mutex> lk(mu);
        int best = -1;
        for (int i = 0; i < (int)kept.size(); ++i)
            if (kept[i].bytes >= bytes && kept[i].bytes <= bytes + bytes / 4 + 4096 &&
                (best < 0 || kept[i].bytes < kept[best].bytes))
                best = i;
        if (best < 0) return nullptr;
        void* p = kept[best].p;
        sizes[p] = kept[best].bytes;
        kept.erase(kept.begin() + best);
        return p;
    }
    // true if the block is kept
    bool keep(std::vector<Block>& kept, size_t limit, void* p, size_t bytes) {
        if (budget || bytes > limit / 2) return false;
        int current = device;  // the caller's device stays current, as it does in hipFree
        bool idle = hipGetDevice(&current) == hipSuccess && hipSetDevice(device) == hipSuccess &&
                    hipDeviceSynchronize() == hipSuccess;
        if (current != device) idle = hipSetDevice(current) == hipSuccess && idle;
        if (!idle) return false;
        std::vector<Block> oldest;  // make room
        {
            std::lock_guard<std::mutex> lk(mu);
            auto it = sizes.find(p);
            if (it != sizes.end()) {
                bytes = it->second;  // the block's own size, if it had been reused
                sizes.erase(it);
            }
            size_t total = bytes;
            for (const Block& b : kept) total += b.bytes;
            size_t out = 0;
            while (total > limit && out < kept.size()) total -= kept[out++].bytes;
            oldest.assign(kept.begin(), kept.begin() + out);
            kept.erase(kept.begin(), kept.begin() + out);
            kept.push_back({p, bytes});
        }
        for (const Block& b : oldest) (void)(&kept == &kept_host ? hipHostFree(b.p) : hipFree(b.p));
        return true;
    }
    std::map<void*, size_t> sizes;  // reused blocks in use that are larger than asked for
    bool give_back() {
        std::vector<Block> d, h;
        {
            std::lock_guard<std::mutex> lk(mu);
            d.swap(kept_device);
            h.swap(kept_host);
        }
        for (const Block& b : d) (void)hipFree(b.p);
        for (const Block& b : h) (void)hipHostFree(b.p);
        return !d.empty();
    }
    // Device memory without a charge to the budget; `must`: the call fails without it, so what
    // pairs and engines only keep to be faster makes room.
    hipError_t raw_alloc(void** p, size_t bytes, bool must) {
        if (!bytes) bytes = 1;
        if ((*p = take(kept_device, bytes))) return hipSuccess;
        hipError_t err = hipSetDevice(device);
        if (err == hipSuccess) err = hipMalloc(p, bytes);
        if (err != hipSuccess) {  // again without the kept blocks
            (void)hipGetLastError();
            give_back();
            err = hipMalloc(p, bytes);
        }
        while (err == hipErrorOutOfMemory && must && reclaim(device)) {
            (void)hipGetLastError();
            err = hipMalloc(p, bytes);
        }
        return err;
    }
    void raw_free(void* p, size_t bytes) {
        if (p && !keep(kept_device, kKeepDevice, p, bytes ? bytes : 1)) {
            forget(p);
            (void)hipFree(p);
        }
    }
    // Mapped, coherent pinned host memory.
    hipError_t host_alloc(void** p, size_t bytes) {
        if ((*p = take(kept_host, bytes))) return hipSuccess;
        hipError_t err = hipHostMalloc(p, bytes, hipHostMallocMapped | hipHostMallocCoherent);
        if (err != hipSuccess) {
            (void)hipGetLastError();
            give_back();
            err = hipHostMalloc(p, bytes, hipHostMallocMapped | hipHostMallocCoherent);
        }
        return err;
    }
    void host_free(void* p, size_t bytes) {
        if (p && !keep(kept_host, kKeepHost, p, bytes)) {
            forget(p);
            (void)hipHostFree(p);
        }
    }
    // Words that an upload's checks set (2, pinned, zeroed), kept with the engine whether or not it has
    // a budget: making them takes longer than a small upload.
    std::vector<int*> flags;  // free ones, guarded by mu
    hipError_t take_flags(int** f) {
        {
            std::lock_guard<std::mutex> lk(mu);
            if (!flags.empty()) {
                *f = flags.back();
                flags.pop_back();
            }
        }
        const hipError_t err = *f ? hipSuccess : hipHostMalloc((void**)f, 2 * sizeof(int), hipHostMallocMapped | hipHostMallocCoherent);
        if (err == hipSuccess) (*f)[0] = (*f)[1] = 0;
        return err;
    }
    void give_flags(int* f) {
        if (!f) return;
        std::lock_guard<std::mutex> lk(mu);
        flags.push_back(f);
    }
    void forget(void* p) {
        std::lock_guard<std::mutex> lk(mu);
        sizes.erase(p);
    }

    int alloc(void** p, size_t bytes) {
        {
            std::lock_guard<std::mutex> lk(mu);
            if (budget && used + bytes > budget)
                return fail(LC2E_ERR_BUDGET, "HBM budget exceeded: %zu used + %zu requested > %zu",
                            used, bytes, budget);
            used += bytes;  // reserved before the allocation, returned if it fails
        }
        const hipError_t err = raw_alloc(p, bytes, true);
        if (err != hipSuccess) {
            std::lock_guard<std::mutex> lk(mu);
            used -= bytes;
            return fail(LC2E_ERR_HIP, "hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(err));
        }
        return LC2E_OK;
    }
    void release(void* p, size_t bytes) {
        if (p) {
            raw_free(p, bytes);
            std::lock_guard<std::mutex> lk(mu);
            used -= bytes;
        }
    }
};

struct lc2e_volume {
    lc2e_engine* e = nullptr;
    void* d = nullptr;
    size_t bytes = 0;
    int f16 = 0;
    bool large = false;  // a voxel exceeds kHalfRange
    lc2e_geom g{};
};

struct GraphEntry {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

struct lc2e_pair {
    lc2e_engine* e = nullptr;
    lc2e_volume* fixed = nullptr;
    lc2e_volume* moving = nullptr;
    lc2e_pair_info info{};
    lc2e::VGeom v{};
    lc2e::SGeom sg{};
    float* stat_img = nullptr;
    float* stat_grad = nullptr;
    double* ustat = nullptr;  // [2][V]: patch mean and centred energy of a static ultrasound
    size_t vbytes = 0;
    // 3D z-chunk: forced for every launch (lc2e_pair_set_tuning), else the value tuned for
    // the launch's batch size (lc2e_pair_autotune / lc2e_pair_set_tuning_n), else a model
    int zchunk_forced = 0;
    std::map<int, int> tuned;
    std::map<int, int> model_cache;  // the launch model's z-chunk per batch size
    int last_zchunk = 0;
    // batch buffers
    int cap = 0;
    int part_bpp = 0;  // partial sums per pose the partials buffer holds
    float* d_mats = nullptr;
    double* d_partials = nullptr;
    float* h_mats = nullptr;   // pinned, mapped and coherent; with h_out a block of h_bytes
    double* h_out = nullptr;
    size_t h_bytes = 0;
    float* h_mats_dev = nullptr;   // their device addresses
    double* h_out_dev = nullptr;
    double* h_part = nullptr;      // pinned, mapped and coherent: kHostPartials partials
    double* h_part_dev = nullptr;
    size_t cap_bytes = 0;
    bool use_graph = false;
    std::map<int, GraphEntry> graphs;
    // changes whenever captured launches of this pair go stale (buffers or decomposition
    // changed); unique across pairs, so a graph cached by address is never reused for
    // another pair
    std::atomic<unsigned long long> gen = 0;
    // mutual information (patchSize 0): extremes of the static image, per-pose extremes,
    // joint histograms and results, sized for mi_cap poses of mi_bins counters
    int* mi_ext_stat = nullptr;
    bool mi_stat_ready = false;
    int mi_cap = 0;
    size_t mi_bins = 0;
    int* mi_ext = nullptr;
    unsigned* mi_hist = nullptr;
    double* mi_out = nullptr;
    float* mi_warp = nullptr;  // warped images of mi_warp_poses poses
    int mi_warp_poses = 0;
    int mi_refused = 0;  // > 0: memory for that many was not to be had
    // two-kernel path: the warped moving image of ws_poses poses (ws_bytes each) and, if the
    // static image is the high-resolution one, its statistics; kept with the pair (see
    // make_two_kernel)
    bool two = false;
    bool two_charged = false;  // the memory below counts against the engine's budget
    bool two_required = false;  // no other path evaluates the pair
    void* ws = nullptr;
    size_t ws_bytes = 0;
    int ws_poses = 0;
    int users = 0;        // calls in progress (guarded by g_registry_mu)
    int ws_refused = 0;   // > 0: memory for that many poses was not to be had
    bool pinned = false;  // a caller's graph holds launches that use the workspace
    bool na = false;  // counted in the engine's na_pairs
    double* istat = nullptr;
    int resident_per_cu = 0;  // work-groups of the evaluation one CU holds at once (0: not queried yet)
    // separable path (radius beyond the fused kernels): grids and box-sum buffers, made at
    // pair creation
    bool sep = false;
    float* sep_grids = nullptr;    // [2][V] f32: moving image, its |Sobel|
    double* sep_sums = nullptr;    // [2][channels][V] f64
    size_t sep_grid_bytes = 0, sep_sum_bytes = 0;
    // kernel timing (eager path)
    bool profile = false;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    double prof_ms = 0.0;
    long long prof_launches = 0;

    int mats_per_pose() const { return info.per_frame_matrices ? info.n_frames : 1; }
    int role() const {
        return info.high_res_is_moving ? lc2e::kRoleMovingImage
               : istat || info.grid_ndim == 3 ? lc2e::kRoleStaticImage : lc2e::kRoleStaticImageFull;
    }
    size_t voxels() const { return vbytes / sizeof(float); }
};

namespace {

std::atomic<unsigned long long> g_generation{1};

// The pairs and engines that hold memory they can do without, for reclaim(). A pair in a call
// (users > 0) keeps its own.
std::mutex g_registry_mu;
std::set<lc2e_pair*> g_pairs;
std::set<lc2e_engine*> g_engines;
struct Use {
    lc2e_pair* p;
    explicit Use(lc2e_pair* pair) : p(pair) {
        std::lock_guard<std::mutex> lk(g_registry_mu);
        ++p->users;
    }
    ~Use() {
        std::lock_guard<std::mutex> lk(g_registry_mu);
        --p->users;
    }
};

void drop_graphs(lc2e_pair* p) {
    for (auto& kv : p->graphs) {
        if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
        if (kv.second.graph) (void)hipGraphDestroy(kv.second.graph);
    }
    p->graphs.clear();
    p->gen = g_generation.fetch_add(1);
}

// Work decomposition of one launch.
struct Tiling {
    int zchunk = 1, ntx = 0, nty = 0, nzc = 0;
    int tiles = 0;  // work-groups per pose
    int bpp = 0;    // partial sums per pose
};

int round_zchunk(int c) { return (c + lc2e::kZBlock - 1) / lc2e::kZBlock * lc2e::kZBlock; }

lc2e::FusedArgs make_args(lc2e_pair* p, const float* d_mats, double* d_partials, const Tiling& t);

// 2D launches that warp in the moments kernel itself: all of a pair without a workspace, and
// those too small to fill the device, where a second launch costs more than warping each
// pixel of the moments' row halos again (static high-resolution image, 256x256, 64 poses: 42 us
// in place, 58 us through the grid; moving, 128 frames 512x384, r = 6, 3 poses: 1.99 ms in
// place, 1.59 ms through the grid). The same values either way, bit for bit.
constexpr long long kInPlaceWaves = 2048;
struct Workspace {
    void* d;
    int poses;
};
// Launches of more poses than the workspace holds go through it in equal parts; `part` is their
// size, and what decides on a launch's shape.
int part(const Workspace& w, int n) {
    const int parts = w.poses > 0 ? (n + w.poses - 1) / w.poses : 1;
    return (n + parts - 1) / parts;
}
bool in_place(const lc2e_pair* p, const Workspace& w, int tiles, int n) {
    return p->info.grid_ndim == 2 && (!w.d || (long long)tiles * 4 * part(w, n) < kInPlaceWaves);
}

// The pair's evaluation kernels for n poses: the moments kernels after a warp into the workspace
// (or in place), the fused kernel, or the separable path.
hipError_t launch_eval(lc2e_pair* p, const lc2e::FusedArgs& a, int n, hipStream_t st, const Workspace& w) {
    if (p->two && in_place(p, w, a.tiles, n)) {
        lc2e::FusedArgs s = a;
        s.in_place = 1;
        return lc2e::launch_moments(s, p->info.grid_ndim, p->role(), n, st);
    }
    if (p->two) {
        // (a launch has less than 2^32 work-items, of which the moments kernels take up to 1024
        // per tile and pose)
        const long long tiles8 = (a.tiles + lc2e::kXcds - 1) / lc2e::kXcds * (long long)lc2e::kXcds;
        const int most = (int)std::max(1LL, std::min<long long>(1 << 30, ((1LL << 22) - 1) / std::max(1LL, tiles8)));
        const int step = std::min(part(w, n), most);
        for (int b = 0; b < n; b += step) {
            const int m = std::min(step, n - b);
            lc2e::FusedArgs s = a;
            s.warp2 = static_cast<float2*>(w.d);
            s.warp1 = static_cast<float*>(w.d);
            s.mats = a.mats + (size_t)b * a.mats_per_pose * 12;
            if (b) s.inline_mat = 0;
            s.partials = a.partials + (size_t)b * a.blocks_per_pose * 2;
            hipError_t err = lc2e::launch_warp_grid(s, p->info.grid_ndim, p->info.src_ndim,
                                                    p->info.high_res_is_moving, m, st);
            if (err == hipSuccess) err = lc2e::launch_moments(s, p->info.grid_ndim, p->role(), m, st);
            if (err != hipSuccess) return err;
        }
        return hipSuccess;
    }
    if (p->sep)
        return lc2e::launch_sep(a, p->info.grid_ndim, p->info.src_ndim, p->info.high_res_is_moving, n,
                                st);
    if (p->info.grid_ndim == 2) return lc2e::launch_fused2(a, p->info.src_ndim, n, st);
    return lc2e::launch_fused(a, p->info.high_res_is_moving, n, st);
}

// Fused work-groups one CU holds at once for this pair's kernel (queried once, then kept).
int resident_per_cu(lc2e_pair* p) {
    if (p->sep) return 1;  // the separable path's launches fill the device by themselves
    if (p->resident_per_cu <= 0) {
        const lc2e::FusedArgs a = make_args(p, nullptr, nullptr, Tiling{});
        int per_cu = 0;
        const hipError_t err =
            p->two ? lc2e::moments_resident_per_cu(a, p->info.grid_ndim, p->role(), &per_cu)
            : p->info.grid_ndim == 2 ? lc2e::fused2_resident_per_cu(a, p->info.src_ndim, &per_cu)
                                     : lc2e::fused_resident_per_cu(a, p->info.high_res_is_moving, &per_cu);
        if (err != hipSuccess || per_cu <= 0)
            per_cu = 1;
        p->resident_per_cu = per_cu;
    }
    return p->resident_per_cu;
}

// z-chunk for a launch of n poses when nothing is tuned. A work-group of chunk c marches
// min(c, planes left) + 2R + 4 plane steps (fused kernel), or as many planes and its pipeline's
// fill (two-kernel path: 4 planes' worth with a moving high-resolution image, 8 with a static
// one; against every chunk at 588 launches of 7 grids, radii 1 to 6, 1 to 32 poses the choice is
// 0.5% off the fastest on average and 7% and 13% at worst, 8 planes for both 1.1% and 21%).
// Work-groups go to the XCDs round-robin by id and, within an XCD, to the first free slot in id
// order (map_block: tile-major, the poses of a tile consecutive; tiles ordered by z-chunk), each
// CU holding resident_per_cu of them. The model replays that dispatch with a min-heap of slot finishing times per XCD and takes
// the latest finish; launches of more than 32 rounds fall back to rounds x steps. Minimise
// over the chunk lengths (multiples of kZBlock; ties: longer chunks). Cached per launch size.
int model_zchunk(lc2e_pair* p, int n) {
    auto hit = p->model_cache.find(n);
    if (hit != p->model_cache.end()) return hit->second;
    const int r = p->info.patch_radius;
    const int ez = p->v.Z - 2 * r;
    int ntx, nty, nzc;
    if (ez <= 0 || lc2e::fused_blocks_3d(p->v, r, ez, &ntx, &nty, &nzc) <= 0) return lc2e::kZBlock;
    const long long cols = (long long)ntx * nty;
    const int cus = p->e->cus > 0 ? p->e->cus : 256;
    const int per_xcd = std::max(1, cus / lc2e::kXcds * resident_per_cu(p));
    const int cmax = round_zchunk(ez);
    const double extra = !p->two ? 2 * r + 4.0 : p->info.high_res_is_moving ? 4.0 : 8.0;
    int best = cmax;
    double best_cost = -1.0;
    std::vector<double> heap;
    for (int c = cmax; c >= lc2e::kZBlock; c -= lc2e::kZBlock) {
        const int chunks = (ez + c - 1) / c;
        const long long tiles = cols * chunks;
        const long long tiles8 = (tiles + lc2e::kXcds - 1) / lc2e::kXcds * lc2e::kXcds;
        const long long rounds = (tiles8 / lc2e::kXcds * n + per_xcd - 1) / per_xcd;
        double cost = 0.0;
        if (rounds > 32) {
            cost = (double)rounds * (c + extra);
        } else {
            for (int x = 0; x < lc2e::kXcds; ++x) {
                heap.assign(per_xcd, 0.0);  // a min-heap of slot finishing times
                for (long long t = x; t < tiles8; t += lc2e::kXcds) {
                    const double len = t >= tiles ? 0.5
                        : (double)std::min<long long>(c, ez - (t / cols) * c) + extra;
                    for (int k = 0; k < n; ++k) {
                        std::pop_heap(heap.begin(), heap.end(), std::greater<double>());
                        heap.back() += len;
                        std::push_heap(heap.begin(), heap.end(), std::greater<double>());
                    }
                }
                cost = std::max(cost, *std::max_element(heap.begin(), heap.end()));
            }
        }
        if (best_cost < 0.0 || cost < best_cost) {
            best_cost = cost;
            best = c;
        }
    }
    p->model_cache[n] = best;
    return best;
}

// `poses`: what the launch's workspace holds (0: it has none). The partial sums do not depend on
// n or poses.
Tiling tiling_for(lc2e_pair* p, int n, int poses) {
    Tiling t;
    const int r = p->info.patch_radius;
    if (p->sep) {  // one partial per 256 output voxels
        t.tiles = t.bpp = lc2e::sep_blocks(p->v, r, p->info.grid_ndim);
        return t;
    }
    if (p->info.grid_ndim == 3) {
        auto it = p->tuned.find(n);
        t.zchunk = round_zchunk(p->zchunk_forced > 0 ? p->zchunk_forced
                                : it != p->tuned.end() ? it->second
                                : model_zchunk(p, p->two ? part({nullptr, poses}, n) : n));
        t.tiles = lc2e::fused_blocks_3d(p->v, r, t.zchunk, &t.ntx, &t.nty, &t.nzc);
        t.bpp = lc2e::fused_partials_3d(p->v, r);
        p->last_zchunk = t.zchunk;
    } else {
        // one work-group and one partial per tile and run of kFrameRun frames (fixed, so
        // that the summation order does not depend on the batch)
        const int tf = lc2e::fused_blocks_2d(p->v, r, &t.ntx, &t.nty);
        t.zchunk = p->v.Z < lc2e::kFrameRun ? p->v.Z : lc2e::kFrameRun;
        t.nzc = tf > 0 ? (p->v.Z + t.zchunk - 1) / t.zchunk : 0;
        t.tiles = t.bpp = t.ntx * t.nty * t.nzc;
    }
    if (p->two) {
        lc2e::FusedArgs a{};
        a.v = p->v;
        a.r = r;
        a.zchunk = t.zchunk;
        lc2e::moments_tiling(&a, p->info.grid_ndim, p->role());
        t.zchunk = a.zchunk;
        t.ntx = a.ntx;
        t.nty = a.nty;
        t.nzc = a.nzc;
        t.tiles = a.tiles;
        t.bpp = a.blocks_per_pose;
    }
    return t;
}

// Partial sums per pose by which the allocation-free entry point admits a call, of the kernels it
// was specified with: one per 16x16 tile and 16 frames (2D), per wave of a 16x16 tile and 8 planes
// (3D), or per 256 outputs (radii beyond both). What is admitted does not depend on the kernel.
size_t admitted_partials(const lc2e_pair* p) {
    const int r = p->info.patch_radius;
    if (p->sep || (p->info.grid_ndim == 3 && r > lc2e::kMaxR3)) return lc2e::sep_blocks(p->v, r, p->info.grid_ndim);
    if (p->info.grid_ndim == 3) return lc2e::fused_partials_3d(p->v, r);
    int ntx, nty;
    lc2e::fused_blocks_2d(p->v, r, &ntx, &nty);
    return (size_t)ntx * nty * ((p->v.Z + lc2e::kFrameRun - 1) / lc2e::kFrameRun);
}

// The partial sums per pose of every launch of the pair (tiling_for without a choice of chunks; 0:
// no patch centre fits).
int partials_per_pose(lc2e_pair* p) {
    if (p->sep || p->info.grid_ndim == 2) {
        const Tiling t = tiling_for(p, 1, 0);
        return t.tiles > 0 ? t.bpp : 0;
    }
    if (!p->two) return lc2e::fused_partials_3d(p->v, p->info.patch_radius);
    lc2e::FusedArgs a{};
    a.v = p->v;
    a.r = p->info.patch_radius;
    a.zchunk = lc2e::kZBlock;
    lc2e::moments_tiling(&a, 3, p->role());
    return a.tiles > 0 ? a.blocks_per_pose : 0;
}

// Launches of at most kHostPartials partials, kHostPose per pose, add them up on the host
// (enqueue_batch).
constexpr int kDirectPoses = 32;
constexpr int kHostPose = 256;
constexpr size_t kHostPartials = 2048;

void free_batch(lc2e_pair* p) {
    drop_graphs(p);
    lc2e_engine* e = p->e;
    if (p->d_mats) e->release(p->d_mats, (size_t)p->cap * p->mats_per_pose() * 12 * sizeof(float));
    if (p->d_partials) e->release(p->d_partials, (size_t)p->cap * p->part_bpp * 2 * sizeof(double));
    e->host_free(p->h_mats, p->h_bytes);
    e->host_free(p->h_part, kHostPartials * 2 * sizeof(double));
    p->h_part = nullptr;
    p->h_part_dev = nullptr;
    p->d_mats = nullptr;
    p->d_partials = nullptr;
    p->h_mats = nullptr;
    p->h_out = nullptr;
    p->h_mats_dev = nullptr;
    p->h_out_dev = nullptr;
    p->cap = 0;
    p->part_bpp = 0;
    p->pinned = false;  // captured launches hold these buffers too
}

void free_mi_warp(lc2e_pair* p) {
    if (p->mi_warp) p->e->raw_free(p->mi_warp, (size_t)p->mi_warp_poses * p->voxels() * sizeof(float));
    p->mi_warp = nullptr;
    p->mi_warp_poses = 0;
}

void free_mi(lc2e_pair* p) {
    lc2e_engine* e = p->e;
    if (p->mi_ext) e->release(p->mi_ext, (size_t)p->mi_cap * 2 * sizeof(int));
    if (p->mi_hist) e->release(p->mi_hist, (size_t)p->mi_cap * p->mi_bins * sizeof(unsigned));
    if (p->mi_out) e->release(p->mi_out, (size_t)p->mi_cap * sizeof(double));
    p->mi_ext = nullptr;
    p->mi_hist = nullptr;
    p->mi_out = nullptr;
    p->mi_cap = 0;
    p->mi_bins = 0;
}

// Memory of the two-kernel path beside the budgeted buffers.
int two_alloc(lc2e_pair* p, void** d, size_t bytes) {
    if (p->two_charged) return p->e->alloc(d, bytes);
    if (p->e->raw_alloc(d, bytes, p->two_required) == hipSuccess) return LC2E_OK;
    (void)hipGetLastError();
    return fail(LC2E_ERR_HIP, "workspace of %zu bytes", bytes);
}
void two_free(lc2e_pair* p, void* d, size_t bytes) {
    if (!d) return;
    if (p->two_charged) p->e->release(d, bytes);
    else p->e->raw_free(d, bytes);  // waits for launches that use it
}

// The workspace for n poses, up to kWorkspaceBytes (at least one pose); larger launches go
// through it in parts. Only an engine without an HBM budget grows it past one pose.
constexpr size_t kWorkspaceBytes = size_t(1) << 30;
constexpr size_t kMiWarpBytes = size_t(1) << 28;  // warped images of the mutual information
// The allocation-free entry point's workspace is made with the pair, so its size cannot follow the
// batches: 64 poses within 512 MiB, at least one. A fresh pair's first call, 32 poses: 64^3, R = 3
// 1820 -> 166 us against parts of one pose (148 in a batch); 192x192x160 4.45 -> 3.10 ms (3.19 with
// 256 MiB, 2.78 in a batch).
constexpr size_t kNoallocBytes = size_t(1) << 29;
constexpr int kNoallocPoses = 64;
int grow_workspace(lc2e_pair* p, int n) {
    if (p->e->budget) {
        if (!p->two_charged) return LC2E_OK;
        n = 1;
    }
    const size_t per = p->voxels() * (p->info.high_res_is_moving ? sizeof(float2) : sizeof(float));
    const int want = (int)std::min<size_t>((size_t)std::max(n, 1), std::max<size_t>(1, kWorkspaceBytes / per));
    if (want <= p->ws_poses || p->pinned || (p->ws_refused && want >= p->ws_refused)) return LC2E_OK;
    void* d = nullptr;
    const int rc = two_alloc(p, &d, (size_t)want * per);
    if (rc < 0) {
        p->ws_refused = want;  // not tried again on every call
        return p->ws ? LC2E_OK : rc;  // what is there still serves
    }
    if (p->ws) {
        drop_graphs(p);
        two_free(p, p->ws, (size_t)p->ws_poses * p->ws_bytes);
    }
    p->ws = d;
    p->ws_bytes = per;
    p->ws_poses = want;
    return LC2E_OK;
}

std::mutex& noalloc_lock(int device) {
    static std::mutex locks[64];
    return locks[device & 63];
}

// Room in the engine's workspace of the allocation-free entry point for poses of the pair.
// Its calls do not touch the pair's own workspace, which launches on a caller's stream may be
// using at the same time.
int reserve_noalloc(lc2e_pair* p) {
    lc2e_engine* e = p->e;
    std::lock_guard<std::mutex> lk(noalloc_lock(e->device));
    const size_t most = std::max(p->ws_bytes, std::min(kNoallocBytes, kNoallocPoses * p->ws_bytes));
    for (size_t bytes : {most, p->ws_bytes}) {
        if (e->na_bytes >= bytes) break;
        void* d = nullptr;
        if (e->raw_alloc(&d, bytes, false) != hipSuccess) {
            (void)hipGetLastError();
            continue;
        }
        e->raw_free(e->na, e->na_bytes);
        e->na = d;
        e->na_bytes = bytes;
    }
    if (e->na_bytes < p->ws_bytes) return fail(LC2E_ERR_HIP, "workspace of %zu bytes", p->ws_bytes);
    p->na = true;
    ++e->na_pairs;
    return LC2E_OK;
}
void release_noalloc(lc2e_pair* p) {
    if (!p->na) return;
    lc2e_engine* e = p->e;
    std::lock_guard<std::mutex> lk(noalloc_lock(e->device));
    p->na = false;
    if (--e->na_pairs || e->na_bytes <= kNoallocBytes) return;  // kept for the next pair
    e->raw_free(e->na, e->na_bytes);
    e->na = nullptr;
    e->na_bytes = 0;
}
// Under noalloc_lock. Without a reservation: 2D launches warp in place; the others share the
// pair's workspace, as radii beyond the fused kernels share their box-sum buffers.
Workspace noalloc_workspace(const lc2e_pair* p) {
    const size_t poses = p->na ? p->e->na_bytes / p->ws_bytes : 0;
    if (poses) return {p->e->na, (int)std::min<size_t>(poses, 1 << 20)};
    if (p->info.grid_ndim == 2) return {nullptr, 0};
    return {p->ws, p->ws_poses};
}

void free_two(lc2e_pair* p) {
    release_noalloc(p);
    two_free(p, p->ws, (size_t)p->ws_poses * p->ws_bytes);
    two_free(p, p->istat, lc2e::kImageStats * p->voxels() * sizeof(double));
    p->ws = nullptr;
    p->istat = nullptr;
    p->ws_poses = 0;
    p->two = false;
}

// Gives back memory of an idle pair (under g_registry_mu): the mutual information's warped images
// and the workspace beyond one pose, whose absence changes no value; with `all` the rest of the
// two-kernel path's, after which 2D pairs warp in place (the same bits) and 3D pairs run the fused
// kernel (the same to rounding). False if there was nothing.
bool shrink(lc2e_pair* p, bool all) {
    if (p->mi_warp) {
        free_mi_warp(p);
        p->mi_refused = 1;
        return true;
    }
    if (p->two_charged || p->pinned) return false;
    if (!all && p->ws_poses > 1) {
        drop_graphs(p);
        two_free(p, p->ws, (size_t)p->ws_poses * p->ws_bytes);
        p->e->give_back();
        p->ws = nullptr;
        p->ws_poses = 0;
        p->ws_refused = 2;
        if (hipMalloc(&p->ws, p->ws_bytes) == hipSuccess) {
            p->ws_poses = 1;
        } else {
            (void)hipGetLastError();
            p->ws = nullptr;
            free_two(p);
            p->two = p->info.grid_ndim == 2;
        }
        return true;
    }
    if (!all || p->two_required || (!p->ws && !p->istat)) return false;
    drop_graphs(p);
    free_two(p);
    p->two = p->info.grid_ndim == 2;
    p->resident_per_cu = 0;
    p->model_cache.clear();
    return true;
}

// The allocation-free entry point's workspace down to one pose of the pairs that use it.
bool shrink_noalloc(lc2e_engine* e) {
    size_t one = 0;
    for (const lc2e_pair* p : g_pairs)
        if (p->e == e && p->na) one = std::max(one, p->ws_bytes);
    std::lock_guard<std::mutex> lk(noalloc_lock(e->device));
    if (e->na_bytes <= one) return false;
    e->raw_free(e->na, e->na_bytes);
    e->give_back();
    e->na = nullptr;
    e->na_bytes = 0;
    if (!one) return true;
    if (hipMalloc(&e->na, one) == hipSuccess) e->na_bytes = one;
    else (void)hipGetLastError(), e->na = nullptr;
    return true;
}

bool reclaim(int device) {
    std::lock_guard<std::mutex> lk(g_registry_mu);
    for (lc2e_engine* e : g_engines)
        if (e->device == device && (e->give_back() || shrink_noalloc(e))) return true;
    for (bool all : {false, true})
        for (lc2e_pair* p : g_pairs)
            if (p->e->device == device && !p->users && shrink(p, all)) return true;
    return false;
}

lc2e::FusedArgs make_args(lc2e_pair* p, const float* d_mats, double* d_partials, const Tiling& t);

// A role of the two-kernel path's moments that writes statistics of a static image.
hipError_t launch_stats(lc2e_pair* p, int role, hipStream_t st) {
    lc2e::FusedArgs a = make_args(p, nullptr, nullptr, Tiling{});
    a.zchunk = 32;  // planes per work-group (3D)
    a.istat_out = p->istat;
    a.ustat_mean_out = p->ustat;
    a.ustat_cyy_out = p->ustat + p->voxels();
    lc2e::moments_tiling(&a, p->info.grid_ndim, role);
    return lc2e::launch_moments(a, p->info.grid_ndim, role, 1, st);
}

// Sets the moments path up. 2D pairs use it from the radii on at which it is faster than the
// fused kernel (with a static high-resolution image always), and do without its memory where
// there is none (in_place). 3D radii beyond the fused kernel need its memory, which is less than the
// separable path's and charged to the budget. Other 3D radii use it on an engine without a
// budget only: under one the fused kernel, which needs no workspace, evaluates the pair, so
// what a budget admits is what it admitted without this path.
int make_two_kernel(lc2e_pair* p, bool required) {
    const bool two_d = p->info.grid_ndim == 2;
    if (two_d && p->info.high_res_is_moving && p->info.patch_radius <= lc2e::kMaxRFused2) return LC2E_OK;
    p->two_charged = required && p->e->budget;
    p->two_required = required;
    p->two = two_d;
    if (!required && p->e->budget) return LC2E_OK;
    p->two = true;
    const bool grid = !two_d || p->info.high_res_is_moving;  // else warped in place
    int rc = grid ? grow_workspace(p, 1) : LC2E_OK;
    if (rc >= 0 && p->ws && !p->two_charged && reserve_noalloc(p) < 0 && !two_d && !required) rc = LC2E_ERR_HIP;
    if (rc >= 0 && !p->info.high_res_is_moving)
        rc = two_alloc(p, (void**)&p->istat, lc2e::kImageStats * p->voxels() * sizeof(double));
    if (rc < 0) {
        free_two(p);
        p->two = two_d;
    }
    return rc < 0 && required ? rc : LC2E_OK;
}

// Batch buffers for n poses whose launches use up to bpp work-groups per pose.
int ensure_batch(lc2e_pair* p, int n, int bpp) {
    if (bpp < 1) bpp = 1;
    if (n <= p->cap && bpp <= p->part_bpp) return LC2E_OK;
    int cap = p->cap > 1 ? p->cap : 1;
    while (cap < n) cap *= 2;
    if (bpp < p->part_bpp) bpp = p->part_bpp;
    free_batch(p);
    lc2e_engine* e = p->e;
    const int mpp = p->mats_per_pose();
    int rc;
    if ((rc = e->alloc((void**)&p->d_mats, (size_t)cap * mpp * 12 * sizeof(float))) < 0) return rc;
    if ((rc = e->alloc((void**)&p->d_partials, (size_t)cap * bpp * 2 * sizeof(double))) < 0) {
        e->release(p->d_mats, (size_t)cap * mpp * 12 * sizeof(float));
        p->d_mats = nullptr;
        return rc;
    }
    p->cap = cap;  // free_batch returns the device bytes by these sizes
    p->part_bpp = bpp;
    // Mapped and coherent: small launches read their matrices from here and every launch's
    // reduction writes its results here, with no copy command (enqueue_batch). Two blocks: an
    // engine with a budget makes and frees them with every pair, 30 us each (with the partial sums
    // in the first one too, 4 poses 256x256, r = 3, take 0.6 us longer).
    const size_t mats_b = ((size_t)cap * mpp * 12 * sizeof(float) + 255) / 256 * 256;
    void *h = nullptr, *d = nullptr, *hp = nullptr, *dp = nullptr;
    p->h_bytes = mats_b + (size_t)cap * 3 * sizeof(double);
    hipError_t he = e->host_alloc(&h, p->h_bytes);
    p->h_mats = static_cast<float*>(h);
    if (he == hipSuccess) he = e->host_alloc(&hp, kHostPartials * 2 * sizeof(double));
    p->h_part = static_cast<double*>(hp);
    if (he == hipSuccess) he = hipHostGetDevicePointer(&d, h, 0);
    if (he == hipSuccess) he = hipHostGetDevicePointer(&dp, hp, 0);
    if (he == hipSuccess) {
        p->h_out = reinterpret_cast<double*>(static_cast<char*>(h) + mats_b);
        p->h_mats_dev = static_cast<float*>(d);
        p->h_out_dev = reinterpret_cast<double*>(static_cast<char*>(d) + mats_b);
        p->h_part_dev = static_cast<double*>(dp);
    }
    if (he != hipSuccess) {
        free_batch(p);  // no half-made buffers: the next call allocates again
        return fail(LC2E_ERR_HIP, "pinned staging allocation of %d poses failed: %s", cap,
                    hipGetErrorString(he));
    }
    return LC2E_OK;
}

// The same for launches of the pair's kernels, and the workspace. A launch that a caller captures
// takes the workspace as it is (nothing may be allocated then), and keeps it where it is.
int ensure_capacity(lc2e_pair* p, int n, bool captured = false) {
    const int rc = ensure_batch(p, n, partials_per_pose(p));
    if (rc < 0 || !p->ws) return rc;
    if (captured) p->pinned = true;
    else (void)grow_workspace(p, n);
    return rc;
}

lc2e::FusedArgs make_args(lc2e_pair* p, const float* d_mats, double* d_partials, const Tiling& t) {
    lc2e::FusedArgs a{};
    a.v = p->v;
    a.s = p->sg;
    a.src = p->moving->d;
    a.src_f16 = p->moving->f16;
    a.stat_img = p->stat_img;
    a.stat_grad = p->stat_grad;
    const size_t V = p->vbytes / sizeof(float);
    a.ustat_mean = p->ustat;
    a.ustat_cyy = p->ustat ? p->ustat + V : nullptr;
    a.mats = d_mats;
    a.partials = d_partials;
    a.wmap = nullptr;
    a.mmap = nullptr;
    a.r = p->info.patch_radius;
    a.zchunk = t.zchunk;
    a.ntx = t.ntx;
    a.nty = t.nty;
    a.nzc = t.nzc;
    a.blocks_per_pose = t.bpp;
    a.tiles = t.tiles;
    a.mats_per_pose = p->mats_per_pose();
    a.istat = p->istat;
    a.src3 = p->info.src_ndim == 3 ? 1 : 0;
    a.in_place = p->two && !p->ws && p->info.grid_ndim == 2 ? 1 : 0;
    a.istat_stride = (long long)V;
    if (p->sep) {
        const size_t V = p->vbytes / sizeof(float);
        a.sep_img = p->sep_grids;
        a.sep_grad = p->sep_grids + V;
        a.sep_a = p->sep_sums;
        a.sep_b = p->sep_sums + (size_t)lc2e::kSepChannels(p->info.high_res_is_moving != 0) * V;
    }
    return a;
}

// Enqueue: the staged matrices to the device, the evaluation, the reduction into the pinned
// result buffer. Each launch command costs several microseconds, so small launches (up to
// kDirectPoses poses of one matrix each, on a single volume or image: each work-group reads its
// pose's 12 floats once) read the pinned matrices in place instead of copying them (13 poses
// 1.5 us less, 32 poses 2 us), and the reduction always writes the results in place: two
// commands less per batch. Where a launch is not captured, up to kInlineMats such matrices go
// with the arguments of the kernels that read them there (all but the 2D fused kernel; a read from
// pinned memory takes 1.2 us at a kernel's start: 4 poses 194x248, r = 5, 33.4 -> 31.6 us), and few
// partials go straight to pinned memory for the host to add up (*host_sum), a launch less: 13 poses
// 96x96, r = 9, 34.0 -> 30.9 us, 256x256, r = 3, static image, 37.8 -> 34.6; sums of 512 to 4096
// partials took the same.
int enqueue_batch(lc2e_pair* p, int n, const Tiling& t, hipStream_t st, bool captured, bool* host_sum) {
    const int mpp = p->mats_per_pose();
    const bool direct = !p->sep && mpp == 1 && n <= kDirectPoses &&
                        (p->info.grid_ndim == 3 || p->v.Z == 1);
    const bool host = !captured && t.tiles > 0 && t.bpp <= kHostPose && (size_t)n * t.bpp <= kHostPartials;
    *host_sum = host;
    if (!direct)
        HIP_TRY(hipMemcpyAsync(p->d_mats, p->h_mats, (size_t)n * mpp * 12 * sizeof(float),
                               hipMemcpyHostToDevice, st));
    if (t.tiles > 0) {
        lc2e::FusedArgs a = make_args(p, direct ? p->h_mats_dev : p->d_mats, host ? p->h_part_dev : p->d_partials, t);
        if (direct && n <= lc2e::kInlineMats && !captured && (p->two || p->info.grid_ndim == 3)) {
            a.inline_mat = 1;
            std::memcpy(a.m0, p->h_mats, (size_t)n * 12 * sizeof(float));
        }
        // timed launches are eager (run_batch), the events bracket the evaluation
        const bool timed = p->profile;
        if (timed) HIP_TRY(hipEventRecord(p->ev0, st));
        HIP_TRY(launch_eval(p, a, n, st, {p->ws, p->ws_poses}));
        if (timed) HIP_TRY(hipEventRecord(p->ev1, st));
        if (!host) HIP_TRY(lc2e::launch_reduce(p->d_partials, t.bpp, n, p->h_out_dev, st));
    } else {
        // no patch centre fits in the grid: every sum is zero
        HIP_TRY(lc2e::launch_reduce(p->d_partials, 0, n, p->h_out_dev, st));
    }
    return LC2E_OK;
}

// The sums of k_reduce from the partials of n poses on the host, added in its order: 256 running sums of
// every 256th partial, then halves (here at most one partial each; halvings that would only add
// the zeros past the last partial are left out).
void sum_partials(const double* partials, int n, int bpp, double* out) {
    double m[kHostPose], w[kHostPose];
    int top = 1;
    while (top < bpp) top *= 2;
    for (int i = 0; i < n; ++i) {
        const double* s = partials + (size_t)i * bpp * 2;
        for (int k = 0; k < top; ++k) {
            m[k] = k < bpp ? 0.0 + s[2 * k] : 0.0;
            w[k] = k < bpp ? 0.0 + s[2 * k + 1] : 0.0;
        }
        for (int h = top / 2; h > 0; h >>= 1)
            for (int k = 0; k < h; ++k) {
                m[k] += m[k + h];
                w[k] += w[k + h];
            }
        double l = m[0] / w[0];
        if (!std::isfinite(l)) l = 0.0;
        out[3 * i] = m[0];
        out[3 * i + 1] = w[0];
        out[3 * i + 2] = l;
    }
}

// Runs a batch of n poses staged in h_mats; the buffers must already fit tiling t.
int run_batch(lc2e_pair* p, int n, const Tiling& t) {
    hipStream_t st = p->e->stream;
    bool host_sum = false;
    if (p->use_graph && !p->profile) {
        auto it = p->graphs.find(n);
        if (it == p->graphs.end()) {
            GraphEntry g;
            HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            int rc = enqueue_batch(p, n, t, st, true, &host_sum);
            hipGraph_t graph = nullptr;
            hipError_t ce = hipStreamEndCapture(st, &graph);
            if (rc >= 0 && ce == hipSuccess) ce = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
            if (rc < 0 || ce != hipSuccess) {
                if (graph) (void)hipGraphDestroy(graph);
                if (rc < 0) return rc;
                return fail(LC2E_ERR_HIP, "graph capture failed: %s", hipGetErrorString(ce));
            }
            g.graph = graph;
            it = p->graphs.emplace(n, g).first;
        }
        HIP_TRY(hipGraphLaunch(it->second.exec, st));
    } else {
        int rc = enqueue_batch(p, n, t, st, false, &host_sum);
        if (rc < 0) return rc;
    }
    HIP_TRY(hipStreamSynchronize(st));
    if (host_sum) sum_partials(p->h_part, n, t.bpp, p->h_out);
    if (p->profile && t.tiles > 0) {
        float ms = 0.0f;
        HIP_TRY(hipEventElapsedTime(&ms, p->ev0, p->ev1));
        p->prof_ms += ms;
        p->prof_launches += 1;
    }
    return LC2E_OK;
}

}  // namespace

namespace lc2e {
// Sets the calling thread's lc2e_last_error() text (the serving loop hands a worker
// thread's message to the client that collects the request).
void set_last_error(const std::string& msg) { g_last_error = msg; }
// Device memory charged to the engine's HBM budget, for the serving loop's launch slots.
int engine_alloc(lc2e_engine* e, void** p, size_t bytes) { return e->alloc(p, bytes); }
void engine_release(lc2e_engine* e, void* p, size_t bytes) { e->release(p, bytes); }
int engine_device(lc2e_engine* e) { return e->device; }
// The share of the device one launch of n poses occupies: its work-groups over the
// work-groups all CUs hold at once (>= 1: it fills the GPU by itself). The serving loop
// runs launches side by side only while their shares add up to at most 1.
// Generation of the pair's launch state: graphs captured under another generation are stale.
unsigned long long pair_generation(lc2e_pair* p) { return p->gen; }
// Make the pair's batch buffers fit n poses now, so that a following
// lc2e_eval_batch_async of n poses allocates nothing (e.g. under stream capture).
int pair_prepare(lc2e_pair* p, int n) {
    Use use(p);
    const int rc = ensure_capacity(p, n);
    if (rc >= 0 && p->ws) {  // once captured it stays as it is
        (void)grow_workspace(p, p->cap);
        p->pinned = true;
    }
    return rc;
}
double launch_share(lc2e_pair* p, int n) {
    Use use(p);
    const Tiling t = tiling_for(p, n, p->ws_poses);
    if (t.tiles <= 0 || n <= 0) return 0.0;
    const int per_cu = resident_per_cu(p);
    const bool fused2 = p->info.grid_ndim == 2 && !p->two && !p->sep;
    const int prun = fused2 ? pose_run(p->v, p->info.src_ndim, p->mats_per_pose(), t.tiles, n) : 1;
    const double wgs = (double)((t.tiles + kXcds - 1) / kXcds * kXcds) * ((n + prun - 1) / prun);
    const int cus = p->e->cus > 0 ? p->e->cus : 256;
    return wgs / ((double)cus * per_cu);
}
}  // namespace lc2e

extern "C" {

const char* lc2e_last_error(void) { return g_last_error.c_str(); }

int lc2e_create(int device, size_t hbm_budget_bytes, lc2e_engine** out) {
    if (!out) return fail(LC2E_ERR_INVALID, "null output handle");
    int ndev = 0;
    HIP_TRY(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev)
        return fail(LC2E_ERR_INVALID, "device %d out of range (%d devices)", device, ndev);
    auto* e = new lc2e_engine();
    e->device = device;
    e->budget = hbm_budget_bytes;
    hipError_t err = hipSetDevice(device);
    if (err == hipSuccess)
        err = hipDeviceGetAttribute(&e->cus, hipDeviceAttributeMultiprocessorCount, device);
    if (err == hipSuccess) err = hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking);
    if (err != hipSuccess) {
        delete e;
        return fail(LC2E_ERR_HIP, "stream creation failed: %s", hipGetErrorString(err));
    }
    // the allocation-free entry point's device scratch: its address on this device, looked
    // up once per device (with the device current) and kept
    const hipError_t se = lc2e::scratch_address(device, &e->scratch);
    if (se != hipSuccess) {
        e->scratch = nullptr;
        e->scratch_error = hipGetErrorString(se);
    }
    {
        std::lock_guard<std::mutex> lk(g_registry_mu);
        g_engines.insert(e);
    }
    *out = e;
    return LC2E_OK;
}

void lc2e_destroy(lc2e_engine* e) {
    if (!e) return;
    {
        std::lock_guard<std::mutex> lk(g_registry_mu);
        g_engines.erase(e);
    }
    (void)hipSetDevice(e->device);
    (void)hipStreamSynchronize(e->stream);
    (void)hipStreamDestroy(e->stream);
    e->raw_free(e->na, e->na_bytes);
    e->give_back();
    for (int* f : e->flags) (void)hipHostFree(f);
    delete e;
}

int lc2e_memory(lc2e_engine* e, size_t* used, size_t* budget) {
    if (!e) return fail(LC2E_ERR_INVALID, "null engine");
    std::lock_guard<std::mutex> lk(e->mu);
    if (used) *used = e->used;
    if (budget) *budget = e->budget;
    return LC2E_OK;
}

int lc2e_volume_upload(lc2e_engine* e, const void* host, lc2e_dtype dtype, const lc2e_geom* geom,
                       lc2e_dtype storage, lc2e_volume** out) {
    if (!e || !host || !geom || !out) return fail(LC2E_ERR_INVALID, "null argument");
    const int dsz = dtype_size(dtype);
    if (!dsz) return fail(LC2E_ERR_INVALID, "unknown dtype %d", (int)dtype);
    for (int a = 0; a < 3; ++a) {
        if (geom->dims[a] <= 0) return fail(LC2E_ERR_INVALID, "dims must be positive");
        // the samplers form row and voxel offsets with 24-bit multiplies
        if (geom->dims[a] >= (1 << 24))
            return fail(LC2E_ERR_UNSUPPORTED, "dimension %d exceeds 2^24 - 1", geom->dims[a]);
        if (!(geom->spacing[a] > 0.0f)) return fail(LC2E_ERR_INVALID, "spacing must be positive");
    }
    const long long n = (long long)geom->dims[0] * geom->dims[1] * geom->dims[2];
    if (n >= (1LL << 31)) return fail(LC2E_ERR_UNSUPPORTED, "volume exceeds 2^31 voxels");
    if (storage != LC2E_STORE_AUTO && storage != LC2E_F16 && storage != LC2E_F32)
        return fail(LC2E_ERR_INVALID, "storage must be F16, F32 or AUTO");
    HIP_TRY(hipSetDevice(e->device));
    // The raw voxels on the device (also its conversion's input) and two words that the kernels
    // set where a voxel is out of range (launch_check): the device reads them at the memory's rate,
    // where a scan on the host took half of an upload.
    struct Scope {
        lc2e_engine* e;
        void* staging = nullptr;
        size_t bytes = 0;
        int* flag = nullptr;
        ~Scope() {
            e->raw_free(staging, bytes);
            if (idle) e->give_flags(flag);  // no kernel of a failed upload may still set it
            else if (flag && hipDeviceSynchronize() == hipSuccess) e->give_flags(flag);
        }
        bool idle = false;
    } tmp{e};
    HIP_TRY(e->take_flags(&tmp.flag));
    void* flag_dev = nullptr;
    HIP_TRY(hipHostGetDevicePointer(&flag_dev, tmp.flag, 0));
    auto stage = [&]() {
        tmp.bytes = (size_t)n * dsz;
        hipError_t err = e->raw_alloc(&tmp.staging, tmp.bytes, true);
        if (err == hipSuccess)
            err = hipMemcpyAsync(tmp.staging, host, tmp.bytes, hipMemcpyHostToDevice, e->stream);
        return err;
    };
    int f16;
    if (storage == LC2E_STORE_AUTO) {
        f16 = (dtype == LC2E_U8 || dtype == LC2E_F16) ? 1 : 0;
        if (dtype == LC2E_I16) {
            // every integer in [-2048, 2048] is exact in half precision (11-bit significand),
            // which covers CT in Hounsfield units: half storage is then lossless. The first voxels
            // are looked at here: all of a small volume, and often enough to tell.
            constexpr long long kFirst = 32768;
            const short* h = static_cast<const short*>(host);
            f16 = 1;
            for (long long i = 0; i < std::min(n, kFirst) && f16; ++i)
                if (h[i] < -2048 || h[i] > 2048) f16 = 0;
            if (f16 && n > kFirst) {
                hipError_t err = stage();
                if (err == hipSuccess)
                    err = lc2e::launch_check(tmp.staging, dtype, n, 2048.0f, (int*)flag_dev, e->stream);
                if (err == hipSuccess) err = hipStreamSynchronize(e->stream);
                if (err != hipSuccess) return fail(LC2E_ERR_HIP, "volume upload failed: %s", hipGetErrorString(err));
                f16 = *tmp.flag ? 0 : 1;
                *tmp.flag = 0;
            }
        }
    }
    else f16 = storage == LC2E_F16;
    // the samplers address a volume and its zeroed tail with 32-bit byte offsets
    const long long pad = lc2e::volume_pad_elems(geom->dims[0], geom->dims[1]);
    if ((n + pad) * (f16 ? 2 : 4) > 0xffffffffLL)
        return fail(LC2E_ERR_UNSUPPORTED,
                    "volume of %lld voxels (plus a %lld-voxel zeroed tail) exceeds the 4 GiB "
                    "that %s storage can address%s", n, pad, f16 ? "f16" : "f32",
                    f16 ? "" : "; store it as F16");
    // The samplers rely on finite voxels (a zero-weight corner must contribute exactly 0): the
    // largest magnitude admitted, and the error that names the first voxel past it.
    const float lim = dtype == LC2E_F32 && !f16 ? 3.4028235e38f : 65504.0f;
    const bool check = dtype == LC2E_F32 || dtype == LC2E_F16;
    auto bad_voxel = [&]() {
        if (dtype == LC2E_F32) {
            const float* h = static_cast<const float*>(host);
            for (long long i = 0; i < n; ++i)
                if (!(std::fabs(h[i]) <= lim))
                    return fail(LC2E_ERR_INVALID, "value %g at %lld is not finite%s", h[i], i,
                                f16 ? " in half storage" : "");
        } else if (dtype == LC2E_F16) {
            const unsigned short* h = static_cast<const unsigned short*>(host);
            for (long long i = 0; i < n; ++i)
                if ((h[i] & 0x7c00u) == 0x7c00u)
                    return fail(LC2E_ERR_INVALID, "half value 0x%04x at %lld is not finite", h[i], i);
        }
        return LC2E_OK;
    };
    auto* v = new lc2e_volume();
    v->e = e;
    v->g = *geom;
    v->f16 = f16;
    const size_t esz = f16 ? 2 : 4;
    v->bytes = (size_t)(n + pad) * esz;
    int rc = e->alloc(&v->d, v->bytes);
    if (rc < 0) {
        delete v;
        const std::string why = g_last_error;
        const int bad = bad_voxel();  // an invalid volume is invalid whether it fits or not
        if (bad >= 0) g_last_error = why;
        return bad < 0 ? bad : rc;
    }
    // zeroed tail (lc2e::volume_pad_elems): the samplers' reads past the last voxel
    hipError_t err = hipMemsetAsync(static_cast<char*>(v->d) + (size_t)n * esz, 0, (size_t)pad * esz, e->stream);
    if (dtype == (f16 ? LC2E_F16 : LC2E_F32)) {  // stored as it comes
        if (err == hipSuccess)
            err = hipMemcpyAsync(v->d, host, (size_t)n * dsz, hipMemcpyHostToDevice, e->stream);
        if (err == hipSuccess) err = lc2e::launch_check(v->d, dtype, n, lim, (int*)flag_dev, e->stream);
    } else {
        if (err == hipSuccess && !tmp.staging) err = stage();
        if (err == hipSuccess && check)
            err = lc2e::launch_check(tmp.staging, dtype, n, lim, (int*)flag_dev, e->stream);
        if (err == hipSuccess)
            err = lc2e::launch_convert(tmp.staging, (int)dtype, v->d, f16, n, e->stream);
    }
    if (err == hipSuccess) err = hipStreamSynchronize(e->stream);
    tmp.idle = err == hipSuccess;
    if (err != hipSuccess || *tmp.flag) {
        e->release(v->d, v->bytes);
        delete v;
        if (err == hipSuccess && (rc = bad_voxel()) < 0) return rc;
        return fail(LC2E_ERR_HIP, "volume upload failed: %s", hipGetErrorString(err));
    }
    v->large = tmp.flag[1] != 0;
    *out = v;
    return LC2E_OK;
}

void lc2e_volume_destroy(lc2e_volume* v) {
    if (!v) return;
    (void)hipStreamSynchronize(v->e->stream);
    v->e->release(v->d, v->bytes);
    delete v;
}

int lc2e_pair_create(lc2e_engine* e, lc2e_volume* fixed, lc2e_volume* moving,
                     const float resampled_spacing[3], int high_res_is_moving,
                     int center_overlaid, int patch_radius, int dim, lc2e_pair** out) {
    if (!e || !fixed || !moving || !resampled_spacing || !out)
        return fail(LC2E_ERR_INVALID, "null argument");
    if (fixed->e != e || moving->e != e) return fail(LC2E_ERR_INVALID, "volume of another engine");
    if (dim != 2 && dim != 3) return fail(LC2E_ERR_INVALID, "dim must be 2 or 3");
    if (patch_radius < 1) return fail(LC2E_ERR_INVALID, "patch radius must be >= 1 (0 selects MI, unsupported)");
    if (patch_radius > lc2e::kMaxRSep)
        return fail(LC2E_ERR_UNSUPPORTED, "patch radius %d > %d", patch_radius, lc2e::kMaxRSep);
    // radii beyond the fused kernels, and 3D sources whose slices hold 2^24 voxels or more
    // (beyond the fused samplers' 24-bit offsets), take the separable path
    const bool big_slices = moving->g.dims[2] > 1 &&
                            (long long)moving->g.dims[0] * moving->g.dims[1] >= lc2e::kMaxFusedSlice;
    const bool small_r = patch_radius <= (dim == 3 ? lc2e::kMaxR3 : lc2e::kMaxR2);
    const int two_max = dim == 3 ? lc2e::kMaxRMom3 : lc2e::kMaxR2;
    const int src_ndim = moving->g.dims[2] > 1 ? 3 : 2;
    if (dim == 3 && (src_ndim != 3 || fixed->g.dims[2] < 1))
        return fail(LC2E_ERR_INVALID, "3D LC2 needs a 3D moving volume");
    for (int a = 0; a < dim; ++a)
        if (!(resampled_spacing[a] > 0.0f)) return fail(LC2E_ERR_INVALID, "resampled spacing must be positive");

    lc2e::PairGeometry pg = lc2e::make_pair_geometry(fixed->g, moving->g, resampled_spacing, dim,
                                                     src_ndim, center_overlaid != 0);
    const long long V = (long long)pg.virt.dims[0] * pg.virt.dims[1] * pg.virt.dims[2];
    if (V >= (1LL << 31)) return fail(LC2E_ERR_UNSUPPORTED, "virtual grid exceeds 2^31 voxels");

    // (the 3D moments kernel addresses a plane of the grid with 32-bit byte offsets; where two
    // voxels may differ by more than single precision holds, the separable path's sampler, which
    // reads only the neighbours a sample needs, keeps the radii beyond the fused kernels)
    const bool big_plane = dim == 3 && (long long)pg.virt.dims[0] * pg.virt.dims[1] >= (1LL << 28);
    const bool moments = patch_radius <= two_max && !big_plane && (small_r || !moving->large);
    const bool sep = big_slices || (!small_r && !moments);
    auto* p = new lc2e_pair();
    p->gen = g_generation.fetch_add(1);
    p->e = e;
    p->fixed = fixed;
    p->moving = moving;
    p->info.virt = pg.virt;
    for (int a = 0; a < 3; ++a) {
        p->info.fixed_center[a] = pg.fixed_center[a];
        p->info.shift[a] = pg.shift[a];
    }
    p->info.grid_ndim = dim;
    p->info.src_ndim = src_ndim;
    p->info.high_res_is_moving = high_res_is_moving ? 1 : 0;
    p->info.patch_radius = patch_radius;
    p->info.n_frames = dim == 2 ? pg.virt.dims[2] : 1;
    p->info.per_frame_matrices = 0;
    const lc2e_geom& vg = pg.virt;
    p->v = lc2e::VGeom{vg.dims[0], vg.dims[1], vg.dims[2], vg.spacing[0], vg.spacing[1],
                       vg.spacing[2], vg.origin[0], vg.origin[1], vg.origin[2]};
    const lc2e_geom& mg = moving->g;
    p->sg = lc2e::make_sgeom(mg.dims, mg.spacing, mg.origin);
    p->vbytes = (size_t)V * sizeof(float);
    int rc = e->alloc((void**)&p->stat_img, p->vbytes);
    if (rc < 0) {
        delete p;
        return rc;
    }
    if (sep) {
        p->sep = true;
        p->sep_grid_bytes = 2 * (size_t)V * sizeof(float);
        p->sep_sum_bytes = 2 * (size_t)lc2e::kSepChannels(high_res_is_moving != 0) * V * sizeof(double);
        if ((rc = e->alloc((void**)&p->sep_grids, p->sep_grid_bytes)) < 0 ||
            (rc = e->alloc((void**)&p->sep_sums, p->sep_sum_bytes)) < 0) {
            if (p->sep_grids) e->release(p->sep_grids, p->sep_grid_bytes);
            e->release(p->stat_img, p->vbytes);
            delete p;
            return rc;
        }
    }
    const lc2e_geom& fg = fixed->g;
    lc2e::SGeom fsg = lc2e::make_sgeom(fg.dims, fg.spacing, fg.origin);
    hipError_t err = lc2e::launch_warp_static(fixed->d, fixed->f16, fsg, p->v, dim, src_ndim,
                                              p->stat_img, e->stream);
    if (err == hipSuccess && !sep && moments && (rc = make_two_kernel(p, !small_r)) < 0) {
        lc2e_pair_destroy(p);
        return rc;
    }
    if (err == hipSuccess && high_res_is_moving) {
        // the fixed image is the ultrasound: its patch statistics are pose-independent
        rc = e->alloc((void**)&p->ustat, 2 * (size_t)V * sizeof(double));
        if (rc < 0) {
            lc2e_pair_destroy(p);
            return rc;
        }
        err = moments ? launch_stats(p, lc2e::kRoleUsStats, e->stream)
                    : lc2e::launch_ustats(p->stat_img, p->v, dim, patch_radius, p->ustat, p->ustat + V,
                                          p->sep_sums, p->sep ? p->sep_sums + (size_t)lc2e::kSepChannels(true) * V : nullptr,
                                          e->stream);
    }
    if (err == hipSuccess && !high_res_is_moving) {
        // the fixed image is the high-resolution one: its |Sobel| is pose-independent
        rc = e->alloc((void**)&p->stat_grad, p->vbytes);
        if (rc < 0) {
            lc2e_pair_destroy(p);
            return rc;
        }
        err = lc2e::launch_sobel(p->stat_img, p->v, dim, p->stat_grad, e->stream);
        if (err == hipSuccess && p->istat) err = launch_stats(p, lc2e::kRoleImageStats, e->stream);
    }
    if (err == hipSuccess) err = hipStreamSynchronize(e->stream);
    if (err != hipSuccess) {
        lc2e_pair_destroy(p);
        return fail(LC2E_ERR_HIP, "pair set-up failed: %s", hipGetErrorString(err));
    }
    {
        std::lock_guard<std::mutex> lk(g_registry_mu);
        g_pairs.insert(p);
    }
    *out = p;
    return LC2E_OK;
}

void lc2e_pair_destroy(lc2e_pair* p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> lk(g_registry_mu);
        g_pairs.erase(p);
    }
    (void)hipStreamSynchronize(p->e->stream);
    free_batch(p);
    free_mi(p);
    free_mi_warp(p);
    if (p->mi_ext_stat) p->e->release(p->mi_ext_stat, 2 * sizeof(int));
    if (p->ev0) (void)hipEventDestroy(p->ev0);
    if (p->ev1) (void)hipEventDestroy(p->ev1);
    p->e->release(p->stat_img, p->vbytes);
    if (p->stat_grad) p->e->release(p->stat_grad, p->vbytes);
    if (p->ustat) p->e->release(p->ustat, 2 * (p->vbytes / sizeof(float)) * sizeof(double));
    if (p->sep_grids) p->e->release(p->sep_grids, p->sep_grid_bytes);
    if (p->sep_sums) p->e->release(p->sep_sums, p->sep_sum_bytes);
    free_two(p);
    delete p;
}

int lc2e_pair_get_info(lc2e_pair* p, lc2e_pair_info* info) {
    if (!p || !info) return fail(LC2E_ERR_INVALID, "null argument");
    *info = p->info;
    return LC2E_OK;
}

int lc2e_pair_set_per_frame(lc2e_pair* p, int per_frame) {
    if (!p) return fail(LC2E_ERR_INVALID, "null pair");
    if (p->info.grid_ndim != 2 && per_frame)
        return fail(LC2E_ERR_INVALID, "per-frame matrices need a 2D frame stack");
    Use use(p);
    free_batch(p);
    p->info.per_frame_matrices = per_frame ? 1 : 0;
    return LC2E_OK;
}

int lc2e_pose_to_matrix(lc2e_pair* p, const double* params, int n, float out12[12]) {
    if (!p || !params || !out12) return fail(LC2E_ERR_INVALID, "null argument");
    int rc = lc2e::pose_to_matrix(p->info, params, n, out12);
    if (rc < 0) return fail(rc, "pose_to_matrix: %d parameters not valid for this pair", n);
    return LC2E_OK;
}

int lc2e_eval_batch(lc2e_pair* p, int n, const float* mats, double* lc2, double* sum_measure,
                    double* sum_w) {
    if (!p || !mats || n < 0) return fail(LC2E_ERR_INVALID, "invalid argument");
    if (n == 0) return LC2E_OK;
    Use use(p);
    HIP_TRY(hipSetDevice(p->e->device));
    const int mpp = p->mats_per_pose();
    const int chunk_max = 65535;
    int status = LC2E_OK;
    for (int base = 0; base < n; base += chunk_max) {
        const int m = (n - base) < chunk_max ? (n - base) : chunk_max;
        int rc = ensure_capacity(p, m);
        if (rc < 0) return rc;
        const Tiling t = tiling_for(p, m, p->ws_poses);
        std::memcpy(p->h_mats, mats + (size_t)base * mpp * 12, (size_t)m * mpp * 12 * sizeof(float));
        rc = run_batch(p, m, t);
        if (rc < 0) return rc;
        for (int i = 0; i < m; ++i) {
            const double sm = p->h_out[3 * i], sw = p->h_out[3 * i + 1], l = p->h_out[3 * i + 2];
            if (lc2) lc2[base + i] = l;
            if (sum_measure) sum_measure[base + i] = sm;
            if (sum_w) sum_w[base + i] = sw;
            if (!(sw > 0.0) || !std::isfinite(sm / sw)) status = LC2E_OK_DEGENERATE;
        }
    }
    return status;
}

int lc2e_eval(lc2e_pair* p, const float* m12, double* lc2) {
    return lc2e_eval_batch(p, 1, m12, lc2, nullptr, nullptr);
}

int lc2e_eval_batch_noalloc(lc2e_pair* p, int n, const float* mats, double* lc2,
                            double* sum_measure, double* sum_w) {
    if (!p || !mats || n < 0) return fail(LC2E_ERR_INVALID, "invalid argument");
    if (n == 0) return LC2E_OK;
    Use use(p);
    lc2e_engine* e = p->e;
    if (!e->scratch)
        return fail(LC2E_ERR_HIP, "device scratch unavailable: %s", e->scratch_error.c_str());
    // One device array serves every call on the device: calls are serialised here, so a
    // call that overlaps another one on the same device waits for it.
    std::lock_guard<std::mutex> lk(noalloc_lock(e->device));
    HIP_TRY(hipSetDevice(e->device));
    hipStream_t st = e->stream;
    const int mpp = p->mats_per_pose();
    const Workspace ws = noalloc_workspace(p);
    // scratch layout: results [m][3] f64, matrices [m][mpp][12] f32, partials [m][bpp][2] f64
    auto up256 = [](size_t b) { return (b + 255) / 256 * 256; };
    auto bytes = [&](size_t m, size_t bpp) {
        return up256(m * 3 * sizeof(double)) + up256(m * mpp * 12 * sizeof(float)) + m * bpp * 2 * sizeof(double);
    };
    const size_t bpp = partials_per_pose(p);
    const size_t need = bytes(n, admitted_partials(p));
    if (need > lc2e::kScratchBytes || bytes(1, bpp) > lc2e::kScratchBytes)
        return fail(LC2E_ERR_INVALID,
                    "%d poses need %zu bytes of device scratch; the allocation-free entry point "
                    "has %zu (use lc2e_eval_batch or fewer poses per call)",
                    n, need, lc2e::kScratchBytes);
    // an admitted call whose partial sums take more than the scratch holds runs in parts
    int most = n;
    while (bytes(most, bpp) > lc2e::kScratchBytes) most = (most + 1) / 2;
    char* base = static_cast<char*>(e->scratch);
    int status = LC2E_OK;
    for (int b0 = 0; b0 < n; b0 += most) {
        const int nb = std::min(most, n - b0);
        double* d_out = reinterpret_cast<double*>(base);
        float* d_mats = reinterpret_cast<float*>(base + up256((size_t)nb * 3 * sizeof(double)));
        double* d_part = reinterpret_cast<double*>(reinterpret_cast<char*>(d_mats) +
                                                   up256((size_t)nb * mpp * 12 * sizeof(float)));
        const Tiling t = tiling_for(p, nb, ws.poses);
        // few matrices go with the kernels' arguments, where one launch takes all poses
        const bool inline_mats = p->two && mpp == 1 && nb <= lc2e::kInlineMats &&
                                 (p->info.grid_ndim == 3 || p->v.Z == 1) &&
                                 (in_place(p, ws, t.tiles, nb) || part(ws, nb) == nb);
        if (!inline_mats)
            HIP_TRY(hipMemcpyAsync(d_mats, mats + (size_t)b0 * mpp * 12, (size_t)nb * mpp * 12 * sizeof(float),
                                   hipMemcpyHostToDevice, st));
        if (t.tiles > 0) {
            // every partial slot is written by the kernels before k_reduce reads it, so the
            // previous call's contents need no clearing
            lc2e::FusedArgs a = make_args(p, d_mats, d_part, t);
            if (inline_mats) {
                a.inline_mat = 1;
                std::memcpy(a.m0, mats + (size_t)b0 * 12, (size_t)nb * 12 * sizeof(float));
            }
            HIP_TRY(launch_eval(p, a, nb, st, ws));
        }
        // results back through a fixed host buffer, a chunk of poses at a time; few partials come
        // back themselves and are added up here, a launch less
        constexpr int kChunk = 128;
        constexpr size_t kFew = 256;
        double h[kChunk * 3], few[kFew * 2];
        const bool host = t.tiles > 0 && bpp <= kHostPose && nb <= kChunk && nb * bpp <= kFew;
        if (!host) HIP_TRY(lc2e::launch_reduce(d_part, (int)bpp, nb, d_out, st));
        for (int b = 0; b < nb; b += kChunk) {
            const int m = nb - b < kChunk ? nb - b : kChunk;
            HIP_TRY(host ? hipMemcpyAsync(few, d_part, nb * bpp * 2 * sizeof(double), hipMemcpyDeviceToHost, st)
                         : hipMemcpyAsync(h, d_out + (size_t)b * 3, (size_t)m * 3 * sizeof(double),
                                          hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
            if (host) sum_partials(few, nb, (int)bpp, h);
            for (int i = 0; i < m; ++i) {
                const double sm = h[3 * i], sw = h[3 * i + 1], l = h[3 * i + 2];
                const int k = b0 + b + i;
                if (lc2) lc2[k] = l;
                if (sum_measure) sum_measure[k] = sm;
                if (sum_w) sum_w[k] = sw;
                if (!(sw > 0.0) || !std::isfinite(sm / sw)) status = LC2E_OK_DEGENERATE;
            }
        }
    }
    return status;
}

int lc2e_eval_batch_async(lc2e_pair* p, int n, const float* d_mats, double* d_out, void* stream) {
    if (!p || !d_mats || !d_out || n <= 0) return fail(LC2E_ERR_INVALID, "invalid argument");
    Use use(p);
    hipStream_t st = stream ? static_cast<hipStream_t>(stream) : p->e->stream;
    // partials are per pair; size them for n
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    HIP_TRY(hipStreamIsCapturing(st, &capture));
    int rc = ensure_capacity(p, n, capture != hipStreamCaptureStatusNone);
    if (rc < 0) return rc;
    const Tiling t = tiling_for(p, n, p->ws_poses);
    if (t.tiles > 0) {
        lc2e::FusedArgs a = make_args(p, d_mats, p->d_partials, t);
        HIP_TRY(launch_eval(p, a, n, st, {p->ws, p->ws_poses}));
    }
    HIP_TRY(lc2e::launch_reduce(p->d_partials, t.tiles > 0 ? t.bpp : 0, n, d_out, st));
    return LC2E_OK;
}

int lc2e_eval_mi_batch(lc2e_pair* p, int n, const float* mats, int bins_us, int bins_hr,
                       double* nmi) {
    if (!p || !mats || !nmi || n < 0) return fail(LC2E_ERR_INVALID, "invalid argument");
    if (n == 0) return LC2E_OK;
    if (bins_us < 2 || bins_hr < 2 || bins_us > lc2e::kMiMaxBins || bins_hr > lc2e::kMiMaxBins)
        return fail(LC2E_ERR_INVALID, "histogram bins must lie in [2, %d]", lc2e::kMiMaxBins);
    Use use(p);
    HIP_TRY(hipSetDevice(p->e->device));
    lc2e_engine* e = p->e;
    hipStream_t st = e->stream;
    const int mpp = p->mats_per_pose();
    const size_t nb = (size_t)lc2e::mi_hist_size(bins_us, bins_hr);
    int rc;
    if (!p->mi_ext_stat) {
        if ((rc = e->alloc((void**)&p->mi_ext_stat, 2 * sizeof(int))) < 0) return rc;
        p->mi_stat_ready = false;
    }
    const int chunk_max = 64;
    const Tiling t = tiling_for(p, 1, 0);
    // Without a budget the warped image is kept between the two passes over it (3D), a float per
    // voxel and pose; what does not fit goes in parts. A buffer of its own: evaluations on a
    // caller's stream may be using the pair's workspace.
    // (Sources of large slices are beyond the pipelined sampler's offsets, those of large voxels
    // beyond its range: warped twice.)
    int step = std::min(n, chunk_max);
    if (!e->budget && p->info.grid_ndim == 3 && !p->moving->large && (long long)p->sg.X * p->sg.Y < lc2e::kMaxFusedSlice) {
        const size_t per = p->voxels() * sizeof(float);
        const int want = (int)std::min<size_t>((size_t)step, std::max<size_t>(1, kMiWarpBytes / per));
        if (want > p->mi_warp_poses && (!p->mi_refused || want < p->mi_refused)) {
            void* d = nullptr;
            if (e->raw_alloc(&d, (size_t)want * per, false) == hipSuccess) {
                free_mi_warp(p);
                p->mi_warp = static_cast<float*>(d);
                p->mi_warp_poses = want;
            } else {
                (void)hipGetLastError();
                p->mi_refused = want;
            }
        }
        if (p->mi_warp) step = std::min(step, p->mi_warp_poses);
    }
    for (int base = 0; base < n; base += step) {
        const int m = (n - base) < step ? (n - base) : step;
        if ((rc = ensure_batch(p, m, t.bpp)) < 0) return rc;
        if (m > p->mi_cap || nb != p->mi_bins) {
            free_mi(p);
            const int cap = m > 8 ? chunk_max : 8;
            if ((rc = e->alloc((void**)&p->mi_ext, (size_t)cap * 2 * sizeof(int))) < 0) return rc;
            p->mi_cap = cap;
            p->mi_bins = nb;
            if ((rc = e->alloc((void**)&p->mi_hist, (size_t)cap * nb * sizeof(unsigned))) < 0 ||
                (rc = e->alloc((void**)&p->mi_out, (size_t)cap * sizeof(double))) < 0) {
                free_mi(p);
                return rc;
            }
        }
        std::memcpy(p->h_mats, mats + (size_t)base * mpp * 12, (size_t)m * mpp * 12 * sizeof(float));
        HIP_TRY(hipMemcpyAsync(p->d_mats, p->h_mats, (size_t)m * mpp * 12 * sizeof(float),
                               hipMemcpyHostToDevice, st));
        lc2e::FusedArgs a = make_args(p, p->d_mats, p->d_partials, t);
        a.warp1 = p->mi_warp;
        // the static image is U when the moving image is the high-resolution one
        const int us_static = p->info.high_res_is_moving;
        HIP_TRY(lc2e::launch_mi(a, p->info.grid_ndim, p->info.src_ndim, us_static, m, bins_us,
                                bins_hr, p->stat_img,
                                p->mi_ext_stat, p->mi_stat_ready ? 1 : 0, p->mi_ext, p->mi_hist,
                                p->mi_out, st));
        p->mi_stat_ready = true;
        HIP_TRY(hipMemcpyAsync(p->h_out, p->mi_out, (size_t)m * sizeof(double),
                               hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        for (int i = 0; i < m; ++i) nmi[base + i] = p->h_out[i];
    }
    return LC2E_OK;
}

int lc2e_sync(lc2e_engine* e) {
    if (!e) return fail(LC2E_ERR_INVALID, "null engine");
    HIP_TRY(hipSetDevice(e->device));
    HIP_TRY(hipDeviceSynchronize());
    return LC2E_OK;
}

int lc2e_debug_fetch(lc2e_pair* p, lc2e_stage stage, const float* m12, void* host) {
    if (!p || !host || !m12) return fail(LC2E_ERR_INVALID, "null argument");
    Use use(p);
    HIP_TRY(hipSetDevice(p->e->device));
    hipStream_t st = p->e->stream;
    const long long V = (long long)p->v.X * p->v.Y * p->v.Z;
    const int mpp = p->mats_per_pose();
    int rc = ensure_capacity(p, 1);
    if (rc < 0) return rc;
    const Tiling t = tiling_for(p, 1, p->ws_poses);
    HIP_TRY(hipMemcpy(p->d_mats, m12, (size_t)mpp * 12 * sizeof(float), hipMemcpyHostToDevice));
    lc2e::FusedArgs a = make_args(p, p->d_mats, p->d_partials, t);
    const bool movi = p->info.high_res_is_moving != 0;
    if (stage == LC2E_STAGE_WARP_I || stage == LC2E_STAGE_WARP_US || stage == LC2E_STAGE_GRAD) {
        const bool want_moving = (stage == LC2E_STAGE_WARP_I) == movi || (stage == LC2E_STAGE_GRAD && movi);
        float* buf = nullptr;
        float* buf2 = nullptr;
        lc2e_engine* e = p->e;
        HIP_TRY(e->raw_alloc((void**)&buf, V * sizeof(float), true));
        hipError_t err = hipSuccess;
        const float* src = p->stat_img;
        if (stage == LC2E_STAGE_GRAD && !movi) {
            src = p->stat_grad;
        } else if (want_moving) {
            err = lc2e::launch_warp_moving(a, p->info.grid_ndim, p->info.src_ndim, buf, st);
            src = buf;
            if (err == hipSuccess && stage == LC2E_STAGE_GRAD) {
                err = e->raw_alloc((void**)&buf2, V * sizeof(float), true);
                if (err == hipSuccess) err = lc2e::launch_sobel(buf, p->v, p->info.grid_ndim, buf2, st);
                src = buf2;
            }
        }
        if (err == hipSuccess) err = hipMemcpyAsync(host, src, V * sizeof(float), hipMemcpyDeviceToHost, st);
        if (err == hipSuccess) err = hipStreamSynchronize(st);
        e->raw_free(buf, V * sizeof(float));
        e->raw_free(buf2, V * sizeof(float));
        if (err != hipSuccess) return fail(LC2E_ERR_HIP, "debug fetch failed: %s", hipGetErrorString(err));
        return LC2E_OK;
    }
    if (stage != LC2E_STAGE_W && stage != LC2E_STAGE_MEASURE)
        return fail(LC2E_ERR_INVALID, "unknown stage %d", (int)stage);
    double* maps = nullptr;
    HIP_TRY(p->e->raw_alloc((void**)&maps, 2 * V * sizeof(double), true));
    hipError_t err = hipMemsetAsync(maps, 0, 2 * V * sizeof(double), st);
    a.wmap = maps;
    a.mmap = maps + V;
    if (err == hipSuccess && t.tiles > 0)
        err = launch_eval(p, a, 1, st, {p->ws, p->ws_poses});
    if (err == hipSuccess)
        err = hipMemcpyAsync(host, stage == LC2E_STAGE_W ? a.wmap : a.mmap, V * sizeof(double),
                             hipMemcpyDeviceToHost, st);
    if (err == hipSuccess) err = hipStreamSynchronize(st);
    p->e->raw_free(maps, 2 * V * sizeof(double));
    if (err != hipSuccess) return fail(LC2E_ERR_HIP, "debug fetch failed: %s", hipGetErrorString(err));
    return LC2E_OK;
}

int lc2e_pair_set_tuning(lc2e_pair* p, int zchunk) {
    if (!p || zchunk < 0) return fail(LC2E_ERR_INVALID, "invalid argument");
    Use use(p);
    (void)hipStreamSynchronize(p->e->stream);
    drop_graphs(p);  // captured launches carry the old decomposition
    p->zchunk_forced = zchunk > 0 ? round_zchunk(zchunk) : 0;
    return LC2E_OK;
}

int lc2e_pair_set_tuning_n(lc2e_pair* p, int n, int zchunk) {
    if (!p || n <= 0 || zchunk < 0) return fail(LC2E_ERR_INVALID, "invalid argument");
    Use use(p);
    (void)hipStreamSynchronize(p->e->stream);
    drop_graphs(p);
    if (zchunk == 0) p->tuned.erase(n);
    else p->tuned[n] = round_zchunk(zchunk);
    return LC2E_OK;
}

int lc2e_pair_autotune(lc2e_pair* p, int n, const float* mats, int iters, int* best_zchunk,
                       double* best_ms) {
    if (!p || !mats || n <= 0 || iters <= 0) return fail(LC2E_ERR_INVALID, "invalid argument");
    Use use(p);
    HIP_TRY(hipSetDevice(p->e->device));
    if (p->info.grid_ndim != 3 || p->sep) {
        if (best_zchunk) *best_zchunk = 1;
        if (best_ms) *best_ms = 0.0;
        return LC2E_OK;
    }
    const int ez = p->v.Z - 2 * p->info.patch_radius;
    // chunks shorter than the column, then the whole column in one chunk
    std::vector<int> cand;
    for (int zc : {8, 16, 24, 32, 48, 64, 96, 128, 192, 256})
        if (zc < ez) cand.push_back(zc);
    cand.push_back(ez > 0 ? round_zchunk(ez) : lc2e::kZBlock);
    struct Events {
        hipEvent_t e0 = nullptr, e1 = nullptr;
        ~Events() {
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
        }
    } ev;
    HIP_TRY(hipEventCreate(&ev.e0));
    HIP_TRY(hipEventCreate(&ev.e1));
    hipEvent_t e0 = ev.e0, e1 = ev.e1;
    int best = 0;
    double bms = 1e300;
    hipStream_t st = p->e->stream;
    drop_graphs(p);
    const int forced = p->zchunk_forced;
    for (int zc : cand) {
        int rc = ensure_capacity(p, n);
        if (rc < 0) return rc;
        p->zchunk_forced = zc;
        const Tiling t = tiling_for(p, n, p->ws_poses);
        p->zchunk_forced = forced;
        HIP_TRY(hipMemcpy(p->d_mats, mats, (size_t)n * p->mats_per_pose() * 12 * sizeof(float),
                          hipMemcpyHostToDevice));
        lc2e::FusedArgs a = make_args(p, p->d_mats, p->d_partials, t);
        HIP_TRY(launch_eval(p, a, n, st, {p->ws, p->ws_poses}));
        HIP_TRY(hipEventRecord(e0, st));
        for (int it = 0; it < iters; ++it) HIP_TRY(launch_eval(p, a, n, st, {p->ws, p->ws_poses}));
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipEventSynchronize(e1));
        float ms = 0.0f;
        HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
        if (ms / (double)iters < bms) {
            bms = ms / (double)iters;
            best = zc;
        }
    }
    p->zchunk_forced = forced;  // a forced z-chunk keeps precedence over the tuned value
    p->tuned[n] = best;
    if (best_zchunk) *best_zchunk = best;
    if (best_ms) *best_ms = bms;
    return LC2E_OK;
}

int lc2e_pair_get_tuning(lc2e_pair* p, int* zchunk) {
    if (!p || !zchunk) return fail(LC2E_ERR_INVALID, "invalid argument");
    *zchunk = p->zchunk_forced > 0 ? p->zchunk_forced
              : p->last_zchunk > 0 ? p->last_zchunk
              : (p->info.grid_ndim == 3 ? round_zchunk(model_zchunk(p, 1)) : 1);
    return LC2E_OK;
}

int lc2e_pair_profile(lc2e_pair* p, int enable) {
    if (!p) return fail(LC2E_ERR_INVALID, "null pair");
    if ((enable != 0) != p->profile) (void)hipStreamSynchronize(p->e->stream);
    if (enable && !p->ev0) {
        HIP_TRY(hipEventCreate(&p->ev0));
        HIP_TRY(hipEventCreate(&p->ev1));
    }
    p->profile = enable != 0;
    p->prof_ms = 0.0;
    p->prof_launches = 0;
    return LC2E_OK;
}

int lc2e_pair_profile_read(lc2e_pair* p, double* kernel_ms, long long* launches) {
    if (!p) return fail(LC2E_ERR_INVALID, "null pair");
    if (kernel_ms) *kernel_ms = p->prof_ms;
    if (launches) *launches = p->prof_launches;
    return LC2E_OK;
}

int lc2e_pair_use_graph(lc2e_pair* p, int enable) {
    if (!p) return fail(LC2E_ERR_INVALID, "null pair");
    Use use(p);
    if (!enable) drop_graphs(p);
    p->use_graph = enable != 0;
    return LC2E_OK;
}

}  // extern "C"
