// Scenarios of the engine's host code (lc2e_engine.cpp and the kernels' launchers) on the fake
// runtime; the name of one is the argument.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "fake_hip.hpp"
#include "lc2e.h"

namespace {

#define CHECK(x)                                                                  \
    do {                                                                          \
        if (!(x)) {                                                               \
            std::printf("%s:%d: %s (%s)\n", __FILE__, __LINE__, #x, lc2e_last_error()); \
            std::exit(1);                                                         \
        }                                                                         \
    } while (0)

constexpr size_t GB = size_t(1) << 30, MB = size_t(1) << 20;

lc2e_engine* engine(size_t budget = 0, int device = 0) {
    lc2e_engine* e = nullptr;
    CHECK(lc2e_create(device, budget, &e) == LC2E_OK);
    return e;
}

// A pair on a grid of the given size: the images are as small as they can be, the grid's
// spacing does the rest.
struct Pair {
    lc2e_volume *f = nullptr, *m = nullptr;
    lc2e_pair* p = nullptr;
    int frames = 1;

    Pair(lc2e_engine* e, int dim, int x, int y, int z, int movi, int r, bool src3, bool tracked = false) {
        CHECK(make(e, dim, x, y, z, movi, r, src3, tracked) >= 0);
    }
    Pair() = default;
    Pair(const Pair&) = delete;
    int make(lc2e_engine* e, int dim, int x, int y, int z, int movi, int r, bool src3, bool tracked = false) {
        const bool stack = dim == 2 && z > 1;
        std::vector<float> img(size_t(stack ? z : 1) * 64 + 4096, 1.0f);
        lc2e_geom g{};
        const int d[3] = {4, 4, dim == 3 ? 4 : z};
        const int n[3] = {x, y, z};
        float rs[3] = {1, 1, 1};
        for (int a = 0; a < 3; ++a) {
            g.dims[a] = d[a];
            g.spacing[a] = 1.0f;
            if (a < dim) rs[a] = (float)d[a] / ((float)n[a] - 0.5f);  // the grid's size is rounded up
        }
        int rc = lc2e_volume_upload(e, img.data(), LC2E_F32, &g, LC2E_STORE_AUTO, &f);
        if (rc < 0) return rc;
        lc2e_geom h{};
        for (int a = 0; a < 3; ++a) {
            h.dims[a] = a < 2 || src3 ? 8 : 1;
            h.spacing[a] = 1.0f;
        }
        if ((rc = lc2e_volume_upload(e, img.data(), LC2E_F32, &h, LC2E_STORE_AUTO, &m)) < 0) return rc;
        if ((rc = lc2e_pair_create(e, f, m, rs, movi, 0, r, dim, &p)) < 0) return rc;
        lc2e_pair_info info{};
        CHECK(lc2e_pair_get_info(p, &info) == LC2E_OK);
        for (int a = 0; a < 3; ++a) CHECK(info.virt.dims[a] == n[a]);
        if (tracked) CHECK(lc2e_pair_set_per_frame(p, 1) == LC2E_OK);
        frames = tracked ? z : 1;
        return LC2E_OK;
    }
    std::vector<float> mats(int n) const { return std::vector<float>(size_t(n) * frames * 12, 0.0f); }
    int batch(int n) { return lc2e_eval_batch(p, n, mats(n).data(), nullptr, nullptr, nullptr); }
    int noalloc(int n) { return lc2e_eval_batch_noalloc(p, n, mats(n).data(), nullptr, nullptr, nullptr); }
    int async(int n, hipStream_t st) {
        static float d_mats[64 * 12];
        static double d_out[64 * 3];
        return lc2e_eval_batch_async(p, n, d_mats, d_out, st);
    }
    int mi(int n, int bins = 256) {
        std::vector<double> out(n);
        return lc2e_eval_mi_batch(p, n, mats(n).data(), bins, bins, out.data());
    }
    ~Pair() {
        if (p) lc2e_pair_destroy(p);
        if (m) lc2e_volume_destroy(m);
        if (f) lc2e_volume_destroy(f);
    }
};

// The allocation-free entry point may run while a launch of the same pair is in flight on a
// caller's stream: they must not write the same warped image.
void noalloc_has_its_own_workspace() {
    lc2e_engine* e = engine();
    hipStream_t st = nullptr;
    CHECK(hipStreamCreateWithFlags(&st, 0) == hipSuccess);
    struct {
        int dim, x, y, z, movi, r;
        bool src3;
    } cases[] = {{3, 64, 64, 64, 1, 3, true}, {3, 64, 64, 64, 0, 2, true}, {3, 48, 48, 48, 1, 5, true},
                 {2, 512, 512, 1, 1, 5, false}, {2, 256, 200, 40, 1, 9, true}};
    for (const auto& c : cases) {
        Pair p(e, c.dim, c.x, c.y, c.z, c.movi, c.r, c.src3);
        const size_t bytes = size_t(c.x) * c.y * c.z * (c.movi ? 8 : 4);
        fake::launches().clear();
        CHECK(p.async(20, st) >= 0);
        CHECK(p.noalloc(20) >= 0);
        int own = 0, callers = 0;
        for (const auto& a : fake::launches()) {
            if (!a.is("k_moments") || !a.a.warp1 || a.a.in_place) continue;
            (a.stream == st ? callers : own)++;
            for (const auto& b : fake::launches())
                if (b.is("k_warp") && (a.stream == st) != (b.stream == st)) {
                    const char *u = (const char*)a.a.warp1, *v = (const char*)b.a.warp1;
                    CHECK(u + bytes <= v || v + bytes <= u);
                }
        }
        CHECK(callers > 0 && own > 0);
    }
    hipStreamDestroy(st);
    lc2e_destroy(e);
    CHECK(fake::used(0) == 0);
}

// A fresh pair's allocation-free call: as few launches as the reserve allows, 2D launches through
// the grid only in parts that fill the device, and chunks chosen for the parts.
void noalloc_runs_in_large_parts() {
    lc2e_engine* e = engine();
    {
        Pair p(e, 3, 64, 64, 64, 1, 3, true);  // 2 MiB a pose
        fake::launches().clear();
        CHECK(p.noalloc(32) >= 0);
        CHECK(fake::count("k_warp_grad3") == 1 && fake::count("k_moments3d") == 1);
        CHECK(fake::launches()[0].a.npose == 32 || fake::launches()[1].a.npose == 32);
    }
    {
        Pair p(e, 3, 192, 192, 160, 1, 3, true);  // 45 MiB a pose: 11 in the reserve
        fake::launches().clear();
        CHECK(p.noalloc(32) >= 0);
        CHECK(fake::count("k_moments3d") == 3);
        const int chunk = fake::launches()[1].a.zchunk;
        fake::launches().clear();
        CHECK(p.noalloc(11) >= 0);  // one part of the same size
        CHECK(fake::count("k_moments3d") == 1 && fake::launches()[1].a.zchunk == chunk);
    }
    {
        // 93 MiB a pose, five in the reserve: a batch of 8 goes through the grid, and so do its
        // parts of four poses, of 2048 waves and more
        Pair p(e, 2, 300, 200, 204, 1, 5, true);
        fake::launches().clear();
        CHECK(p.noalloc(8) >= 0);
        CHECK(fake::count("k_warp2") == 2 && fake::count("k_moments2d") == 2);
    }
    {
        // where there was no memory for more than one pose, whose launch would not fill the
        // device: warped in place, all poses in one launch
        fake::reset(24 * MB);
        Pair p(e, 2, 256, 256, 1, 1, 5, false);
        fake::launches().clear();
        CHECK(p.noalloc(64) >= 0);
        CHECK(fake::count("k_warp2") == 0 && fake::count("k_moments2d") == 1);
    }
    lc2e_destroy(e);
    CHECK(fake::used(0) == 0);
}

// A launch captured by the caller allocates and frees nothing where the pair's batch buffers
// fit, and what it uses stays in place for its replays until a larger batch replaces those.
void captured_launches_keep_their_workspace() {
    lc2e_engine* e = engine();
    hipStream_t st = nullptr;
    hipGraph_t graph = nullptr;
    CHECK(hipStreamCreateWithFlags(&st, 0) == hipSuccess);
    {
        Pair p(e, 3, 64, 64, 64, 1, 3, true);
        CHECK(p.mi(4) >= 0);  // sizes the batch buffers alone
        CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) == hipSuccess);
        fake::launches().clear();
        CHECK(p.async(4, st) >= 0);
        CHECK(hipStreamEndCapture(st, &graph) == hipSuccess);
        CHECK(fake::in_capture() == 0);
        const float* ws = fake::launches()[0].a.warp1;
        fake::launches().clear();
        CHECK(p.batch(4) >= 0);
        CHECK(fake::launches()[0].is("k_warp") && fake::launches()[0].a.warp1 == ws);
        CHECK(p.batch(32) >= 0);  // replaces the batch buffers, as documented
        fake::launches().clear();
        CHECK(p.batch(32) >= 0 && fake::count("k_warp") == 1);
    }
    CHECK(hipGraphDestroy(graph) == hipSuccess);
    CHECK(hipStreamDestroy(st) == hipSuccess);
    lc2e_destroy(e);
}

// Where a larger workspace is not to be had, calls go on with the one there is and do not ask
// for memory each time.
void a_refused_workspace_is_not_asked_for_again() {
    lc2e_engine* e = engine();
    {
        fake::reset(300 * MB);  // 192x192x160: 45 MiB a pose
        Pair p(e, 3, 192, 192, 160, 1, 3, true);
        CHECK(p.batch(8) >= 0);
        const long long asked = fake::attempts();
        fake::launches().clear();
        CHECK(p.batch(8) >= 0 && p.batch(8) >= 0);
        CHECK(fake::attempts() == asked);
        CHECK(fake::count("k_moments3d") > 2);
    }
    lc2e_destroy(e);
}

// Memory that pairs and engines keep only to be faster never makes a call fail: with 200 MiB,
// pairs of a 64^3 grid (4 MiB each without it, 15 with it, and more for batches and mutual
// information) fit as if there were none, on this engine and on another, and all of them
// evaluate; a pair that a caller's graph uses is left alone.
void kept_memory_makes_room() {
    fake::reset(200 * MB);
    lc2e_engine *e = engine(), *other = engine();
    hipStream_t st = nullptr;
    hipGraph_t graph = nullptr;
    CHECK(hipStreamCreateWithFlags(&st, 0) == hipSuccess);
    std::vector<Pair> pairs(44);
    Pair held(e, 3, 64, 64, 64, 1, 3, true);
    CHECK(held.batch(2) >= 0);
    CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) == hipSuccess);
    fake::launches().clear();
    CHECK(held.async(2, st) >= 0);
    CHECK(hipStreamEndCapture(st, &graph) == hipSuccess);
    const float* ws = fake::launches()[0].a.warp1;
    for (size_t i = 0; i < pairs.size(); ++i) {
        CHECK(pairs[i].make(i % 2 ? other : e, 3, 64, 64, 64, 0, i % 3 ? 3 : 4, true) >= 0);
        CHECK(pairs[i].batch(4) >= 0);
        CHECK(pairs[i].mi(2) >= 0);
    }
    for (Pair& p : pairs) CHECK(p.batch(4) >= 0 && p.noalloc(3) >= 0 && p.mi(2) >= 0);
    fake::launches().clear();
    CHECK(held.batch(2) >= 0 && fake::launches()[0].a.warp1 == ws);
    // and the other way round: a volume that needs what they keep
    lc2e_volume* v = nullptr;
    lc2e_geom g{};
    for (int a = 0; a < 3; ++a) g.dims[a] = a < 2 ? 160 : 100, g.spacing[a] = 1.0f;
    std::vector<unsigned char> img(size_t(160) * 160 * 100);
    CHECK(lc2e_volume_upload(e, img.data(), LC2E_U8, &g, LC2E_STORE_AUTO, &v) == LC2E_OK);
    lc2e_volume_destroy(v);
    pairs.clear();
    CHECK(hipGraphDestroy(graph) == hipSuccess);
    CHECK(hipStreamDestroy(st) == hipSuccess);
}

// Giving memory back does not change the calling thread's device, as hipFree does not.
void releases_leave_the_current_device() {
    lc2e_engine* e = engine(0, 0);
    int device = 0;
    {
        Pair p(e, 3, 64, 64, 64, 1, 3, true);
        CHECK(p.batch(4) >= 0);
        CHECK(hipSetDevice(1) == hipSuccess);
    }
    CHECK(hipGetDevice(&device) == hipSuccess && device == 1);
    lc2e_destroy(e);
    CHECK(fake::used(0) == 0);
}

// Kernels of more than 64 KB of LDS need their limit raised on each device they run on.
void every_device_gets_its_lds_limit() {
    for (int device : {0, 1}) {
        lc2e_engine* e = engine(0, device);
        for (int r : {1, 3, 4, 6, 12}) {
            Pair p(e, 3, 48, 48, 48, r % 2, r, true);
            CHECK(p.batch(2) >= 0);
            CHECK(p.mi(1) >= 0);
        }
        CHECK(Pair(e, 2, 256, 256, 1, 0, 64, false).batch(1) >= 0);
        lc2e_destroy(e);
    }
}

// Many poses of a tiny grid: no launch of 2^32 work-items or more.
void launches_stay_below_the_runtime_limit() {
    lc2e_engine* e = engine();
    {
        Pair p(e, 3, 3, 3, 3, 1, 1, true), q(e, 2, 9, 9, 1, 1, 4, false);
        CHECK(p.async(800000, nullptr) >= 0);
        CHECK(q.async(800000, nullptr) >= 0);
    }
    lc2e_destroy(e);
}

// The allocation-free entry point admits by the sizes it was specified with, whatever the kernels'
// own partial sums take.
void noalloc_admits_what_it_did() {
    lc2e_engine* e = engine();
    {
        // one output voxel per plane: 100 / 256 -> 1 sum per pose, where the kernel writes more
        Pair p(e, 3, 11, 11, 110, 1, 5, true);
        fake::launches().clear();
        CHECK(p.noalloc(100000) >= 0);
        CHECK(fake::count("k_reduce") >= 1);
        CHECK(p.noalloc(200000) == LC2E_ERR_INVALID);
        // 256 tiles of 16x16 outputs per pose, which the kernel covers with fewer
        Pair q(e, 2, 262, 262, 1, 0, 3, false);
        CHECK(q.noalloc(4000) >= 0);
        CHECK(q.noalloc(4100) == LC2E_ERR_INVALID);
    }
    lc2e_destroy(e);
}

// A 2D launch that leaves the chip idle runs in twice the waves of half the chain each; one of
// more than a work-group per CU does not.
void small_2d_launches_have_short_waves() {
    lc2e_engine *e = engine(), *b = engine(GB);
    for (lc2e_engine* x : {e, b})
        for (int movi : {0, 1}) {
            Pair p(x, 2, 256, 256, 1, movi, 5, false);
            fake::launches().clear();
            CHECK(p.batch(1) >= 0 && p.batch(64) >= 0);
            std::vector<unsigned> threads;
            for (const auto& l : fake::launches())
                if (l.is("k_moments2d")) threads.push_back(l.threads);
            CHECK(threads.size() == 2 && threads[0] == 512 && threads[1] == 256);
        }
    lc2e_destroy(b);
    lc2e_destroy(e);
}

// One pose of a stack spreads over the chip, with no more partial sums than 16x16 tiles over 16
// frames each had (by which memory and the allocation-free entry point are sized).
void one_pose_of_a_stack_fills_the_device() {
    lc2e_engine *e = engine(), *b = engine(8 * GB);
    struct {
        int x, y, z, r, groups;
    } cases[] = {{256, 200, 40, 4, 400}, {256, 200, 40, 9, 400}, {512, 384, 128, 5, 1024}, {90, 70, 100, 10, 64}, {21, 22, 50, 10, 4}};
    for (lc2e_engine* x : {e, b})
        for (const auto& c : cases)
            for (int movi : {0, 1}) {
                Pair p(x, 2, c.x, c.y, c.z, movi, c.r, true, true);
                fake::launches().clear();
                CHECK(p.batch(1) >= 0);
                const int ex = c.x - 2 * c.r, ey = c.y - 2 * c.r;
                const int most = (ex + 15) / 16 * ((ey + 15) / 16) * ((c.z + 15) / 16);
                for (const auto& l : fake::launches())
                    if (l.is("k_moments2d")) {
                        CHECK(l.a.tiles >= c.groups);
                        CHECK(l.a.blocks_per_pose <= most);
                    }
                CHECK(fake::count("k_moments2d") == 1);
            }
    lc2e_destroy(b);
    lc2e_destroy(e);
}

// Small calls: no reduction launch where the host adds up few partial sums, and matrices in the
// arguments of the kernels that read them there, without allocation too.
void small_calls_have_few_commands() {
    lc2e_engine* e = engine();
    {
        Pair p(e, 2, 96, 96, 1, 1, 9, false), f(e, 2, 96, 96, 1, 1, 3, false), v(e, 3, 64, 64, 64, 1, 3, true);
        fake::launches().clear();
        CHECK(p.batch(13) >= 0 && f.batch(13) >= 0 && fake::count("k_reduce") == 0);
        fake::launches().clear();
        CHECK(p.noalloc(8) >= 0 && v.noalloc(8) >= 0);
        for (const auto& l : fake::launches())
            if (l.is("k_moments") || l.is("k_warp")) CHECK(l.a.inline_mat == 1);
        fake::launches().clear();
        CHECK(p.noalloc(9) >= 0 && v.noalloc(9) >= 0 && f.noalloc(2) >= 0 && f.batch(2) >= 0);
        for (const auto& l : fake::launches())
            if (l.is("k_moments") || l.is("k_warp") || l.is("k_fused")) CHECK(l.a.inline_mat == 0);
    }
    lc2e_destroy(e);
}

// A small 3D launch is cut into short chunks, and calls of up to 32 poses copy no matrices.
void small_3d_launches_are_spread_out() {
    lc2e_engine* e = engine();
    {
        Pair p(e, 3, 64, 64, 64, 1, 1, true);
        CHECK(p.batch(32) >= 0);
        fake::launches().clear();
        const long long copies = fake::copies();
        CHECK(p.batch(4) >= 0);
        for (const auto& l : fake::launches())
            if (l.is("k_warp_grad3")) CHECK(l.groups >= 512);  // 2 x 4 columns, 4 poses, 16 chunks
        CHECK(p.batch(13) >= 0 && p.batch(32) >= 0);
        CHECK(fake::copies() == copies);
    }
    lc2e_destroy(e);
}

// The chunk model's overhead per work-group is that of the kernels that run: one plane per step at
// radii from 4 with a moving high-resolution image, whose short chunks cost little.
void chunks_fit_the_kernel_that_runs() {
    lc2e_engine* e = engine();
    {
        struct {
            int x, y, z, r, n, most;
        } cases[] = {{48, 48, 48, 4, 13, 32}, {64, 64, 64, 6, 17, 32}, {64, 64, 64, 5, 9, 24}};
        for (const auto& c : cases) {
            Pair p(e, 3, c.x, c.y, c.z, 1, c.r, true);
            CHECK(p.batch(c.n) >= 0);
            int zchunk = 0;
            CHECK(lc2e_pair_get_tuning(p.p, &zchunk) == LC2E_OK && zchunk <= c.most);
        }
    }
    lc2e_destroy(e);
}

// Mutual information without a kept warp gathers every voxel in the joint histogram: a large
// launch of small histograms has many work-groups, the others one round of the CUs.
void joint_histograms_that_warp_again_spread_out() {
    lc2e_engine *e = engine(), *b = engine(8 * GB);
    {
        Pair kept(e, 3, 128, 128, 128, 1, 2, true), again(b, 3, 128, 128, 128, 1, 2, true);
        struct {
            Pair& p;
            int n, bins;
            unsigned long long least, most;
        } cases[] = {{kept, 30, 32, 200, 256}, {again, 30, 256, 200, 256}, {again, 40, 32, 1024, 2048}, {again, 5, 32, 200, 256}};
        for (const auto& c : cases) {
            fake::launches().clear();
            CHECK(c.p.mi(c.n, c.bins) >= 0);
            for (const auto& l : fake::launches())
                if (l.is("k_mi_joint")) CHECK(l.groups >= c.least && l.groups <= c.most);
            CHECK(fake::count("k_mi_joint") == 1);
        }
    }
    lc2e_destroy(b);
    lc2e_destroy(e);
}

// Freed blocks are kept up to a limit; past it the oldest go, so what a program frees now is there
// for its next object of that size whatever it freed before.
void old_blocks_make_room_for_new_ones() {
    lc2e_engine* e = engine();
    for (int side : {400, 440, 480}) {  // 0.26 to 0.44 GB each, in single precision
        lc2e_volume* v = nullptr;
        lc2e_geom g{};
        for (int a = 0; a < 3; ++a) g.dims[a] = side, g.spacing[a] = 1.0f;
        std::vector<float> img(size_t(side) * side * side);
        CHECK(lc2e_volume_upload(e, img.data(), LC2E_F32, &g, LC2E_STORE_AUTO, &v) == LC2E_OK);
        lc2e_volume_destroy(v);
        CHECK(fake::used(0) <= GB);
    }
    { Pair p(e, 3, 128, 128, 128, 0, 3, true); }
    const long long mallocs = fake::mallocs();
    { Pair p(e, 3, 128, 128, 128, 0, 3, true); }
    CHECK(fake::mallocs() == mallocs);
    lc2e_destroy(e);
    CHECK(fake::used(0) == 0);
}

// After the first one an upload makes no pinned memory, with a budget or without, and a small int16
// volume's storage is settled without the device.
void small_uploads_make_nothing_pinned() {
    for (size_t budget : {size_t(0), GB}) {
        lc2e_engine* e = engine(budget);
        std::vector<short> img(33 * 32 * 32);
        long long pinned = 0;
        for (int k = 0; k < 4; ++k) {
            lc2e_volume* v = nullptr;
            lc2e_geom g{};
            for (int a = 0; a < 3; ++a) g.dims[a] = a ? 32 : k < 2 ? 32 : 33, g.spacing[a] = 1.0f;
            if (k == 3) img[32 * 32 * 32] = 3000;  // past the voxels that the host looks at
            fake::launches().clear();
            size_t used0 = 0, used = 0;
            CHECK(lc2e_memory(e, &used0, nullptr) == LC2E_OK);
            CHECK(lc2e_volume_upload(e, img.data(), LC2E_I16, &g, LC2E_STORE_AUTO, &v) == LC2E_OK);
            CHECK(lc2e_memory(e, &used, nullptr) == LC2E_OK);
            const size_t n = size_t(g.dims[0]) * 32 * 32, pad = size_t(g.dims[0]) * 33 + 64;
            CHECK(used - used0 == (n + pad) * 2);  // (kernels do not run here: nothing is flagged)
            CHECK(fake::count("k_check") == (k < 2 ? 0 : 1));
            lc2e_volume_destroy(v);
            if (k == 0) pinned = fake::pinned();
        }
        CHECK(fake::pinned() == pinned);
        lc2e_destroy(e);
    }
}

// Pinned memory takes longer to make than a small pair's first call: two blocks for all of it.
void a_pair_makes_two_pinned_blocks() {
    lc2e_engine* e = engine(GB);
    {
        Pair p(e, 2, 96, 96, 1, 1, 3, false);
        const long long before = fake::pinned();
        CHECK(p.batch(4) >= 0 && p.batch(4) >= 0 && p.mi(3) >= 0);
        CHECK(fake::pinned() == before + 2);
    }
    lc2e_destroy(e);
    CHECK(fake::used(0) == 0);
}

//@SCENARIOS

const std::map<std::string, std::function<void()>> kScenarios = {
    {"noalloc_has_its_own_workspace", noalloc_has_its_own_workspace},
    {"noalloc_runs_in_large_parts", noalloc_runs_in_large_parts},
    {"captured_launches_keep_their_workspace", captured_launches_keep_their_workspace},
    {"a_refused_workspace_is_not_asked_for_again", a_refused_workspace_is_not_asked_for_again},
    {"kept_memory_makes_room", kept_memory_makes_room},
    {"releases_leave_the_current_device", releases_leave_the_current_device},
    {"every_device_gets_its_lds_limit", every_device_gets_its_lds_limit},
    {"launches_stay_below_the_runtime_limit", launches_stay_below_the_runtime_limit},
    {"noalloc_admits_what_it_did", noalloc_admits_what_it_did},
    {"small_2d_launches_have_short_waves", small_2d_launches_have_short_waves},
    {"one_pose_of_a_stack_fills_the_device", one_pose_of_a_stack_fills_the_device},
    {"small_calls_have_few_commands", small_calls_have_few_commands},
    {"small_3d_launches_are_spread_out", small_3d_launches_are_spread_out},
    {"chunks_fit_the_kernel_that_runs", chunks_fit_the_kernel_that_runs},
    {"joint_histograms_that_warp_again_spread_out", joint_histograms_that_warp_again_spread_out},
    {"old_blocks_make_room_for_new_ones", old_blocks_make_room_for_new_ones},
    {"small_uploads_make_nothing_pinned", small_uploads_make_nothing_pinned},
    {"a_pair_makes_two_pinned_blocks", a_pair_makes_two_pinned_blocks},
//@TABLE
};

}  // namespace

int main(int argc, char** argv) {
    const auto it = kScenarios.find(argc > 1 ? argv[1] : "");
    if (it == kScenarios.end()) return std::printf("no such scenario\n"), 2;
    fake::reset(64 * GB);
    it->second();
    std::printf("%s passed\n", argv[1]);
    return 0;
}
