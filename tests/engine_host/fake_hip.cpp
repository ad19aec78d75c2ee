#include "fake_hip.hpp"

#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <utility>

namespace {

thread_local int t_device = 0;
thread_local hipError_t t_error = hipSuccess;  // a refused launch's
struct Block {
    size_t bytes;
    int device;
};
// In a function: the library registers its kernels before this file's globals are made.
struct State {
    std::recursive_mutex mu;
    size_t limit = size_t(1) << 40;
    size_t used[2] = {0, 0};
    std::map<void*, Block> blocks;
    std::vector<fake::Launch> launches;
    std::map<const void*, std::string> names;               // kernel handle -> mangled name
    std::map<std::pair<const void*, int>, int> lds;         // (kernel, device) -> allowed dynamic LDS
    std::map<const void*, size_t> vars;                     // device variable -> size
    std::map<std::pair<const void*, int>, void*> var_addr;  // (variable, device) -> address
    std::set<hipStream_t> capturing;
    int in_capture = 0;
    long long mallocs = 0, attempts = 0, copies = 0, pinned = 0;
};
State& g() {
    static State* s = new State();
    return *s;
}

struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
thread_local std::vector<Config> t_configs;

void* map_bytes(size_t n) {
    void* p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return p == MAP_FAILED ? nullptr : p;
}
void note_capture() {
    if (!g().capturing.empty()) ++g().in_capture;
}

}  // namespace

namespace fake {

void reset(size_t device_bytes) {
    std::lock_guard<std::recursive_mutex> lk(g().mu);
    g().limit = device_bytes;
    g().launches.clear();
    g().in_capture = 0;
    g().mallocs = g().attempts = g().copies = g().pinned = 0;
}
std::vector<Launch>& launches() { return g().launches; }
int in_capture() { return g().in_capture; }
size_t used(int device) { return g().used[device]; }
long long mallocs() { return g().mallocs; }
long long attempts() { return g().attempts; }
long long copies() { return g().copies; }
long long pinned() { return g().pinned; }
bool live(const void* p) {
    std::lock_guard<std::recursive_mutex> lk(g().mu);
    for (const auto& b : g().blocks)
        if (p >= b.first && p < static_cast<char*>(b.first) + b.second.bytes) return true;
    return false;
}
int count(const char* part) {
    int n = 0;
    for (const Launch& l : g().launches) n += l.is(part);
    return n;
}

}  // namespace fake

#define LOCK std::lock_guard<std::recursive_mutex> lk(g().mu)

extern "C" {

hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = t_device, hipSuccess; }
hipError_t hipSetDevice(int d) { return d < 0 || d > 1 ? hipErrorInvalidDevice : (t_device = d, hipSuccess); }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() {
    const hipError_t e = t_error;
    t_error = hipSuccess;
    return e;
}

hipError_t hipMalloc(void** p, size_t n) {
    LOCK;
    note_capture();
    ++g().attempts;
    if (g().used[t_device] + n > g().limit) return *p = nullptr, hipErrorOutOfMemory;
    if (!(*p = map_bytes(n))) return hipErrorOutOfMemory;
    g().blocks[*p] = {n, t_device};
    g().used[t_device] += n;
    ++g().mallocs;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    LOCK;
    note_capture();
    if (!p) return hipSuccess;
    auto it = g().blocks.find(p);
    if (it == g().blocks.end()) std::abort();  // not an allocation
    g().used[it->second.device] -= it->second.bytes;
    munmap(p, it->second.bytes ? it->second.bytes : 1);
    g().blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    LOCK;
    ++g().pinned;
    return (*p = std::calloc(1, n ? n : 1)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    LOCK;
    ++g().copies;
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(std::malloc(1)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() {
    LOCK;
    note_capture();
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    LOCK;
    g().capturing.insert(s);
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* out) {
    LOCK;
    g().capturing.erase(s);
    *out = reinterpret_cast<hipGraph_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    LOCK;
    *st = g().capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *x = reinterpret_cast<hipGraphExec_t>(std::malloc(1)), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t x) { return std::free(x), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return std::free(x), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(std::malloc(1)), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

void** __hipRegisterFatBinary(const void*) {
    static void* handle[1];
    return handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    LOCK;
    g().names[fn] = name;
}
void __hipRegisterVar(void**, void* var, char*, const char*, int, size_t bytes, int, int) {
    LOCK;
    g().vars[var] = bytes;
}
hipError_t hipGetSymbolAddress(void** p, const void* var) {
    LOCK;
    void*& a = g().var_addr[{var, t_device}];
    if (!a) a = map_bytes(g().vars[var]);
    return *p = a, hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* fn, hipFuncAttribute, int v) {
    LOCK;
    g().lds[{fn, t_device}] = v;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t lds) { return *n = lds > 80 * 1024 ? 1 : 2, hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    t_configs.push_back({grid, block, lds, st});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
    const Config c = t_configs.back();
    t_configs.pop_back();
    *grid = c.grid, *block = c.block, *lds = c.lds, *st = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t st) {
    LOCK;
    fake::Launch l;
    l.kernel = g().names[fn];
    l.groups = (unsigned long long)grid.x * grid.y * grid.z;
    l.threads = block.x * block.y * block.z;
    l.lds = lds;
    l.device = t_device;
    l.stream = st;
    l.captured = g().capturing.count(st) != 0;
    if ((unsigned long long)grid.x * block.x >= (1ULL << 32)) return t_error = hipErrorInvalidConfiguration;
    const auto it = g().lds.find({fn, t_device});
    if (lds > 65536 && (it == g().lds.end() || (size_t)it->second < lds)) return t_error = hipErrorInvalidValue;
    for (const char* k : {"k_moments", "k_warp_grad3", "k_warp_us3", "k_warp2", "k_fused", "k_mi_warp3", "k_mi_joint"})
        if (l.is(k)) std::memcpy(&l.a, args[0], sizeof(l.a));
    g().launches.push_back(l);
    return hipSuccess;
}

}  // extern "C"
