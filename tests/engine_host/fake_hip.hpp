// A stand-in for the HIP runtime under the built engine library: "device" memory is host memory
// of a limited amount, copies are immediate, kernels do not run but their launches are recorded
// with their arguments, and calls that the runtime refuses (allocation during a capture, a launch
// beyond a kernel's LDS limit or of 2^32 work-items) are refused or counted. Test infrastructure
// only; no GPU is touched.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

#include "lc2e_kernels.hpp"

namespace fake {

struct Launch {
    std::string kernel;  // mangled name
    unsigned long long groups = 0;
    unsigned threads = 0;
    size_t lds = 0;
    int device = 0;
    hipStream_t stream = nullptr;
    bool captured = false;
    lc2e::FusedArgs a{};  // the first argument of the kernels that take one
    bool is(const char* part) const { return kernel.find(part) != std::string::npos; }
};

void reset(size_t device_bytes);  // forgets the launches and counts; memory limit per device
std::vector<Launch>& launches();
int in_capture();                   // allocations, frees and device waits during a capture
size_t used(int device);            // device bytes allocated
bool live(const void* p);           // p lies in an allocation of device memory
long long mallocs();                // hipMalloc calls that succeeded
long long attempts();               // all
long long copies();                 // asynchronous ones
long long pinned();                 // hipHostMalloc calls
int count(const char* kernel_part);  // launches whose kernel's name holds the text

}  // namespace fake
