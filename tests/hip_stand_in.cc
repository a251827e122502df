// The HIP runtime calls libccdecode.so makes, without a GPU: device memory is
// host memory, copies copy, kernels do nothing but leave their names in a
// log. Preloaded before the library's own runtime (test_host_path.py), it
// runs the library's host side on the CPU: what a pass launches, and what it
// does when the runtime reports an error.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
std::map<const void*, std::string> names;
std::vector<std::string> launches;
std::string joined;
long fail_at = -1;   // the launch, counted from the last reset, that fails
hipError_t last = hipSuccess;
dim3 cfg_grid, cfg_block;
size_t cfg_lds;
hipStream_t cfg_stream;
}  // namespace

extern "C" {
void stand_in_reset(long fail) {
    launches.clear();
    fail_at = fail;
}
// The launches since the last reset: mangled kernel names, one a line.
const char* stand_in_launches() {
    joined.clear();
    for (const std::string& n : launches) joined += n + "\n";
    return joined.c_str();
}

void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*,
                           int*) {
    names[host] = device;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *st = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    launches.push_back(names[f]);
    if ((long)launches.size() - 1 == fail_at) return last = hipErrorLaunchFailure;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }

hipError_t hipMalloc(void** p, size_t n) {
    *p = calloc(n ? n : 1, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return hipMalloc(p, (size_t)4 << 20); }

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
}
