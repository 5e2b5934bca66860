// A HIP runtime without a GPU, for tests of what the library does on the host. Preloaded in front of the
// real one: device memory is host memory of a limited size, kernels are not run but listed, and a named
// call can be made to fail. Memory starts as zeros, so a scene of one triangle loads.
#include <hip/hip_runtime_api.h>

#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

std::map<void*, size_t> blocks;
std::map<const void*, std::string> kernels;
size_t capacity = (size_t)1 << 40, used = 0, peak = 0;
std::string failing, launched;
hipError_t failure = hipSuccess, last = hipSuccess;
std::vector<dim3> configs;
float clockMs = 0;

hipError_t result(const char* call) {
    if (failing != call) return hipSuccess;
    last = failure;
    return failure;
}

}  // namespace

extern "C" {

// ---- controls
void fake_hip_limit(size_t bytes) { capacity = bytes; peak = used; }
size_t fake_hip_used() { return used; }
size_t fake_hip_peak() { return peak; }
void fake_hip_fail(const char* call, int error) { failing = call; failure = (hipError_t)error; }
// "kernel grid block" of every launch since the last call, also of captured ones, and "graph" for a replay, one a line
const char* fake_hip_launched() {
    static std::string out;
    out.swap(launched);
    launched.clear();
    return out.c_str();
}

// ---- runtime
hipError_t hipMalloc(void** p, size_t bytes) {
    *p = nullptr;
    if (used + bytes > capacity) return last = hipErrorOutOfMemory;
    void* m = mmap(nullptr, bytes + 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return last = hipErrorOutOfMemory;
    blocks[m] = bytes;
    used += bytes;
    if (used > peak) peak = used;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = blocks.find(p);
    if (it == blocks.end()) return p ? last = hipErrorInvalidValue : hipSuccess;
    used -= it->second;
    munmap(p, it->second + 1);
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { *p = calloc(1, bytes); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "injected"; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 1; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* symbol) { *p = (void*)symbol; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)8; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)8; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *e = (hipGraphExec_t)8;
    return result("hipGraphInstantiate");
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    launched += "graph\n";
    return result("hipGraphLaunch");
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)8; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = clockMs += 1; return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
    launched += kernels[f] + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + "\n";
    return result("hipLaunchKernel");
}
void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
    configs.push_back(grid);
    configs.push_back(block);
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *block = configs.back(); configs.pop_back();
    *grid = configs.back(); configs.pop_back();
    *shared = 0;
    *stream = (hipStream_t)8;
    return hipSuccess;
}

}  // extern "C"
