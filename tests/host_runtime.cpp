// A stand-in for the HIP runtime functions that libpqb_perm.so calls, for tests of the
// engine's host side without a GPU: memory is the host's, copies are made, kernel launches
// are written down by name and do nothing, and a function can be told to fail.  Loaded with
// global visibility before the engine, whose references then resolve here.

#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

std::map<const void*, std::string> kernels;
std::string launched;   // names, one a line
std::string failing;    // function whose calls fail from the `failing_from`-th on
int failing_from = 0;
struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
std::vector<Config> configs;
int token;  // any handle

hipError_t called(const char* name) {
    return failing == name && --failing_from <= 0 ? hipErrorUnknown : hipSuccess;
}

}  // namespace

extern "C" {

void host_runtime_fail(const char* name, int from) {
    failing = name;
    failing_from = from;
}

// the kernels launched since the last call, one name a line
const char* host_runtime_launched() {
    static std::string out;
    out.swap(launched);
    launched.clear();
    return out.c_str();
}

void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(&token); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, uint3*, uint3*, dim3*, dim3*,
                           int*) {
    kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    configs.push_back({grid, block, shared, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = configs.back().grid;
    *block = configs.back().block;
    *shared = configs.back().shared;
    *stream = configs.back().stream;
    configs.pop_back();
    return hipSuccess;
}

static hipError_t last = hipSuccess;
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    launched += kernels[f] + "\n";
    return last = called("hipLaunchKernel");
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "failed as told"; }

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->maxSharedMemoryPerMultiProcessor = 160 * 1024;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    return *n = 3, hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) {
    std::memset(a, 0, sizeof(*a));
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) { return *p = std::calloc(n, 1), called("hipMalloc"); }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::calloc(n, 1), called("hipHostMalloc"); }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(to, from, n);
    return called("hipMemcpyAsync");
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = nullptr, hipErrorUnknown; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    return *s = reinterpret_cast<hipStream_t>(&token), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return called("hipStreamSynchronize"); }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(&token), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return called("hipStreamBeginCapture"); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    return *g = reinterpret_cast<hipGraph_t>(&token), hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *x = reinterpret_cast<hipGraphExec_t>(&token), called("hipGraphInstantiate");
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return called("hipGraphLaunch"); }

}  // extern "C"
