// A HIP runtime for the engine's host code on a machine without a GPU: device
// memory is host memory, copies copy, and a kernel launch only records the
// kernel's name -- or fails, if the test asked for that.
#include "fake_hip.hpp"

#include <cstdlib>
#include <cstring>
#include <map>

namespace fake {
std::vector<std::string> launched;
std::string fail_next;
void (*on_graph_launch)() = nullptr;
void (*on_copy)(void* dst, const void* src, size_t bytes, int kind) = nullptr;
static std::map<const void*, std::string>& names() {   // (kernels are registered before main)
    static std::map<const void*, std::string> m;
    return m;
}
static hipError_t last = hipSuccess;
}  // namespace fake
using namespace fake;

extern "C" {
void** __hipRegisterFatBinary(const void*) { return (void**)&names(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names()[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = *b = dim3(1);
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    const std::string& n = names()[f];
    if (!fail_next.empty() && n.find(fail_next) != std::string::npos) {
        fail_next.clear();
        return last = hipErrorLaunchFailure;
    }
    launched.push_back(n);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "error"; }

hipError_t hipMalloc(void** p, size_t n) { return (*p = calloc(n ? n : 1, 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
    memcpy(d, s, n);
    if (on_copy) on_copy(d, s, n, (int)kind);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind kind) { return hipMemcpyAsync(d, s, n, kind, nullptr); }
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
    launched.push_back("set");
    return hipMemset(p, v, n);
}

hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->name, "host");
    strcpy(p->gcnArchName, "gfx950");
    p->totalGlobalMem = 1ull << 32;
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = const_cast<void*>(s); return hipSuccess; }

static int token;
hipError_t hipStreamCreate(hipStream_t* s) { *s = (hipStream_t)&token; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)&token; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)&token; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = (hipGraphExec_t)&token;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    launched.push_back("graph");
    if (on_graph_launch) on_graph_launch();
    return hipSuccess;
}
}
