// A stand-in for the HIP calls libtgx.so makes, for CPU tests of its host side: device memory is the
// host's, kernels are counted and not run, and the null stream is as late as HIP allows. A clear by
// hipMemset, or a hipMemsetAsync on the null stream, runs only once the host waits for that stream (a
// hipStreamSynchronize of it, a hipDeviceSynchronize, a blocking hipMemcpy, a hipFree) or the test
// settles it. What is queued on another stream runs at once, and is a violation where a clear that
// has not run could still overtake it: a copy into or out of the memory it clears, or any kernel.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

namespace {

struct Clear {
    char* p;
    int value;
    size_t bytes;
};
std::vector<Clear> clears;  // queued on the null stream and not run yet
int violations = 0, graphs = 0, last_nodes = 0;
bool capturing = false;
int captured = 0;

void settle() {
    for (const Clear& c : clears) std::memset(c.p, c.value, c.bytes);
    clears.clear();
}
void violation(const char* what) {
    ++violations;
    std::fprintf(stderr, "hip_model: %s while a clear of its memory may still run\n", what);
}
void copy(void* dst, const void* src, size_t bytes, hipStream_t stream) {
    if (!stream) settle();
    for (const Clear& c : clears)
        for (const char* p : {(const char*)dst, (const char*)src})
            if (p < c.p + c.bytes && c.p < p + bytes) violation("a copy");
    std::memmove(dst, src, bytes);
}
void kernel(hipStream_t stream) {
    if (capturing) {
        ++captured;
        return;
    }
    if (!stream) settle();
    if (!clears.empty()) violation("a kernel");
}
template <typename T>
hipError_t give(T* out) {  // a handle of its own
    *out = (T)std::calloc(1, 64);
    return hipSuccess;
}
int& nodes_of(void* handle) { return *(int*)handle; }

}  // namespace

extern "C" {

int hip_model_violations() { return violations; }
int hip_model_pending() { return (int)clears.size(); }  // clears that may still run
void hip_model_settle() { settle(); }
int hip_model_graphs() { return graphs; }          // instantiated so far
int hip_model_last_nodes() { return last_nodes; }  // kernels in the graph launched last

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // hip_runtime_api.h names its versioned symbol
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->sharedMemPerBlock = 160 << 10;
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipDeviceSynchronize() { settle(); return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "hip_model"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) { std::memset(a, 0, sizeof *a); return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* scratch = std::calloc(1, 32 << 20);
    *p = scratch;
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t bytes) {
    *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
    std::memset(*p, 0xa5, bytes);  // as a freed allocation left it
    return hipSuccess;
}
hipError_t hipFree(void* p) { settle(); std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }

hipError_t hipMemset(void* p, int value, size_t bytes) { clears.push_back({(char*)p, value, bytes}); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int value, size_t bytes, hipStream_t s) {
    if (!s) return hipMemset(p, value, bytes);
    std::memset(p, value, bytes);
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind) { copy(dst, src, bytes, nullptr); return hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t s) {
    if (!capturing) copy(dst, src, bytes, s);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t height, hipMemcpyKind,
                            hipStream_t s) {
    for (size_t i = 0; i < height && !capturing; ++i) copy((char*)dst + i * dpitch, (const char*)src + i * spitch, width, s);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return give(s); }
hipError_t hipStreamDestroy(hipStream_t s) { std::free((void*)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { if (!s) settle(); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return give(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return give(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }

static thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } call;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) { call = {grid, block, lds, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    *grid = call.grid, *block = call.block, *lds = call.lds, *s = call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s) { kernel(s); return hipSuccess; }
hipError_t hipExtLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s, hipEvent_t, hipEvent_t, int) { kernel(s); return hipSuccess; }
void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { capturing = true; captured = 0; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    capturing = false;
    give(g);
    nodes_of(*g) = captured;
    return hipSuccess;
}
hipError_t hipGraphCreate(hipGraph_t* g, unsigned) { return give(g); }
hipError_t hipGraphAddKernelNode(hipGraphNode_t* n, hipGraph_t g, const hipGraphNode_t*, size_t, const hipKernelNodeParams*) {
    ++nodes_of(g);
    return give(n);
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    ++graphs;
    give(e);
    nodes_of(*e) = nodes_of(g);
    return hipSuccess;
}
hipError_t hipGraphUpload(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
    kernel(s);
    last_nodes = nodes_of(e);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { std::free((void*)g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { std::free((void*)e); return hipSuccess; }

}  // extern "C"
