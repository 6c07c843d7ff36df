// A HIP runtime for host tests on the CPU: a program that includes this defines
// the runtime calls that the library makes (the executable's definitions come
// before libamdhip64's), with host memory for device memory, launches that run
// nothing, a limit on the device's memory and a launch that fails.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>

namespace {
hipError_t g_pending = hipSuccess;  // what hipGetLastError returns
size_t g_limit = ~size_t{0}, g_used = 0;
std::map<void*, size_t> g_blocks;
long g_launches = 0, g_fail_at = -1;
dim3 g_grid;  // the last launch's

hipError_t fail(hipError_t e) {
    g_pending = e;
    return e;
}
template <class T>
hipError_t handle(T* out) {
    *out = reinterpret_cast<T>(std::malloc(1));
    return hipSuccess;
}
template <class T>
hipError_t drop(T h) {
    std::free(reinterpret_cast<void*>(h));
    return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t __hipPushCallConfiguration(dim3 g, dim3, size_t, hipStream_t) {
    return g_grid = g, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = g_grid;
    *b = dim3(1);
    *lds = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    return g_launches++ == g_fail_at ? fail(hipErrorLaunchOutOfResources) : hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_pending;
    g_pending = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (n > g_limit - g_used) return fail(hipErrorOutOfMemory);
    *p = std::malloc(n);
    if (!*p) return fail(hipErrorOutOfMemory);
    g_blocks[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    g_used -= g_blocks[p];
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    return std::memset(d, v, n), hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return drop(s); }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return drop(e); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return handle(x);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return drop(g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return drop(x); }
}
