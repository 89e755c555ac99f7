// HIP runtime entry points for a process without a GPU (TEST INFRASTRUCTURE
// ONLY): loaded with global symbols before the library, they take the place
// of the runtime's.  Memory is host memory, launches are counted and do
// nothing; xth_fail(what, n) lets the next n calls of one entry point fail
// and leave the error that hipGetLastError reports, as the runtime's do.
#include <cstdlib>
#include <cstring>
#include <string>

#include <hip/hip_runtime_api.h>

namespace {
std::string g_what;
int g_fail = 0, g_kernels = 0, g_module_kernels = 0;
hipError_t g_last = hipSuccess;

hipError_t result(const char *what) {
    if (g_fail > 0 && g_what == what) {
        g_fail--;
        return g_last = hipErrorOutOfMemory;
    }
    return hipSuccess;
}
}  // namespace

#pragma GCC visibility push(default)
extern "C" {
void xth_fail(const char *what, int n) { g_what = what; g_fail = n; }
int xth_kernels(void) { return g_kernels; }
int xth_module_kernels(void) { return g_module_kernels; }

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return result("hipSetDevice"); }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipPeekAtLastError(void) { return g_last; }
const char *hipGetErrorString(hipError_t) { return "planted failure"; }
hipError_t hipMalloc(void **p, size_t n) {
    const hipError_t e = result("hipMalloc");
    *p = e == hipSuccess ? std::malloc(n ? n : 1) : nullptr;
    return e;
}
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    const hipError_t e = result("hipMemcpy");
    if (e == hipSuccess) std::memcpy(d, s, n);
    return e;
}
hipError_t hipModuleLoadData(hipModule_t *m, const void *) {
    *m = reinterpret_cast<hipModule_t>(1);
    return result("hipModuleLoadData");
}
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t, const char *) {
    *f = reinterpret_cast<hipFunction_t>(1);
    return result("hipModuleGetFunction");
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) {
    *c = hipStreamCaptureStatusNone;
    return result("hipStreamIsCapturing");
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) {
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
    g_kernels++;
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t, unsigned, unsigned, unsigned, unsigned, unsigned,
                                 unsigned, unsigned, hipStream_t, void **, void **) {
    g_module_kernels++;
    return hipSuccess;
}
}
#pragma GCC visibility pop
