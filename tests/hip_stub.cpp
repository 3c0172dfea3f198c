// Host-only stand-in for the part of the HIP runtime that libps3d_gpu.so uses, for tests of
// its host code without a GPU: device memory is host memory, kernels do nothing, streams run
// at once.  Two devices with a current one per thread; an event is recorded on streams of its
// own device only; a failed call leaves its error for hipGetLastError.
// STUB_HOST_ALLOCS: how many hipHostMalloc calls succeed (default: all).
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <cstring>

namespace {
thread_local int cur = 0;
thread_local hipError_t last = hipSuccess;
std::atomic<int> host_calls{0}, launches{0};
struct Obj { int dev; };
hipError_t ret(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
template <class T>
hipError_t make(T *out) {
    *out = reinterpret_cast<T>(new Obj{cur});
    return hipSuccess;
}
int dev(const void *p) { return static_cast<const Obj *>(p)->dev; }
hipError_t alloc(void **p, size_t n) {
    *p = std::calloc(n ? n : 1, 1);
    return ret(*p ? hipSuccess : hipErrorOutOfMemory);
}
}  // namespace

extern "C" {
int stub_host_calls() { return host_calls; }
int stub_launches() { return launches; }

hipError_t hipGetDevice(int *d) { return *d = cur, hipSuccess; }
hipError_t hipSetDevice(int d) { return d < 0 || d > 1 ? ret(hipErrorInvalidDevice) : (cur = d, hipSuccess); }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorInvalidHandle ? "invalid handle" : e == hipErrorOutOfMemory ? "out of memory" : "error"; }

hipError_t hipMalloc(void **p, size_t n) { return alloc(p, n); }
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    const char *k = std::getenv("STUB_HOST_ALLOCS");
    if (host_calls++ >= (k ? std::atoi(k) : 1 << 30)) return ret(hipErrorOutOfMemory);
    return alloc(p, n);
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind) {
    for (size_t i = 0; i < h; ++i) std::memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return make(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return delete reinterpret_cast<Obj *>(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return make(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return make(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<Obj *>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return ret(dev(e) == dev(s) ? hipSuccess : hipErrorInvalidHandle); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }

hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return ++launches, hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static double scratch[8];
    return *p = scratch, hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return ret(hipErrorNotSupported); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return ret(hipErrorNotSupported); }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return ret(hipErrorNotSupported); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return ret(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}
