// A stand-in for the HIP runtime on host memory, for tests of the library's
// error paths without a GPU: allocations are malloc's, copies happen at once,
// kernels don't run.  Calls that touch a stream are logged, and the n-th
// allocation or launch of a kernel can be made to fail.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

static std::map<const void *, std::string> names;
static std::string calls, fail_name;
static int fail_in = 0;
static hipError_t last = hipSuccess;

static hipError_t note(const std::string &what, hipError_t error) {
    const bool fails = !fail_name.empty() && what.find(fail_name) != std::string::npos && --fail_in == 0;
    calls += what + (fails ? " failed\n" : "\n");
    if (fails) last = error;
    return fails ? error : hipSuccess;
}

extern "C" {

const char *host_hip_calls() { return calls.c_str(); }
// Forgets the calls so far; the n-th call from here whose name holds `name` fails.
void host_hip_fail(const char *name, int n) {
    calls.clear();
    fail_name = name;
    fail_in = n;
}

void **__hipRegisterFatBinary(const void *) {
    static void *p;
    return &p;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s) {
    *g = *b = dim3(1);
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
    return note("launch " + names[f], hipErrorLaunchFailure);
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }
hipError_t hipMalloc(void **p, size_t n) {
    const hipError_t e = note("malloc", hipErrorOutOfMemory);
    *p = e == hipSuccess ? std::malloc(n ? n : 1) : nullptr;
    return e;
}
hipError_t hipFree(void *p) {
    std::free(p);
    return note("free", hipSuccess);
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::malloc(n ? n : 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return note("copy", hipErrorInvalidValue);
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return note("synchronize", hipErrorUnknown); }

}  // extern "C"
