// A HIP runtime without a device, for the library's error handling on the CPU: loaded (globally) before the
// library, it takes the library's calls. Device memory is host memory, kernels do nothing, and a chosen call
// or launch fails with a chosen error, as it would on a device.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

#include <hip/hip_runtime_api.h>

namespace {
std::mutex m;
std::map<const void *, std::string> kernels;
std::map<std::string, long> counts;          // calls by name; launches also as "launch"
std::string failWhat;
long failAt = -1;
hipError_t failWith = hipSuccess;
hipError_t last = hipSuccess;                 // (one for all threads, where the runtime has one each)
bool placesBad = false;
int refusePinned = 0;
unsigned long long handle = 1;
void *symbol = nullptr;

// counts a call of `name` (kernels by a part of their name) and tells whether it is the one to fail
hipError_t called(const char *name, const std::string &kernel = std::string()) {
    std::lock_guard<std::mutex> lk(m);
    counts[name]++;
    if (!kernel.empty()) counts[kernel]++;
    const bool hit = failAt >= 0 && (kernel.empty() ? failWhat == name : kernel.find(failWhat) != std::string::npos);
    if (hit && failAt-- == 0) return last = failWith;
    return hipSuccess;
}
template <typename T> void give(T *out) { *out = reinterpret_cast<T>(handle += 16); }
}  // namespace

extern "C" {
// the test's side
void stand_in_fail(const char *what, long nth, int error) {
    std::lock_guard<std::mutex> lk(m);
    failWhat = what;
    failAt = nth;
    failWith = (hipError_t)error;
    last = hipSuccess;
}
void stand_in_refuse_pinned(int calls) { refusePinned = calls; }
void stand_in_places_outside(int on) { placesBad = on != 0; }
long stand_in_count(const char *part) {
    std::lock_guard<std::mutex> lk(m);
    long n = 0;
    for (auto &kv : counts) n += kv.first.find(part) != std::string::npos ? kv.second : 0;
    return n;
}

// the library's side
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t size, int, int) { symbol = calloc(size, 1); }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) {
    const std::string &name = kernels[f];
    if (placesBad && name.find("k_places") != std::string::npos) **static_cast<int **>(args[4]) = 1;
    return called("launch", name);
}
hipError_t hipMalloc(void **p, size_t n) {
    *p = calloc(n ? n : 1, 1);
    return called("hipMalloc");
}
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (refusePinned > 0) {
        refusePinned--;
        return last = hipErrorOutOfMemory;
    }
    *p = calloc(n, 1);
    return called("hipHostMalloc");
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    if (!d || !s) return last = hipErrorInvalidValue;
    memmove(d, s, n);
    return called("hipMemcpy");
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    if (!d || !s) return last = hipErrorInvalidValue;
    memmove(d, s, n);
    return called("hipMemcpyAsync");
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return called("hipMemsetAsync"); }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)1 << 34; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 4; return hipSuccess; }
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipPeekAtLastError(void) { return last; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorInvalidValue ? "invalid argument" : "stand-in error"; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = symbol; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
    memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { give(s); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return called("hipStreamSynchronize"); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { give(g); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *g, hipGraph_t, hipGraphNode_t *, char *, size_t) { give(g); return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return called("hipGraphLaunch"); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { give(e); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { give(e); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return called("hipEventRecord"); }
hipError_t hipEventSynchronize(hipEvent_t) { return called("hipEventSynchronize"); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
}
