// A HIP runtime without a GPU, for tests/test_host_runtime.py: device memory is
// host memory (zeroed), copies are done at once, kernels are only counted by
// name.  Loaded with RTLD_GLOBAL before libvkzg.so, whose HIP calls then come
// here, so the library's host code (allocations, plans, caches, accounting, what
// it does after a failed call) runs on any machine.  Results have no meaning.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex mu;
std::map<const void *, std::string> kernels;  // host stub -> device name
std::map<std::string, uint64_t> launches;
std::map<void *, size_t> dev, pinned;
uint64_t live = 0, limit = 288ull << 30, copies = 0;
int64_t fail_in = 0;  // the fail_in-th allocation from now on fails
thread_local hipError_t last = hipSuccess;
thread_local struct {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
} config;

bool alloc_fails(size_t bytes) {
    if (fail_in > 0 && --fail_in == 0) return true;
    return live + bytes > limit;
}
void *handle() { return std::malloc(16); }
}  // namespace

extern "C" {

// ------------------------------------------------------------- for the test
void host_fail_alloc(int64_t n) { fail_in = n; }
int64_t host_fail_left() { return fail_in; }
void host_limit(uint64_t bytes) { limit = bytes; }
uint64_t host_live() { return live; }
uint64_t host_copies() { return copies; }
// Launches of kernels whose name holds `part`.
uint64_t host_launches(const char *part) {
    std::lock_guard<std::mutex> lock(mu);
    uint64_t n = 0;
    for (const auto &l : launches)
        if (l.first.find(part) != std::string::npos) n += l.second;
    return n;
}

// ------------------------------------------------------------ registration
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *stub, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    std::lock_guard<std::mutex> lock(mu);
    kernels[stub] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s) {
    config = {grid, block, shmem, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, hipStream_t *s) {
    *grid = config.grid;
    *block = config.block;
    *shmem = config.shmem;
    *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *stub, dim3 grid, dim3 block, void **, size_t, hipStream_t) {
    std::lock_guard<std::mutex> lock(mu);
    const auto k = kernels.find(stub);
    if (k == kernels.end() || grid.x == 0 || block.x == 0 || block.x > 1024) return last = hipErrorInvalidValue;
    launches[k->second]++;
    return hipSuccess;
}

// ------------------------------------------------------------------ memory
hipError_t hipMalloc(void **p, size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    *p = nullptr;
    if (alloc_fails(bytes)) return last = hipErrorOutOfMemory;
    void *m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return last = hipErrorOutOfMemory;
    dev[m] = bytes;
    live += bytes;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lock(mu);
    if (!p) return hipSuccess;
    const auto d = dev.find(p);
    if (d == dev.end()) return last = hipErrorInvalidValue;
    munmap(p, d->second);
    live -= d->second;
    dev.erase(d);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    std::lock_guard<std::mutex> lock(mu);
    pinned[*p] = bytes;
    return *p == MAP_FAILED ? last = hipErrorOutOfMemory : hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::lock_guard<std::mutex> lock(mu);
    const auto h = pinned.find(p);
    if (h == pinned.end()) return last = hipErrorInvalidValue;
    munmap(p, h->second);
    pinned.erase(h);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total) {
    std::lock_guard<std::mutex> lock(mu);
    *free_bytes = live < limit ? limit - live : 0;
    *total = limit;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t) {
    if (bytes) std::memcpy(dst, src, bytes);
    std::lock_guard<std::mutex> lock(mu);
    copies++;
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t bytes) {
    std::memset(p, v, bytes);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t bytes, hipStream_t) { return hipMemset(p, v, bytes); }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *m = std::calloc(1, 16u << 20);
    *p = m;
    return hipSuccess;
}

// ---------------------------------------------------- devices, streams, graphs
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 1;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->name, "host");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = static_cast<hipStream_t>(handle());
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) {
    *c = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = static_cast<hipGraph_t>(handle());
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = static_cast<hipGraphExec_t>(handle());
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = static_cast<hipEvent_t>(handle());
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    static uint32_t x = 1;  // different times, so that a tuner chooses
    x = x * 1664525u + 1013904223u;
    *ms = 1.0f + (float)(x >> 8) / (1 << 24);
    return hipSuccess;
}

}  // extern "C"
