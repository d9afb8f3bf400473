// Host stand-in for the HIP runtime calls of libemptyroom.so, for CPU tests of
// the host code around the kernels.  Loaded with RTLD_GLOBAL before the library,
// it takes the place of the real runtime: two devices, device memory from malloc,
// kernels that only take time (fake_kernel_ms on their stream), copies that are
// done when their stream gets there.  What HIP refuses and the tests rely on is
// refused: an event recorded on a stream of another device.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <thread>

using Clock = std::chrono::steady_clock;

namespace {
struct Stream {
    int device;
    Clock::time_point busy = Clock::now();
};
struct Event {
    int device;
    Clock::time_point at = Clock::now();
};
std::mutex mu;
std::map<void *, size_t> device_memory;
std::set<char *> pinned;  // slots of 2 MiB and more
size_t device_used = 0, device_limit = (size_t)64 << 30;
std::atomic<int> kernel_ms{0}, frees{0}, mallocs{0}, host_throws{0}, ring_copies{0};
thread_local int device = 0;
Stream *S(hipStream_t s) { return reinterpret_cast<Stream *>(s); }
Event *E(hipEvent_t e) { return reinterpret_cast<Event *>(e); }
}  // namespace

extern "C" {

// --- what a test sets and reads ------------------------------------------------
void fake_kernel_ms(int ms) { kernel_ms = ms; }
void fake_device_limit(size_t bytes) { device_limit = bytes; }
void fake_host_malloc_throws(int on) { host_throws = on; }
size_t fake_device_used() { return device_used; }
int fake_ring_copies() { return ring_copies; }  // copies into pinned blocks of 2 MiB
int fake_mallocs() { return mallocs; }
int fake_frees() { return frees; }

// --- devices and memory ----------------------------------------------------------
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return hipErrorInvalidDevice;
    device = d;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total) {
    std::lock_guard<std::mutex> lk(mu);
    *total = device_limit;
    *free_bytes = device_limit - device_used;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> lk(mu);
    mallocs++;
    *p = nullptr;
    if (device_used + n > device_limit || !(*p = std::calloc(1, n))) return hipErrorOutOfMemory;
    device_memory[*p] = n;
    device_used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lk(mu);
    frees++;
    auto it = device_memory.find(p);
    if (it == device_memory.end()) return hipErrorInvalidValue;
    device_used -= it->second;
    device_memory.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (host_throws) throw std::bad_alloc();  // as the library's own host memory can
    *p = std::calloc(1, n);
    std::lock_guard<std::mutex> lk(mu);
    if (n == (2u << 20)) pinned.insert((char *)*p);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
    std::lock_guard<std::mutex> lk(mu);
    pinned.erase((char *)p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *m = std::calloc(1, (size_t)64 << 20);
    *p = m;
    return hipSuccess;
}

// --- streams and events ------------------------------------------------------------
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(new Stream{device});
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { delete S(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::this_thread::sleep_until(S(s)->busy);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new Event{device});
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete E(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (E(e)->device != S(s)->device) return hipErrorInvalidHandle;
    E(e)->at = S(s)->busy;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    return Clock::now() < E(e)->at ? hipErrorNotReady : hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(to, from, n);
    std::lock_guard<std::mutex> lk(mu);
    if (pinned.count((char *)to)) ring_copies++;
    return hipSuccess;
}

// --- kernels and graphs ------------------------------------------------------------
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s) {
    Stream *t = S(s);
    const auto now = Clock::now();
    t->busy = (t->busy > now ? t->busy : now) + std::chrono::milliseconds(kernel_ms);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 4;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = reinterpret_cast<hipGraph_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *x = reinterpret_cast<hipGraphExec_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { std::free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { std::free(x); return hipSuccess; }

hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake"; }
const char *hipGetErrorName(hipError_t) { return "fake"; }

// --- what the compiler's launch stubs and module constructors call --------------------
thread_local dim3 call_grid, call_block;
thread_local size_t call_lds;
thread_local hipStream_t call_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    call_grid = g;
    call_block = b;
    call_lds = lds;
    call_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = call_grid;
    *b = call_block;
    *lds = call_lds;
    *s = call_stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *,
                           void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}
