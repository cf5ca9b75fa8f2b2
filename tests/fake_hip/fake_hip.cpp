// A stand-in for the HIP runtime, for CPU tests of the plugin's host code on its error paths: the
// plugin's .hip files compiled for the host alone link against this instead of libamdhip64. Device memory
// is zeroed host memory. Launches are queued and run when the stream is waited for; a kernel does nothing
// but publish: the traversal that opens round r of a bounce loop reports paths while r <= fake_rounds.
// Allocations and launches can be made to fail.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {

struct Launch {
    std::string name;
    unsigned long long *word = nullptr;  // where the kernel publishes, if it does
    uint32_t tag = 0;
};
// (Objects that the plugin's own static destructors still use are never destroyed.)
std::mutex &gLock = *new std::mutex;
std::deque<Launch> &gQueue = *new std::deque<Launch>;
std::set<void *> &gLive = *new std::set<void *>;
// Filled by the kernels' registration, which runs before this file's initialisers may have.
std::map<const void *, std::string> &Names() {
    static auto *m = new std::map<const void *, std::string>;
    return *m;
}
std::map<const void *, void *> &Vars() {
    static auto *m = new std::map<const void *, void *>;
    return *m;
}
long gMallocs = 0, gFailMalloc = 0, gFailLaunch = 0, gLaunches = 0, gNullCounters = 0;
int gRounds = 1, gLazy = 0;
std::string gFailName;
hipError_t gLast = hipSuccess;

void Run(const Launch &l) {
    ++gLaunches;
    if (l.word)
        __atomic_store_n(l.word, (uint64_t(l.tag) << 32) | uint64_t(int(l.tag) <= gRounds ? 1 : 0), __ATOMIC_RELAXED);
}
void Drain() {
    for (; !gQueue.empty(); gQueue.pop_front()) Run(gQueue.front());
}

}  // namespace

extern "C" {

extern const char __hip_fatbin[16] __attribute__((visibility("default")));
const char __hip_fatbin[16] = {0};

// ---- what a test sets and reads ------------------------------------------------------------------
#define FAKE __attribute__((visibility("default")))
FAKE void fake_rounds(int n) { gRounds = n; }
FAKE void fake_lazy(int on) { gLazy = on; }                  // launches wait for a synchronisation
FAKE void fake_fail_malloc(long k) { gFailMalloc = k; }      // the k-th allocation from now fails (0: none)
FAKE void fake_fail_launch(const char *name, long k) {       // the k-th launch of a kernel from now fails
    gFailName = name;
    gFailLaunch = k;
}
FAKE long fake_pending() { return long(gQueue.size()); }     // launches that nothing has waited for
FAKE long fake_live() { return long(gLive.size()); }         // device allocations
FAKE long fake_mallocs() { return gMallocs; }                // allocations so far
FAKE long fake_launches() { return gLaunches; }              // launches run so far
FAKE long fake_null_counters() { return gNullCounters; }     // counting traversals launched without counters

// ---- the runtime ----------------------------------------------------------------------------------
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    Names()[host] = name;
}
void __hipRegisterVar(void **, void *host, char *, char *, int, size_t size, int, int) {
    Vars()[host] = std::calloc(1, size);
}
struct CallConfig {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
static thread_local CallConfig gConfig;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
    gConfig = {g, b, l, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s) {
    *g = gConfig.grid, *b = gConfig.block, *l = gConfig.lds, *s = gConfig.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) {
    std::lock_guard<std::mutex> lock(gLock);
    Launch l;
    l.name = Names()[f];
    if (gFailLaunch > 0 && l.name.find(gFailName) != std::string::npos && --gFailLaunch == 0)
        return gLast = hipErrorLaunchFailure;
    const bool bounce = l.name.find("k_trace_bounce") != std::string::npos || l.name.find("k_intersect") != std::string::npos;
    if (bounce) {  // (scene, buffers, queue, publish, counters)
        struct Publish {
            unsigned long long *word;
            uint32_t tag;
        };
        const Publish p = *static_cast<const Publish *>(args[3]);
        l.word = p.word;
        l.tag = p.tag;
        if (l.name.find("ILb1E") != std::string::npos && !*static_cast<void **>(args[4])) ++gNullCounters;
    }
    gQueue.push_back(l);
    if (!gLazy) Drain();
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = gLast;
    gLast = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "fake HIP error"; }
hipError_t hipMalloc(void **p, size_t n) {
    ++gMallocs;
    if (gFailMalloc > 0 && --gFailMalloc == 0) return hipErrorOutOfMemory;
    *p = std::calloc(1, n);
    gLive.insert(*p);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
    Drain();
    gLive.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind kind, hipStream_t) {
    if (!d || !s) return hipErrorInvalidValue;
    if (kind == hipMemcpyDeviceToHost) Drain();  // (an upload is staged: it waits for nothing)
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipStreamSynchronize(hipStream_t) {
    std::lock_guard<std::mutex> lock(gLock);
    Drain();
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) { return hipStreamSynchronize(s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(new int(0));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    delete reinterpret_cast<int *>(s);
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->name, "fake");
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 4;
    p->totalGlobalMem = size_t(1) << 30;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *symbol) {
    *p = Vars()[symbol];
    return *p ? hipSuccess : hipErrorInvalidSymbol;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = reinterpret_cast<hipEvent_t>(new int(0));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<int *>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0;
    return hipSuccess;
}
// Not used by the tests that run on this.
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t *, size_t *, hipDeviceptr_t) { return hipErrorInvalidValue; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
