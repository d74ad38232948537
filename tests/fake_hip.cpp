// A stand-in for the HIP runtime on a machine without a GPU, for tests of the library's host side: it runs no kernel, counts
// memory, and does every queued copy as late as the calls made allow, so that a copy whose source was changed too early is seen.
// Loaded globally in front of the library, whose calls then land here.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Copy {
    void* dst;
    const void* src;
    std::string was;  // the source when the copy was queued
    long number;
};
struct Event {
    int stream = 0;
    long number = 0;
};
long g_number = 0, g_late = 0, g_malloc_failures = 0;
std::map<int, std::vector<Copy>> g_queue;         // per stream, in order
std::map<void*, size_t> g_device;
size_t g_used = 0, g_budget = ~(size_t)0, g_fail_lo = 1, g_fail_hi = 0;
hipError_t g_last = hipSuccess;
std::map<const void*, std::string> g_names;       // host stub -> kernel
std::map<const void*, size_t> g_vars;
std::map<const void*, void*> g_symbols;
std::string g_log;
int g_streams = 0;

int id_of(hipStream_t s) { return (int)(reinterpret_cast<uintptr_t>(s) & 0xffff); }

void drain(int stream, long upto) {
    auto& q = g_queue[stream];
    size_t n = 0;
    while (n < q.size() && q[n].number <= upto) {
        g_late += std::memcmp(q[n].src, q[n].was.data(), q[n].was.size()) != 0;
        std::memcpy(q[n].dst, q[n].was.data(), q[n].was.size());
        ++n;
    }
    q.erase(q.begin(), q.begin() + n);
}
void drain_all() {
    for (auto& q : g_queue) drain(q.first, g_number);
}
}  // namespace

extern "C" {
// ---- for the tests
void fake_set_budget(size_t bytes) { g_budget = bytes; }
void fake_fail_sizes(size_t lo, size_t hi) { g_fail_lo = lo, g_fail_hi = hi; }
size_t fake_used() { return g_used; }
long fake_late_copies() { return g_late; }
long fake_malloc_failures() { return g_malloc_failures; }
long fake_pending(int stream) { return (long)g_queue[stream].size(); }
const char* fake_log() { return g_log.c_str(); }
void fake_clear_log() { g_log.clear(); }

// ---- the runtime
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e == hipSuccess ? "no error" : "error"; }
hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (g_used + n > g_budget || (n >= g_fail_lo && n <= g_fail_hi)) {
        ++g_malloc_failures;
        return g_last = hipErrorOutOfMemory;
    }
    if (posix_memalign(p, 256, n ? n : 1)) return g_last = hipErrorOutOfMemory;
    g_log += "malloc " + std::to_string(n) + "\n";
    g_device[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    drain_all();
    auto it = g_device.find(p);
    if (it == g_device.end()) return p ? g_last = hipErrorInvalidValue : hipSuccess;
    g_used -= it->second;
    g_device.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = nullptr;
    if (n >= g_fail_lo && n <= g_fail_hi) return g_last = hipErrorOutOfMemory;
    return posix_memalign(p, 256, n ? n : 1) ? g_last = hipErrorOutOfMemory : hipSuccess;
}
hipError_t hipHostFree(void* p) {
    drain_all();  // (as the runtime's does)
    return std::free(p), hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = (size_t)1 << 38, *t = (size_t)1 << 38, hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
    g_queue[id_of(s)].push_back({dst, src, std::string(static_cast<const char*>(src), n), ++g_number});
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) {
    drain_all();
    return std::memcpy(dst, src, n), hipSuccess;
}
hipError_t hipMemsetAsync(void* dst, int v, size_t n, hipStream_t s) {
    drain(id_of(s), g_number);
    return std::memset(dst, v, n), hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>((uintptr_t)(100 + g_streams++)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) { return *c = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    g_log += "sync " + std::to_string(id_of(s)) + "\n";
    return drain(id_of(s), g_number), hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    g_log += "wait " + std::to_string(id_of(s)) + " " + std::to_string(reinterpret_cast<Event*>(e)->stream) + "\n";
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    g_log += "sync all\n";
    return drain_all(), hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(new Event()), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<Event*>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return *reinterpret_cast<Event*>(e) = {id_of(s), ++g_number}, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) {
    const Event* v = reinterpret_cast<Event*>(e);
    return drain(v->stream, v->number), hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) { return std::memset(a, 0, sizeof(*a)), hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    void*& at = g_symbols[symbol];
    if (!at && posix_memalign(&at, 256, g_vars[symbol] ? g_vars[symbol] : 1)) return hipErrorOutOfMemory;
    return *p = at, hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, hipStream_t s) {
    g_log += "run " + std::to_string(id_of(s)) + " " + g_names[f] + " " + std::to_string((long)grid.x * grid.y * grid.z) + " " + std::to_string(block.x) + "\n";
    return hipSuccess;
}
struct Call {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
static thread_local std::vector<Call> g_calls;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { return g_calls.push_back({g, b, lds, s}), hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    const Call c = g_calls.back();
    g_calls.pop_back();
    return *g = c.grid, *b = c.block, *lds = c.lds, *s = c.stream, hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { g_names[f] = name; }
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) { g_vars[var] = size; }
}
