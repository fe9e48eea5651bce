// hip_host_stub.cpp -- a HIP runtime without a GPU, for the library's host side: linked with the
// library's own objects in place of libamdhip64, so a call runs all of its host code, with kernel
// launches that do nothing.  Device memory is zeroed host memory under a limit the test sets; every
// handle that a call passes (pointer, stream, event, graph) has to be alive, and what is not is noted.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {
struct State {
    std::mutex m;
    std::map<char *, size_t> mem;
    std::set<void *> streams, events, graphs, execs;
    std::map<std::string, long> calls;
    std::map<const void *, std::string> kernels;
    size_t used = 0, limit = ~size_t(0), most = 0;
    std::string faults;
};
State &st() {
    static State *s = new State;  // outlives the library's static objects
    return *s;
}
char g_symbol[64 << 20];
thread_local dim3 t_grid, t_block;
thread_local size_t t_lds;
thread_local hipStream_t t_stream;

struct Call {
    std::lock_guard<std::mutex> lk{st().m};
    const char *name;
    explicit Call(const char *n) : name(n) { ++st().calls[n]; }
    void need(bool ok, const char *what) {
        if (!ok) st().faults += std::string(name) + ": " + what + "; ";
    }
    void stream(hipStream_t s) { need(!s || st().streams.count(s), "not a stream"); }
    void event(hipEvent_t e) { need(st().events.count(e), "not an event"); }
    bool inside(const void *p, size_t n) {
        auto it = st().mem.upper_bound((char *)p);
        if (it == st().mem.begin()) return false;
        --it;
        return (char *)p + n <= it->first + it->second;
    }
};
template <typename H>
hipError_t fresh(std::set<void *> &live, H *out) {
    void *h = new char;  // never reused: a stale handle stays recognisable
    live.insert(h);
    *out = (H)h;
    return hipSuccess;
}
}  // namespace

extern "C" {
// ---- the test's side
void stub_limit(size_t bytes) { st().limit = bytes; }
size_t stub_used() { return st().used; }
size_t stub_most() {  // the largest use since the last call of this
    const size_t v = st().most;
    st().most = st().used;
    return v;
}
long stub_calls(const char *name) { return st().calls[name]; }
long stub_launches(const char *kernel) {  // launches of the kernels whose mangled name holds `kernel`
    long n = 0;
    for (auto &c : st().calls)
        if (c.first.compare(0, 2, "_Z") == 0 && c.first.find(kernel) != std::string::npos) n += c.second;
    return n;
}
const char *stub_faults() { return st().faults.c_str(); }

// ---- registration and launches
void **__hipRegisterFatBinary(const void *) { return new void *; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *) {
    st().kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    t_grid = g, t_block = b, t_lds = lds, t_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = t_grid, *b = t_block, *lds = t_lds, *s = t_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t lds, hipStream_t s) {
    Call c("hipLaunchKernel");
    c.stream(s);
    ++st().calls[st().kernels[f]];
    c.need(g.x && g.y && g.z && b.x && b.x * b.y * b.z <= 1024 && lds <= 160 * 1024, "launch shape");
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 2;
    return hipSuccess;
}

// ---- device
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {  // (the header renames it)
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }

// ---- memory
hipError_t hipMalloc(void **p, size_t n) {
    Call c("hipMalloc");
    if (n > st().limit - (st().used < st().limit ? st().used : st().limit)) return hipErrorOutOfMemory;
    const size_t pages = (n + 4095) & ~size_t(4095);
    *p = mmap(nullptr, pages ? pages : 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    st().mem[(char *)*p] = n;
    st().used += n;
    if (st().used > st().most) st().most = st().used;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    Call c("hipFree");
    if (!p) return hipSuccess;
    auto it = st().mem.find((char *)p);
    c.need(it != st().mem.end(), "not an allocation");
    if (it == st().mem.end()) return hipErrorInvalidValue;
    const size_t pages = (it->second + 4095) & ~size_t(4095);
    munmap(p, pages ? pages : 4096);
    st().used -= it->second;
    st().mem.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    *p = g_symbol;
    return hipSuccess;
}
static hipError_t copy(Call &c, void *d, const void *s, size_t n, hipMemcpyKind k) {
    if (k == hipMemcpyDeviceToHost) c.need(c.inside(s, n), "source outside device memory");
    if (k == hipMemcpyHostToDevice) c.need(c.inside(d, n), "destination outside device memory");
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
    Call c("hipMemcpy");
    return copy(c, d, s, n, k);
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t q) {
    Call c("hipMemcpyAsync");
    c.stream(q);
    return copy(c, d, s, n, k);
}
hipError_t hipMemset(void *p, int v, size_t n) {
    Call c("hipMemset");
    c.need(c.inside(p, n), "outside device memory");
    memset(p, v, n);
    return hipSuccess;
}

// ---- streams, events, graphs
#define STUB_END(set_, h_)                            \
    c.need(st().set_.erase((void *)h_), "not alive"); \
    return hipSuccess
hipError_t hipStreamCreate(hipStream_t *s) {
    Call c("hipStreamCreate");
    return fresh(st().streams, s);
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    Call c("hipStreamCreateWithFlags");
    return fresh(st().streams, s);
}
hipError_t hipStreamDestroy(hipStream_t s) {
    Call c("hipStreamDestroy");
    STUB_END(streams, s);
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    Call c("hipStreamSynchronize");
    c.stream(s);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    Call c("hipStreamWaitEvent");
    c.stream(s);
    c.event(e);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
    Call c("hipEventCreate");
    return fresh(st().events, e);
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    Call c("hipEventCreateWithFlags");
    return fresh(st().events, e);
}
hipError_t hipEventDestroy(hipEvent_t e) {
    Call c("hipEventDestroy");
    STUB_END(events, e);
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Call c("hipEventRecord");
    c.stream(s);
    c.event(e);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    Call c("hipEventSynchronize");
    c.event(e);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
    Call c("hipEventElapsedTime");
    c.event(a);
    c.event(b);
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    Call c("hipStreamBeginCapture");
    c.stream(s);
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    Call c("hipStreamEndCapture");
    return fresh(st().graphs, g);
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    Call c("hipGraphInstantiate");
    return fresh(st().execs, e);
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
    Call c("hipGraphLaunch");
    c.stream(s);
    c.need(st().execs.count(e), "not alive");
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    Call c("hipGraphExecDestroy");
    STUB_END(execs, e);
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    Call c("hipGraphDestroy");
    STUB_END(graphs, g);
}
}  // extern "C"
