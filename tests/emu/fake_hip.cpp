// A HIP runtime without a device, for tests of the engine's host side (tests/test_host_calls.py).
// Loaded ahead of liblnt.so with RTLD_GLOBAL, it takes the library's HIP calls: device memory is
// host memory, kernels do nothing, and every call that orders or launches work is written to a
// log ("launch stream kernel", "graph stream nodes", "capture stream nodes", "record stream event",
// "wait stream event", "copy stream bytes", "sync stream", "stream stream" where one is made).  A launch can be made to fail.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
std::string g_log;
std::map<const void *, std::string> g_names;
std::map<hipStream_t, hipGraph_t> g_capturing;  // streams under capture
std::map<hipGraph_t, int> g_nodes;              // kernel nodes of a graph
std::map<hipEvent_t, hipGraph_t> g_captured;    // events last recorded in a capture
uintptr_t g_next = 1;
std::string g_fail_kind;
int g_fail_in = 0;
hipError_t g_last = hipSuccess;

void note(const char *what, void *stream, const std::string &more = "") {
    g_log += std::string(what) + " " + std::to_string((uintptr_t)stream) + (more.empty() ? "" : " " + more) + "\n";
}
template <class T>
T handle() {
    return (T)(g_next++);
}
bool fails(const char *kind) { return g_fail_in > 0 && g_fail_kind == kind && --g_fail_in == 0; }

struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
std::vector<Config> g_configs;
}  // namespace

extern "C" {

const char *fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }
// The nth following call of a kind ("launch": a kernel, "graph": a graph launch, "copy") fails.
void fake_fail(const char *kind, int nth) {
    g_fail_kind = kind;
    g_fail_in = nth;
}

void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, uint3 *, uint3 *, dim3 *,
                           dim3 *, int *) {
    g_names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    g_configs.push_back({grid, block, shared, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    const Config c = g_configs.back();
    g_configs.pop_back();
    *grid = c.grid, *block = c.block, *shared = c.shared, *stream = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t s) {
    auto c = g_capturing.find(s);
    if (c != g_capturing.end()) return g_nodes[c->second]++, hipSuccess;
    if (fails("launch")) return g_last = hipErrorLaunchFailure;
    note("launch", s, g_names[f]);
    return hipSuccess;
}

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof *p);
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = nullptr, hipErrorInvalidSymbol; }

hipError_t hipMalloc(void **p, size_t n) { return *p = std::calloc(1, n), *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (fails("copy")) return hipErrorUnknown;
    note("copy", st, std::to_string(n));
    return std::memmove(d, s, n), hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = handle<hipStream_t>();
    return note("stream", *s), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return note("sync", s), hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    auto c = g_captured.find(e);
    if (c != g_captured.end())
        g_capturing[s] = c->second;  // the stream joins the capture
    else
        note("wait", s, std::to_string((uintptr_t)e));
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    auto c = g_capturing.find(s);
    if (c != g_capturing.end()) return g_captured[e] = c->second, hipSuccess;
    g_captured.erase(e);
    return note("record", s, std::to_string((uintptr_t)e)), hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    g_capturing[s] = handle<hipGraph_t>();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
    *g = g_capturing[s];
    for (auto i = g_capturing.begin(); i != g_capturing.end();) i = i->second == *g ? g_capturing.erase(i) : std::next(i);
    for (auto i = g_captured.begin(); i != g_captured.end();) i = i->second == *g ? g_captured.erase(i) : std::next(i);
    return note("capture", s, std::to_string(g_nodes[*g])), hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    return *e = (hipGraphExec_t)g, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
    if (fails("graph")) return hipErrorLaunchFailure;
    return note("graph", s, std::to_string(g_nodes[(hipGraph_t)e])), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
