// Stand-in for the HIP runtime, loaded before libshockx.so so that the library's host code runs on the
// CPU: device memory is host memory, kernels do not run, copies and fills are checked against the
// allocations they touch (an overrun is counted and left undone), and a captured graph keeps the three
// arguments of a batch launch (records, work list, blocks) for graph_bad to check on every launch.
#include <dlfcn.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <map>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace {
struct Node { char *rec, *work; int total; };
struct Graph { std::vector<Node> nodes; };
std::mutex mu;
std::map<char *, size_t> device, pinned;
size_t pinned_now = 0;
int overruns = 0, graph_bad = 0, graph_nodes = 0, capture_fails = 0, host_allocs = 0, events = 0;
bool capturing = false, no_threads = false;
Graph *captured = nullptr;
thread_local int current = 0;
thread_local struct { uint64_t g[3], b[3]; size_t sh; void *st; } call;

// n bytes at p stay inside one live allocation (host memory outside all of them is the caller's)
bool inside(const std::map<char *, size_t> &m, const void *p, size_t n, bool must)
{
    char *q = (char *)p;
    auto it = m.upper_bound(q);
    if (it == m.begin()) return !must;
    --it;
    if (q >= it->first + it->second) return !must;
    return q + n <= it->first + it->second;
}
int copy(void *d, const void *s, size_t n)
{
    std::lock_guard<std::mutex> l(mu);
    if (!inside(device, d, n, false) || !inside(device, s, n, false) || !inside(pinned, d, n, false) ||
        !inside(pinned, s, n, false)) { overruns++; return 0; }
    memmove(d, s, n);
    return 0;
}
int take(std::map<char *, size_t> &m, void **p, size_t n)
{
    *p = calloc(1, n ? n : 1);
    std::lock_guard<std::mutex> l(mu);
    m[(char *)*p] = n;
    return 0;
}
}

void std::thread::_M_start_thread(_State_ptr st, void (*dep)())
{
    if (no_threads) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
    using F = void (*)(std::thread *, _State_ptr, void (*)());
    static const F real = (F)dlsym(dlopen("libstdc++.so.6", RTLD_NOW),
        "_ZNSt6thread15_M_start_threadESt10unique_ptrINS_6_StateESt14default_deleteIS1_EEPFvvE");
    real(this, std::move(st), dep);
}

extern "C" {
int stub_overruns() { return overruns; }
int stub_graph_bad() { return graph_bad; }
int stub_graph_nodes() { return graph_nodes; }
int stub_events() { return events; }
long stub_pinned() { return (long)pinned_now; }
void stub_no_threads(int on) { no_threads = on; }
void stub_fail_captures(int n) { capture_fails = n; }

int hipGetDeviceCount(int *n) { *n = 2; return 0; }
int hipGetDevice(int *d) { *d = current; return 0; }
int hipSetDevice(int d) { current = d; return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 256; return 0; }
const char *hipGetErrorString(int) { return "stub"; }
int hipGetLastError() { return 0; }
int hipMalloc(void **p, size_t n) { return take(device, p, n); }
int hipFree(void *p)
{
    std::lock_guard<std::mutex> l(mu);
    if (p) { device.erase((char *)p); free(p); }
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned)
{
    host_allocs++;
    int rc = take(pinned, p, n);
    pinned_now += n;
    return rc;
}
int hipHostFree(void *p)
{
    std::lock_guard<std::mutex> l(mu);
    if (p) { pinned_now -= pinned[(char *)p]; pinned.erase((char *)p); free(p); }
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) { return copy(d, s, n); }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { return copy(d, s, n); }
int hipMemsetAsync(void *d, int v, size_t n, void *)
{
    std::lock_guard<std::mutex> l(mu);
    if (!inside(device, d, n, true)) { overruns++; return 0; }
    memset(d, v, n);
    return 0;
}
int hipEventCreate(void **e) { *e = malloc(1); events++; return 0; }
int hipEventCreateWithFlags(void **e, unsigned) { *e = malloc(1); events++; return 0; }
int hipEventDestroy(void *e) { free(e); events--; return 0; }
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) { *ms = 1.f; return 0; }
int hipStreamCreate(void **s) { *s = malloc(1); return 0; }
int hipStreamCreateWithFlags(void **s, unsigned) { *s = malloc(1); return 0; }
int hipStreamDestroy(void *s) { free(s); return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipGetSymbolAddress(void **p, const void *) { *p = nullptr; return 1; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return 0; }

struct Dim { unsigned x, y, z; };
int hipLaunchKernel(const void *, Dim, Dim, void **args, size_t, void *)
{
    if (capturing) captured->nodes.push_back({*(char **)args[0], *(char **)args[1], *(int *)args[2]});
    return 0;
}
int hipStreamBeginCapture(void *, int) { captured = new Graph; capturing = true; return 0; }
int hipStreamEndCapture(void *, void **g) { *g = captured; capturing = false; return 0; }
int hipGraphInstantiate(void **x, void *g, void *, void *, size_t)
{
    if (capture_fails > 0) { capture_fails--; return 2; }
    *x = new Graph(*(Graph *)g);
    return 0;
}
int hipGraphDestroy(void *g) { delete (Graph *)g; return 0; }
int hipGraphExecDestroy(void *x) { delete (Graph *)x; return 0; }
int hipGraphLaunch(void *x, void *)
{
    if (!x) return 1;
    std::lock_guard<std::mutex> l(mu);
    graph_nodes = (int)((Graph *)x)->nodes.size();
    for (const Node &n : ((Graph *)x)->nodes) {
        // the work list of `total` entries (case, x, y, z), its case indices small, on the device
        bool ok = inside(device, n.rec, 1, true) && inside(device, n.work, 16 * (size_t)n.total, true);
        for (int q = 0; ok && q < n.total; q++) ok = ((int *)n.work)[4 * q] >= 0 && ((int *)n.work)[4 * q] < 64;
        if (!ok) graph_bad++;
    }
    return 0;
}
int __hipPushCallConfiguration(Dim g, Dim b, size_t sh, void *st)
{
    memcpy(call.g, &g, sizeof g); memcpy(call.b, &b, sizeof b); call.sh = sh; call.st = st;
    return 0;
}
int __hipPopCallConfiguration(Dim *g, Dim *b, size_t *sh, void **st)
{
    memcpy(g, call.g, sizeof *g); memcpy(b, call.b, sizeof *b); *sh = call.sh; *st = call.st;
    return 0;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}
