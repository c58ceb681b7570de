// hip_stub.cpp -- a HIP runtime that runs nothing, for tests of the engine's
// host side on a machine without a GPU.  Device memory is host memory (filled
// with 0xa5, as an allocation holds anything), launches are only written down.
// Loaded with global symbols before libcgocn.so, its entry points take the
// place of the runtime's; the log has one line per call.
#include <cxxabi.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::string g_log;
std::map<void*, size_t> g_live;          // allocations, device and pinned
std::map<const void*, std::string> g_kernel;
std::map<void*, std::string> g_stream;   // s1, s2, .. in order of creation
std::map<void*, long> g_time;            // events: the work launched before them
long g_work = 0;                         // 1 per launch of a flux split by levels, 10 per other launch
long g_fail_malloc = -1, g_fail_event = -1, g_fail_capture = -1;  // calls until one fails, -1 never

std::string stream(void* s) { return s ? g_stream[s] : "null"; }
void line(const std::string& t) { g_log += t + "\n"; }
bool fails(long& n) {
    if (n < 0) return false;
    return n-- == 0;
}
int alloc(void** p, size_t n, const char* what) {
    if (fails(g_fail_malloc)) return 2;
    *p = malloc(n ? n : 1);
    memset(*p, 0xa5, n);
    g_live[*p] = n;
    line(std::string(what) + " " + std::to_string(n));
    return 0;
}
int release(void* p, const char* what) {
    if (!p) return 0;
    if (!g_live.erase(p)) {
        line("bad " + std::string(what));
        return 1;
    }
    free(p);
    line(what);
    return 0;
}
struct dim3 {
    uint32_t x, y, z;
};
struct {
    dim3 g, b;
    size_t lds;
    void* s;
} g_cfg;
}  // namespace

extern "C" {
// what the tests read and set
const char* stub_log() { return g_log.c_str(); }
void stub_clear() { g_log.clear(); }
long stub_live() { return (long)g_live.size(); }
void stub_fail(const char* what, long n) {
    (!strcmp(what, "malloc") ? g_fail_malloc : !strcmp(what, "event") ? g_fail_event : g_fail_capture) = n;
}

void* __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void*) {}
void __hipRegisterFunction(void*, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    int st = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    std::string t = st == 0 ? d : name;
    free(d);
    if (t.rfind("void ", 0) == 0) t = t.substr(5);
    if (t.rfind("cgo::", 0) == 0) t = t.substr(5);
    std::string nosp;
    for (char c : t.substr(0, t.find('(')))
        if (c != ' ') nosp += c;
    g_kernel[host] = nosp;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s) {
    g_cfg = {g, b, lds, s};
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) {
    *g = g_cfg.g;
    *b = g_cfg.b;
    *lds = g_cfg.lds;
    *s = g_cfg.s;
    return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, void* s) {
    line("launch " + g_kernel[f] + " " + std::to_string(g.x) + "x" + std::to_string(g.y) + "x" + std::to_string(g.z) + " " +
         std::to_string(b.x) + " " + stream(s));
    const std::string& k = g_kernel[f];
    g_work += k.rfind("k_flux", 0) == 0 && k.substr(k.size() - 3) == ",3>" ? 1 : 10;
    return g.x && g.y && g.z && b.x ? 0 : 1;
}
int hipGetDeviceCount(int* n) {
    *n = 1;
    return 0;
}
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 163840;
    return 0;
}
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "stub error"; }
int hipMalloc(void** p, size_t n) { return alloc(p, n, "malloc"); }
int hipFree(void* p) { return release(p, "free"); }
int hipHostMalloc(void** p, size_t n, unsigned) { return alloc(p, n, "hostmalloc"); }
int hipHostFree(void* p) { return release(p, "hostfree"); }
// a fill of device memory is queued on the null stream, a copy waits for it
int hipMemset(void* p, int v, size_t n) {
    memset(p, v, n);
    line("memset null");
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
    memcpy(d, s, n);
    line("sync null");
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) {
    *s = malloc(1);
    g_live[*s] = 1;
    g_stream[*s] = "s" + std::to_string(g_stream.size() + 1);
    return 0;
}
int hipStreamDestroy(void* s) { return release(s, "streamdestroy"); }
int hipStreamSynchronize(void* s) {
    line("sync " + stream(s));
    return 0;
}
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipEventCreateWithFlags(void** e, unsigned) {
    if (fails(g_fail_event)) return 2;
    *e = malloc(1);
    g_live[*e] = 1;
    return 0;
}
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) { return release(e, "eventdestroy"); }
int hipEventRecord(void* e, void*) {
    g_time[e] = g_work;
    return 0;
}
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) {
    *ms = (float)(g_time[b] - g_time[a]);
    return 0;
}
int hipStreamBeginCapture(void*, int) { return fails(g_fail_capture) ? 2 : 0; }
int hipStreamEndCapture(void*, void** g) {
    if (fails(g_fail_capture)) return 2;
    *g = malloc(1);
    g_live[*g] = 1;
    return 0;
}
int hipGraphInstantiate(void** x, void*, void**, char*, size_t) {
    if (fails(g_fail_capture)) return 2;
    *x = malloc(1);
    g_live[*x] = 1;
    return 0;
}
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphExecDestroy(void* x) { return release(x, "execdestroy"); }
int hipGraphDestroy(void* g) { return release(g, "graphdestroy"); }
}
