// A stand-in for the HIP runtime on the host, for tests of the library's host
// code: two devices whose memory is the host's, streams and events that
// remember their device, kernels that do nothing.  It refuses what HIP refuses
// (an event recorded on another device's stream, more dynamic LDS than a
// kernel was allowed on the stream's device) and counts what is made.  Loaded
// with global symbols before the library, whose calls then come here.
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

typedef int hipError_t;
struct Dim3 { unsigned x, y, z; };
struct Stream { int dev; };
struct Event { int dev; int at; };

static std::mutex g_lock;
static thread_local int t_dev = 0;
static thread_local hipError_t t_error = 0;  // of a launch
static std::map<const void*, std::string> g_names;
static std::map<std::pair<const void*, int>, int> g_lds;  // (kernel, device) -> dynamic LDS allowed
static std::map<void*, int> g_owner;                       // memory -> device
static std::map<std::string, long long> g_count;
static std::vector<std::string> g_launches;
static std::atomic<int> g_fail_host_malloc{0}, g_fail_new{0};
static std::atomic<int> g_marks{0};
static float (*g_elapsed)(int, int) = nullptr;
// a block-step launch's partition (its eighth argument: boxes along x, y, z,
// steps, threads), a one-step sweep's tiles (its second: along z, y, x, planes)
struct Grid { int v[5]; };
static std::vector<Grid> g_grids;
struct Call { Dim3 grid, block; size_t lds; Stream* stream; };
static thread_local Call t_call;

// The stand-in's own allocations never fail.
static thread_local int t_inside = 0;
struct Inside {
    Inside() { t_inside++; }
    ~Inside() { t_inside--; }
};

static void count(const char* what, int dev) {
    Inside in;
    std::lock_guard<std::mutex> l(g_lock);
    g_count[what]++;
    g_count[std::string(what) + "@" + std::to_string(dev)]++;
}
static int dev_of(Stream* s) { return s ? s->dev : t_dev; }

extern "C" {
// ---- what a test asks ----
long long host_count(const char* what) {
    std::lock_guard<std::mutex> l(g_lock);
    return g_count[what];
}
int host_launches() { return (int)g_launches.size(); }
const char* host_launch(int i) { return g_launches[(size_t)i].c_str(); }
void host_grid(int i, int* out) { memcpy(out, &g_grids[(size_t)i], sizeof(Grid)); }
void host_fail_host_malloc(int on) { g_fail_host_malloc = on; }
void host_fail_new(int on) { g_fail_new = on; }
void host_elapsed(float (*f)(int, int)) { g_elapsed = f; }

// ---- devices ----
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return 101;
    t_dev = d;
    return 0;
}
hipError_t hipGetDevice(int* d) { *d = t_dev; return 0; }
hipError_t hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
hipError_t hipGetDevicePropertiesR0600(void*, int) { return 101; }
const char* hipGetErrorString(hipError_t) { return "refused by the stand-in runtime"; }
hipError_t hipGetLastError() {
    const hipError_t e = t_error;
    t_error = 0;
    return e;
}

// ---- memory ----
static hipError_t take(void** p, size_t n, const char* what) {
    *p = calloc(1, n ? n : 1);
    count(what, t_dev);
    Inside in;
    std::lock_guard<std::mutex> l(g_lock);
    g_owner[*p] = t_dev;
    return 0;
}
hipError_t hipMalloc(void** p, size_t n) { return take(p, n, "malloc"); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (g_fail_host_malloc) return 2;
    return take(p, n, "host_malloc");
}
static hipError_t drop(void* p, const char* what) {
    count(what, t_dev);
    std::lock_guard<std::mutex> l(g_lock);
    g_owner.erase(p);
    free(p);
    return 0;
}
hipError_t hipFree(void* p) { return drop(p, "free"); }
hipError_t hipHostFree(void* p) { return drop(p, "host_free"); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, Stream*) { memcpy(d, s, n); return 0; }
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, Stream*) { memset(d, v, n); return 0; }
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, int, Stream*) { return 1; }

// ---- streams and events ----
hipError_t hipStreamCreateWithFlags(Stream** s, unsigned) {
    Inside in;
    count("stream", t_dev);
    *s = new Stream{t_dev};
    return 0;
}
hipError_t hipStreamDestroy(Stream* s) { count("stream_destroy", s->dev); delete s; return 0; }
hipError_t hipStreamSynchronize(Stream*) { return 0; }
hipError_t hipStreamWaitEvent(Stream*, Event*, unsigned) { return 0; }
hipError_t hipEventCreateWithFlags(Event** e, unsigned) {
    Inside in;
    count("event", t_dev);
    *e = new Event{t_dev, 0};
    return 0;
}
hipError_t hipEventDestroy(Event* e) { delete e; return 0; }
hipError_t hipEventRecord(Event* e, Stream* s) {
    if (e->dev != dev_of(s)) return 400;  // an event of another device
    e->at = ++g_marks;
    return 0;
}
hipError_t hipEventSynchronize(Event*) { return 0; }
hipError_t hipEventElapsedTime(float* ms, Event* a, Event* b) {
    *ms = g_elapsed ? g_elapsed(a->at, b->at) : 1.0f;
    return 0;
}

// ---- kernels ----
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    g_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t hipGetSymbolAddress(void** p, const void*) { static char room[64]; *p = room; return 0; }
hipError_t __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, Stream* s) { t_call = {g, b, lds, s}; return 0; }
hipError_t __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, Stream** s) {
    *g = t_call.grid; *b = t_call.block; *lds = t_call.lds; *s = t_call.stream;
    return 0;
}
hipError_t hipFuncSetAttribute(const void* f, int, int v) {
    Inside in;
    std::lock_guard<std::mutex> l(g_lock);
    g_lds[{f, t_dev}] = v;
    return 0;
}
hipError_t hipLaunchKernel(const void* f, Dim3, Dim3, void** args, size_t lds, Stream* s) {
    const int dev = dev_of(s);
    Inside in;
    count("launch", dev);
    if (lds > 65536) count("large_lds", dev);
    std::lock_guard<std::mutex> l(g_lock);
    g_launches.push_back(g_names[f]);
    g_grids.push_back({});
    if (g_names[f].find("k_block_steps") != std::string::npos) memcpy(&g_grids.back(), args[7], 5 * sizeof(int));
    if (g_names[f].find("k_sweep_tiled") != std::string::npos) memcpy(&g_grids.back(), args[1], 4 * sizeof(int));
    auto room = g_lds.find({f, dev});
    if ((long long)lds > (room == g_lds.end() ? 65536 : room->second)) return t_error = 1;
    return 0;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return 0; }

// ---- graphs ----
hipError_t hipStreamBeginCapture(Stream*, int) { return 0; }
hipError_t hipStreamEndCapture(Stream*, void** g) { *g = (void*)1; return 0; }
hipError_t hipGraphInstantiate(void** e, void*, void*, char*, size_t) { *e = (void*)1; return 0; }
hipError_t hipGraphLaunch(void*, Stream*) { return 0; }
hipError_t hipGraphExecDestroy(void*) { return 0; }
hipError_t hipGraphDestroy(void*) { return 0; }
}

// Allocations of the library's C++ code fail after host_fail_new(1).
void* operator new(size_t n) {
    if (g_fail_new && !t_inside) throw std::bad_alloc();
    if (void* p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
