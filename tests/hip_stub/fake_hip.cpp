// fake_hip.cpp -- TEST INFRASTRUCTURE: the HIP runtime functions that
// libupdec.so calls, without a device.  Loaded into a process's global scope
// before the library, so that the library's calls bind to these: "device"
// memory is host memory, kernels do nothing, and every call that depends on
// the current device or on a stream capture is written to a log.  It lets the
// CPU suite look at what the host code asks of the runtime -- on which
// device, in which order, and with how much memory -- where a real run could
// only be seen to work.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex mu;
std::string text;                        // the log, one call a line
size_t room = ~(size_t)0;                // bytes hipMalloc still gives
bool capturing = false;                  // a stream of some thread is being captured
std::map<void*, size_t> sizes;
std::vector<void*> pinned;
std::map<const void*, std::string> kernels;
thread_local int device = 0;
thread_local int capture_mode = 0;       // hipStreamCaptureModeGlobal
void say(const char* what, const std::string& rest = "")
{
    text += std::string(what) + " dev" + std::to_string(device) + (rest.empty() ? "" : " " + rest) + "\n";
}
constexpr int kInvalid = 1, kNoMemory = 2, kCapture = 900;
int take(void** p, size_t n)
{
    if (n > room) return kNoMemory;
    room -= n;
    *p = calloc(1, n ? n : 1);
    sizes[*p] = n;
    return 0;
}
int give(void* p)
{
    auto it = sizes.find(p);
    if (it == sizes.end()) return kInvalid;
    room += it->second;
    sizes.erase(it);
    // not returned to the allocator: the test may compare addresses
    return 0;
}
struct Dim3 { uint32_t x, y, z; };
struct Shape { Dim3 grid, block; size_t lds; void* stream; };
thread_local std::vector<Shape> shapes;
}  // namespace

extern "C" {
// ---- the test's side
const char* fake_log() { return text.c_str(); }
void fake_clear() { text.clear(); }
void fake_room(size_t n) { room = n; }
void fake_capturing(int on) { capturing = on != 0; }
void* fake_pinned(int i) { return i < (int)pinned.size() ? pinned[i] : nullptr; }

// ---- devices
int hipGetDevice(int* d) { *d = device; return 0; }
int hipSetDevice(int d) { device = d; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipGetDevicePropertiesR0600(void*, int) { return kInvalid; }
int hipMemGetInfo(size_t* f, size_t* t) { *f = room; *t = ~(size_t)0; return 0; }
const char* hipGetErrorString(int e) { return e == kNoMemory ? "out of memory" : e == kCapture ? "not permitted while a stream is capturing" : "error"; }
int hipGetLastError() { return 0; }
int hipDeviceSynchronize() { std::lock_guard<std::mutex> g(mu); say("hipDeviceSynchronize"); return 0; }

// ---- memory
int hipMalloc(void** p, size_t n)
{
    std::lock_guard<std::mutex> g(mu);
    const int rc = capturing && capture_mode != 2 ? kCapture : take(p, n);
    say("hipMalloc", std::to_string(n) + " -> " + std::to_string(rc));
    return rc;
}
int hipFree(void* p)
{
    std::lock_guard<std::mutex> g(mu);
    if (!p) return 0;
    say("hipFree", std::to_string(sizes.count(p) ? sizes[p] : 0));
    return give(p);
}
int hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> g(mu);
    *p = calloc(1, n ? n : 1);
    pinned.push_back(*p);
    return 0;
}
int hipHostFree(void*) { return 0; }
int hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return 0; }
int hipMallocAsync(void** p, size_t n, void*) { std::lock_guard<std::mutex> g(mu); return take(p, n); }
int hipFreeAsync(void* p, void*) { std::lock_guard<std::mutex> g(mu); return give(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::lock_guard<std::mutex> g(mu); say("hipMemcpy"); memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::lock_guard<std::mutex> g(mu); say("hipMemcpyAsync"); memcpy(d, s, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { memset(d, v, n); return 0; }
int hipGetSymbolAddress(void** p, const void*) { static char room_for_it[64]; *p = room_for_it; return 0; }

// ---- streams, events, graphs
int hipStreamCreate(void** s) { *s = malloc(1); return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { std::lock_guard<std::mutex> g(mu); say("hipStreamCreateWithFlags"); *s = malloc(1); return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { std::lock_guard<std::mutex> g(mu); say("hipStreamSynchronize"); return 0; }
int hipStreamIsCapturing(void*, int* status) { *status = capturing ? 1 : 0; return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { *g = malloc(1); return 0; }
int hipThreadExchangeStreamCaptureMode(int* m) { const int was = capture_mode; capture_mode = *m; *m = was; return 0; }
int hipEventCreate(void** e) { *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = malloc(1); return 0; }
int hipEventDestroy(void*) { return 0; }
int hipEventQuery(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0; return 0; }
int hipGraphInstantiate(void** x, void*, void*, void*, size_t) { *x = malloc(1); return 0; }
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }

// ---- kernels
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { kernels[f] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t lds, void* s) { shapes.push_back({g, b, lds, s}); return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* lds, void** s)
{
    const Shape x = shapes.back();
    shapes.pop_back();
    *g = x.grid; *b = x.block; *lds = x.lds; *s = x.stream;
    return 0;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3, void**, size_t, void*)
{
    std::lock_guard<std::mutex> l(mu);
    say("launch", kernels[f] + " grid " + std::to_string(g.x));
    return 0;
}
int hipModuleLoadData(void** m, const void*) { *m = malloc(1); return 0; }
int hipModuleUnload(void*) { return 0; }
int hipModuleGetFunction(void** f, void*, const char*) { *f = malloc(1); return 0; }
int hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int* n, void*, int, size_t) { *n = 4; return 0; }
int hipModuleLaunchKernel(void*, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, void*, void**, void**) { std::lock_guard<std::mutex> g(mu); say("launch module"); return 0; }
}
