// The HIP entry points that libvoxel_hip.so calls, as host memory and a log:
// what the library queues, in which order, and what it does when a call fails
// can then be checked without a GPU.  Loaded with RTLD_GLOBAL before the
// library, whose calls then bind here.  Kernels are logged by name and do
// nothing; fresh memory is filled with 0xA5; a call on a capturing stream is
// logged as captured and does nothing either.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
struct Dim3 {
    uint32_t x, y, z;
};
constexpr int kOk = 0, kFailed = 999, kUnsupported = 900;
std::string g_log, g_fail;
std::map<const void *, std::string> g_kernels;
void *g_capturing = nullptr;  // the capturing stream
void *g_captured = nullptr;   // the last that was
void *g_synced = nullptr;     // the last stream waited for
int g_capture_mode = 0;
Dim3 g_grid, g_block;
size_t g_shared;
void *g_stream;
uintptr_t g_handles = 0x1000;

// Logs a call; true if it is the one that calls_fail named.
bool call(const std::string &name, const void *stream = nullptr) {
    g_log += (g_capturing && stream == g_capturing ? "captured:" : "") + name + "\n";
    if (g_fail != name) return false;
    g_fail.clear();
    return true;
}
bool captured(const void *stream) { return g_capturing && stream == g_capturing; }
int make(void **out) {
    *out = (void *)(g_handles += 0x10);
    return kOk;
}
}  // namespace

extern "C" {
// ---- for the test
const char *calls_log() { return g_log.c_str(); }
void calls_clear() { g_log.clear(); }
void calls_fail(const char *name) { g_fail = name; }  // the next call of that name fails
void *calls_capture_stream() { return g_captured; }
void *calls_synced_stream() { return g_synced; }

// ---- HIP
int hipGetDeviceCount(int *n) { return *n = 1, kOk; }
int hipSetDevice(int) { return kOk; }
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, kOk; }
int hipGetLastError() { return kOk; }
const char *hipGetErrorString(int) { return "failed by the test"; }
int hipMalloc(void **p, size_t n) {
    if (call("hipMalloc")) return 2;
    if (g_capturing && g_capture_mode != 2) return kUnsupported;
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    memset(*p, 0xA5, n);
    return kOk;
}
int hipFree(void *p) { return free(p), kOk; }
int hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(1, n), kOk; }
int hipHostFree(void *p) { return free(p), kOk; }
int hipMemcpy(void *d, const void *s, size_t n, int) { return memcpy(d, s, n), kOk; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *st) {
    if (call("hipMemcpyAsync", st)) return kFailed;
    if (!captured(st)) memcpy(d, s, n);
    return kOk;
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) {
    if (call("hipMemsetAsync", st)) return kFailed;
    if (!captured(st)) memset(d, v, n);
    return kOk;
}
int hipStreamCreateWithFlags(void **s, unsigned) { return make(s); }
int hipStreamDestroy(void *) { return kOk; }
int hipStreamSynchronize(void *s) {
    g_synced = s;
    if (call("hipStreamSynchronize", s)) return kFailed;
    return captured(s) ? kUnsupported : kOk;
}
int hipStreamWaitEvent(void *s, void *, unsigned) { return call("hipStreamWaitEvent", s) ? kFailed : kOk; }
int hipEventCreate(void **e) { return make(e); }
int hipEventCreateWithFlags(void **e, unsigned) { return make(e); }
int hipEventDestroy(void *) { return kOk; }
int hipEventRecord(void *, void *s) { return call("hipEventRecord", s) ? kFailed : kOk; }
int hipEventQuery(void *) { return kOk; }
int hipEventSynchronize(void *) { return call("hipEventSynchronize") ? kFailed : kOk; }
int hipEventElapsedTime(float *ms, void *, void *) { return *ms = 1.0f, kOk; }
int hipStreamBeginCapture(void *s, int mode) {
    if (call("hipStreamBeginCapture") || g_capturing) return kFailed;
    g_capturing = g_captured = s;
    g_capture_mode = mode;
    return kOk;
}
int hipStreamEndCapture(void *, void **g) {
    g_capturing = nullptr;
    if (call("hipStreamEndCapture")) return *g = nullptr, kFailed;
    return make(g);
}
int hipStreamIsCapturing(void *s, int *status) { return *status = captured(s), kOk; }
int hipGraphInstantiate(void **x, void *, void **, char *, size_t) {
    return call("hipGraphInstantiate") ? kFailed : make(x);
}
int hipGraphLaunch(void *, void *s) { return call("hipGraphLaunch", s) ? kFailed : kOk; }
int hipGraphDestroy(void *) { return kOk; }
int hipGraphExecDestroy(void *) { return kOk; }
int hipGetSymbolAddress(void **p, const void *) {
    static uint32_t words[4096];
    return *p = words, kOk;
}
int hipLaunchKernel(const void *f, Dim3 g, Dim3, void **, size_t, void *s) {
    char grid[16];
    snprintf(grid, sizeof grid, " %u", g.x);
    return call(g_kernels[f] + grid, s) ? kFailed : kOk;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t n, void *s) {
    g_grid = g, g_block = b, g_shared = n, g_stream = s;
    return kOk;
}
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *n, void **s) {
    *g = g_grid, *b = g_block, *n = g_shared, *s = g_stream;
    return kOk;
}
void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *,
                           void *, void *, int *) {
    // _ZN2vx11fill_kernelILi32EEE... -> fill_kernel
    std::string s = name;
    if (s.rfind("_ZN2vx", 0) == 0) {
        char *rest;
        const unsigned long n = strtoul(name + 6, &rest, 10);
        s.assign(rest, n);
    }
    g_kernels[f] = s;
}
}
