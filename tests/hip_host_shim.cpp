// A HIP runtime without a GPU, for tests of the host side on the CPU: memory is host memory, copies and
// fills are done at once, kernels are not run, and every stream-ordered call is noted in a text log, a
// line each. Loaded with RTLD_GLOBAL before the library, whose HIP calls then come here.
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
std::string g_log;
std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m;
    return m;
}
size_t g_refuse = 0;  // pinned allocations of this size fail
intptr_t g_handles = 0x1000;
Dim3 g_grid, g_block;
void* g_stream;

void note(const char* fmt, auto... args) {
    char line[256];
    snprintf(line, sizeof(line), fmt, args...);
    g_log += line;
    g_log += '\n';
}
int handle(void** p) {
    *p = reinterpret_cast<void*>(g_handles += 16);
    return 0;
}
}  // namespace

extern "C" {
const char* shim_log() { return g_log.c_str(); }
void shim_clear() { g_log.clear(); }
void shim_refuse_pinned(size_t bytes) { g_refuse = bytes; }

int hipGetDeviceCount(int* n) { return *n = 1, 0; }
int hipGetDevice(int* d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipGetLastError() { return 0; }
int hipPeekAtLastError() { return 0; }
const char* hipGetErrorString(int) { return "shim"; }
int hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = (size_t)64 << 30, 0; }
int hipMalloc(void** p, size_t n) { return (*p = calloc(n, 1)) ? 0 : 2; }
int hipFree(void* p) { return free(p), 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { return n == g_refuse ? 2 : hipMalloc(p, n); }
int hipHostFree(void* p) { return free(p), 0; }
int hipGetSymbolAddress(void** p, const void*) {
    static char zero[1 << 20];
    return *p = zero, 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) { return memcpy(d, s, n), 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* st) {
    note("copy %p stream %p", d, st);
    return memcpy(d, s, n), 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return memset(d, v, n), 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return handle(s); }
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void* s) { return note("sync stream %p", s), 0; }
int hipStreamWaitEvent(void* s, void* e, unsigned) { return note("wait %p stream %p", e, s), 0; }
int hipEventCreate(void** e) { return handle(e); }
int hipEventCreateWithFlags(void** e, unsigned) { return handle(e); }
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void* e, void* s) { return note("record %p stream %p", e, s), 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 1.f, 0; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) { return handle(e); }
int hipGraphLaunch(void*, void*) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { return handle(g); }
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t, void* s) {
    g_grid = g;
    g_block = b;
    g_stream = s;
    return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* sh, void** s) {
    *g = g_grid;
    *b = g_block;
    *sh = 0;
    *s = g_stream;
    return 0;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3 b, void** args, size_t, void* s) {
    const std::string& name = names()[f];
    // the refit kernels: how many of the first 14 words of the device state are set (up to the KEEP records)
    int set = 0;
    if (name.find("k_refit") != std::string::npos)
        for (int i = 0; i < 14; ++i)
            set += static_cast<void**>(args[name.find("k_refit_top") != std::string::npos ? 0 : 1])[i] != nullptr;
    note("launch %s grid %u block %u set %d stream %p", name.c_str(), g.x, b.x, set, s);
    return 0;
}
void** __hipRegisterFatBinary(const void*) {
    static void* module;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}
