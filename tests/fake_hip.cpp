// fake_hip.cpp -- the HIP runtime calls libnekcem_hip.so makes, on host
// memory, so that its host side can be driven and watched without a GPU.
// Kernels do not run: a launch is logged with its name, grid, block and
// stream.  Copies and fills are done at once, inside the allocations they
// name; two devices with a settable capacity; the n-th launch from now can be
// made to fail.  Loaded with RTLD_GLOBAL before the library.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cxxabi.h>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Block {
    size_t bytes;
    int device;   // -1: pinned host memory
};
std::mutex mu;
std::map<const char *, Block> blocks;
std::map<const void *, std::string> kernels;
std::string text;
hipError_t last = hipSuccess;
int current = 0;
long fail_in = -1;
size_t cap[2] = {size_t(1) << 40, size_t(1) << 40}, used[2] = {0, 0};
int next_id = 1;

struct Config {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
};
thread_local std::vector<Config> configs;

hipError_t done(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
int id(const void *h) { return (int)(intptr_t)h; }

__attribute__((format(printf, 1, 2))) void note(const char *f, ...) {
    char s[512];
    va_list a;
    va_start(a, f);
    vsnprintf(s, sizeof s, f, a);
    va_end(a);
    text += s;
    text += '\n';
}

const Block *find(const void *p, const char **base) {
    auto it = blocks.upper_bound((const char *)p);
    if (it == blocks.begin()) return nullptr;
    --it;
    if ((const char *)p >= it->first + it->second.bytes) return nullptr;
    *base = it->first;
    return &it->second;
}

// Whether n bytes from p stay inside the allocation p lies in (plain host memory: yes).
bool inside(const void *p, size_t n) {
    const char *base = nullptr;
    const Block *b = find(p, &base);
    return !b || (size_t)((const char *)p - base) + n <= b->bytes;
}

}  // namespace

extern "C" {

// ---- what the tests use ----
void fake_clear_log() { std::lock_guard<std::mutex> l(mu); text.clear(); }
const char *fake_log() { return text.c_str(); }
void fake_fail_launch(long n) { fail_in = n; }
void fake_set_capacity(int dev, size_t bytes) { cap[dev] = bytes; }
size_t fake_used(int dev) { return used[dev]; }

// ---- the runtime ----
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> l(mu);
    if (used[current] + n > cap[current]) return done(hipErrorOutOfMemory);
    void *m = nullptr;
    if (posix_memalign(&m, 256, n ? n : 1)) return done(hipErrorOutOfMemory);
    memset(m, 0x7f, n);      // nothing a caller may rely on
    blocks[(const char *)m] = {n, current};
    used[current] += n;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> l(mu);
    if (!p) return hipSuccess;
    auto it = blocks.find((const char *)p);
    if (it == blocks.end() || it->second.device < 0) return done(hipErrorInvalidValue);
    used[it->second.device] -= it->second.bytes;
    blocks.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    std::lock_guard<std::mutex> l(mu);
    *p = malloc(n);
    memset(*p, 0xff, n);     // what a check that finds nothing writes
    blocks[(const char *)*p] = {n, -1};
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::lock_guard<std::mutex> l(mu);
    blocks.erase((const char *)p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *fr, size_t *tot) {
    *tot = cap[current];
    *fr = cap[current] - used[current];
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *n, hipDeviceptr_t p) {
    std::lock_guard<std::mutex> l(mu);
    const char *at = nullptr;
    const Block *b = find(p, &at);
    if (!b || b->device < 0) return done(hipErrorInvalidValue);
    *base = (hipDeviceptr_t)at;
    *n = b->bytes;
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    std::lock_guard<std::mutex> l(mu);
    const char *base = nullptr;
    const Block *b = find(p, &base);
    if (!b) return done(hipErrorInvalidValue);
    memset(a, 0, sizeof *a);
    a->type = b->device < 0 ? hipMemoryTypeHost : hipMemoryTypeDevice;
    a->device = b->device < 0 ? 0 : b->device;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    std::lock_guard<std::mutex> l(mu);
    note("copy %zu stream %d", n, id(st));
    if (!inside(d, n) || !inside(s, n)) return done(hipErrorInvalidValue);
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, s, n, k, nullptr); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
    std::lock_guard<std::mutex> l(mu);
    note("fill %zu stream %d", n, id(st));
    if (!inside(d, n)) return done(hipErrorInvalidValue);
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { return hipMemsetAsync(d, v, n, nullptr); }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)(intptr_t)next_id++; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { note("wait %d", id(s)); return hipSuccess; }
hipError_t hipDeviceSynchronize() { note("wait all"); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    note("stream %d waits for event %d", id(s), id(e));
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)(intptr_t)next_id++; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { note("event %d on stream %d", id(e), id(s)); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "a failure made by the test"; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return hipMalloc(p, 1 << 20); }

void **__hipRegisterFatBinary(const void *) { static void *m; return &m; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    int rc = 0;
    char *s = abi::__cxa_demangle(name, nullptr, nullptr, &rc);
    std::string n = s ? s : name;
    free(s);
    // without the return type and the argument list
    if (n.back() == ')') {
        size_t i = n.size();
        for (int depth = 0; i > 0 && (depth += n[i - 1] == ')' ? 1 : n[i - 1] == '(' ? -1 : 0);) --i;
        n.resize(i ? i - 1 : 0);
    }
    if (n.rfind("void ", 0) == 0) n = n.substr(5);
    kernels[f] = n;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
    configs.push_back({g, b, sh, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s) {
    const Config c = configs.back();
    configs.pop_back();
    *g = c.grid;
    *b = c.block;
    *sh = c.shmem;
    *s = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t s) {
    std::lock_guard<std::mutex> l(mu);
    if (fail_in >= 0 && fail_in-- == 0) {
        note("failed launch stream %d", id(s));
        return done(hipErrorLaunchFailure);
    }
    note("launch %s grid %u %u block %u stream %d", kernels[f].c_str(), g.x, g.y, b.x, id(s));
    return hipSuccess;
}

}  // extern "C"
