// A HIP runtime for tests of host code on a machine without a GPU: device
// memory is host memory, copies are done at once, kernels do nothing.  It
// keeps a log of the calls, can refuse allocations, report a stream as being
// captured, sleep where the host waits for the device, and call back there.
// Loaded with RTLD_GLOBAL before libanalisi_hip.so, whose HIP calls bind to it.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <unistd.h>

namespace {
std::mutex mu;
std::map<const void *, std::string> names;   // kernels
std::map<char *, size_t> blocks;             // live device allocations
std::string lines;                           // the log
uint64_t refuse_from = UINT64_MAX;           // bytes of a device allocation that is refused
uint64_t refuse_after = UINT64_MAX;          // device allocations that still succeed
unsigned wait_us = 0;                        // of every wait of the host
unsigned launch_us = 0;                      // of every launch
int fill = 0;                                // byte that device memory is filled with
unsigned dump = 0;                           // bytes of a launch's first argument in the log
bool capturing = false;
void (*on_wait)() = nullptr;                 // called at every wait of the host
thread_local bool in_wait = false;
struct Config {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
};
thread_local Config config;

unsigned long tid() { return (unsigned long)std::hash<std::thread::id>()(std::this_thread::get_id()); }
template <class... A>
void log(const char *fmt, A... a) {
    char s[4096];
    std::snprintf(s, sizeof s, fmt, a...);
    std::lock_guard<std::mutex> l(mu);
    lines += std::to_string(tid()) + " " + s + "\n";
}
hipError_t wait(const char *what, const void *on) {
    log("%s %p", what, on);
    if (wait_us) usleep(wait_us);
    if (on_wait && !in_wait) {
        in_wait = true;
        on_wait();
        in_wait = false;
    }
    return hipSuccess;
}
}  // namespace

extern "C" {
// control
void fake_refuse(uint64_t from_bytes, uint64_t after) {
    std::lock_guard<std::mutex> l(mu);
    refuse_from = from_bytes;
    refuse_after = after;
}
void fake_wait(unsigned us, void (*callback)()) {
    wait_us = us;
    on_wait = callback;
}
void fake_launch_time(unsigned us) { launch_us = us; }
void fake_dump(unsigned bytes) { dump = bytes; }
void fake_fill(int byte) { fill = byte; }
void fake_capture(int on) { capturing = on != 0; }
size_t fake_log(char *out, size_t cap) {  // takes the log when it fits
    std::lock_guard<std::mutex> l(mu);
    const size_t n = lines.size();
    if (out && n < cap) {
        std::memcpy(out, lines.c_str(), n + 1);
        lines.clear();
    }
    return n;
}
uint64_t fake_live() {
    std::lock_guard<std::mutex> l(mu);
    return blocks.size();
}

// kernels
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    std::lock_guard<std::mutex> l(mu);
    names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
    config = Config{g, b, sh, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s) {
    *g = config.grid;
    *b = config.block;
    *sh = config.shmem;
    *s = config.stream;
    return hipSuccess;
}
static thread_local hipError_t last = hipSuccess;
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t s) {
    std::string bufs;
    char p[32];
    {
        // the device allocations that the first argument points into, if it is
        // a structure or a pointer (its first 160 bytes)
        std::lock_guard<std::mutex> l(mu);
        for (int k = 0; args && k < 20; k++) {
            char *v;
            std::memcpy(&v, (char *)args[0] + 8 * k, 8);
            auto it = blocks.upper_bound(v);
            if (it == blocks.begin()) continue;
            --it;
            if (v < it->first + it->second) {
                std::snprintf(p, sizeof p, " %d:%p", k, (void *)v);
                bufs += p;
            }
        }
        bufs = (names.count(f) ? names[f] : "?") + bufs;
        if (dump) bufs += " =";
        for (unsigned k = 0; args && k < dump; k++) {
            std::snprintf(p, sizeof p, "%02x", ((unsigned char *)args[0])[k]);
            bufs += p;
        }
    }
    log("launch %p %u,%u,%u %u %s", (void *)s, g.x, g.y, g.z, b.x * b.y * b.z, bufs.c_str());
    if (launch_us) usleep(launch_us);
    // the dispatch packet holds 32 bits of threads a dimension: the real runtime
    // runs the number modulo 2^32
    const bool bad = (uint64_t)g.x * b.x > UINT32_MAX || (uint64_t)g.y * b.y > UINT32_MAX ||
                     (uint64_t)g.z * b.z > UINT32_MAX || g.x == 0 || g.y == 0 || g.z == 0 || g.y > 65535 * 1024u;
    return last = bad ? hipErrorInvalidConfiguration : hipSuccess;
}

// memory
hipError_t hipMalloc(void **p, size_t n) {
    log("malloc %zu", n);
    std::lock_guard<std::mutex> l(mu);
    if (n >= refuse_from || refuse_after == 0) return last = hipErrorOutOfMemory;
    if (refuse_after != UINT64_MAX) refuse_after--;
    char *q = (char *)std::calloc(1, n + 64);
    if (!q) return last = hipErrorOutOfMemory;
    if (fill) std::memset(q, fill, n);
    blocks[q] = n;
    *p = q;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    log("free %p", p);
    std::lock_guard<std::mutex> l(mu);
    if (!blocks.erase((char *)p)) return last = hipErrorInvalidValue;
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(1, n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
    if (p) log("hostfree %p", p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
    log("memcpy %d %zu", (int)k, n);
    std::memcpy(d, s, n);
    return k == hipMemcpyDeviceToHost ? wait("copied", d) : hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
    log("memcpyasync %d %zu %p", (int)k, n, (void *)st);
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = *t = 64ull << 30;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char *room = (char *)std::calloc(1, 64u << 20);
    *p = room;
    return hipSuccess;
}

// waits, streams, events, graphs
hipError_t hipDeviceSynchronize(void) { return wait("devicesync", nullptr); }
hipError_t hipStreamSynchronize(hipStream_t s) { return wait("streamsync", s); }
hipError_t hipEventSynchronize(hipEvent_t e) { return wait("eventsync", e); }
static void *token() {
    static uintptr_t n = 0x1000;
    std::lock_guard<std::mutex> l(mu);
    return (void *)(n += 16);
}
hipError_t hipStreamCreate(hipStream_t *s) {
    *s = (hipStream_t)token();
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) {
    *c = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    log("waitevent %p %p", (void *)s, (void *)e);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t)token();
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    log("record %p %p", (void *)e, (void *)s);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = (hipGraph_t)token();
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = (hipGraphExec_t)token();
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

// the device
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError(void) {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
}
