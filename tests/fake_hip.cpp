// A stand-in for the HIP runtime on the host: two devices, streams, events,
// memory and kernel launches that do nothing but keep the runtime's rules, so
// that the engine's host code can be checked on them without a GPU.
//   * work goes to a stream only while its device is the calling thread's, but
//     for copies, clears and graph launches; an event is recorded only on a
//     stream of its own device
//   * memory freed on a stream can be had again on it, and elsewhere once the
//     stream was waited for
//   * device memory has a limit; every timed interval is shorter than the last
// Loaded with RTLD_GLOBAL before the engine, its symbols come first.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace {
enum { OK = 0, INVALID_VALUE = 1, OUT_OF_MEMORY = 2, INVALID_HANDLE = 400 };
struct Stream {
    int dev;
    size_t freed;  // bytes freed on it since it was waited for last
    bool capturing;
};
struct Event {
    int dev;
};
struct Dim3 {
    uint32_t x, y, z;
};
std::mutex mu;
thread_local int current = 0, last_error = OK;
size_t limit = ~(size_t)0, used = 0;  // device bytes: allowed; allocated or not yet reusable
std::map<void *, size_t> device, host;
long intervals = 0, launches[2] = {0, 0};
thread_local struct {
    Dim3 grid, block;
    size_t shared;
    void *stream;
} config;

int take(void **p, size_t n, Stream *s = nullptr) {
    std::lock_guard<std::mutex> lk(mu);
    if (s) {  // what was freed on it is its own again
        used -= s->freed;
        s->freed = 0;
    }
    if (used + n > limit) return OUT_OF_MEMORY;
    *p = std::calloc(1, n ? n : 1);
    device[*p] = n;
    used += n;
    return OK;
}
int give(void *p, Stream *s) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = device.find(p);
    if (it == device.end()) return INVALID_VALUE;
    if (s)
        s->freed += it->second;
    else
        used -= it->second;
    device.erase(it);
    std::free(p);
    return OK;
}
}  // namespace

extern "C" {
// control
void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_used() { return used; }
size_t fake_host() {
    size_t n = 0;
    for (auto &h : host) n += h.second;
    return n;
}
long fake_launches(int dev) { return launches[dev]; }

int hipGetDevice(int *d) { return *d = current, OK; }
int hipSetDevice(int d) { return d < 0 || d > 1 ? INVALID_VALUE : (current = d, OK); }
const char *hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : e == INVALID_HANDLE ? "invalid handle" : "error"; }
int hipGetLastError() {
    const int e = last_error;
    last_error = OK;
    return e;
}

int hipMalloc(void **p, size_t n) { return take(p, n); }
int hipMallocAsync(void **p, size_t n, void *s) { return ((Stream *)s)->dev != current ? INVALID_HANDLE : take(p, n, (Stream *)s); }
int hipFree(void *p) { return p ? give(p, nullptr) : OK; }
int hipFreeAsync(void *p, void *s) { return give(p, (Stream *)s); }
int hipHostMalloc(void **p, size_t n, unsigned) {
    std::lock_guard<std::mutex> lk(mu);
    *p = std::calloc(1, n);
    host[*p] = n;
    return OK;
}
int hipHostFree(void *p) {
    std::lock_guard<std::mutex> lk(mu);
    host.erase(p);
    std::free(p);
    return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int) { return std::memcpy(d, s, n), OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { return std::memcpy(d, s, n), OK; }
int hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), OK; }
int hipMemsetAsync(void *d, int v, size_t n, void *) { return std::memset(d, v, n), OK; }
int hipDeviceGetDefaultMemPool(void **p, int) { return *p = nullptr, OK; }
int hipMemPoolSetAttribute(void *, int, void *) { return OK; }

int hipStreamCreateWithFlags(void **s, unsigned) { return *s = new Stream{current, 0, false}, OK; }
int hipStreamCreate(void **s) { return hipStreamCreateWithFlags(s, 0); }
int hipStreamSynchronize(void *s) {
    std::lock_guard<std::mutex> lk(mu);
    used -= ((Stream *)s)->freed;
    ((Stream *)s)->freed = 0;
    return OK;
}
int hipStreamDestroy(void *s) {
    hipStreamSynchronize(s);
    delete (Stream *)s;
    return OK;
}
int hipStreamBeginCapture(void *s, int) { return ((Stream *)s)->capturing = true, OK; }
int hipStreamEndCapture(void *s, void **g) { return ((Stream *)s)->capturing = false, *g = s, OK; }
int hipGraphInstantiate(void **x, void *g, void *, void *, size_t) { return *x = g, OK; }
int hipGraphLaunch(void *, void *) { return OK; }
int hipGraphDestroy(void *) { return OK; }
int hipGraphExecDestroy(void *) { return OK; }

int hipEventCreateWithFlags(void **e, unsigned) { return *e = new Event{current}, OK; }
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { return delete (Event *)e, OK; }
int hipEventRecord(void *e, void *s) { return ((Event *)e)->dev == ((Stream *)s)->dev ? OK : INVALID_HANDLE; }
int hipEventSynchronize(void *) { return OK; }
int hipEventQuery(void *) { return OK; }
int hipEventElapsedTime(float *ms, void *, void *) { return *ms = 1000.f / (float)++intervals, OK; }

int hipFuncSetAttribute(const void *, int, int) { return OK; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 4, OK; }
int hipGetSymbolAddress(void **, const void *) { return INVALID_VALUE; }
int hipLaunchKernel(const void *, Dim3, Dim3, void **, size_t, void *s) {
    const int dev = ((Stream *)s)->dev;
    if (dev != current) return last_error = INVALID_HANDLE;
    std::lock_guard<std::mutex> lk(mu);
    ++launches[dev];
    return OK;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void *s) { return config = {g, b, sh, s}, OK; }
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *sh, void **s) {
    return *g = config.grid, *b = config.block, *sh = config.shared, *s = config.stream, OK;
}
void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}
