// A HIP runtime of host memory for tests of the library's host code on a
// machine without a GPU (loaded before the real one): device allocations are
// host ones and can be refused, copies happen at once, kernels do not run but
// their launches are recorded.
#include <hip/hip_runtime.h>

#include <pthread.h>

#include <dlfcn.h>
#include <errno.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <new>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex m;
std::map<void *, size_t> device;
std::map<const void *, std::string> names;
std::vector<size_t> sizes;
std::string launches;
std::vector<size_t> refused;
size_t held = 0, most = 0, capacity = SIZE_MAX;
bool no_threads = false;
int started = 0;
size_t most_new = SIZE_MAX;
int live = 0, most_live = 0;
long waits = 0;
bool then_fail = false;
struct Start {
    void *(*f)(void *);
    void *arg;
};
void *run_thread(void *p) {
    const Start s = *(Start *) p;
    free(p);
    {
        std::lock_guard<std::mutex> lock(m);
        if (++live > most_live) most_live = live;
    }
    void *r = s.f(s.arg);
    std::lock_guard<std::mutex> lock(m);
    live--;
    return r;
}
}  // namespace

extern "C" {

// --- what tests ask -----------------------------------------------------------
void host_reset() {
    std::lock_guard<std::mutex> lock(m);
    sizes.clear();
    launches.clear();
    most = held;
}
void host_refuse(const size_t *v, int n) {  // device allocations of these sizes fail
    std::lock_guard<std::mutex> lock(m);
    refused.assign(v, v + n);
}
int host_sizes(size_t *out, int most_out) {  // device allocations since the reset
    std::lock_guard<std::mutex> lock(m);
    for (int i = 0; i < most_out && i < (int) sizes.size(); i++) out[i] = sizes[i];
    return (int) sizes.size();
}
void host_capacity(size_t n) { capacity = n; }  // bytes of device memory
size_t host_held() { return held; }
size_t host_most() { return most; }
const char *host_launches() { return launches.c_str(); }  // "name x y z threads lds\n" each
void host_no_threads(int on) { no_threads = on != 0; }
void host_most_new(size_t n) { most_new = n; }  // larger host allocations throw
int host_most_live() { return most_live; }  // threads at one time
// the next n event queries are not ready, the others done or (fail) an error
void host_events(long n, int fail) { waits = n, then_fail = fail != 0; }
int host_started() { return started; }

// --- threads --------------------------------------------------------------------
int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    static auto real = (int (*)(pthread_t *, const pthread_attr_t *, void *(*) (void *), void *))
        dlsym(RTLD_NEXT, "pthread_create");
    if (no_threads) return EAGAIN;
    __atomic_fetch_add(&started, 1, __ATOMIC_RELAXED);
    Start *s = (Start *) malloc(sizeof(Start));
    s->f = f, s->arg = arg;
    return real(t, a, run_thread, s);
}

// --- memory ---------------------------------------------------------------------
}
void *operator new(size_t n) {
    void *p = n <= most_new ? malloc(n ? n : 1) : nullptr;
    if (p == nullptr) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
extern "C" {

// --- the runtime ----------------------------------------------------------------
void **__hipRegisterFatBinary(const void *) { return (void **) malloc(8); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
    names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof(*p));
    p->sharedMemPerBlock = 160 * 1024;
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> lock(m);
    for (size_t r : refused) {
        if (r == n) return *p = nullptr, hipErrorOutOfMemory;
    }
    if (n > capacity || held > capacity - n) return *p = nullptr, hipErrorOutOfMemory;
    *p = calloc(1, n);
    device[*p] = n;
    sizes.push_back(n);
    held += n;
    if (held > most) most = held;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lock(m);
    held -= device[p];
    device.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    return *p = calloc(1, n), hipSuccess;
}
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    return memcpy(d, s, n), hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    std::lock_guard<std::mutex> lock(m);
    auto it = device.upper_bound((void *) p);
    if (it == device.begin()) return hipErrorInvalidValue;
    --it;
    if ((const char *) p >= (const char *) it->first + it->second) return hipErrorInvalidValue;
    memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    return *s = (hipStream_t) malloc(8), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t) malloc(8), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return free(e), hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) {
    std::lock_guard<std::mutex> lock(m);
    if (waits > 0) return waits--, hipErrorNotReady;
    return then_fail ? hipErrorUnknown : hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { return *p = (void *) s, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }

// A launch of 2^32 threads or more in a dimension, or beyond the grid's
// limits in y and z, is refused as the runtime refuses it.
static thread_local struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} config;
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    config.grid = grid, config.block = block, config.lds = lds, config.stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = config.grid, *block = config.block, *lds = config.lds, *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t lds,
                           hipStream_t) {
    std::lock_guard<std::mutex> lock(m);
    launches += names[f];
    for (size_t v : {(size_t) grid.x, (size_t) grid.y, (size_t) grid.z, (size_t) block.x, lds}) {
        launches += " " + std::to_string(v);
    }
    launches += "\n";
    const bool ok = grid.x && grid.y && grid.z && grid.y < 65536 && grid.z < 65536 &&
                    (unsigned long long) grid.x * block.x < (1ull << 32);
    return ok ? hipSuccess : hipErrorInvalidConfiguration;
}
}
