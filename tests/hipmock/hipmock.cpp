// Test double of the HIP runtime for libsssi's host code: device memory is
// host memory (zeroed), copies and fills are done at once, kernels are not run
// but noted by name, with their grid and the bytes of chosen arguments.  Loaded
// with global visibility before libsssi.so, its symbols take the runtime's
// place.  hipmock_* steer it.
#include <hip/hip_runtime.h>
#include <unistd.h>

#include <new>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex mu;
std::map<const void *, std::string> kernels;
std::map<const void *, size_t> sizes;  // device allocations
struct Launch {
    std::string name;
    unsigned grid[3], block[3];
    std::vector<std::vector<char>> args;
};
std::vector<Launch> launches;
std::string watch;             // kernels whose arguments are kept
std::vector<size_t> watch_arg;  // bytes of each argument
std::atomic<long> fail_in{-1};  // device allocations until one fails
std::atomic<long> sync_us{0};   // what a stream synchronisation waits
std::atomic<long> n_malloc{0}, n_host{0}, n_copied{0}, copy_limit{1L << 62};
std::atomic<size_t> mem_free{(size_t)1 << 38};
dim3 cfg_grid, cfg_block;
int dummy;

// hipGetLastError's: the thread's last failure, until it is asked for (a call
// that succeeds does not clear it)
thread_local hipError_t last = hipSuccess;
thread_local long new_in = -1;  // this thread's operator new calls until one throws

hipError_t take(void **p, size_t n) {
    ++n_malloc;
    if (fail_in >= 0 && fail_in-- == 0) return last = hipErrorOutOfMemory;
    *p = std::calloc(n ? n : 1, 1);
    std::lock_guard<std::mutex> lk(mu);
    sizes[*p] = n;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
void drop(void *p) {
    {
        std::lock_guard<std::mutex> lk(mu);
        sizes.erase(p);
    }
    std::free(p);
}
hipError_t copy(void *d, const void *s, size_t n) {
    n_copied += (long)n;
    if ((long)n <= copy_limit) std::memcpy(d, s, n);
    return hipSuccess;
}
}  // namespace

void *operator new(size_t n) {
    if (new_in >= 0 && new_in-- == 0) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}

extern "C" {
// the calling thread's k-th operator new from here on throws; what is left of k
void hipmock_fail_new(long k) { new_in = k; }
long hipmock_new_left() { return new_in; }
void hipmock_fail_malloc(long k) { fail_in = k; }
void hipmock_sync_us(long us) { sync_us = us; }
void hipmock_copy_limit(long n) { copy_limit = n; }
void hipmock_mem_free(size_t n) { mem_free = n; }
long hipmock_mallocs() { return n_malloc; }
// bytes of the device allocation at p (0: none)
size_t hipmock_size(const void *p) {
    std::lock_guard<std::mutex> lk(mu);
    auto it = sizes.find(p);
    return it == sizes.end() ? 0 : it->second;
}
long hipmock_host_mallocs() { return n_host; }
void hipmock_watch(const char *name, const size_t *bytes, int n) {
    watch = name;
    watch_arg.assign(bytes, bytes + n);
}
void hipmock_clear() { launches.clear(); }
long hipmock_count(const char *name) {
    std::lock_guard<std::mutex> lk(mu);
    long n = 0;
    for (auto &l : launches) n += l.name.find(name) != std::string::npos;
    return n;
}
// argument a of the k-th watched launch into out; its size, or -1
long hipmock_arg(long k, int a, void *out) {
    std::lock_guard<std::mutex> lk(mu);
    for (auto &l : launches)
        if (!l.args.empty() && k-- == 0) {
            std::memcpy(out, l.args[a].data(), l.args[a].size());
            return (long)l.args[a].size();
        }
    return -1;
}
// grid and block of the k-th launch of a kernel of that name
int hipmock_dims(const char *name, long k, unsigned *out) {
    std::lock_guard<std::mutex> lk(mu);
    for (auto &l : launches)
        if (l.name.find(name) != std::string::npos && k-- == 0) {
            std::memcpy(out, l.grid, 12);
            std::memcpy(out + 3, l.block, 12);
            return 0;
        }
    return -1;
}

void **__hipRegisterFatBinary(const void *) { return (void **)&dummy; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
    kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
    cfg_grid = g;
    cfg_block = b;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s) {
    *g = cfg_grid;
    *b = cfg_block;
    *sh = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    Launch l{kernels[f], {g.x, g.y, g.z}, {b.x, b.y, b.z}, {}};
    if (!watch.empty() && l.name.find(watch) != std::string::npos)
        for (size_t a = 0; a < watch_arg.size(); ++a)
            l.args.emplace_back((char *)args[a], (char *)args[a] + watch_arg[a]);
    launches.push_back(std::move(l));
    // (the runtime's limit: fewer than 2^32 threads in a dimension)
    const bool fits = (unsigned long long)g.x * b.x < (1ull << 32) && g.x && g.y && g.z;
    if (!fits) last = hipErrorInvalidConfiguration;
    return fits ? hipSuccess : hipErrorInvalidConfiguration;
}
hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return take(p, n); }
hipError_t hipFree(void *p) { drop(p); return hipSuccess; }
hipError_t hipFreeAsync(void *p, hipStream_t) { drop(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    ++n_host;
    *p = std::calloc(n ? n : 1, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = mem_free;
    *t = (size_t)288 << 30;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return copy(d, s, n); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    return copy(d, s, n);
}
hipError_t hipMemset(void *d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    if (sync_us > 0) usleep((useconds_t)sync_us);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)std::malloc(8);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { *d = 0; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)std::malloc(8); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    p->sharedMemPerBlock = 160 << 10;
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = std::calloc(64 << 20, 1); return hipSuccess; }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t *p, int) { *p = nullptr; return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }
}
