// common.cpp -- host helpers shared by the propagators (see common.h).
#include "common.h"

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <map>
#include <mutex>
#include <system_error>

namespace sssi {

static thread_local std::string g_last_error;
static thread_local hipStream_t g_alloc_stream = nullptr;

hipStream_t &alloc_stream() { return g_alloc_stream; }

void set_last_error(const char *msg) { g_last_error = msg ? msg : ""; }

const char *last_error_text() { return g_last_error.c_str(); }

static int64_t gcd64(int64_t a, int64_t b) {
    if (a < 0) a = -a;
    if (b < 0) b = -b;
    while (b) {
        const int64_t t = a % b;
        a = b;
        b = t;
    }
    return a;
}

void staggered_coefficients(int N, double *c) {
    if (N < 1 || N > 8) fail(SSSI_EINVAL, "nDiffOrder must be in 1..8 (got %d)", N);
    for (int j = 1; j <= N; ++j) {
        int64_t num = 1, den = 2 * j - 1;
        bool neg = false;
        for (int m = 1; m <= N; ++m) {
            if (m == j) continue;
            const int64_t a = (int64_t)(2 * m - 1) * (2 * m - 1);
            int64_t b = a - (int64_t)(2 * j - 1) * (2 * j - 1);
            if (b < 0) { neg = !neg; b = -b; }
            const int64_t g1 = gcd64(a, den), g2 = gcd64(num, b);
            num = (num / g2) * (a / g1);
            den = (den / g1) * (b / g2);
            const int64_t g = gcd64(num, den);
            num /= g;
            den /= g;
        }
        c[j - 1] = (neg ? -1.0 : 1.0) * ((double)num / (double)den);
    }
}

// fwdTimeCpmlFor2dAw_mex.c:100-145 with dampPml (finiteDifference.c:253-280):
// d0 = -(3 v)/(2 L) log(1e-6), d = d0 (u/L)(u/L), b = exp(-d dt).
static inline float bm1_of(double v, double u, double L, double dt) {
    const double d0 = -(3.0 * v) / (2 * L) * std::log(1e-6);
    const double d = d0 * (u / L) * (u / L);
    return (float)(std::exp(-d * dt) - 1.0);
}

float cpml2d_bm1_x(const double *v, int64_t nz, int64_t nx, int nB, double dx, double dt,
                   int64_t q) {
    const int64_t i = q / (2 * nB), xs = q % (2 * nB);
    const double L = nB * dx;
    if (xs < nB) return bm1_of(v[xs * nz + i], (nB - xs) * dx, L, dt);         // left
    const int64_t j = xs - nB;
    return bm1_of(v[(nx - nB + j) * nz + i], (j + 1) * dx, L, dt);              // right
}

float cpml2d_bm1_z(const double *v, int64_t nz, int64_t nx, int nB, double dz, double dt,
                   int64_t q) {
    const int64_t i = q / nx, j = q % nx;
    return bm1_of(v[j * nz + (nz - nB + i)], (i + 1) * dz, nB * dz, dt);      // bottom
}

void cpml2d_bm1(const double *v, int64_t nz, int64_t nx, int nB, double dz, double dx, double dt,
                std::vector<float> &zbm1, std::vector<float> &xbm1) {
    zbm1.assign((size_t)nB * nx, 0.f);
    xbm1.assign((size_t)nz * 2 * nB, 0.f);
    if (nB == 0) return;
    for (int64_t q = 0; q < (int64_t)xbm1.size(); ++q)
        xbm1[q] = cpml2d_bm1_x(v, nz, nx, nB, dx, dt, q);
    for (int64_t q = 0; q < (int64_t)zbm1.size(); ++q)
        zbm1[q] = cpml2d_bm1_z(v, nz, nx, nB, dz, dt, q);
}

void validate_common(int dim, int64_t nz, int64_t nx, int64_t ny, int64_t nt, int N, int nB,
                     double dz, double dx, double dy, double dt, bool need_N) {
    if (nz < 1 || nx < 1 || ny < 1)
        fail(SSSI_EINVAL, "grid must be non-empty (nz=%lld nx=%lld ny=%lld)", (long long)nz,
             (long long)nx, (long long)ny);
    if (nz > (1 << 24) || nx > (1 << 24) || ny > (1 << 24) || nz * nx > (int64_t)1 << 30)
        fail(SSSI_EINVAL, "grid too large for the 2-D index space");
    if (nt < 1) fail(SSSI_EINVAL, "nt must be >= 1 (got %lld)", (long long)nt);
    if (need_N && (N < 1 || N > 8)) fail(SSSI_EINVAL, "nDiffOrder must be in 1..8 (got %d)", N);
    if (nB < 0) fail(SSSI_EINVAL, "nBoundary must be >= 0 (got %d)", nB);
    if ((int64_t)nB > nz) fail(SSSI_EINVAL, "nBoundary=%d exceeds nz=%lld", nB, (long long)nz);
    if (2 * (int64_t)nB > nx)
        fail(SSSI_EINVAL, "2*nBoundary=%d exceeds nx=%lld", 2 * nB, (long long)nx);
    if ((dim == 3 || ny > 1) && 2 * (int64_t)nB > ny)
        fail(SSSI_EINVAL, "2*nBoundary=%d exceeds ny=%lld", 2 * nB, (long long)ny);
    if (!(dz > 0) || !(dx > 0) || !(dy > 0) || !(dt > 0) || !std::isfinite(dz) ||
        !std::isfinite(dx) || !std::isfinite(dy) || !std::isfinite(dt))
        fail(SSSI_EINVAL, "dz, dx, dy and dt must be positive and finite");
}

void validate_velocity(const double *v, int64_t n, const char *name) {
    if (!v) fail(SSSI_EINVAL, "%s must not be NULL", name);
    std::atomic<int64_t> bad{-1};
    parallel_ranges(n, [&](int64_t a, int64_t b) {
        for (int64_t q = a; q < b; ++q)
            if (!(v[q] > 0.0) || !std::isfinite(v[q])) {
                int64_t want = -1;
                bad.compare_exchange_strong(want, q);
                return;
            }
    }, 1 << 16);
    const int64_t q = bad.load();
    if (q >= 0)
        fail(SSSI_EINVAL, "%s must be finite and positive (element %lld is %g)", name,
             (long long)q, v[q]);
}

double max_velocity(const double *v, int64_t n) {
    std::mutex mu;
    double vmax = 0.0;
    parallel_ranges(n, [&](int64_t a, int64_t b) {
        double m[4] = {0.0, 0.0, 0.0, 0.0};  // independent chains
        int64_t q = a;
        for (; q + 4 <= b; q += 4)
            for (int k = 0; k < 4; ++k) m[k] = std::max(m[k], v[q + k]);
        for (; q < b; ++q) m[0] = std::max(m[0], v[q]);
        std::lock_guard<std::mutex> lk(mu);
        vmax = std::max({vmax, m[0], m[1], m[2], m[3]});
    }, (int64_t)1 << 18);
    return vmax;
}

namespace {
std::mutex g_stream_mu;
std::map<int, std::vector<hipStream_t>> g_streams;  // idle pool streams per device
}  // namespace

hipStream_t stream_acquire() {
    int dev = 0;
    SSSI_HIP(hipGetDevice(&dev));
    {
        std::lock_guard<std::mutex> lk(g_stream_mu);
        auto &v = g_streams[dev];
        if (!v.empty()) {
            hipStream_t s = v.back();
            v.pop_back();
            return s;
        }
    }
    hipStream_t s = nullptr;
    SSSI_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    return s;
}

void stream_release(hipStream_t s) {
    if (!s) return;
    int dev = 0;
    // an idle stream goes back to its own device's list; one that cannot be
    // drained or placed is destroyed
    if (hipStreamSynchronize(s) != hipSuccess || hipStreamGetDevice(s, &dev) != hipSuccess) {
        (void)hipStreamDestroy(s);
        return;
    }
    std::lock_guard<std::mutex> lk(g_stream_mu);
    g_streams[dev].push_back(s);
}

namespace {
// Pinned chunks kept for the next download (hipHostMalloc takes about 0.1 ms
// per MB): at most kKept of them idle in the process, the rest are freed.  A
// call takes two: with 4 kept, four and eight threads bringing 24 MB each to
// the host at once took 4.4 and 7.4 ms, with 16 kept 2.5 and 4.8.
constexpr size_t kChunkBytes = (size_t)8 << 20;
constexpr size_t kKept = 16;
std::mutex g_chunk_mu;
std::vector<void *> g_chunks;

struct PinnedChunk {
    void *p = nullptr;
    PinnedChunk() = default;
    PinnedChunk(const PinnedChunk &) = delete;
    PinnedChunk &operator=(const PinnedChunk &) = delete;
    ~PinnedChunk() {
        if (!p) return;
        {
            std::lock_guard<std::mutex> lk(g_chunk_mu);
            if (g_chunks.size() < kKept) {
                g_chunks.push_back(p);
                return;
            }
        }
        (void)hipHostFree(p);
    }
    void acquire() {
        {
            std::lock_guard<std::mutex> lk(g_chunk_mu);
            g_chunks.reserve(kKept);  // (giving one back does not allocate)
            if (!g_chunks.empty()) {
                p = g_chunks.back();
                g_chunks.pop_back();
                return;
            }
        }
        // usable with every device, whichever is current when it is taken again
        SSSI_HIP(hipHostMalloc(&p, kChunkBytes, hipHostMallocPortable));
    }
};

// What stream_to_host's workers share: they sleep on `go` until the next chunk
// has come (or `stop`), the caller on `through` until a buffer is free again.
struct Relay {
    std::mutex mu;
    std::condition_variable go, through;
    std::atomic<bool> stop{false};
    std::atomic<size_t> ready{0};  // chunks that have come
    long team = -1;                // workers that take part (-1: not decided)
    // A chunk that is on its way comes within 0.2 ms: a worker looks for it that
    // long before it goes to sleep, as waking 15 takes 50 us.
    void look(size_t c) const {
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
        while (ready.load() <= c && !stop.load() && std::chrono::steady_clock::now() < until)
            std::this_thread::yield();
    }
    std::vector<size_t> done;    // workers that are through with a chunk
};

// Workers of all calls of the process at a time: they widen and page in
// results, which is bound by the host's memory and its page tables.  Four and
// eight threads bringing 24 MB each to the host: 2.5 and 4.8 ms with 15 workers
// a call, 1.9 and 2.4 with 15 in all.  They are started while the stream still
// computes (starting 15 takes 0.3 ms) and asleep until it is done, and only then
// is it decided how many take part.
constexpr long kWorkers = 15, kAsleep = 60;
std::atomic<long> g_workers{0}, g_asleep{0};

// The workers; left early (an exception), they are told to stop and joined.
struct Crew {
    Relay &r;
    std::vector<std::thread> th;
    long held = 0, taken = 0;  // of kAsleep, of kWorkers
    template <class F>
    void start(size_t want, F &f) {
        held = (long)want;
        const long n = std::min<long>(held, kAsleep - g_asleep.fetch_add(held));
        if (n < 2) return;
        try {
            th.reserve((size_t)n);
            for (size_t k = 0; k < (size_t)n; ++k) th.emplace_back([&f, k] { f(k); });
        } catch (const std::system_error &) {  // no more threads: those there do it
        } catch (const std::bad_alloc &) {
        }
    }
    // How many take part (0: the caller does it); the others leave.
    long decide() {
        taken = (long)th.size();
        const long n = std::min<long>(taken, kWorkers - g_workers.fetch_add(taken));
        const long team = n < 2 ? 0 : n;
        {
            std::lock_guard<std::mutex> lk(r.mu);
            r.team = team;
        }
        r.go.notify_all();
        return team;
    }
    void join() {
        for (auto &t : th)
            if (t.joinable()) t.join();
    }
    ~Crew() {
        {
            std::lock_guard<std::mutex> lk(r.mu);
            r.stop = true;
        }
        r.go.notify_all();
        join();
        g_workers -= taken;
        g_asleep -= held;
    }
};
}  // namespace

void stream_to_host(const void *dev, size_t n, size_t elem, hipStream_t s, const HostUse &use) {
    if (n == 0) return;
    const char *src = (const char *)dev;
    const size_t per = std::max<size_t>(1, kChunkBytes / elem), nchunk = (n + per - 1) / per;
    PinnedChunk buf[2];
    buf[0].acquire();
    if (nchunk > 1) buf[1].acquire();
    auto fetch = [&](size_t c) {
        SSSI_HIP(hipMemcpyAsync(buf[c & 1].p, src + c * per * elem,
                                std::min(per, n - c * per) * elem, hipMemcpyDeviceToHost, s));
        SSSI_HIP(hipStreamSynchronize(s));
    };
    // a worker per MB, up to 15; none for a small result
    const size_t want = std::min<size_t>({15, n * elem >> 20,
                                          std::max(1u, std::thread::hardware_concurrency())});
    Relay r;
    r.done.assign(nchunk, 0);
    auto work = [&](size_t k) {
        std::unique_lock<std::mutex> lk(r.mu);
        r.go.wait(lk, [&] { return r.stop || r.team >= 0; });
        const long team = r.team;
        if (r.stop || (long)k >= team) return;
        const size_t T = (size_t)team;
        for (size_t c = 0; c < nchunk; ++c) {
            lk.unlock();
            r.look(c);
            lk.lock();
            r.go.wait(lk, [&] { return r.stop || r.ready > c; });
            if (r.stop) return;
            lk.unlock();
            const size_t m = std::min(per, n - c * per), a = m * k / T, b = m * (k + 1) / T;
            if (b > a) use((const char *)buf[c & 1].p + a * elem, c * per + a, b - a);
            lk.lock();
            if (++r.done[c] == T) r.through.notify_one();
        }
    };
    Crew crew{r};  // (last: joined before anything the workers use is gone)
    size_t T = 0;  // that take part
    if (want > 1) {
        crew.start(want, work);
        SSSI_HIP(hipStreamSynchronize(s));  // what the stream still computes
        T = (size_t)crew.decide();
    }
    for (size_t c = 0; c < nchunk; ++c) {
        if (T > 0 && c >= 2) {  // the buffer's last chunk has been used
            std::unique_lock<std::mutex> lk(r.mu);
            r.through.wait(lk, [&] { return r.done[c - 2] == T; });
        }
        fetch(c);
        if (T > 0) {
            {
                std::lock_guard<std::mutex> lk(r.mu);
                r.ready = c + 1;
            }
            r.go.notify_all();
        } else {
            use(buf[c & 1].p, c * per, std::min(per, n - c * per));
        }
    }
    crew.join();
}

void copy_to_host(void *dst, const void *dev, size_t bytes, hipStream_t s) {
    stream_to_host(dev, bytes, 1, s, [dst](const void *src, size_t first, size_t count) {
        std::memcpy((char *)dst + first, src, count);
    });
}

void widen_to_host(double *dst, const float *dev, size_t n, hipStream_t s) {
    stream_to_host(dev, n, sizeof(float), s, [dst](const void *src, size_t first, size_t count) {
        const float *f = (const float *)src;
        for (size_t q = 0; q < count; ++q) dst[first + q] = f[q];
    });
}

}  // namespace sssi
