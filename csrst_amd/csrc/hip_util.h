// hip_util.h -- error handling, device buffers and reductions shared by the
// CSRST kernel library.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

namespace hu {

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define HU_CHECK(expr)                                                                               \
    do {                                                                                             \
        hipError_t e_ = (expr);                                                                      \
        if (e_ != hipSuccess)                                                                        \
            throw hu::Error(-3, std::string(#expr) + ": " + hipGetErrorString(e_) + " (" + __FILE__ + \
                                    ":" + std::to_string(__LINE__) + ")");                           \
    } while (0)

#define HU_LAUNCH_CHECK() HU_CHECK(hipGetLastError())

// Last error of a call that had no handle to store it in (one per thread,
// shared by every translation unit of the library).
inline std::string &global_error()
{
    static thread_local std::string e;
    return e;
}

inline std::string fmt(const char *f, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, f);
    vsnprintf(buf, sizeof(buf), f, ap);
    va_end(ap);
    return buf;
}

// What frees the idle device memory that the library keeps between calls
// (csrst_sf.hip's workspaces), if it keeps any.
inline std::atomic<void (*)()> &give_back()
{
    static std::atomic<void (*)()> f{nullptr};
    return f;
}

// hipMalloc that gives idle memory back before it fails, and leaves no error
// for the next launch check to find.
inline hipError_t device_alloc(void **p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    void (*f)() = give_back().load();
    if (e == hipErrorOutOfMemory && f) {
        f();
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
    }
    return e;
}

// Owning device buffer.
template <class T>
struct DBuf {
    T *p = nullptr;
    size_t n = 0;
    DBuf() = default;
    DBuf(const DBuf &) = delete;
    DBuf &operator=(const DBuf &) = delete;
    ~DBuf() { release(); }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    void alloc(size_t count)
    {
        if (count == n && p) return;
        release();
        if (count == 0) return;
        if (device_alloc((void **)&p, count * sizeof(T)) != hipSuccess)
            throw Error(-2, fmt("hipMalloc of %zu bytes failed", count * sizeof(T)));
        n = count;
    }
    void zero(hipStream_t s) { if (n) HU_CHECK(hipMemsetAsync(p, 0, n * sizeof(T), s)); }
    size_t bytes() const { return n * sizeof(T); }
};

// Copies between pageable host memory and the device through pinned buffers.
//
// The runtime's own path copies 13 GB/s (33.5 MB in 2.4 ms): one thread at a
// time moves the data to or from pinned memory, page faults of a fresh result
// array included.  Here kThreads threads do, each with two buffers of its own,
// so that one is filled or emptied while the other is on the link.
// 4 x 1024 x 2048 floats in and out: 4.9 ms before, 3.8 now, and no faster with 6
// or 8 threads or with chunks of 0.5 or 2 MiB: the transfers themselves bound it.
// Transfers below kMin stay with the runtime: a call that makes its own Stage
// pays for the buffers too (a Poisson solve's three arrays of 4 MiB 0.07 ms slower,
// of 11.4 MiB 0.07 ms faster, of 16 MiB 0.4, of 64 MiB 1.5).  So does host
// memory that is already pinned.
//
// One Stage serves one stream at a time: it belongs to the object or call whose
// transfers it makes and frees its buffers (8 MiB) with it.
class Stage {
public:
    Stage() = default;
    Stage(const Stage &) = delete;
    Stage &operator=(const Stage &) = delete;
    ~Stage()
    {
        for (Slot &t : slot_)
            if (t.ev) {
                (void)hipEventSynchronize(t.ev);
                (void)hipEventDestroy(t.ev);
            }
        if (pin_) (void)hipHostFree(pin_);
    }
    // dst (device) = src (host).  Pageable memory may be reused when the call
    // returns; pinned memory only once the stream has been waited for, as the
    // callers do before they return.
    void in(void *dst, const void *src, size_t bytes, hipStream_t s)
    {
        if (!staged(src, bytes)) {
            HU_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
            return;
        }
        run(bytes, [=](Slot *two, std::atomic<size_t> &next) -> hipError_t {
            hipError_t e = hipSuccess;
            size_t k;
            for (int i = 0; (k = next.fetch_add(1)) * kChunk < bytes; i ^= 1) {
                const size_t n = std::min(kChunk, bytes - k * kChunk);
                if ((e = hipEventSynchronize(two[i].ev)) != hipSuccess) return e;   // its last transfer has ended
                memcpy(two[i].p, (const char *)src + k * kChunk, n);
                if ((e = hipMemcpyAsync((char *)dst + k * kChunk, two[i].p, n, hipMemcpyHostToDevice, s)) != hipSuccess) return e;
                if ((e = hipEventRecord(two[i].ev, s)) != hipSuccess) return e;
            }
            return e;
        });
    }
    // dst (host) = src (device) as the stream's work so far leaves it; complete when the call returns
    void out(void *dst, const void *src, size_t bytes, hipStream_t s)
    {
        if (!staged(dst, bytes)) {
            HU_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
            HU_CHECK(hipStreamSynchronize(s));
            return;
        }
        run(bytes, [=](Slot *two, std::atomic<size_t> &next) -> hipError_t {
            hipError_t e = hipSuccess;
            size_t at[2] = {bytes, bytes};                                          // offsets on their way, bytes: none
            for (int i = 0;; i ^= 1) {
                const size_t o = next.fetch_add(1) * kChunk;
                if (o < bytes) {
                    if ((e = hipMemcpyAsync(two[i].p, (const char *)src + o, std::min(kChunk, bytes - o), hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
                    if ((e = hipEventRecord(two[i].ev, s)) != hipSuccess) return e;
                    at[i] = o;
                }
                const size_t q = at[i ^ 1];
                if (q < bytes) {
                    if ((e = hipEventSynchronize(two[i ^ 1].ev)) != hipSuccess) return e;
                    memcpy((char *)dst + q, two[i ^ 1].p, std::min(kChunk, bytes - q));
                    at[i ^ 1] = bytes;
                }
                if (at[i] >= bytes) return e;
            }
        });
    }

private:
    static constexpr size_t kChunk = 1 << 20, kMin = 8 * kChunk;
    static constexpr int kThreads = 4;
    struct Slot {
        char *p = nullptr;
        hipEvent_t ev = nullptr;
    };
    Slot slot_[2 * kThreads];
    void *pin_ = nullptr;

    bool staged(const void *host, size_t bytes)
    {
        if (bytes < kMin) return false;
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, host) != hipSuccess) (void)hipGetLastError();   // unknown to the runtime: pageable
        else if (a.type != hipMemoryTypeUnregistered) return false;
        if (!pin_) {
            if (hipHostMalloc(&pin_, 2 * kThreads * kChunk, hipHostMallocDefault) != hipSuccess) {
                (void)hipGetLastError();
                pin_ = nullptr;
                return false;
            }
            for (int k = 0; k < 2 * kThreads; ++k) slot_[k].p = (char *)pin_ + k * kChunk;
        }
        for (Slot &t : slot_)
            if (!t.ev) HU_CHECK(hipEventCreateWithFlags(&t.ev, hipEventDisableTiming));
        return true;
    }
    template <class F>
    void run(size_t bytes, F work)
    {
        int dev = 0;
        HU_CHECK(hipGetDevice(&dev));
        std::atomic<size_t> next{0};
        hipError_t err[kThreads];
        std::thread th[kThreads];
        for (hipError_t &e : err) e = hipSuccess;
        try {
            for (int t = 1; t < kThreads; ++t)
                th[t] = std::thread([&, t] {
                    err[t] = hipSetDevice(dev);
                    if (err[t] == hipSuccess) err[t] = work(slot_ + 2 * t, next);
                });
        } catch (const std::exception &) {   // no more threads: those that run, and this one, do it all
        }
        err[0] = work(slot_, next);
        for (std::thread &t : th)
            if (t.joinable()) t.join();
        for (hipError_t e : err) HU_CHECK(e);
    }
};

// Monotone mapping of doubles onto unsigned 64-bit integers so that min/max
// reductions can use integer atomics (order-independent, hence deterministic).
__device__ __forceinline__ unsigned long long ord(double v)
{
    unsigned long long u = __double_as_longlong(v);
    return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}
__host__ __device__ __forceinline__ double unord(unsigned long long u)
{
    u = (u & 0x8000000000000000ull) ? (u & 0x7fffffffffffffffull) : ~u;
    double d;
    memcpy(&d, &u, sizeof(d));
    return d;
}

// Wave-level (64-lane) reductions.
template <class T>
__device__ __forceinline__ T wave_min(T v)
{
    for (int o = 32; o > 0; o >>= 1) {
        T w = __shfl_xor(v, o, 64);
        v = w < v ? w : v;
    }
    return v;
}
template <class T>
__device__ __forceinline__ T wave_max(T v)
{
    for (int o = 32; o > 0; o >>= 1) {
        T w = __shfl_xor(v, o, 64);
        v = w > v ? w : v;
    }
    return v;
}

}  // namespace hu
