// host_copy.hip -- large copies between the caller's (pageable) arrays and
// device memory.
//
// A pageable hipMemcpy to the host runs at 18 GB/s, and the FP32 form's
// conversion was one more pass over a buffer allocated for it.  Here the array
// goes in 2 MB pieces through two pinned buffers: while one is on the bus the
// other is copied, or converted, on the host.  137 MB to the host: FP64 7.7 ->
// 5.1 ms, FP32 21.3 -> 4.5; FP32 from the host 19.6 -> 3.7.  FP64 from the host
// stays with hipMemcpy (4.6 ms, staged 4.7), and so does FP64 into an array that
// the runtime knows (pinned by the caller, managed): 2.4 ms, staged 4.8.  More
// host threads (2 to 8) brought 3.5 ms on an idle host and 5 to 7 beside a
// spinning OpenMP pool, so the calling thread does it alone.
//
// The buffers belong to the process: allocated by the first large copy, shared
// by every context (a copy that finds them taken goes the plain way) and freed
// with the last context.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "host_copy.hpp"

namespace fen {

namespace {

constexpr size_t kPiece = 2u << 20;      // bytes of a pinned buffer
constexpr size_t kLeast = 2 * kPiece;    // smaller copies go the plain way

struct Staging {
    std::mutex busy;   // held by the copy that uses the buffers
    std::mutex users_lock;
    int users = 0;     // contexts
    void *piece[2] = {nullptr, nullptr};

    bool allocate()
    {
        for (void *&p : piece)
            if (!p && hipHostMalloc(&p, kPiece) != hipSuccess) {
                (void)hipGetLastError();
                p = nullptr;
                return false;
            }
        return true;
    }
    void release()
    {
        for (void *&p : piece) {
            if (p) (void)hipHostFree(p);
            p = nullptr;
        }
    }
};

Staging &staging()
{
    static Staging *s = new Staging();   // never destroyed: contexts may outlive static objects
    return *s;
}

void check(hipError_t e)
{
    if (e != hipSuccess) throw std::runtime_error(std::string("host copy: ") + hipGetErrorString(e));
}

void to_host(double *dst, const void *src, size_t n, size_t es)
{
    if (es == sizeof(double)) {
        std::memcpy(dst, src, n * sizeof(double));
    } else {
        const float *f = static_cast<const float *>(src);
        for (size_t q = 0; q < n; q++) dst[q] = (double)f[q];
    }
}

void from_host(float *dst, const double *src, size_t n)   // (FP64 arrays come the plain way)
{
    for (size_t q = 0; q < n; q++) dst[q] = (float)src[q];
}

// The stream's device is current while this lives: the copy's events have to
// belong to it, and the caller may have another one current.
struct OnDeviceOf {
    int before = 0;
    bool ok = false, changed = false;
    explicit OnDeviceOf(hipStream_t s)
    {
        hipDevice_t dev = 0;
        ok = hipGetDevice(&before) == hipSuccess && hipStreamGetDevice(s, &dev) == hipSuccess;
        if (ok && dev != before) ok = changed = hipSetDevice(dev) == hipSuccess;
        if (!ok) (void)hipGetLastError();
    }
    ~OnDeviceOf()
    {
        if (changed) (void)hipSetDevice(before);
    }
};

// The copy through the two buffers, one piece on the bus while the other is on
// the host; everything it queued is done when it returns or throws.
struct Pipe {
    hipStream_t stream;
    hipEvent_t ev[2] = {nullptr, nullptr};
    explicit Pipe(hipStream_t s) : stream(s) {}
    ~Pipe()
    {
        (void)hipStreamSynchronize(stream);
        for (auto e : ev)
            if (e) (void)hipEventDestroy(e);
    }

    void run(void *const *piece, char *devp, double *host, size_t n, size_t es, bool out)
    {
        const size_t per = kPiece / es;
        size_t at[2] = {0, 0};
        bool flying[2] = {false, false};
        auto finish = [&](int b) {
            if (!flying[b]) return;
            flying[b] = false;
            check(hipEventSynchronize(ev[b]));
            if (out) to_host(host + at[b], piece[b], std::min(per, n - at[b]), es);
        };
        for (auto &e : ev) check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        int b = 0;
        for (size_t a = 0; a < n; a += per, b ^= 1) {
            finish(b);
            at[b] = a;
            const size_t m = std::min(per, n - a);
            if (out) {
                check(hipMemcpyAsync(piece[b], devp + a * es, m * es, hipMemcpyDeviceToHost, stream));
            } else {
                from_host(static_cast<float *>(piece[b]), host + a, m);
                check(hipMemcpyAsync(devp + a * es, piece[b], m * es, hipMemcpyHostToDevice, stream));
            }
            check(hipEventRecord(ev[b], stream));
            flying[b] = true;
        }
        finish(b);
        finish(b ^ 1);
    }
};

// Whether the runtime knows the array (by its first element): pinned, managed,
// or a device's.
bool registered(const void *host)
{
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, host) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type != hipMemoryTypeUnregistered;
}

// Whether the staged way took the copy.
bool staged(hipStream_t stream, void *devp, double *host, size_t n, size_t es, bool out)
{
    if (n * es < kLeast || (es == sizeof(double) && registered(host))) return false;
    Staging &s = staging();
    std::unique_lock<std::mutex> lock(s.busy, std::try_to_lock);
    if (!lock.owns_lock() || !s.allocate()) return false;
    OnDeviceOf device(stream);
    if (!device.ok) return false;
    Pipe(stream).run(s.piece, static_cast<char *>(devp), host, n, es, out);
    return true;
}

}  // namespace

void host_copy_user(int change)
{
    Staging &s = staging();
    std::lock_guard<std::mutex> l(s.users_lock);
    s.users += change;
    if (s.users > 0) return;
    std::lock_guard<std::mutex> b(s.busy);
    s.release();
}

void queue_to_host(hipStream_t stream, double *dst, const double *src, size_t n)
{
    if (staged(stream, const_cast<double *>(src), dst, n, sizeof(double), true)) return;
    check(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToHost, stream));
}

void queue_to_device(hipStream_t stream, double *dst, const double *src, size_t n)
{
    check(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyHostToDevice, stream));
}

void copy_to_host(hipStream_t stream, double *dst, const void *src, size_t n, size_t es)
{
    if (es == sizeof(double)) {
        queue_to_host(stream, dst, static_cast<const double *>(src), n);
        check(hipStreamSynchronize(stream));
        return;
    }
    if (staged(stream, const_cast<void *>(src), dst, n, es, true)) return;
    std::vector<float> h(n);
    check(hipMemcpyAsync(h.data(), src, n * es, hipMemcpyDeviceToHost, stream));
    check(hipStreamSynchronize(stream));
    to_host(dst, h.data(), n, es);
}

void copy_to_device(hipStream_t stream, void *dst, const double *src, size_t n, size_t es)
{
    if (es == sizeof(double)) {
        queue_to_device(stream, static_cast<double *>(dst), src, n);
        check(hipStreamSynchronize(stream));
        return;
    }
    if (staged(stream, dst, const_cast<double *>(src), n, es, false)) return;
    std::vector<float> h(n);
    from_host(h.data(), src, n);
    check(hipMemcpyAsync(dst, h.data(), n * es, hipMemcpyHostToDevice, stream));
    check(hipStreamSynchronize(stream));
}

}  // namespace fen
