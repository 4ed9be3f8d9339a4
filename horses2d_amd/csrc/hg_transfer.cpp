// Transfers between a caller's (pageable) arrays and the device, through pinned staging buffers.
//
// The runtime's own path for pageable memory brings a state back at 10.5 GB/s into fresh memory (one
// thread's page faults and copies: a seventh of a pass of 200 steps at 134 MB), 205 kB in 97 us and four
// values in 22 us.  Here up to four threads each move a share of a large array, every one with two
// pinned buffers, so that the copy out of one overlaps the transfer into the other and the page
// faults are taken in parallel; short arrays and single values are written into the pinned buffer by
// a kernel, without the copy engine's start and signals (205 kB: 21 us, four values 14 us).  Uploads are
// staged up to a MiB; the runtime maps longer arrays in place, at 30 GB/s.
//
// The staging sets belong to a process-wide pool: a set is taken for one share of one transfer, at
// most kIdleSets are kept, and the last handle's destruction frees them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <functional>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "hg_device.h"
#include "hg_handle.h"

namespace {

constexpr size_t kBuffer = size_t(2) << 20;     // bytes of one pinned buffer
// A share moves in chunks of kShort, half a buffer from kShare and a buffer from kLong on: a
// transfer's start costs 10 us, and the first chunk's copy waits for its transfer.
constexpr size_t kShort = size_t(512) << 10;
constexpr size_t kLong = size_t(8) << 20;
constexpr size_t kShare = size_t(2) << 20;       // a thread's smallest share
constexpr int kThreads = 4;
// A share of at most this many chunks moves by a kernel that reads or writes the pinned buffer
// itself, without the copy engine's start and its signals.
constexpr size_t kByKernel = 2;
constexpr size_t kIdleSets = 8;                  // 32 MiB of pinned memory

struct Staging {
    int device = -1;
    void *buf[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};     // the last transfer of each buffer
    bool used[2] = {false, false};
};

std::mutex g_mutex;
std::vector<Staging *> g_idle;
int g_handles = 0;

void release_set(Staging *s) {
    if (!s) return;
    for (int b = 0; b < 2; ++b) {
        if (s->used[b]) (void)hipEventSynchronize(s->done[b]);
        if (s->done[b]) (void)hipEventDestroy(s->done[b]);
        if (s->buf[b]) (void)hipHostFree(s->buf[b]);
    }
    delete s;
}

// A set for a device (current in this thread); null where pinned memory or an event is not to be had.
Staging *take_set(int device) {
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        for (size_t k = g_idle.size(); k-- > 0;)
            if (g_idle[k]->device == device) {
                Staging *s = g_idle[k];
                g_idle.erase(g_idle.begin() + (long)k);
                return s;
            }
    }
    Staging *s = new (std::nothrow) Staging();
    if (!s) return nullptr;
    s->device = device;
    hipError_t e = hipSuccess;
    for (int b = 0; b < 2 && e == hipSuccess; ++b) {
        // kernels write these buffers and the host reads them after the event
        e = hipHostMalloc(&s->buf[b], kBuffer, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&s->done[b], hipEventDisableTiming | hipEventReleaseToSystem);
        else s->buf[b] = nullptr;
        if (e != hipSuccess) s->done[b] = nullptr;
    }
    if (e == hipSuccess) return s;
    release_set(s);
    (void)hipGetLastError();   // the caller goes another way
    return nullptr;
}

void give_set(Staging *s) {
    if (!s) return;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_handles > 0 && g_idle.size() < kIdleSets) {
            g_idle.push_back(s);
            return;
        }
    }
    release_set(s);
}

// After a failed transfer: whatever it left on the stream may still use the buffers, and no event
// marks its end, so the set does not go back to the pool.  The caller reports the error; it does not
// stay for the next launch's hipGetLastError.
void discard_set(Staging *s, hipStream_t stream) {
    (void)hipStreamSynchronize(stream);
    release_set(s);
    (void)hipGetLastError();
}

hipError_t wait_buffer(Staging *s, int b) {
    if (!s->used[b]) return hipSuccess;
    const hipError_t e = hipEventSynchronize(s->done[b]);
    if (e == hipSuccess) s->used[b] = false;
    return e;
}

// Makes the handle's device current in the calling thread, and back again.
struct OnDevice {
    int before = -1;
    hipError_t err;
    explicit OnDevice(int device) {
        err = hipGetDevice(&before);
        if (err == hipSuccess && before != device) err = hipSetDevice(device);
        else before = -1;
    }
    ~OnDevice() {
        if (before >= 0) (void)hipSetDevice(before);
    }
};

// One share, between host and dev; without a staging set, by the runtime's own path.
hipError_t move_share(int device, hipStream_t stream, char *host, char *dev, size_t bytes, bool to_dev) {
    OnDevice on(device);
    hipError_t e = on.err;
    if (e != hipSuccess) return e;
    Staging *s = take_set(device);
    if (!s) {
        e = to_dev ? hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, stream)
                   : hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream);
        return e == hipSuccess ? hipStreamSynchronize(stream) : e;
    }
    const size_t chunk = bytes < kShare ? kShort : bytes < kLong ? kBuffer / 2 : kBuffer, n = (bytes + chunk - 1) / chunk;
    auto len = [&](size_t k) { return std::min(chunk, bytes - k * chunk); };
    for (size_t k = 0; k < n + (to_dev ? 0 : 1) && e == hipSuccess; ++k) {
        const int b = (int)(k & 1);
        if (k < n) {
            e = wait_buffer(s, b);
            if (to_dev && e == hipSuccess) std::memcpy(s->buf[b], host + k * chunk, len(k));
            if (e == hipSuccess)
                e = n <= kByKernel && len(k) % 16 == 0
                        ? hg::launch_copy(to_dev ? s->buf[b] : dev + k * chunk, to_dev ? dev + k * chunk : s->buf[b],
                                          len(k), stream)
                    : to_dev ? hipMemcpyAsync(dev + k * chunk, s->buf[b], len(k), hipMemcpyHostToDevice, stream)
                             : hipMemcpyAsync(s->buf[b], dev + k * chunk, len(k), hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(s->done[b], stream);
            if (e == hipSuccess) s->used[b] = true;
        }
        if (!to_dev && k > 0 && e == hipSuccess) {
            // the chunk before, while this one's transfer runs
            e = wait_buffer(s, b ^ 1);
            if (e == hipSuccess) std::memcpy(host + (k - 1) * chunk, s->buf[b ^ 1], len(k - 1));
        }
    }
    if (e == hipSuccess) give_set(s);   // a buffer whose upload still runs is waited for by its next user
    else discard_set(s, stream);
    return e;
}

hipError_t move(hg_handle *h, char *host, char *dev, size_t bytes, bool to_dev) {
    std::atomic<int> err{(int)hipSuccess};
    hg::in_shares((int64_t)((bytes + kShort - 1) / kShort), (int64_t)(kShare / kShort), [&](int64_t c0, int64_t c1) {
        const size_t a = (size_t)c0 * kShort, b = std::min(bytes, (size_t)c1 * kShort);
        hipError_t e = hipErrorOutOfMemory;
        try {
            e = move_share(h->device, h->stream, host + a, dev + a, b - a, to_dev);
        } catch (const std::exception &) {
        }
        if (e != hipSuccess) err = (int)e;
    });
    return (hipError_t)err.load();
}

}  // namespace

namespace hg {

void in_shares(int64_t n, int64_t least, const std::function<void(int64_t, int64_t)> &f) {
    if (n <= 0) return;
    const int64_t nt = std::max<int64_t>(1, std::min<int64_t>(kThreads, n / least)), per = (n + nt - 1) / nt;
    std::vector<std::thread> th;
    th.reserve((size_t)nt);
    int64_t here = 0;   // the shares this thread does: [0, per), and those no thread was to be had for
    for (int64_t k = nt - 1; k > 0; --k) {
        const int64_t a = std::min(n, k * per), b = std::min(n, a + per);
        if (a >= b) continue;
        try {
            th.emplace_back(std::cref(f), a, b);
        } catch (const std::exception &) {
            here = b;
            break;
        }
    }
    f(0, std::max(here, std::min(n, per)));
    for (auto &t : th) t.join();
}

void transfers_open() {
    std::lock_guard<std::mutex> lock(g_mutex);
    ++g_handles;
}

void transfers_close() {
    std::vector<Staging *> idle;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (--g_handles > 0) return;
        idle.swap(g_idle);
    }
    for (Staging *s : idle) release_set(s);
}

hipError_t copy_to_host(hg_handle *h, void *dst, const void *src, size_t bytes) {
    try {
        return move(h, (char *)dst, (char *)const_cast<void *>(src), bytes, false);
    } catch (const std::exception &) {
        return hipErrorOutOfMemory;
    }
}

hipError_t copy_to_device(hg_handle *h, void *dst, const void *src, size_t bytes) {
    if (bytes > kByKernel * kShort) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, h->stream);
        return e == hipSuccess ? hipStreamSynchronize(h->stream) : e;
    }
    try {
        return move(h, (char *)const_cast<void *>(src), (char *)dst, bytes, true);
    } catch (const std::exception &) {
        return hipErrorOutOfMemory;
    }
}

hipError_t read_values(hg_handle *h, double *dst, const double *src, int n, int stride) {
    if (n <= 0) return hipSuccess;
    if (stride == 1 && n > 1024) return copy_to_host(h, dst, src, n * sizeof(double));
    if ((size_t)n * sizeof(double) > kBuffer) return hipErrorInvalidValue;
    OnDevice on(h->device);
    hipError_t e = on.err;
    if (e != hipSuccess) return e;
    Staging *s = take_set(h->device);
    if (!s) {
        const int m = stride == 1 ? 1 : n;   // copies
        for (int i = 0; i < m && e == hipSuccess; ++i)
            e = hipMemcpyAsync(dst + i, src + (int64_t)i * stride, (n / m) * sizeof(double), hipMemcpyDeviceToHost,
                               h->stream);
        return e == hipSuccess ? hipStreamSynchronize(h->stream) : e;
    }
    e = wait_buffer(s, 0);
    if (e == hipSuccess) e = launch_store_values(src, n, stride, (double *)s->buf[0], h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e == hipSuccess) {
        std::memcpy(dst, s->buf[0], n * sizeof(double));
        give_set(s);
    } else {
        discard_set(s, h->stream);
    }
    return e;
}

}  // namespace hg
