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
// The staging sets belong to a process-wide pool of at most kSets per device: a transfer takes what is
// idle or may still be made, up to one per share, and goes the runtime's way when that is none.  The
// last handle's destruction frees them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
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
// Sets of a device, 32 MiB of pinned memory.  Making one takes longer than a short transfer: with the sets
// beyond eight freed after use, eight threads' states of 25.7 MB took 8.8 ms instead of the runtime's 5.2.
constexpr int kSets = 8;

struct Staging {
    int device = -1;
    bool busy = true;                            // a transfer has it
    void *buf[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};     // the last transfer of each buffer
    bool used[2] = {false, false};
};

std::mutex g_mutex;
std::vector<Staging *> g_sets;   // of every device
int g_handles = 0;

void release_set(Staging *s) {
    for (int b = 0; b < 2; ++b) {
        if (s->used[b]) (void)hipEventSynchronize(s->done[b]);
        if (s->done[b]) (void)hipEventDestroy(s->done[b]);
        if (s->buf[b]) (void)hipHostFree(s->buf[b]);
    }
    delete s;
}

void drop_set(Staging *s) {
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        const auto at = std::find(g_sets.begin(), g_sets.end(), s);
        if (at != g_sets.end()) g_sets.erase(at);
    }
    release_set(s);
}

bool make_buffers(Staging *s) {
    for (int b = 0; b < 2; ++b) {
        // kernels write these buffers and the host reads them after the event
        if (hipHostMalloc(&s->buf[b], kBuffer, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) !=
            hipSuccess) {
            s->buf[b] = nullptr;
            return false;
        }
        if (hipEventCreateWithFlags(&s->done[b], hipEventDisableTiming | hipEventReleaseToSystem) != hipSuccess) {
            s->done[b] = nullptr;
            return false;
        }
    }
    return true;
}

// Up to `want` sets of a device (current in this thread); fewer, or none, where other transfers have them
// or pinned memory or an event is not to be had.
int take_sets(int device, int want, Staging **out) {
    int got = 0, fresh;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        int live = 0;
        for (Staging *s : g_sets) {
            if (s->device != device) continue;
            ++live;
            if (s->busy || got == want) continue;
            s->busy = true;
            out[got++] = s;
        }
        fresh = got;
        try {
            for (; got < want && live < kSets; ++live) {
                g_sets.reserve(g_sets.size() + 1);
                out[got] = new Staging();
                out[got]->device = device;
                g_sets.push_back(out[got++]);
            }
        } catch (const std::bad_alloc &) {   // what there is
        }
    }
    for (int k = fresh; k < got; ++k)
        if (!make_buffers(out[k])) {
            (void)hipGetLastError();   // the caller goes another way
            for (int j = k; j < got; ++j) drop_set(out[j]);
            got = k;
        }
    return got;
}

void give_set(Staging *s) {
    std::lock_guard<std::mutex> lock(g_mutex);
    s->busy = false;
}

// After a failed transfer: whatever it left on the stream may still use the buffers, and no event
// marks its end, so the set does not go back to the pool.  The caller reports the error; it does not
// stay for the next launch's hipGetLastError.
void discard_set(Staging *s, hipStream_t stream) {
    (void)hipStreamSynchronize(stream);
    drop_set(s);
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

// One share, between host and dev, through a staging set.
hipError_t move_share(Staging *s, hipStream_t stream, char *host, char *dev, size_t bytes, bool to_dev) {
    OnDevice on(s->device);
    hipError_t e = on.err;
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

// By up to kThreads threads, one of them the caller's.
hipError_t move(hg_handle *h, char *host, char *dev, size_t bytes, bool to_dev) {
    if (bytes == 0) return hipSuccess;
    OnDevice on(h->device);
    if (on.err != hipSuccess) return on.err;
    const size_t chunks = (bytes + kShort - 1) / kShort;
    Staging *sets[kThreads];
    const int want = (int)std::max<size_t>(1, std::min<size_t>(kThreads, chunks / (kShare / kShort)));
    const int n = take_sets(h->device, want, sets);
    if (n == 0) {
        const hipError_t e = to_dev ? hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, h->stream)
                                    : hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, h->stream);
        return e == hipSuccess ? hipStreamSynchronize(h->stream) : e;
    }
    const size_t per = (chunks + n - 1) / n * kShort;
    std::atomic<int> err{(int)hipSuccess};
    auto share = [&](int k) {
        const size_t a = std::min(bytes, k * per), b = std::min(bytes, a + per);
        const hipError_t e = move_share(sets[k], h->stream, host + a, dev + a, b - a, to_dev);
        if (e != hipSuccess) err = (int)e;
    };
    std::thread th[kThreads];
    int k = n - 1;
    try {
        for (; k > 0; --k) th[k] = std::thread(share, k);
    } catch (const std::exception &) {   // no more threads: the shares up to k are this one's
    }
    for (; k >= 0; --k) share(k);
    for (std::thread &t : th)
        if (t.joinable()) t.join();
    return (hipError_t)err.load();
}

}  // namespace

namespace hg {

void transfers_open() {
    std::lock_guard<std::mutex> lock(g_mutex);
    ++g_handles;
}

void transfers_close() {
    std::vector<Staging *> idle;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (--g_handles > 0) return;
        idle.swap(g_sets);
    }
    for (Staging *s : idle) release_set(s);
}

hipError_t copy_to_host(hg_handle *h, void *dst, const void *src, size_t bytes) {
    return move(h, (char *)dst, (char *)const_cast<void *>(src), bytes, false);
}

hipError_t copy_to_device(hg_handle *h, void *dst, const void *src, size_t bytes) {
    if (bytes > kByKernel * kShort) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, h->stream);
    return move(h, (char *)const_cast<void *>(src), (char *)dst, bytes, true);
}

hipError_t read_values(hg_handle *h, double *dst, const double *src, int n, int stride) {
    if (n <= 0) return hipSuccess;
    if (stride == 1 && n > 1024) return copy_to_host(h, dst, src, n * sizeof(double));
    if ((size_t)n * sizeof(double) > kBuffer) return hipErrorInvalidValue;
    OnDevice on(h->device);
    hipError_t e = on.err;
    if (e != hipSuccess) return e;
    Staging *s = nullptr;
    if (!take_sets(h->device, 1, &s)) {
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
