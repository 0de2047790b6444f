// Copies between device memory and the caller's ordinary (pageable) host
// arrays, pipelined through pinned buffers.
//
// A pageable hipMemcpyAsync is staged by one thread inside the runtime (17
// GB/s down, 29 GB/s up here, 4 GB/s down into pages not touched yet).  Here
// the array moves in slices: a kernel fills or drains one pinned slot over
// the link while host threads copy others to or from the array, so the link's
// rate is the bound: 53 GB/s down and 54 up, 45 and 41 when the copy engine
// moved the slices (kernels that make the values, macrovar and the checkpoint,
// store into the slots themselves).  1.81 GB of fields: 40.9 -> 34.3 ms; 11.2
// MB 480 -> 340 us.
//
// The pinned slots belong to the process, not to a handle: up to HOST_WORKERS
// x HOST_DEPTH slots of HOST_SLICE bytes (48 MiB), each allocated by the first
// copy that needs it and freed with the last handle (retain / release).  One
// copy uses them at a time; a copy that finds them taken by another thread, or
// cannot allocate them, goes the plain way.  So does one whose array the runtime
// knows (runtime_array): it moves a pinned array at the link's rate by itself
// (us through the slots / by the runtime: 11.2 MB of fields 329 / 256, 10 MB of
// populations down 318 / 205, up 256 / 204).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>

namespace d3q19 {

constexpr int HOST_WORKERS = 6, HOST_DEPTH = 2;
constexpr size_t HOST_SLICE = 4u << 20;
constexpr size_t HOST_MIN = 64u << 10; // smaller copies go the plain way

// Bytes of a slice of a copy of `total` bytes: downloads in smaller slices
// below 64 MiB, so that the host's part overlaps the link's (us with 1 / 2 / 4
// MiB: 2.1 MB of fields 87 / 104 / 106, 11.2 MB 381 / 416 / 473, 53 MB of
// populations 1 560 / 1 411 / 1 736); uploads in whole ones, whose kernels
// need the waves to hide the link's latency (53 MB 1 651 / 1 253 / 1 162).
inline size_t host_slice(size_t total, bool down)
{
    return !down || total >= 64u << 20 ? HOST_SLICE : total >= 16u << 20 ? HOST_SLICE / 2 : HOST_SLICE / 4;
}

// Uploads below this size take three threads, which are as fast as six there
// (33 MB in four arrays 908 us with three, 917-954 with six, 82 MB 1 893 / 1 865,
// 184 MB 3 884 / 3 727) and need half of the slots, whose allocation the first
// copy pays for.
constexpr size_t HOST_UP_ALL = 96u << 20;

// Threads for a copy of `total` bytes: one (no thread is started) for downloads
// below 8 MiB and uploads below 24 MiB.  Two keep up with the link where the
// array's pages are there, as an upload's are (11.5 MB 0.46 ms with one, 0.52
// with four); more share the faults of a new array (11.2 MB of fields
// into one 1 570 us with two, 1 060 with four; 28 MB of viscosities 837 us with
// three, 780 with six).
inline int host_workers(size_t total, bool down)
{
    if (total < (down ? 8u : 24u) << 20)
        return 1;
    const size_t most = down || total >= HOST_UP_ALL ? HOST_WORKERS : 3;
    return (int)std::min<size_t>(most, 2 + (total >> 22));
}

// Whole arrays from the host that go the plain way although they are large
// enough: one thread fills the slots no faster than the runtime its own pinned
// buffers from 2 MiB on, and several do from 26 MiB on (us from arrays not seen
// before, runtime / slots: 0.5 MB 31 / 35, 2.1 MB in four 102 / 103, 2.9 MB 114 /
// 136, 4.4 MB 153 / 183, 17.6 MB in four 607 / 905, 24.6 MB in four 867 / 1 091,
// 29 MB 1 080 / 866, 33 MB in four 1 207 / 954, 41 MB 1 571 / 1 147).
constexpr size_t HOST_UP_PLAIN = 2u << 20, HOST_UP_MANY = 26u << 20;

// Copies with at least this many threads (16 MiB) use two streams.
constexpr int HOST_SIDE_WORKERS = 6;

struct HostPool {
    std::mutex mu;      // held by the copy that uses the slots
    std::mutex life_mu; // users
    int users = 0;
    int device = -1;    // device of the events and the side stream
    char *slot[HOST_WORKERS * HOST_DEPTH] = {};
    hipEvent_t ev[HOST_WORKERS * HOST_DEPTH] = {};
    hipStream_t side = nullptr; // of this device, created by the first large copy

    void drop_events()
    {
        if (side)
            (void)hipStreamDestroy(side);
        side = nullptr;
        for (hipEvent_t &e : ev) {
            if (e)
                (void)hipEventDestroy(e);
            e = nullptr;
        }
        device = -1;
    }
    // The slots of `workers` threads and this device's events (called with mu
    // held).
    bool ready(int dev, int workers)
    {
        for (int k = 0; k < workers * HOST_DEPTH; k++)
            if (!slot[k] && hipHostMalloc((void **)&slot[k], HOST_SLICE, hipHostMallocPortable) != hipSuccess) {
                slot[k] = nullptr;
                (void)hipGetLastError();
                return false;
            }
        if (device != dev) {
            drop_events();
            for (hipEvent_t &e : ev)
                if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                    e = nullptr;
                    (void)hipGetLastError();
                    drop_events();
                    return false;
                }
            device = dev;
        }
        if (workers >= HOST_SIDE_WORKERS && !side &&
            hipStreamCreateWithFlags(&side, hipStreamNonBlocking) != hipSuccess) {
            side = nullptr;
            (void)hipGetLastError();
            return false;
        }
        return true;
    }
    // The stream of odd slices: the side stream for large copies, so that the
    // link is not idle between the end of one slice's kernel and the start of
    // the next (1.81 GB down 36.2 -> 34.3 ms, 1.08 GB up 20.9 -> 20.0 ms); 2 MB
    // took 105 us with two streams, 90 with one.
    hipStream_t other(hipStream_t s, int workers) const { return workers >= HOST_SIDE_WORKERS ? side : s; }
    void retain()
    {
        std::lock_guard<std::mutex> l(life_mu);
        users++;
    }
    // The last user gives everything back (no copy of another user can run), while
    // its own stream is still there: with the side stream destroyed last, the
    // runtime's own copies on the next handle's stream took 4-6 ms longer (64x128x80,
    // upload and first steps 1 260 us, 6 820 after such a life; 13 MB of samples
    // into a trainer 390 / 4 650).
    void release()
    {
        std::lock_guard<std::mutex> l(life_mu);
        if (--users > 0)
            return;
        std::lock_guard<std::mutex> c(mu);
        drop_events();
        for (char *&p : slot) {
            if (p)
                (void)hipHostFree(p);
            p = nullptr;
        }
    }
};

inline HostPool &host_pool()
{
    static HostPool *p = new HostPool(); // outlives every handle, also at exit
    return *p;
}

// Slices 0 .. n-1 from the device: enqueue(k, slot, pinned, stream) puts what
// fills the pinned slot on the stream, consume(k, pinned) reads it on the host.
// Called with the pool's lock held, its slots ready and stream s idle; returns
// the first error.  Everything enqueued has finished when it returns.
template <class Enqueue, class Consume>
hipError_t host_slices_out(HostPool &pool, int device, hipStream_t s, size_t n, int workers, Enqueue enqueue,
                           Consume consume)
{
    const hipStream_t odd = pool.other(s, workers);
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&](int w) {
        size_t held[HOST_DEPTH];
        int first = 0, count = 0;
        hipError_t e = hipSetDevice(device);
        while (e == hipSuccess && err.load() == (int)hipSuccess) {
            while (count < HOST_DEPTH) {
                const size_t k = next.fetch_add(1);
                if (k >= n)
                    break;
                const int q = (first + count) % HOST_DEPTH, slot = w * HOST_DEPTH + q;
                const hipStream_t on = k % 2 ? odd : s;
                e = enqueue(k, slot, pool.slot[slot], on);
                if (e == hipSuccess)
                    e = hipEventRecord(pool.ev[slot], on);
                if (e != hipSuccess)
                    break;
                held[q] = k;
                count++;
            }
            if (e != hipSuccess || count == 0)
                break;
            const int slot = w * HOST_DEPTH + first;
            e = hipEventSynchronize(pool.ev[slot]);
            if (e != hipSuccess)
                break;
            consume(held[first], pool.slot[slot]);
            first = (first + 1) % HOST_DEPTH;
            count--;
        }
        int ok = (int)hipSuccess;
        if (e != hipSuccess)
            err.compare_exchange_strong(ok, (int)e);
    };
    std::thread t[HOST_WORKERS];
    int started = 1;
    try {
        for (; started < workers; started++)
            t[started] = std::thread(work, started);
    } catch (...) { // no more threads: those that run take all slices
    }
    work(0);
    for (int w = 1; w < HOST_WORKERS; w++)
        if (t[w].joinable())
            t[w].join();
    const hipError_t e = hipStreamSynchronize(s), e2 = odd == s ? e : hipStreamSynchronize(odd);
    return err.load() != (int)hipSuccess ? (hipError_t)err.load() : e != hipSuccess ? e : e2;
}

// Slices 0 .. n-1 to the device: produce(k, pinned) fills the pinned slot on
// the host, enqueue(k, slot, pinned, stream) puts what reads it on the stream.
template <class Produce, class Enqueue>
hipError_t host_slices_in(HostPool &pool, int device, hipStream_t s, size_t n, int workers, Produce produce,
                          Enqueue enqueue)
{
    const hipStream_t odd = pool.other(s, workers);
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&](int w) {
        hipError_t e = hipSetDevice(device);
        for (int i = 0; e == hipSuccess && err.load() == (int)hipSuccess; i++) {
            const size_t k = next.fetch_add(1);
            if (k >= n)
                break;
            const int slot = w * HOST_DEPTH + i % HOST_DEPTH;
            if (i >= HOST_DEPTH)
                e = hipEventSynchronize(pool.ev[slot]);
            if (e != hipSuccess)
                break;
            produce(k, pool.slot[slot]);
            const hipStream_t on = k % 2 ? odd : s;
            e = enqueue(k, slot, pool.slot[slot], on);
            // the only worker's last slices are not waited for one by one
            if (e == hipSuccess && (workers > 1 || k + HOST_DEPTH < n))
                e = hipEventRecord(pool.ev[slot], on);
        }
        int ok = (int)hipSuccess;
        if (e != hipSuccess)
            err.compare_exchange_strong(ok, (int)e);
    };
    std::thread t[HOST_WORKERS];
    int started = 1;
    try {
        for (; started < workers; started++)
            t[started] = std::thread(work, started);
    } catch (...) { // no more threads: those that run take all slices
    }
    work(0);
    for (int w = 1; w < HOST_WORKERS; w++)
        if (t[w].joinable())
            t[w].join();
    const hipError_t e = hipStreamSynchronize(s), e2 = odd == s ? e : hipStreamSynchronize(odd);
    return err.load() != (int)hipSuccess ? (hipError_t)err.load() : e != hipSuccess ? e : e2;
}

// Copy between device memory and a pinned slot, 16 bytes a lane and four in
// flight; `tail` bytes (below 16) follow the n vectors.
typedef uint32_t LinkVec __attribute__((ext_vector_type(4)));
constexpr int LINK_BLOCK = 256, LINK_UNROLL = 4;
// blocks of a copy, measured in 4 MiB pieces (GB/s with 8 / 32 / 128 / 512
// blocks): down 48.3 / 53.3 / 54.7 / 54.9, up 54.7 / 54.5 / 49.1 / 41.4, where
// more reads in flight than the link takes get in each other's way.  The copy
// engine: 50.3 either way.
constexpr size_t LINK_DOWN_BLOCKS = 256, LINK_UP_BLOCKS = 32;

static __global__ void __launch_bounds__(LINK_BLOCK) k_link_copy(const LinkVec *__restrict__ src, LinkVec *__restrict__ dst,
                                                                 size_t n, uint32_t tail)
{
    constexpr size_t STRIDE = LINK_BLOCK * LINK_UNROLL;
    for (size_t i = blockIdx.x * STRIDE + threadIdx.x; i < n; i += gridDim.x * STRIDE) {
        LinkVec v[LINK_UNROLL];
#pragma unroll
        for (int k = 0; k < LINK_UNROLL; k++)
            if (i + k * LINK_BLOCK < n)
                v[k] = __builtin_nontemporal_load(src + i + k * LINK_BLOCK);
#pragma unroll
        for (int k = 0; k < LINK_UNROLL; k++)
            if (i + k * LINK_BLOCK < n)
                dst[i + k * LINK_BLOCK] = v[k];
    }
    if (blockIdx.x == 0 && threadIdx.x < tail)
        ((char *)(dst + n))[threadIdx.x] = ((const char *)(src + n))[threadIdx.x];
}

// One slice between device memory and a pinned slot; addresses that are not on
// 16 bytes take the runtime's copy, unless the tail's bytes are all there is.
inline hipError_t link_copy(void *dst, const void *src, size_t bytes, bool down, hipStream_t s)
{
    if (bytes >= sizeof(LinkVec) && ((uintptr_t)dst | (uintptr_t)src) % sizeof(LinkVec))
        return hipMemcpyAsync(dst, src, bytes, down ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, s);
    const size_t n = bytes / sizeof(LinkVec), per = LINK_BLOCK * LINK_UNROLL;
    const unsigned grid =
        (unsigned)std::max<size_t>(1, std::min<size_t>((n + per - 1) / per, down ? LINK_DOWN_BLOCKS : LINK_UP_BLOCKS));
    hipLaunchKernelGGL(k_link_copy, dim3(grid), dim3(LINK_BLOCK), 0, s, (const LinkVec *)src, (LinkVec *)dst, n,
                       (uint32_t)(bytes % sizeof(LinkVec)));
    return hipGetLastError();
}

// What the runtime knows the caller's array as: pinned (hipMemoryTypeHost),
// managed, a device's, or nothing (hipMemoryTypeUnregistered).  Only the
// runtime's own copies serve all of those.
inline hipMemoryType array_type(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return hipMemoryTypeUnregistered;
    }
    return a.type;
}
inline bool runtime_array(const void *p) { return array_type(p) != hipMemoryTypeUnregistered; }

// One contiguous part of a copy; a null host pointer is skipped.
struct HostPart {
    void *host;
    void *dev;
    size_t bytes;
};

// The parts one after another, `down` from the device or up to it, by at most
// `most` threads; returns when the copy has finished.
inline hipError_t host_copy(int device, hipStream_t s, const HostPart *parts, int nparts, bool down,
                            int most = HOST_WORKERS)
{
    size_t total = 0;
    bool known = false;
    for (int p = 0; p < nparts; p++)
        total += parts[p].host ? parts[p].bytes : 0;
    for (int p = 0; p < nparts && total >= HOST_MIN; p++)
        known = known || (parts[p].host && runtime_array(parts[p].host));
    const bool sliced = total >= HOST_MIN && !known && (down || total < HOST_UP_PLAIN || total >= HOST_UP_MANY);
    HostPool &pool = host_pool();
    std::unique_lock<std::mutex> lock(pool.mu, std::defer_lock);
    if (sliced) {
        // what the stream still computes is waited for before the slots are taken
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess)
            return e;
    }
    const int workers = std::min(most, host_workers(total, down));
    if (!sliced || !lock.try_lock() || !pool.ready(device, workers)) {
        for (int p = 0; p < nparts; p++)
            if (parts[p].host) {
                const hipError_t e =
                    down ? hipMemcpyAsync(parts[p].host, parts[p].dev, parts[p].bytes, hipMemcpyDeviceToHost, s)
                         : hipMemcpyAsync(parts[p].dev, parts[p].host, parts[p].bytes, hipMemcpyHostToDevice, s);
                if (e != hipSuccess)
                    return e;
            }
        return hipStreamSynchronize(s);
    }
    const size_t slice = host_slice(total, down);
    size_t n = 0;
    for (int p = 0; p < nparts; p++)
        n += parts[p].host ? (parts[p].bytes + slice - 1) / slice : 0;
    // slice k: its part and place
    auto find = [&](size_t k, char *&host, char *&dev) -> size_t {
        for (int p = 0; p < nparts; p++) {
            const size_t m = parts[p].host ? (parts[p].bytes + slice - 1) / slice : 0;
            if (k < m) {
                host = (char *)parts[p].host + k * slice;
                dev = (char *)parts[p].dev + k * slice;
                return std::min(slice, parts[p].bytes - k * slice);
            }
            k -= m;
        }
        return 0;
    };
    if (down)
        return host_slices_out(
            pool, device, s, n, workers,
            [&](size_t k, int, char *pinned, hipStream_t on) {
                char *host, *dev;
                const size_t b = find(k, host, dev);
                return link_copy(pinned, dev, b, true, on);
            },
            [&](size_t k, const char *pinned) {
                char *host, *dev;
                const size_t b = find(k, host, dev);
                memcpy(host, pinned, b);
            });
    return host_slices_in(
        pool, device, s, n, workers,
        [&](size_t k, char *pinned) {
            char *host, *dev;
            const size_t b = find(k, host, dev);
            memcpy(pinned, host, b);
        },
        [&](size_t k, int, const char *pinned, hipStream_t on) {
            char *host, *dev;
            const size_t b = find(k, host, dev);
            return link_copy(dev, pinned, b, false, on);
        });
}

} // namespace d3q19
