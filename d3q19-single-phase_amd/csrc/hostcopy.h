// Copies between device memory and the caller's ordinary (pageable) host
// arrays, pipelined through pinned buffers.
//
// A pageable hipMemcpyAsync is staged by one thread inside the runtime (17
// GB/s down, 29 GB/s up here, 4 GB/s down into pages not touched yet).  Here
// the array moves in slices: the copy engine fills or drains one pinned slot
// while host threads copy others to or from the array, so the link's rate is
// the bound (45 GB/s with 4 MiB slices, 20 us of each slice being the copy's
// start; 512 MB down: 31 ms before, 11.5 ms).  Two threads keep up with the
// link; more share the page faults of a new array (184 MB: 46 ms before,
// 13 ms).
//
// The pinned slots belong to the process, not to a handle: HOST_WORKERS x
// HOST_DEPTH slots of HOST_SLICE bytes (48 MiB), allocated by the first large
// copy and freed with the last handle (host_pool_retain / release).  One copy
// uses them at a time; a copy that finds them taken by another thread, or
// cannot allocate them, goes the plain way.
#pragma once

#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>

namespace d3q19 {

constexpr int HOST_WORKERS = 6, HOST_DEPTH = 2;
constexpr size_t HOST_SLICE = 4u << 20;
constexpr size_t HOST_MIN = 1u << 20; // smaller copies go the plain way

struct HostPool {
    std::mutex mu;      // held by the copy that uses the slots
    std::mutex life_mu; // users
    int users = 0;
    int device = -1;    // device of the events
    char *slot[HOST_WORKERS * HOST_DEPTH] = {};
    hipEvent_t ev[HOST_WORKERS * HOST_DEPTH] = {};

    void drop_events()
    {
        for (hipEvent_t &e : ev) {
            if (e)
                (void)hipEventDestroy(e);
            e = nullptr;
        }
        device = -1;
    }
    // Slots and this device's events (called with mu held).
    bool ready(int dev)
    {
        for (char *&p : slot)
            if (!p && hipHostMalloc((void **)&p, HOST_SLICE, hipHostMallocPortable) != hipSuccess) {
                p = nullptr;
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
        return true;
    }
    void retain()
    {
        std::lock_guard<std::mutex> l(life_mu);
        users++;
    }
    // The last user gives everything back (no copy of another user can run).
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

// Slices 0 .. n-1 from the device: enqueue(k, slot, pinned) puts what fills
// the pinned slot on stream s, consume(k, pinned) reads it on the host.
// Called with the pool's lock held and its slots ready; returns the first
// error.  Everything enqueued has finished when it returns.
template <class Enqueue, class Consume>
hipError_t host_slices_out(HostPool &pool, int device, hipStream_t s, size_t n, int workers, Enqueue enqueue,
                           Consume consume)
{
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
                e = enqueue(k, slot, pool.slot[slot]);
                if (e == hipSuccess)
                    e = hipEventRecord(pool.ev[slot], s);
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
    const hipError_t e = hipStreamSynchronize(s);
    return err.load() != (int)hipSuccess ? (hipError_t)err.load() : e;
}

// Slices 0 .. n-1 to the device: produce(k, pinned) fills the pinned slot on
// the host, enqueue(k, slot, pinned) puts what reads it on stream s.
template <class Produce, class Enqueue>
hipError_t host_slices_in(HostPool &pool, int device, hipStream_t s, size_t n, int workers, Produce produce,
                          Enqueue enqueue)
{
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
            e = enqueue(k, slot, pool.slot[slot]);
            if (e == hipSuccess)
                e = hipEventRecord(pool.ev[slot], s);
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
    const hipError_t e = hipStreamSynchronize(s);
    return err.load() != (int)hipSuccess ? (hipError_t)err.load() : e;
}

// Threads for a copy of `bytes`: one (no thread is started) below 8 MiB.
inline int host_workers(size_t bytes)
{
    return (int)std::max<size_t>(1, std::min<size_t>(HOST_WORKERS, bytes / HOST_SLICE / 2));
}

// One contiguous part of a copy; a null host pointer is skipped.
struct HostPart {
    void *host;
    void *dev;
    size_t bytes;
};

// The parts one after another, `down` from the device or up to it; returns
// when the copy has finished.
inline hipError_t host_copy(int device, hipStream_t s, const HostPart *parts, int nparts, bool down)
{
    size_t total = 0;
    for (int p = 0; p < nparts; p++)
        total += parts[p].host ? parts[p].bytes : 0;
    HostPool &pool = host_pool();
    std::unique_lock<std::mutex> lock(pool.mu, std::defer_lock);
    if (total >= HOST_MIN) {
        // what the stream still computes is waited for before the slots are taken
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess)
            return e;
    }
    if (total < HOST_MIN || !lock.try_lock() || !pool.ready(device)) {
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
    // copies below two slices a worker in smaller ones, so that the host's
    // part overlaps the link's
    const size_t slice = total < 2 * HOST_SLICE ? HOST_SLICE / 4 : HOST_SLICE;
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
            pool, device, s, n, host_workers(total),
            [&](size_t k, int, char *pinned) {
                char *host, *dev;
                const size_t b = find(k, host, dev);
                return hipMemcpyAsync(pinned, dev, b, hipMemcpyDeviceToHost, s);
            },
            [&](size_t k, const char *pinned) {
                char *host, *dev;
                const size_t b = find(k, host, dev);
                memcpy(host, pinned, b);
            });
    return host_slices_in(
        pool, device, s, n, host_workers(total),
        [&](size_t k, char *pinned) {
            char *host, *dev;
            const size_t b = find(k, host, dev);
            memcpy(pinned, host, b);
        },
        [&](size_t k, int, const char *pinned) {
            char *host, *dev;
            const size_t b = find(k, host, dev);
            return hipMemcpyAsync(dev, pinned, b, hipMemcpyHostToDevice, s);
        });
}

} // namespace d3q19
