// Device-to-host copies into the caller's ordinary (pageable) memory.
//
// The runtime's own copy into pageable memory runs at 18 GB/s: one thread
// moves what the DMA engine brought into a pinned buffer.  The link does 57.
// Here the DMA fills the slots of a pinned ring in order, and several threads
// empty them into the caller's memory at the same time: 512x512x256 (4.3 GB)
// comes down in 90 ms instead of 250, 64x64x48 (13.6 MB) in 0.48 ms instead of
// 1.1.  One thread empties 28 GB/s, three 46 GB/s, seven or twelve no more.
// Starting them costs some 60 us: below 8 MiB this thread empties the ring itself,
// and all fields that one launch wrote come down as one run, because a copy and an
// event per field cost 20 us each (eight fields of 16x16x12, 0.3 MB: 180 us with
// slots per field, 45 as a run; 32x32x24, 1.9 MB: 210, 107; 48x48x28, 4.8 MB: 263,
// 209).  One array up to 1 MiB takes the runtime's own copy, which needs no second
// copy here (0.6 MB: 58 us, 65 through the ring; 2.1 MB: 175, 152).  Arrays that
// the caller pinned need no ring (copy_direct).
//
// Threads live for one call (they start while the first piece is on its way),
// so nothing runs between calls.  A ring is used by one call at a time; it is
// taken from and put back into a list of at most two, which is emptied when
// the last handle goes.

#include "mhd_copy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace rmhd {

namespace {

constexpr size_t SMALL = 1 << 20, RING = 32 << 20;
constexpr int SLOTS = 8, KEEP = 2, THREADS = 3;
constexpr size_t THREADS_FROM = 8 << 20, PIECE = 1 << 20, DIRECT_FROM = 384 << 10;
static_assert(THREADS_FROM <= RING && SLOTS >= 4, "a result without threads fits the ring");

struct Ring {
    char *base = nullptr;
    int dev = 0;  // device the events belong to
    hipEvent_t ev[SLOTS] = {};
};

std::mutex g_mu;
std::vector<Ring *> g_free;
int g_handles = 0;

void ring_free(Ring *r) {
    for (auto &e : r->ev)
        if (e) (void)hipEventDestroy(e);
    if (r->base) (void)hipHostFree(r->base);
    delete r;
}

hipError_t ring_get(Ring **out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (size_t i = 0; i < g_free.size(); ++i)
            if (g_free[i]->dev == dev) {
                *out = g_free[i];
                g_free.erase(g_free.begin() + (long)i);
                return hipSuccess;
            }
    }
    Ring *r = new Ring;
    r->dev = dev;
    e = hipHostMalloc(reinterpret_cast<void **>(&r->base), RING, hipHostMallocDefault);
    for (int i = 0; i < SLOTS && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&r->ev[i], hipEventDisableTiming);
    if (e != hipSuccess) {
        ring_free(r);
        return e;
    }
    *out = r;
    return hipSuccess;
}

void ring_put(Ring *r) {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_handles > 0 && g_free.size() < (size_t)KEEP) {
            try {
                g_free.push_back(r);
                return;
            } catch (...) {
            }
        }
    }
    ring_free(r);
}

struct Task {
    char *dst;
    size_t bytes;
};

// State shared by the threads of one call.
struct Job {
    Ring *ring;
    const std::vector<Task> *tasks;
    size_t slot_bytes;
    std::atomic<int> queued{0}, next{0}, failed{0};
    std::vector<std::atomic<char>> done;
    explicit Job(size_t n) : done(n) {}
};

// Empties ring slots into the caller's memory until no task is left.
void drain(Job *j) {
    const int n = (int)j->tasks->size();
    for (;;) {
        const int i = j->next.fetch_add(1);
        if (i >= n) return;
        while (j->queued.load(std::memory_order_acquire) <= i) {
            if (j->failed.load()) return;
            std::this_thread::yield();
        }
        if (hipEventSynchronize(j->ring->ev[i % SLOTS]) != hipSuccess) {
            j->failed.store(1);
            return;
        }
        const Task &t = (*j->tasks)[(size_t)i];
        memcpy(t.dst, j->ring->base + (size_t)(i % SLOTS) * j->slot_bytes, t.bytes);
        j->done[(size_t)i].store(1, std::memory_order_release);
    }
}

// One ordinary copy per contiguous run: a small array, spans that overlap, or no
// pinned memory.
hipError_t copy_plain(const HostSpan *spans, int n, FillFn fill, void *ctx, hipStream_t s) {
    std::vector<char> tmp;
    for (int i = 0; i < n;) {
        const char *src = nullptr;
        hipError_t e = hipSuccess;
        const int m = fill(ctx, i, &src, &e);
        if (m < 1) return e != hipSuccess ? e : hipErrorUnknown;
        size_t bytes = 0;
        for (int k = 0; k < m; ++k) bytes += spans[i + k].bytes;
        char *dst = static_cast<char *>(spans[i].dst);
        if (m > 1) {
            tmp.resize(bytes);
            dst = tmp.data();
        }
        e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        if (m > 1)
            for (int k = 0; k < m; ++k) {
                memcpy(spans[i + k].dst, dst, spans[i + k].bytes);
                dst += spans[i + k].bytes;
            }
        i += m;
    }
    return hipSuccess;
}

// Copies n bytes at src into the spans, from byte off of span i on (both moved on).
void scatter(const HostSpan *spans, int &i, size_t &off, const char *src, size_t n) {
    while (n) {
        const size_t m = std::min(n, spans[i].bytes - off);
        memcpy(static_cast<char *>(spans[i].dst) + off, src, m);
        src += m;
        n -= m;
        off += m;
        if (off == spans[i].bytes) {
            ++i;
            off = 0;
        }
    }
}

// Results that fit the ring, without threads: each contiguous run comes down in
// one to four pieces whatever its spans, and this thread copies a piece out
// while the next one is on its way.
hipError_t copy_mid(const HostSpan *spans, int n, FillFn fill, void *ctx, hipStream_t s) {
    Ring *ring = nullptr;
    hipError_t e = ring_get(&ring);
    if (e != hipSuccess) {  // no pinned memory: the runtime's own copies
        (void)hipGetLastError();
        return copy_plain(spans, n, fill, ctx, s);
    }
    for (int i = 0; i < n && e == hipSuccess;) {
        const char *src = nullptr;
        const int m = fill(ctx, i, &src, &e);
        if (m < 1) {
            if (e == hipSuccess) e = hipErrorUnknown;
            break;
        }
        size_t bytes = 0;
        for (int k = 0; k < m; ++k) bytes += spans[i + k].bytes;
        const size_t piece = std::max(PIECE, (bytes / 4 + 4095) / 4096 * 4096);
        int np = 0;
        for (size_t o = 0; o < bytes && e == hipSuccess; o += piece, ++np) {
            e = hipMemcpyAsync(ring->base + o, src + o, std::min(piece, bytes - o), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess && o + piece < bytes) e = hipEventRecord(ring->ev[np], s);
        }
        int at = i;
        size_t off = 0;
        for (int k = 0; k < np && e == hipSuccess; ++k) {
            e = k < np - 1 ? hipEventSynchronize(ring->ev[k]) : hipStreamSynchronize(s);
            const size_t o = (size_t)k * piece;
            if (e == hipSuccess) scatter(spans, at, off, ring->base + o, std::min(piece, bytes - o));
        }
        i += m;
    }
    // nothing may still write into the ring when it is used again
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    ring_put(ring);
    return e;
}

// Whether the runtime copies into the spans itself: where the CPU may not write
// (device memory), and where the caller pinned all of them and they are not short.
bool spans_direct(const HostSpan *spans, int n, size_t total) {
    bool known = true;
    for (int i = 0; i < n; ++i) {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, spans[i].dst) != hipSuccess) {
            (void)hipGetLastError();
            a.type = hipMemoryTypeUnregistered;
        }
        if (a.type == hipMemoryTypeDevice) return true;
        known = known && a.type != hipMemoryTypeUnregistered;
    }
    return known && total >= n * DIRECT_FROM;
}

// Straight into the spans, one wait at the end: the link's rate, without a copy
// by the CPU (eight pinned fields, us through the ring and so: 4.8 MB 215, 179;
// 13.9 MB 489, 336; 141 MB 3357, 2674; one of 1.7 MB 101, 53).  Each copy costs
// 10 us, so that short ones are faster as a run through the ring (eight of 0.1
// MB: 54, 98; of 0.24 MB: 95, 123; the lines cross at 0.4 MB).
hipError_t copy_direct(const HostSpan *spans, int n, FillFn fill, void *ctx, hipStream_t s) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < n && e == hipSuccess;) {
        const char *src = nullptr;
        int m = fill(ctx, i, &src, &e);
        if (m < 1 && e == hipSuccess) e = hipErrorUnknown;
        for (; m > 0 && e == hipSuccess; --m, ++i) {
            e = hipMemcpyAsync(spans[i].dst, src, spans[i].bytes, hipMemcpyDeviceToHost, s);
            src += spans[i].bytes;
        }
    }
    const hipError_t e2 = hipStreamSynchronize(s);
    return e != hipSuccess ? e : e2;
}

// Whether two spans share memory (the same array passed twice): they are then
// copied one after the other, and the later one's bytes stay.
bool spans_overlap(const HostSpan *spans, int n) {
    for (int i = 0; i < n; ++i)
        for (int k = 0; k < i; ++k) {
            const char *const a = static_cast<const char *>(spans[i].dst), *const b = static_cast<const char *>(spans[k].dst);
            if (a < b + spans[k].bytes && b < a + spans[i].bytes) return true;
        }
    return false;
}

hipError_t copy_large(const HostSpan *spans, int n, size_t total, FillFn fill, void *ctx, hipStream_t s) {
    // slots small enough that a result makes several of them, so that the
    // copies out of the ring overlap the DMA into it
    const size_t slot = std::min(RING / SLOTS, std::max((size_t)(256 << 10), (total / 8 + 4095) / 4096 * 4096));
    std::vector<Task> tasks;
    for (int i = 0; i < n; ++i)
        for (size_t o = 0; o < spans[i].bytes; o += slot)
            tasks.push_back({static_cast<char *>(spans[i].dst) + o, std::min(slot, spans[i].bytes - o)});
    Job job(tasks.size());
    job.tasks = &tasks;
    job.slot_bytes = slot;
    hipError_t e = ring_get(&job.ring);
    if (e != hipSuccess) {  // no pinned memory: the runtime's own copies
        (void)hipGetLastError();
        return copy_plain(spans, n, fill, ctx, s);
    }
    std::vector<std::thread> th;
    try {
        th.reserve((size_t)THREADS);
        for (int t = 0; t < THREADS; ++t) th.emplace_back(drain, &job);
    } catch (...) {  // fewer threads: this one empties the rest
    }
    const bool alone = th.empty();
    auto queue_all = [&]() -> hipError_t {
        size_t task = 0;
        for (int i = 0; i < n;) {
            const char *src = nullptr;
            hipError_t r = hipSuccess;
            const int m = fill(ctx, i, &src, &r);
            if (m < 1) return r != hipSuccess ? r : hipErrorUnknown;
            for (int k = 0; k < m; ++k, ++i)
                for (size_t o = 0; o < spans[i].bytes; o += slot, ++task) {
                    // the slot's previous content has been copied out
                    if (task >= SLOTS) {
                        const size_t old = task - SLOTS;
                        if (alone) {
                            r = hipEventSynchronize(job.ring->ev[old % SLOTS]);
                            if (r != hipSuccess) return r;
                            memcpy(tasks[old].dst, job.ring->base + (old % SLOTS) * slot, tasks[old].bytes);
                            job.next.store((int)old + 1);
                        } else {
                            while (!job.done[old].load(std::memory_order_acquire)) {
                                if (job.failed.load()) return hipErrorUnknown;
                                std::this_thread::yield();
                            }
                        }
                    }
                    r = hipMemcpyAsync(job.ring->base + (task % SLOTS) * slot, src + o, tasks[task].bytes,
                                       hipMemcpyDeviceToHost, s);
                    if (r == hipSuccess) r = hipEventRecord(job.ring->ev[task % SLOTS], s);
                    if (r != hipSuccess) return r;
                    job.queued.store((int)task + 1, std::memory_order_release);
                    if (o + slot >= spans[i].bytes) src += spans[i].bytes;
                }
        }
        return hipSuccess;
    };
    e = queue_all();
    if (e != hipSuccess) job.failed.store(1);
    else drain(&job);
    for (auto &t : th) t.join();
    if (e == hipSuccess && job.failed.load()) e = hipErrorUnknown;
    // nothing may still write into the ring when it is used again
    const hipError_t e2 = hipStreamSynchronize(s);
    ring_put(job.ring);
    return e != hipSuccess ? e : e2;
}

}  // namespace

void copy_retain() {
    std::lock_guard<std::mutex> lock(g_mu);
    ++g_handles;
}

void copy_release() {
    std::vector<Ring *> gone;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (--g_handles == 0) gone.swap(g_free);
    }
    for (Ring *r : gone) ring_free(r);
}

hipError_t copy_out(const HostSpan *spans, int n, FillFn fill, void *ctx, hipStream_t s) {
    size_t total = 0;
    for (int i = 0; i < n; ++i) total += spans[i].bytes;
    try {
        if (n == 1 && total <= SMALL) return copy_plain(spans, n, fill, ctx, s);
        if (spans_direct(spans, n, total)) return copy_direct(spans, n, fill, ctx, s);
        if (total < THREADS_FROM) return copy_mid(spans, n, fill, ctx, s);
        if (spans_overlap(spans, n)) return copy_plain(spans, n, fill, ctx, s);
        return copy_large(spans, n, total, fill, ctx, s);
    } catch (...) {  // no host memory for the lists
        return hipErrorOutOfMemory;
    }
}

}  // namespace rmhd
