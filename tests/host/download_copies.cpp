// copy_out (mhd_copy.hip) byte for byte, on host memory: as it runs, where no
// memory can be pinned, and where none or one of its threads can be started.
#include "hip_host.h"

#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <chrono>
#include <thread>

#include "../../rast-3dmhd_amd/csrc/mhd_copy.h"

using namespace rmhd;

// Threads that a call can start (-1: any number), and those left to it.
static int threads_allowed = -1;
static std::atomic<int> threads_left{-1};
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    typedef int (*Create)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static const Create real = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
    if (threads_left == 0) return EAGAIN;
    if (threads_left > 0) --threads_left;
    return real(t, a, f, arg);
}

// A "device" buffer of `room` bytes that each fill overwrites with the next
// spans that fit it; byte b of span i is a function of both.
static int fails_at = -1;  // span whose fill fails
struct Source {
    const HostSpan *spans;
    int n;
    size_t room;
    char *dev;
    static char value(int i, size_t b) { return (char)(b * 131 + (b >> 11) + i * 17 + 1); }
    static int fill(void *ctx, int i, const char **src, hipError_t *e) {
        Source &s = *static_cast<Source *>(ctx);
        if (i == fails_at) {
            *e = hipErrorLaunchFailure;
            return 0;
        }
        size_t at = 0;
        int m = 0;
        for (; i + m < s.n && (m == 0 || at + s.spans[i + m].bytes <= s.room); ++m) {
            for (size_t b = 0; b < s.spans[i + m].bytes; ++b) s.dev[at + b] = value(i + m, b);
            at += s.spans[i + m].bytes;
        }
        *src = s.dev;
        return m;
    }
};

static hipError_t copy_all(const std::vector<HostSpan> &spans, size_t room) {
    size_t most = room;
    for (const HostSpan &s : spans) most = std::max(most, s.bytes);
    void *dev = nullptr;
    (void)hipMalloc(&dev, most);
    Source src{spans.data(), (int)spans.size(), room, static_cast<char *>(dev)};
    threads_left = threads_allowed;
    const hipError_t e = copy_out(spans.data(), (int)spans.size(), Source::fill, &src, nullptr);
    (void)hipFree(dev);
    return e;
}

// Totals on both sides of the limits, from one span to eight, some of them or
// all filled at once; a source that fails for the last of them.
static int sizes() {
    const std::vector<std::vector<size_t>> all = {
        {1}, {1 << 20}, {(1 << 20) + 1}, {9 << 20}, {70 << 20}, {40, 8, 24}, {300000, 8, 5000000, 16, 77777},
        {(8 << 20) - 1}, {8 << 20}, {(4 << 20) - 8, (4 << 20) - 8}, {4 << 20, 4 << 20}, {262144, 262145, 9 << 20, 1, 1 << 18},
        std::vector<size_t>(8, (5 << 20) + 1001)};
    for (const std::vector<size_t> &lens : all)
        for (const size_t room : {(size_t)1, (size_t)6 << 20, (size_t)128 << 20}) {
            std::vector<std::vector<char>> out;
            std::vector<HostSpan> spans;
            for (size_t n : lens) out.emplace_back(n + 1, (char)85);
            for (size_t i = 0; i < lens.size(); ++i) spans.push_back({out[i].data(), lens[i]});
            HH_CHECK(copy_all(spans, room) == hipSuccess);
            for (size_t i = 0; i < lens.size(); ++i) {
                for (size_t b = 0; b < lens[i]; ++b) HH_CHECK(out[i][b] == Source::value((int)i, b));
                HH_CHECK(out[i][lens[i]] == 85);
            }
            if (lens.size() > 1 && room == 1) {
                fails_at = (int)lens.size() - 1;
                HH_CHECK(copy_all(spans, room) == hipErrorLaunchFailure);
                fails_at = -1;
            }
        }
    return 0;
}

// The same array for two spans: as if they were copied one after the other, the
// last one's bytes stay, also when the first event is seen late.
static int same_array() {
    std::atomic<int> waits{0};
    hh::on_event_wait = [&](hipEvent_t) {
        if (waits.fetch_add(1) == 0) std::this_thread::sleep_for(std::chrono::milliseconds(200));
    };
    const size_t n = (5 << 20) + 40;
    std::vector<char> a(n), b(n);
    HH_CHECK(copy_all({{a.data(), n}, {b.data(), n}, {a.data(), n}}, 3 * n) == hipSuccess);
    for (size_t i = 0; i < n; ++i) HH_CHECK(a[i] == Source::value(2, i) && b[i] == Source::value(1, i));
    return 0;
}

// Spans in pinned memory of 384 KiB and more on average are copied to directly,
// without the ring, shorter ones in a run; a pageable one among them is served too.
static int pinned() {
    for (const std::vector<size_t> &sizes : {std::vector<size_t>{3 << 20, 100, 9 << 20}, {2 << 20}, {384 << 10, 384 << 10}, {384 << 10, (384 << 10) - 1}}) {
        for (const size_t room : {(size_t)4 << 20, (size_t)64 << 20})
            for (int pageable = 0; pageable < 2; ++pageable) {
                std::vector<HostSpan> spans;
                std::vector<char> own(sizes.back());
                for (size_t n : sizes) {
                    void *p = nullptr;
                    (void)hipHostMalloc(&p, n, 0);
                    spans.push_back({p, n});
                }
                void *const last = spans.back().dst;
                size_t total = 0;
                for (size_t n : sizes) total += n;
                const bool direct = !pageable && total >= sizes.size() * (384 << 10);
                if (pageable) spans.back().dst = own.data();
                hh::copies.clear();
                HH_CHECK(copy_all(spans, room) == hipSuccess);
                for (size_t i = 0; i < spans.size(); ++i) {
                    for (size_t b = 0; b < spans[i].bytes; ++b)
                        HH_CHECK(static_cast<char *>(spans[i].dst)[b] == Source::value((int)i, b));
                    HH_CHECK(direct == (hh::copies[0].dst == spans[0].dst));
                    if (direct) HH_CHECK(hh::copies.size() == spans.size() && hh::copies[i].dst == spans[i].dst);
                }
                spans.back().dst = last;
                for (const HostSpan &s : spans) (void)hipHostFree(s.dst);
            }
    }
    // memory the CPU may not write, however short
    void *dev = nullptr;
    (void)hipMalloc(&dev, 6000);
    std::vector<char> own(4000);
    const std::vector<HostSpan> spans = {{own.data(), own.size()}, {dev, 6000}};
    hh::copies.clear();
    HH_CHECK(copy_all(spans, 1 << 20) == hipSuccess && hh::copies.size() == 2 && hh::copies[1].dst == dev);
    (void)hipFree(dev);
    return 0;
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    copy_retain();
    int rc = 1;
    hh::no_pinned = what == "no_pinned_memory";
    threads_allowed = what == "no_threads" ? 0 : what == "one_thread" ? 1 : -1;
    if (what == "sizes" || what == "no_pinned_memory" || what == "no_threads" || what == "one_thread") rc = sizes();
    else if (what == "same_array") rc = same_array();
    else if (what == "pinned") rc = pinned();
    else printf("unknown check\n");
    copy_release();
    HH_CHECK(hh::ranges.empty());
    return rc;
}
