// copy_out (mhd_copy.hip) byte for byte, on host memory: totals on both sides
// of its limits, spans of uneven sizes, several of them filled at once.
#include "hip_host.h"

#include <atomic>
#include <chrono>
#include <thread>

#include "../../rast-3dmhd_amd/csrc/mhd_copy.h"

using namespace rmhd;

// A "device" buffer of `room` bytes that each fill overwrites with the next
// spans that fit it; byte b of span i is a function of both.
struct Source {
    const HostSpan *spans;
    int n;
    size_t room;
    char *dev;
    static char value(int i, size_t b) { return (char)(b * 131 + (b >> 11) + i * 17 + 1); }
    static int fill(void *ctx, int i, const char **src, hipError_t *) {
        Source &s = *static_cast<Source *>(ctx);
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
    const hipError_t e = copy_out(spans.data(), (int)spans.size(), Source::fill, &src, nullptr);
    (void)hipFree(dev);
    return e;
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

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    copy_retain();
    int rc = 1;
    if (what == "same_array") rc = same_array();
    else printf("unknown check\n");
    copy_release();
    HH_CHECK(hh::ranges.empty());
    return rc;
}
