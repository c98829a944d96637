// The pinned ring behind the engine's table uploads (upload_async, csrc/api.hip) over
// a model of the runtime: a stream that completes its copies late, in order, and as
// far as the test lets it.  A ring half that is used again, or given back, before its
// copies are done shows as a wrong table.  Prints one line per scenario; the exit
// status is 1 after any failure.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <random>
#include <vector>

#include "common.hpp"

namespace {
struct Op {
    void *dst;
    const void *src;
    size_t bytes;
};
std::deque<Op> queue;
uint64_t done = 0, pushed = 0;  // operations completed and issued
std::map<char *, size_t> pinned;
size_t pinned_now = 0, pinned_most = 0;
int direct = 0, staged = 0, freed_busy = 0;
size_t refuse_from = SIZE_MAX;  // allocations of at least this many bytes fail

bool is_pinned(const void *p) {
    for (auto &kv : pinned)
        if (p >= kv.first && p < kv.first + kv.second) return true;
    return false;
}
void progress(uint64_t to) {
    while (done < to) {
        const Op &o = queue.front();
        if (o.bytes) memcpy(o.dst, o.src, o.bytes);
        queue.pop_front();
        ++done;
    }
}
struct Event {
    uint64_t at = 0;
};
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (n >= refuse_from) return hipErrorOutOfMemory;
    *p = malloc(n);
    pinned[(char *)*p] = n;
    pinned_now += n;
    pinned_most = std::max(pinned_most, pinned_now);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    const size_t n = pinned[(char *)p];
    for (auto &o : queue)
        if (o.src >= p && o.src < (char *)p + n) ++freed_busy;
    memset(p, 0x5a, n);
    pinned_now -= n;
    pinned.erase((char *)p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
    queue.push_back({dst, src, n});
    ++pushed;
    if (!is_pinned(src)) {  // (waits for the stream to reach it)
        ++direct;
        progress(pushed);
    } else {
        ++staged;
    }
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t) new Event;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    queue.push_back({nullptr, nullptr, 0});
    ((Event *)e)->at = ++pushed;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return done >= ((Event *)e)->at ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventSynchronize(hipEvent_t e) {
    progress(((Event *)e)->at);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    progress(pushed);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "refused"; }
}

// `tables` of up to `most` bytes; after each the stream goes on with probability
// `pace`; pinned allocations of `refuse` bytes and more fail from the start or from
// the middle on, and for the last quarter they succeed again
static int scenario(const char *name, int tables, size_t most, double pace, size_t refuse, bool from_start) {
    std::mt19937_64 rng(42);
    ptbgpu_ctx ctx;
    queue.clear();
    done = pushed = 0;
    pinned_now = pinned_most = 0;
    direct = staged = freed_busy = 0;
    refuse_from = from_start ? refuse : SIZE_MAX;
    std::vector<std::vector<char>> want, got;
    int bad = 0, late = 0;
    for (int i = 0; i < tables; ++i) {
        if (i == tables / 2) refuse_from = refuse;
        if (i == tables / 4 * 3) refuse_from = SIZE_MAX, late = staged;
        const size_t n = 1 + rng() % most;
        std::vector<char> t(n);
        for (size_t k = 0; k < n; k += 1 + n / 64) t[k] = (char)rng();
        t[n - 1] = (char)rng();
        want.push_back(t);
        got.emplace_back(n);
        bad += ptb::upload_async(&ctx, got.back().data(), t.data(), n) != PTBGPU_OK;
        std::fill(t.begin(), t.end(), 0x33);  // (the caller's table goes away)
        if (rng() % 1000 < 1000 * pace) progress(done + rng() % (pushed - done + 1));
    }
    progress(pushed);
    for (size_t i = 0; i < want.size(); ++i) bad += want[i] != got[i];
    bad += freed_busy + (pinned_most > (size_t)96 << 20) + (staged == late);
    bad += !ctx.last_error.empty();
    printf("%s: %d staged, %d direct, %zu MB pinned at most, %d failures\n", name, staged, direct,
           pinned_most >> 20, bad);
    for (auto &kv : ctx.host_bufs)
        if (kv.second.ptr) (void)hipHostFree(kv.second.ptr);
    return bad;
}

int main() {
    int bad = 0;
    bad += scenario("past many halves", 4000, 100 << 10, 0.3, SIZE_MAX, false);
    bad += scenario("a stream that stands still", 400, 1 << 20, 0.0, SIZE_MAX, false);
    bad += scenario("large tables", 60, 40 << 20, 0.2, SIZE_MAX, false);
    bad += scenario("growth refused", 2000, 1 << 20, 0.01, 4 << 20, true);
    bad += scenario("no pinned memory at first", 400, 1 << 20, 0.3, 1, true);
    return bad ? 1 : 0;
}
