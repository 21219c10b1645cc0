// mh_stage.hip -- large copies between pageable host memory and the device.
//
// The runtime's own copy of pageable memory stages it through pinned memory on
// one host thread, and images that have to be packed first are copied twice.
// Here a few threads each fill (or empty) their own pinned buffers, the copy
// of one running while the other is filled, and take the images from where
// they lie.  The bound is the link, 57 GB/s in one copy (37 in pieces of 1 MiB).
//
// Measured: a library of 2,000 images of four sizes (37 MB) from a list of
// arrays 15.0 -> 2.8 ms, of which 1.2 are the caller's list; 1,500 images of
// one size (74 MB) 4.0 -> 2.5 ms.  Three threads with 4 MiB buffers: 2.4 ms
// for those 74 MB; 1 MiB buffers 3.0, 256 KiB 6.2; four or six threads the same.
//
// Starting the threads takes 30-60 us and the runtime keeps buffers it has
// copied pinned, so one buffer is only staged from the size where that is no
// slower even for a buffer copied again and again (us, runtime and staged):
// up 6 MiB 228 and 318, 16 MiB 520 and 550, 24 MiB 750 and 750, 48 MiB 1,770
// and 1,400 (buffers not seen before: equal at 12 MiB); down 4 MiB 226 and 240,
// 6 MiB 341 and 290, 64 MiB 3,850 and 1,640.  Images to be gathered come
// through here whatever they sum to, below kLeastShared on one thread: 0.8 MiB
// 137 us (chunks of 512 KiB 161, three threads 175), 3.6 MiB 262 (282, 325), 4.8
// MiB 300 (305, 340).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "mh_internal.hpp"

namespace mh {
namespace host {

namespace {
constexpr size_t kBuffer = (size_t)4 << 20, kLeastChunk = (size_t)1 << 20;
constexpr size_t kLeastUp = (size_t)24 << 20, kLeastDown = (size_t)6 << 20,
                 kLeastShared = (size_t)5 << 20;

// Bytes a buffer is filled with at a time: two rounds a thread for a copy of
// a few MB, whole buffers for a large one (a copy costs 10 us by itself).
size_t chunk_of(size_t total) {
    const size_t share = (total / (2 * kStageThreads) + 0xffff) & ~(size_t)0xffff;
    return std::min(kBuffer, std::max(kLeastChunk, share));
}

int stage_ready(StageBuf& b) {
    if (!b.copied) HIPCHK(hipEventCreateWithFlags(&b.copied, hipEventDisableTiming));
    if (!b.p) HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&b.p), kBuffer, hipHostMallocDefault));
    return MH_OK;
}

// f(thread) on kStageThreads threads, this one among them (on this one alone
// below kLeastShared bytes), and the first error of any of them.  A thread
// that cannot be started is done without: the threads share the chunks.
template <typename F>
int on_threads(mh_context* ctx, size_t total, size_t chunks, F&& f) {
    int rc[kStageThreads] = {};
    std::string text[kStageThreads];
    std::thread helpers[kStageThreads];
    for (int t = 1; t < kStageThreads && (size_t)t < chunks && total >= kLeastShared; ++t) {
        try {
            helpers[t] = std::thread([&, t]() {
                rc[t] = set_device(ctx);
                if (!rc[t]) rc[t] = f(t);
                if (rc[t]) text[t] = mh_last_error();
            });
        } catch (...) {
            break;
        }
    }
    rc[0] = f(0);
    for (std::thread& h : helpers)
        if (h.joinable()) h.join();
    if (rc[0]) return rc[0];
    for (int t = 1; t < kStageThreads; ++t)
        if (rc[t]) return fail(rc[t], "%s", text[t].c_str());
    return MH_OK;
}

// Memory that the runtime knows is copied from or to directly.
bool known_to_runtime(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}
}  // namespace

bool staged_up(const void* host, size_t bytes) {
    return bytes >= kLeastUp && !known_to_runtime(host);
}
bool staged_down(const void* host, size_t bytes) {
    return bytes >= kLeastDown && !known_to_runtime(host);
}

int stage_upload(mh_context* ctx, uint8_t* dst, const std::vector<HostSpan>& spans) {
    std::vector<size_t> at(spans.size() + 1, 0);  // where each span goes
    for (size_t i = 0; i < spans.size(); ++i) at[i + 1] = at[i] + spans[i].bytes;
    const size_t total = at.back(), chunk = chunk_of(total), chunks = (total + chunk - 1) / chunk;
    std::lock_guard<std::mutex> g(ctx->stage_mu);
    std::atomic<size_t> next{0};
    const int rc = on_threads(ctx, total, chunks, [&](int t) -> int {
        for (int k = 0;; k ^= 1) {
            const size_t c = next.fetch_add(1);
            if (c >= chunks) return MH_OK;
            StageBuf& b = ctx->stage[2 * t + k];
            CHK(stage_ready(b));
            HIPCHK(hipEventSynchronize(b.copied));  // (its last copy; none: returns at once)
            const size_t lo = c * chunk, hi = std::min(total, lo + chunk);
            size_t i = (size_t)(std::upper_bound(at.begin(), at.end(), lo) - at.begin()) - 1;
            for (size_t o = lo; o < hi; ++i) {
                const size_t end = std::min(hi, at[i + 1]);
                if (end > o) memcpy(b.p + (o - lo), spans[i].p + (o - at[i]), end - o);
                o = std::max(o, end);
            }
            HIPCHK(hipMemcpyAsync(dst + lo, b.p, hi - lo, hipMemcpyHostToDevice, ctx->stream));
            HIPCHK(hipEventRecord(b.copied, ctx->stream));
        }
    });
    if (!rc) return MH_OK;
    // no pinned memory to be had, perhaps: all of it by the runtime
    (void)hipGetLastError();
    for (size_t i = 0; i < spans.size(); ++i)
        if (spans[i].bytes)
            HIPCHK(hipMemcpyAsync(dst + at[i], spans[i].p, spans[i].bytes, hipMemcpyHostToDevice,
                                  ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MH_OK;
}

int stage_download(mh_context* ctx, uint8_t* host, const uint8_t* src, size_t total) {
    const size_t chunk = chunk_of(total), chunks = (total + chunk - 1) / chunk;
    std::lock_guard<std::mutex> g(ctx->stage_mu);
    std::atomic<size_t> next{0};
    const int rc = on_threads(ctx, total, chunks, [&](int t) -> int {
        size_t mine[2];
        bool busy[2] = {false, false};
        for (int k = 0;; k ^= 1) {
            StageBuf& b = ctx->stage[2 * t + k];
            if (busy[k]) {
                HIPCHK(hipEventSynchronize(b.copied));
                const size_t lo = mine[k] * chunk;
                memcpy(host + lo, b.p, std::min(total, lo + chunk) - lo);
                busy[k] = false;
            }
            const size_t c = next.fetch_add(1);
            if (c >= chunks) {
                if (!busy[k ^ 1]) return MH_OK;
                continue;
            }
            CHK(stage_ready(b));
            HIPCHK(hipEventSynchronize(b.copied));
            const size_t lo = c * chunk;
            HIPCHK(hipMemcpyAsync(b.p, src + lo, std::min(total, lo + chunk) - lo,
                                  hipMemcpyDeviceToHost, ctx->stream));
            HIPCHK(hipEventRecord(b.copied, ctx->stream));
            mine[k] = c;
            busy[k] = true;
        }
    });
    if (!rc) return MH_OK;
    (void)hipGetLastError();
    HIPCHK(hipMemcpyAsync(host, src, total, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MH_OK;
}

void stage_release(mh_context* ctx) {
    for (StageBuf& b : ctx->stage) {
        if (b.copied) hipEventDestroy(b.copied);
        if (b.p) hipHostFree(b.p);
        b = StageBuf{};
    }
}

}  // namespace host
}  // namespace mh
