// Results from the device to the caller's memory.
#include <algorithm>
#include <cstring>
#include <thread>

#include "bh_internal.h"

namespace bh {

// A result leaves through pinned slots of the context, one per copying thread: the thread
// queues the device copy of its next piece, waits for it and stores (or adds) the piece into
// the caller's columns.  What bounds it is the caller's memory, whose pages are new as a rule:
// one thread fills them at a few GB/s, eight at about 29 GB/s (29 MB of complex floats:
// 1.0 ms; hipMemcpy2DAsync to pageable memory took 19.4 ms each way).  A piece is 1 MiB, long
// enough for the copy engine, short enough that a 1.6 MB result takes two threads.
namespace {

struct HostStage {
    static constexpr int kSlots = 8;
    static constexpr size_t kPiece = size_t(1) << 20;
    std::mutex mu;
    char *p = nullptr;
    hipEvent_t ev[kSlots] = {};
    ~HostStage() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (p) (void)hipHostFree(p);
    }
};

template <typename R>
void add_span(char *dst, const char *src, size_t bytes)
{
    // the caller's memory may be aligned to its bytes only
    for (size_t i = 0; i < bytes; i += sizeof(R)) {
        R a, b;
        std::memcpy(&a, dst + i, sizeof(R));
        std::memcpy(&b, src + i, sizeof(R));
        a += b;
        std::memcpy(dst + i, &a, sizeof(R));
    }
}

}  // namespace

void download_block(Ctx &ctx, const void *dev, void *host, size_t pitch, size_t width, int64_t cols, int es, bool add)
{
    const size_t total = width * (size_t)cols;
    if (total == 0) return;
    static std::mutex create;
    std::shared_ptr<void> held;
    {
        std::lock_guard<std::mutex> g(create);
        if (!ctx.host_stage) ctx.host_stage = std::make_shared<HostStage>();
        held = ctx.host_stage;
    }
    HostStage &st = *static_cast<HostStage *>(held.get());
    std::lock_guard<std::mutex> g(st.mu);
    constexpr size_t kBytes = HostStage::kSlots * HostStage::kPiece;
    std::vector<char> pageable;   // where no memory can be pinned: slower, for this call
    if (!st.p && hipHostMalloc((void **)&st.p, kBytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        st.p = nullptr;
        pageable.resize(kBytes);
    }
    char *const slots = st.p ? st.p : pageable.data();
    for (hipEvent_t &e : st.ev)
        if (!e) BH_CHECK_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    const int64_t pieces = (int64_t)((total + HostStage::kPiece - 1) / HostStage::kPiece);
    std::atomic<int64_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int slot) {
        hipError_t e = hipSetDevice(ctx.device);
        char *buf = slots + (size_t)slot * HostStage::kPiece;
        while (e == hipSuccess) {
            const int64_t k = next.fetch_add(1);
            if (k >= pieces) break;
            const size_t at = (size_t)k * HostStage::kPiece, len = std::min(HostStage::kPiece, total - at);
            e = hipMemcpyAsync(buf, (const char *)dev + at, len, hipMemcpyDeviceToHost, ctx.stream);
            if (e == hipSuccess) e = hipEventRecord(st.ev[slot], ctx.stream);
            if (e == hipSuccess) e = hipEventSynchronize(st.ev[slot]);
            if (e != hipSuccess) break;
            for (size_t o = 0; o < len;) {   // the piece's part of each column
                const size_t col = (at + o) / width, in = (at + o) % width, n = std::min(len - o, width - in);
                char *d = (char *)host + col * pitch + in;
                if (!add) std::memcpy(d, buf + o, n);
                else if (es == 8) add_span<double>(d, buf + o, n);
                else add_span<float>(d, buf + o, n);
                o += n;
            }
        }
        if (e != hipSuccess) failed.store((int)e);
    };
    const int want = (int)std::min<int64_t>({pieces, HostStage::kSlots, std::max(1u, std::thread::hardware_concurrency())});
    std::vector<std::thread> th;
    try {
        th.reserve(want);
        for (int t = 1; t < want; ++t) th.emplace_back(work, t);
    } catch (...) {
        // no more threads, or no memory for one: those that run take the pieces (an exception that
        // left them unjoined would end the process)
    }
    work(0);
    for (std::thread &t : th) t.join();
    if (failed.load() != (int)hipSuccess) {
        (void)hipStreamSynchronize(ctx.stream);   // no copy into the slots is left queued
        BH_CHECK_HIP((hipError_t)failed.load());
    }
}

}  // namespace bh
