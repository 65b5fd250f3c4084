// Results to columns of the caller's memory, stored and added, at sizes around the pieces; and
// where memory or threads run out on the way: the block still arrives, or the call says why not.
#include <cstdlib>
#include <cstring>
#include <new>
#include <numeric>

#include "hip_stub.h"

namespace {
std::atomic<int> spare{-1};   // allocations that are still granted (-1: all)
std::atomic<int> copies_left{1 << 30};
bool pin = true;
}  // namespace

void *operator new(size_t n)
{
    if (spare >= 0 && spare-- <= 0) {
        spare = 0;
        throw std::bad_alloc();
    }
    return std::malloc(n ? n : 1);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return pin && (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (copies_left-- <= 0) return hipErrorUnknown;
    return std::memcpy(d, s, n), hipSuccess;
}
}

#include "download.cpp"

using namespace bh;

namespace {

// rows x cols complex entries of two R each into columns `pad` entries longer; 0: as expected
template <typename R>
int run(Ctx &ctx, int64_t rows, int64_t cols, int64_t pad, bool add)
{
    std::vector<R> dev(2 * rows * cols), host(2 * (rows + pad) * cols), want;
    std::iota(dev.begin(), dev.end(), R(1));
    std::iota(host.begin(), host.end(), R(5));
    want = host;
    for (int64_t c = 0; c < cols; ++c)
        for (int64_t i = 0; i < 2 * rows; ++i) {
            R &w = want[2 * (rows + pad) * c + i];
            w = dev[2 * rows * c + i] + (add ? w : R(0));
        }
    try {
        download_block(ctx, dev.data(), host.data(), 2 * (rows + pad) * sizeof(R), 2 * rows * sizeof(R), cols, (int)sizeof(R), add);
    } catch (const Error &e) {
        return e.code;
    }
    return host == want ? 0 : (std::printf("%lld x %lld, pad %lld, add %d\n", (long long)rows, (long long)cols, (long long)pad, add), 1);
}

}  // namespace

int main()
{
    Ctx ctx;
    for (bool add : {false, true})
        for (int64_t pad : {0, 3}) {
            for (auto rc : {std::pair<int64_t, int64_t>{1, 1}, {65536, 1}, {65537, 3}, {7, 40000}, {300, 900}, {200000, 2}})
                if (run<double>(ctx, rc.first, rc.second, pad, add) || run<float>(ctx, rc.first, rc.second, pad, add)) return 1;
        }
    // no memory to pin, then some
    {
        Ctx fresh;
        pin = false;
        if (run<double>(fresh, 700, 1000, 5, false) || run<float>(fresh, 700, 1000, 5, true)) return 1;
        pin = true;
        if (run<double>(fresh, 700, 1000, 5, true)) return 1;
    }
    // memory that runs out while the threads are made
    for (int grant = 0; grant < 12; ++grant) {
        std::vector<double> dev(2 * 700000, 2.0), host(dev.size(), 0.0);
        spare = grant;
        download_block(ctx, dev.data(), host.data(), 16 * 700, 16 * 700, 1000, 8, true);
        spare = -1;
        if (host != dev) return std::printf("%d allocations: wrong block\n", grant), 1;
    }
    // a copy that fails
    copies_left = 3;
    if (run<double>(ctx, 700, 1000, 0, false) != BH_ERR_HIP) return std::printf("expected an error\n"), 1;
    copies_left = 1 << 30;
    return run<double>(ctx, 700, 1000, 0, false);
}
