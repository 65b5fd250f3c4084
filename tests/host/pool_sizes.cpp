// The pool's account against what is allocated: buffers reused by ever smaller requests keep
// their whole size, through every kind of owner.
#include "hip_stub.h"
#include "pool.cpp"

using namespace bh;

int main()
{
    constexpr size_t kMiB = size_t(1) << 20;
    Ctx ctx;
    ctx.pool_limit = 1000 * kMiB;
    auto bad = [&](const char *what, size_t want) {
        if (ctx.pool_bytes == want && stub::live_bytes == want) return false;
        std::printf("%s: pool says %zu, allocated %zu, expected %zu\n", what, ctx.pool_bytes, stub::live_bytes, want);
        return true;
    };
    for (size_t mib : {100, 81, 80}) {
        PoolBuf<char> b(ctx, mib * kMiB);
        b.done();
        if (bad("workspace", 100 * kMiB)) return 1;
    }
    for (size_t mib : {99, 80}) {
        DevBuf<double> b;
        pool_alloc(ctx, b, mib * kMiB / 8);
        DevBuf<double> c(std::move(b)), d;
        d = std::move(c);
        pool_release(ctx, d);
        if (b.p || c.p || bad("matrix", 100 * kMiB)) return 1;
    }
    {
        PoolBuf<char> b(ctx, 79 * kMiB);   // 100 is more than 5/4 of it
        b.done();
        if (bad("a second one", 179 * kMiB)) return 1;
    }
    // the limit holds for what is really there: 20 times, each a little smaller than the one before
    ctx.pool_limit = 300 * kMiB;
    std::vector<PoolBuf<char>> w(4);
    for (int i = 0; i < 20; ++i) {
        for (size_t k = 0; k < w.size(); ++k) w[k].alloc(ctx, (90 - i) * kMiB);
        for (auto &b : w) b.done();
        if (ctx.pool_bytes != stub::live_bytes || stub::live_bytes > ctx.pool_limit)
            return std::printf("round %d: pool says %zu, allocated %zu\n", i, ctx.pool_bytes, stub::live_bytes), 1;
    }
    DevBuf<char> own(7 * kMiB);   // from no pool
    pool_release(ctx, own);
    pool_trim(ctx, 0);
    return stub::live_bytes == 0 && ctx.pool_bytes == 0 ? 0 : (std::printf("not all freed\n"), 1);
}
