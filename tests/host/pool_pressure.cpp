// Allocations of every kind against what the pools of the device's contexts hold: a call that
// fits without them is served, one that does not is refused with the pools of its device empty.
#include "hip_stub.h"
#include "pool.cpp"

using namespace bh;

namespace {

constexpr size_t kMiB = size_t(1) << 20;

void fill(Ctx &ctx, size_t mib)
{
    PoolBuf<char> b(ctx, mib * kMiB);
    b.done();
}

template <typename F>
int code(F f)
{
    try {
        f();
    } catch (const Error &e) {
        return e.code;
    }
    return BH_OK;
}

}  // namespace

int main()
{
    stub::budget = 1000 * kMiB;
    Ctx a, b, other;
    other.device = 1;
    for (Ctx *c : {&a, &b, &other}) pool_register(c);
    auto refill = [&] {
        for (Ctx *c : {&a, &b, &other}) pool_trim(*c, 0);
        fill(a, 400);
        fill(b, 300);
        fill(other, 100);
    };
    refill();
    {
        DevBuf<char> w;
        if (code([&] { w.alloc(500 * kMiB); }) != BH_OK) return std::printf("plain buffer refused\n"), 1;
        if (other.pool_bytes != 100 * kMiB) return std::printf("another device's pool was freed\n"), 1;
    }
    refill();
    {
        DevBuf<double> w;
        if (code([&] { w.ensure(850 * kMiB / 8); }) != BH_OK) return std::printf("both pools' memory refused\n"), 1;
    }
    refill();
    {
        PoolBuf<char> w;   // of a context whose own pool is not enough
        if (code([&] { w.alloc(b, 650 * kMiB); }) != BH_OK) return std::printf("pooled buffer refused\n"), 1;
        w.done();
    }
    refill();
    {
        DevBuf<char> w;
        if (code([&] { w.alloc(950 * kMiB); }) != BH_ERR_OOM || w.p || w.n) return std::printf("expected OOM\n"), 1;
        if (a.pool_bytes || b.pool_bytes) return std::printf("pools kept\n"), 1;
    }
    refill();
    pool_trim(b, 0);
    pool_unregister(&b);   // a context that has ended is not looked at
    {
        DevBuf<char> w;
        if (code([&] { w.alloc(700 * kMiB); }) != BH_OK) return std::printf("refused\n"), 1;
    }
    pool_unregister(&a);
    pool_trim(other, 0);
    pool_unregister(&other);
    return stub::live_bytes == 0 ? 0 : (std::printf("not all freed\n"), 1);
}
