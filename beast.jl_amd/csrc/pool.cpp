// Pool of large device buffers (Ctx::pool).
#include "bh_internal.h"

namespace bh {

namespace {
constexpr size_t kPoolMinBytes = size_t(1) << 20;   // smaller buffers are freed at once
}

PoolMem pool_alloc(Ctx &ctx, size_t bytes)
{
    {
        std::lock_guard<std::mutex> g(ctx.pool_mu);
        int best = -1;
        for (int i = 0; i < (int)ctx.pool.size(); ++i) {
            const size_t b = ctx.pool[i].bytes;
            if (b >= bytes && b - bytes <= bytes / 4 && (best < 0 || b < ctx.pool[best].bytes)) best = i;
        }
        if (best >= 0) {
            const PoolMem m = ctx.pool[best];
            ctx.pool_bytes -= m.bytes;
            ctx.pool.erase(ctx.pool.begin() + best);
            return m;
        }
    }
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) {   // pooled memory may be what is missing
        (void)hipGetLastError();
        pool_trim(ctx, 0);
        e = hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
        set_error("hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(e));
        throw Error{BH_ERR_OOM};
    }
    return {p, bytes};
}

void pool_free(Ctx &ctx, PoolMem m)
{
    if (!m.p) return;
    std::vector<void *> drop;
    {
        std::lock_guard<std::mutex> g(ctx.pool_mu);
        if (m.bytes < kPoolMinBytes || m.bytes > ctx.pool_limit) {
            drop.push_back(m.p);
        } else {
            ctx.pool.push_back(m);
            ctx.pool_bytes += m.bytes;
            while (ctx.pool_bytes > ctx.pool_limit) {   // oldest first
                drop.push_back(ctx.pool.front().p);
                ctx.pool_bytes -= ctx.pool.front().bytes;
                ctx.pool.erase(ctx.pool.begin());
            }
        }
    }
    for (void *q : drop) (void)hipFree(q);
}

void pool_trim(Ctx &ctx, size_t keep_bytes)
{
    std::vector<void *> drop;
    {
        std::lock_guard<std::mutex> g(ctx.pool_mu);
        while (ctx.pool_bytes > keep_bytes && !ctx.pool.empty()) {
            drop.push_back(ctx.pool.front().p);
            ctx.pool_bytes -= ctx.pool.front().bytes;
            ctx.pool.erase(ctx.pool.begin());
        }
    }
    for (void *q : drop) (void)hipFree(q);
}

}  // namespace bh
