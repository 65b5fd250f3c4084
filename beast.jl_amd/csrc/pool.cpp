// Pool of large device buffers (Ctx::pool).
#include <set>

#include "bh_internal.h"

namespace bh {

namespace {
constexpr size_t kPoolMinBytes = size_t(1) << 20;   // smaller buffers are freed at once

// never destroyed: a context may outlive the library's static objects
std::mutex &registry_mutex()
{
    static std::mutex &m = *new std::mutex;
    return m;
}
std::set<Ctx *> &registry()
{
    static std::set<Ctx *> &s = *new std::set<Ctx *>;
    return s;
}
}  // namespace

void pool_register(Ctx *ctx)
{
    std::lock_guard<std::mutex> g(registry_mutex());
    registry().insert(ctx);
}

void pool_unregister(Ctx *ctx)
{
    std::lock_guard<std::mutex> g(registry_mutex());
    registry().erase(ctx);
}

void *device_malloc(size_t bytes)
{
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        int device = -1;
        BH_CHECK_HIP(hipGetDevice(&device));
        {
            std::lock_guard<std::mutex> g(registry_mutex());
            for (Ctx *c : registry())
                if (c->device == device) pool_trim(*c, 0);
        }
        e = hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
        set_error("hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(e));
        throw Error{BH_ERR_OOM};
    }
    return p;
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
    return {device_malloc(bytes), bytes};
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
