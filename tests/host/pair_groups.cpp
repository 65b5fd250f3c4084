// Pair-block groups where memory is short: the search ends, with blocks that fit whatever is
// left, or with none where a row tile and a column tile do not fit.
#include <cstdio>
#include <random>

#include "tile_groups.h"

using namespace bh;

int main()
{
    std::mt19937 rng(5);
    constexpr size_t kEntry = 144;
    for (int round = 0; round < 300; ++round) {
        // tiles of neighbours, some of dofs without shapes: first, last or between
        const int nf = 2000;
        auto tiles = [&](std::vector<int> &ptr, std::vector<int> &cells, int nt) {
            ptr.assign(1, 0);
            cells.clear();
            const int empty = (int)(rng() % 4), base = (int)(rng() % nf);
            for (int t = 0; t < nt; ++t) {
                const bool none = (empty == 1 && t < 3) || (empty == 2 && t > nt - 3) || (empty == 3 && t % 2);
                for (int i = 0; i < (none ? 0 : 128); ++i) cells.push_back((base + 60 * t + i) % nf);
                ptr.push_back((int)cells.size());
            }
        };
        std::vector<int> rp, rc, cp, cc;
        tiles(rp, rc, 1 + (int)(rng() % 20));
        tiles(cp, cc, 1 + (int)(rng() % 20));
        const PairGroups least = pair_groups(rp, rc, nf, cp, cc, nf, kEntry, 0);
        const PairGroups all = pair_groups(rp, rc, nf, cp, cc, nf, kEntry, size_t(2) << 30);
        if (all.rows.groups.size() != 1 || all.cols.groups.size() != 1) return std::printf("split without need\n"), 1;
        if (least.bytes > 128u * 128u * kEntry) return std::printf("smallest groups take %zu bytes\n", least.bytes), 1;
        const size_t rooms[] = {0, least.bytes ? least.bytes - 1 : 0, least.bytes, 3 * least.bytes, all.bytes / 5, all.bytes};
        for (size_t room : rooms) {
            int tries = 0;
            PairGroups r;
            const bool ok = shrink_to_fit(
                r, size_t(2) << 30, [&](size_t budget) { return pair_groups(rp, rc, nf, cp, cc, nf, kEntry, budget); },
                [&](size_t bytes) { return ++tries < 100 && bytes <= room; });
            if (tries >= 100) return std::printf("no end: room for %zu, %zu needed\n", room, least.bytes), 1;
            if (ok != (least.bytes <= room)) return std::printf("room for %zu, %zu needed: %d\n", room, least.bytes, ok), 1;
            if (!ok) continue;
            for (const TileGroup &g : r.rows.groups)
                for (const TileGroup &h : r.cols.groups)
                    if (g.n > r.rows.most || (size_t)(r.rows.most * h.n) * kEntry > room) return std::printf("blocks beyond the room\n"), 1;
            if (r.rows.groups.back().t1 != (int)rp.size() - 1 || r.cols.groups.back().t1 != (int)cp.size() - 1)
                return std::printf("tiles left over\n"), 1;
        }
    }
    return 0;
}
