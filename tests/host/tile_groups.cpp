// Groups of dof tiles: every tile in one group, each group's cells once and those of its tiles,
// places that lead back to the tile's cells, and no group beyond its limit that could be smaller.
#include <climits>
#include <cstdio>
#include <random>
#include <set>

#include "tile_groups.h"

using namespace bh;

int main()
{
    std::mt19937 rng(3);
    for (int round = 0; round < 600; ++round) {
        const int nf = 1 + (int)(rng() % 700), nt = (int)(rng() % 12);
        std::vector<int> ptr(1, 0), cells;
        for (int t = 0; t < nt; ++t) {
            std::set<int> s;   // tiles without shapes, of neighbours, of scattered dofs
            const int kind = (int)(rng() % 3), count = kind ? (int)(rng() % 129) : 0, base = (int)(rng() % nf);
            for (int i = 0; i < count; ++i) s.insert(kind == 1 ? (base + i) % nf : (int)(rng() % nf));
            cells.insert(cells.end(), s.begin(), s.end());
            ptr.push_back((int)cells.size());
        }
        const int pad = rng() % 2 ? 64 : 1;
        const long long limits[] = {0, 64, 200, 1000, LLONG_MAX}, limit = limits[rng() % 5];
        const TileGroups r = tile_groups(ptr, cells, nf, pad, limit);
        int next = 0;
        size_t listed = 0;
        long long most = 0;
        for (const TileGroup &g : r.groups) {
            if (g.t0 != next || g.t1 <= g.t0 || (size_t)g.c0 != listed) return std::printf("groups out of order\n"), 1;
            std::set<int> want;
            for (int k = ptr[g.t0]; k < ptr[g.t1]; ++k) {
                want.insert(cells[k]);
                if (r.loc[k] < 0 || r.loc[k] >= g.n || r.cells[g.c0 + r.loc[k]] != cells[k]) return std::printf("place\n"), 1;
            }
            if ((int)want.size() != g.n) return std::printf("%d cells for %d\n", g.n, (int)want.size()), 1;
            const long long padded = (g.n + pad - 1) / pad * pad;
            if (padded > limit && g.t1 - g.t0 > 1) return std::printf("a group beyond its limit\n"), 1;
            if (limit == LLONG_MAX && r.groups.size() > 1) return std::printf("split without need\n"), 1;
            most = std::max(most, padded);
            next = g.t1;
            listed += g.n;
        }
        if (next != nt || r.most != most || listed != r.cells.size()) return std::printf("tiles left over\n"), 1;
    }
    return 0;
}
