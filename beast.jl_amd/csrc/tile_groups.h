// Dof tiles in groups whose cells are listed once (host).
#pragma once

#include <algorithm>
#include <vector>

namespace bh {

struct TileGroup {
    int t0, t1;   // tiles [t0, t1)
    int c0, n;    // its cells, [c0, c0 + n) of the list
};

struct TileGroups {
    std::vector<TileGroup> groups;
    std::vector<int> cells;   // the groups' cells, each once per group
    std::vector<int> loc;     // for each entry of the tiles' cell lists, the cell's place in its group
    long long most = 0;       // most cells of a group, padded
};

// Tile t touches the cells tcells[tptr[t] .. tptr[t + 1]), each once, out of nf.  Consecutive tiles
// form a group while its cells, padded to a multiple of `pad`, stay within `limit`; a group has
// at least one tile.
inline TileGroups tile_groups(const std::vector<int> &tptr, const std::vector<int> &tcells, long long nf, int pad,
                              long long limit)
{
    TileGroups r;
    r.loc.resize(tcells.size());
    auto padded = [&](long long n) { return (n + pad - 1) / pad * pad; };
    std::vector<int> at(nf, -1);   // place in the list of the cell's last group
    const int nt = (int)tptr.size() - 1;
    for (int t = 0; t < nt;) {
        TileGroup g{t, t, (int)r.cells.size(), 0};
        for (; t < nt; ++t) {
            int more = 0;
            for (int k = tptr[t]; k < tptr[t + 1]; ++k) more += at[tcells[k]] < g.c0;
            if (t > g.t0 && padded(g.n + more) > limit) break;
            for (int k = tptr[t]; k < tptr[t + 1]; ++k) {
                const int c = tcells[k];
                if (at[c] < g.c0) {
                    at[c] = g.c0 + g.n++;
                    r.cells.push_back(c);
                }
                r.loc[k] = at[c] - g.c0;
            }
        }
        g.t1 = t;
        r.most = std::max(r.most, padded(g.n));
        r.groups.push_back(g);
    }
    return r;
}

}  // namespace bh
