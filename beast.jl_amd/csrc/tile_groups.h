// Dof tiles in groups whose cells are listed once (host).
#pragma once

#include <algorithm>
#include <climits>
#include <cstddef>
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

// The row and column groups of a matrix formed from pair blocks of `entry` bytes: all columns
// and as many row tiles as fit `budget` bytes of blocks; the columns are split too where one row
// tile with all of them is too much.  bytes: the blocks of the largest pair of groups, above the
// budget only where a row tile with a column tile is.
struct PairGroups {
    TileGroups rows, cols;
    size_t bytes = 0;
};

inline PairGroups pair_groups(const std::vector<int> &rptr, const std::vector<int> &rcells, long long rnf,
                              const std::vector<int> &cptr, const std::vector<int> &ccells, long long cnf, size_t entry,
                              size_t budget)
{
    constexpr int kRowPad = 64;   // a wave's test cells
    const long long blocks = (long long)(budget / entry);
    PairGroups r;
    r.cols = tile_groups(cptr, ccells, cnf, 1, LLONG_MAX);
    r.rows = tile_groups(rptr, rcells, rnf, kRowPad, r.cols.most ? blocks / r.cols.most : LLONG_MAX);
    if (r.rows.most * r.cols.most > blocks) r.cols = tile_groups(cptr, ccells, cnf, 1, blocks / r.rows.most);
    r.bytes = (size_t)(r.rows.most * r.cols.most) * entry;
    return r;
}

// The groups for the largest of budget, budget / 4, .. whose blocks alloc(bytes) has room for
// (false: none); false if not even the smallest groups do.
template <typename Plan, typename Alloc>
bool shrink_to_fit(PairGroups &r, size_t budget, const Plan &plan, const Alloc &alloc)
{
    for (;; budget /= 4) {
        r = plan(budget);
        if (alloc(r.bytes)) return true;
        if (r.bytes > budget) return false;   // no smaller groups
    }
}

}  // namespace bh
