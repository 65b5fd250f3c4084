// Walks the tournaments of every panel as k_tslu_panel numbers their sets and counters and
// compares with what is allocated for the matrix.
#include <cstdio>
#include <vector>

#include "lu_rules.h"

using namespace bh;

int main()
{
    const int most = 1024;   // first-stage sets: up to 524,288 rows
    for (int count = 1; count <= most; ++count) {
        // the fewest and the most rows that give `count` sets
        const size_t sets = tslu_sets((count - 1) * kTsluRows + 1);
        if (sets != tslu_sets(count * kTsluRows)) return std::printf("%d: row counts of one set count differ\n", count), 1;
        // every shorter panel was walked against its own, smaller allocation
        if (count > 1 && sets < tslu_sets((count - 1) * kTsluRows)) return std::printf("%d sets: fewer than before\n", count), 1;
        int nl = count, off = 0, coff = 0;
        while (nl > 1) {
            const int fan = tslu_fan(nl), groups = tslu_groups(nl);
            std::vector<int> members(groups, 0);
            for (int g = 0; g < nl; ++g) {
                if ((size_t)(off + g) >= sets) return std::printf("%d sets: set %d of %zu\n", count, off + g, sets), 1;
                if (g / fan >= groups || (size_t)(coff + g / fan) >= sets) return std::printf("%d sets: counter %d\n", count, coff + g / fan), 1;
                ++members[g / fan];
            }
            for (int m : members)
                if (m < 1 || m > kTsluFan) return std::printf("%d sets: a group of %d\n", count, m), 1;
            coff += groups;
            off += nl;
            nl = groups;
        }
        if ((size_t)off >= sets) return std::printf("%d sets: last set %d of %zu\n", count, off, sets), 1;
    }
    return 0;
}
