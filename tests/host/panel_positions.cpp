// Rows of an FP64 panel under interchanges that its workgroups do not agree on: some give up a
// wait and have read whatever the slots held, an earlier panel's position or none.  Every row
// stays at a row of the panel [k0, n), so the rows and the row moves are stored inside the matrix.
#include <cstdio>
#include <random>
#include <vector>

#include "lu_rules.h"

using namespace bh;

int main()
{
    std::mt19937 rng(1);
    for (int round = 0; round < 2000; ++round) {
        const int rows_per = 8, G = 2 + (int)(rng() % 6), k0 = 32 * (int)(rng() % 4), n = k0 + kPW + (int)(rng() % (rows_per * G));
        const bool sound = round % 2 == 0;   // nobody late: a permutation results
        std::vector<int> pos(n - k0);
        std::vector<char> used(n - k0, 0);
        for (int r = 0; r < n - k0; ++r) pos[r] = k0 + r;
        for (int j = 0; j < kPW; ++j) {
            const int c = k0 + j;
            std::vector<int> cand;   // positions of the rows left
            for (int r = 0; r < n - k0; ++r)
                if (!used[r]) cand.push_back(pos[r]);
            const int agreed = cand.empty() ? c : cand[rng() % cand.size()];
            std::vector<int> p(G);
            for (int g = 0; g < G; ++g) {
                const bool late = !sound && rng() % 4 == 0;
                p[g] = panel64_pivot(late, !cand.empty(), late ? (int)(rng() % n) : agreed, c);
            }
            for (int r = 0; r < n - k0; ++r) {
                bool u = used[r];
                if (!u) panel64_move(pos[r], u, c, p[r % G]);
                used[r] = u;
                if (pos[r] < k0 || pos[r] >= n) return std::printf("row %d of [%d, %d) at %d\n", k0 + r, k0, n, pos[r]), 1;
            }
        }
        if (!sound) continue;
        std::vector<char> seen(n - k0, 0);
        for (int at : pos) seen[at - k0] = 1;
        for (char s : seen)
            if (!s) return std::printf("no permutation\n"), 1;
    }
    return 0;
}
