// Rules of the LU panels that host and device share: plain integer functions, so that they can
// be checked without a GPU.
#pragma once

#include <algorithm>
#include <cstddef>

#ifdef __HIPCC__
#define BH_HD __host__ __device__
#else
#define BH_HD
#endif

namespace bh {

constexpr int kPW = 32;                       // panel width
constexpr int kTsluT = 256;                   // threads of a tournament workgroup
constexpr int kTsluRows = 2 * kTsluT;         // its rows
constexpr int kTsluFan = kTsluRows / kPW;     // candidate sets merged per workgroup at most

// Groups that nl sets are merged in, as even as they get: the fewest levels, and among
// those groups of at most kTsluFan / 2 sets, whose rows take one register row per thread
// (21 us against 28 us for 32 columns).
BH_HD inline int tslu_groups(int nl)
{
    const int most = nl <= kTsluFan ? kTsluFan : (nl <= kTsluFan * kTsluFan / 2 ? kTsluFan / 2 : kTsluFan);
    return (nl + most - 1) / most;
}
BH_HD inline int tslu_fan(int nl) { return (nl + tslu_groups(nl) - 1) / tslu_groups(nl); }

// candidate sets of all levels of one tournament that begins with nl sets
inline size_t tslu_sets_from(int nl)
{
    for (size_t t = 0;; nl = tslu_groups(nl)) {
        t += nl;
        if (nl <= 1) return t;
    }
}

// Candidate sets that the tournaments of all panels of an n-row matrix take at most.  The
// panels get shorter and the sets of a shorter one can be more: 129 sets merge in 9 groups,
// 128 in 16.  (The group counters of a tournament are fewer than its sets.)
inline size_t tslu_sets(int n)
{
    size_t most = 1;
    for (int nl = (int)(((long long)n + kTsluRows - 1) / kTsluRows); nl > 0; --nl) most = std::max(most, tslu_sets_from(nl));
    return most;
}

// FP64 panels.  Row that a workgroup takes as column c's pivot: pos, the position of the best
// candidate that it read.  Without a candidate none moves, nor after a wait that ran out (late):
// the words read then are of an earlier column, or none, and their position may lie above the panel.
BH_HD inline int panel64_pivot(bool late, bool found, int pos, int c) { return found && !late ? pos : c; }

// The interchange of the positions c and p for a row at pos that has not been a pivot.  Workgroups
// that disagree on p (one of them late) leave two rows in one place: void, but inside the panel.
BH_HD inline void panel64_move(int &pos, bool &used, int c, int p)
{
    if (pos == p) {
        used = true;
        pos = c;
    } else if (pos == c) {
        pos = p;
    }
}

}  // namespace bh
