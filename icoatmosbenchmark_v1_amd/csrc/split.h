// How a kernel's levels are divided among its work-groups (host arithmetic only).
#pragma once

#include <algorithm>

namespace nicam {

// The shortest march that makes no more ranges of kall levels than kper levels
// each do: the levels of a range spread over all of them.
inline int even_split(int kall, int kper)
{
    const int nkr = (kall + std::min(kper, kall) - 1) / std::min(kper, kall);
    return (kall + nkr - 1) / nkr;
}

// Levels per work-group, at most cap, of a kernel whose work-groups march up a
// range of levels: base columns of work-groups over kall levels, slots of them
// on the chip at a time, each paying about one and a half levels to start.  The
// launch costs about rounds * (levels + 1.5): the least of that, the longer march
// on a tie.  An estimate: the kernels say how near it comes.
inline int level_split(long base, int kall, long slots, int cap)
{
    int best = 0;
    double cost = 0.0;
    for (int kper = std::min(cap, kall); kper >= 1; --kper) {
        kper = even_split(kall, kper);
        const int nkr = (kall + kper - 1) / kper;
        const double t = (double)((base * nkr + slots - 1) / slots) * (kper + 1.5);
        if (best == 0 || t < cost) {
            cost = t;
            best = kper;
        }
    }
    return best;
}

}  // namespace nicam
