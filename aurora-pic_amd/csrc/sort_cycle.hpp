// sort_cycle.hpp - when the adaptive policy sorts a species again, from its
// timings alone (no HIP: the host tests run it).
//
// The renewal rule: with a cycle cost C(n) = sort + pushes 1..n and pushes
// that slow down as the cycle ages, the long-run cost per step C(n)/n is
// least at the first n whose push exceeds C(n)/n.  The push compared is the
// mean of the last three timed pushes (timing noise).
#pragma once

#include <algorithm>
#include <cstdint>

namespace aurora {

// The sort in C(n) stands for the one that will end the cycle.  A new state's
// first cycle begins with a general sort (a radix sort, a permutation of every
// array and their allocations) and, unless the caller chose radix sorts, ends
// with a local one: there the sort counts for at most this many of the cycle's
// first push, the local sort's order of cost (2 pushes of 128^3 x 16, 5 of
// 256^2 x 32).  Taken at its own cost it kept a new state unsorted until its
// pushes took 1,640 us (430 freshly sorted) and 338 us (33).  Later cycles count
// the sort that began them in full, also a general one (the method is radix, or
// too many particles move too far for a local sort): the next costs the same.
constexpr double kLocalSortPushes = 4.0;

struct SortCycle {
    double sort_ms = 0.0;         // the sort that began the cycle; 0: not timed
    bool first = false;           // a new state's
    double first_push_ms = 0.0;   // the cycle's first timed push
    double push_ms = 0.0;         // its timed pushes
    int64_t pushes = 0;
    double recent_ms[3] = {0.0, 0.0, 0.0};   // the last three

    // a sort has been queued; its time, if it is timed, comes later (sort_ms)
    void begin(bool first_cycle) {
        sort_ms = 0.0;
        first = first_cycle;
        push_ms = 0.0;
        pushes = 0;
    }
    void pushed(double ms) {
        if (pushes == 0) first_push_ms = ms;
        push_ms += ms;
        recent_ms[2] = recent_ms[1];
        recent_ms[1] = recent_ms[0];
        recent_ms[0] = ms;
        ++pushes;
    }
    // local: the method is the local sort
    bool due(bool local) const {
        if (pushes < 3) return false;
        const double recent = (recent_ms[0] + recent_ms[1] + recent_ms[2]) / 3.0;
        const double sort =
            first && local ? std::min(sort_ms, kLocalSortPushes * first_push_ms) : sort_ms;
        return recent * static_cast<double>(pushes) > sort + push_ms;
    }
};

}  // namespace aurora
