// The host loop of one PCG solve: in which groups its iterations are launched
// and when the host reads the state back. Plain C++, so that the loop runs
// against a simulated device as well.
#pragma once
#include <algorithm>

namespace ifl {

// One strip of up to 128 columns. Level 4 in groups as for larger grids / so:
// 96x64 3176 / 3107 us, 128x64 3714 / 3708, 160x64 4219 / 4222, 200x64
// 5090 / 5113.
inline bool short_iterations(int w, int nstrips) { return nstrips == 1 && w <= 128; }

// Launches iterations 0, 1, ... of a solve that is not over at its entry,
// until the state says that it is or `limit` have been launched. `D` supplies
//   int launch(int it)             queues iteration `it`
//   int post(int slot)             queues a copy of the state after all that
//                                  is queued into host mirror `slot` (0 or 1)
//   int wait(int slot, bool all)   until the copy in `slot` has landed (all:
//                                  until everything queued has run)
//   bool over(int slot)            the mirror's state is the end of the solve
//   bool seen_over(int slot)       the same, read while the copy may still be
//                                  on its way: a hint
// and returns 0 or an error from the first three, which ends the loop. On
// entry mirror 1 holds the state before iteration 0; *last is the mirror that
// holds the final state.
//
// Iterations go out in groups of 4, after 16 of 8; past the exit a launch
// returns at once (~10 us for an iteration's). The host waits for the first
// group's state, since many solves end there, and then stays one group ahead
// of the state it waits for, so the device has work while the host reads. A
// solve that works for 75 iterations (128^2) launches 88; groups doubling
// from 4 to 64 launched 124 and left the device idle at every read.
//
// On a small grid of one strip (`short_its`) an iteration runs for
// about as long as the host takes to launch it, so every launch past the exit
// delays the solve: there the groups stay at 4, and before each launch of a
// group ahead the host looks whether the group before has ended the solve.
// us per solve with the groups above, so, and with doubling groups: level 4
// at 16x16 (25 iterations) 983, 902 and 922; level 7 at 16x16 (27) 926, 840
// and 828; level 3 at 33x33 (26) 949, 869 and 976. Elsewhere the device is the
// slower side, the look finds nothing and the further copies gain nothing.
template <class D>
int run_groups(D& d, int limit, bool short_its, int* last) {
    int launched = 0, group = 0;
    bool ahead = false;  // a group beyond the state waited for is in flight
    *last = 1;
    auto launch_group = [&]() -> int {
        const int nb = std::min(launched < 16 || short_its ? 4 : 8, limit - launched);
        for (int k = 0; k < nb; k++) {
            // the mirror of the group before holds its own state or, until
            // the copy lands, that of two groups before, which was not over;
            // what it says is confirmed by the wait
            if (ahead && short_its && d.seen_over((group + 1) & 1)) {
                ahead = false;
                return 0;
            }
            if (int rc = d.launch(launched)) return rc;
            launched++;
        }
        return d.post(group++ & 1);
    };
    do {
        if (!ahead)
            if (int rc = launch_group()) return rc;
        ahead = launched > 4 && launched < limit;
        if (ahead)
            if (int rc = launch_group()) return rc;
        *last = (ahead ? group - 2 : group - 1) & 1;
        if (int rc = d.wait(*last, !ahead)) return rc;
    } while (!d.over(*last) && (ahead || launched < limit));
    return 0;
}

}  // namespace ifl
