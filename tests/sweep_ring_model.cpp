// A model of the record ring of the LU-SGS sweeps: the copy waves' own loop (ffring.h) with
// events in place of loads, waits and barriers, and the compute waves' reads where ffring.h says
// they are.  Interval i is the time between barriers i - 1 and i: step s's phases are the
// intervals 2s + 1 and 2s + 2, and 0 is the time before the first step.
//
// argv: nsteps, wait (a number added to every bound, or "none"), early (intervals by which the
// copies start earlier).  Prints for each of the kernel's rings what it finds wrong, or "ok".
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../finflo_amd/csrc/ffring.h"

constexpr int READERS = 3;

template <bool FWD, bool F32, int NLD>
static void model(int nsteps, const char *wait_arg, int early)
{
    constexpr int RS = ff::ring_slots<FWD, F32>();
    const bool none = !std::strcmp(wait_arg, "none");
    const int bias = none ? 0 : std::atoi(wait_arg);
    std::vector<int> start(nsteps, -1), there(nsteps, -1), order;
    int now = 0, done = 0, bad = 0, twice = 0;     // done: records whose loads are known to be complete
    auto copy = [&](int s) {
        if (s < 0 || s >= nsteps || start[s] >= 0) twice++;
        else start[s] = std::max(now - early, 0);
        order.push_back(s);
    };
    auto wait = [&](auto n) {
        if (none) return;
        const int flight = decltype(n)::value + bias;                     // loads that may remain
        const int complete = ((int)order.size() * NLD - flight) / NLD;    // whole records, in order
        for (; done < complete; done++) there[order[done]] = now;
    };
    auto sync = [&] { now++; };
    ff::ring_copy_wave<RS, NLD>(nsteps, copy, wait, sync);
    if (now != 1 + 2 * nsteps) { printf("barriers %d ", now); bad++; }
    if (twice) { printf("copied twice or out of range %d ", twice); bad++; }
    for (int s = 0; s < nsteps; s++) {
        int first = 1 << 30, last = -1;
        auto read = [&](int i) { first = std::min(first, i); last = std::max(last, i); };
        read(s > 0 ? 2 * (s - 1) + 2 : 1);                    // the increments' fields (wave 0)
        for (int w = 0; w < READERS; w++) read(2 * s + ff::ring_face_phase(w));
        if (start[s] < 0) { printf("record %d not copied ", s); bad++; continue; }
        // it has arrived in an interval before that of its first read
        if (there[s] < 0 || there[s] >= first) { printf("record %d read before it arrives ", s); bad++; }
        // the next copy into its slot starts in an interval after that of its last read
        if (s + RS < nsteps && start[s + RS] <= last) { printf("record %d overwritten ", s); bad++; }
        if (bad > 3) break;
    }
    printf("%s\n", bad ? "" : "ok");
}

int main(int, char **argv)
{
    const int n = std::atoi(argv[1]), early = std::atoi(argv[3]);
    // the loads of a copy wave per record: the kernel asserts the same numbers
    model<false, false, ff::ring_loads<false, false>()>(n, argv[2], early);
    model<false, true, ff::ring_loads<false, true>()>(n, argv[2], early);
    model<true, false, ff::ring_loads<true, false>()>(n, argv[2], early);
    model<true, true, ff::ring_loads<true, true>()>(n, argv[2], early);
    return 0;
}
