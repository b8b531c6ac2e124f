// When a tile of a waiting sweep (k_sweep_wait) gives up.  Plain C++ (the
// functions are constexpr, so they serve host and device alike).
//
// A wait is counted in polls of its own: while its process is switched out or
// its queue preempted no poll is made, so that time never counts, as it would
// by any clock.  And the count starts again whenever a tile has been started
// anywhere in the sweep: as long as the sweep gets on, nothing gives up.
#pragma once

#include <stdint.h>

namespace bda {

// A wait looks at the sweep's ticket counter after every kWaitLook polls (a
// power of two; a poll is a load past the L2 and a short sleep, 0.5 to 1 us),
// and gives up after kWaitPatience looks in a row at the same count: 4 million
// polls, seconds in which no tile of the sweep was started.
constexpr uint32_t kWaitLook = 256, kWaitPatience = 1u << 14;

// Polls between two looks (less one) and equal looks to give up after, for a
// limit in polls; a limit below kWaitLook looks after every poll.
struct WaitLimit {
    uint32_t mask = kWaitLook - 1, patience = kWaitPatience;
};
constexpr WaitLimit wait_limit(uint32_t polls) {
    WaitLimit l;
    l.mask = polls < kWaitLook ? 0 : kWaitLook - 1;
    l.patience = polls < kWaitLook ? polls : polls / kWaitLook;
    return l;
}

struct WaitCount {
    int32_t tickets = -1;  // at the last look
    uint32_t looks = 0;    // without a change
};

constexpr bool wait_over(WaitCount &c, int32_t tickets, uint32_t patience) {
    if (tickets != c.tickets) {
        c.tickets = tickets;
        c.looks = 0;
        return false;
    }
    return ++c.looks > patience;
}

}  // namespace bda
