// The order of things at the barrier between two steps of the single launch (program.hip), apart from how they are done on the
// device: a workgroup that waits at most so long, and a launch that is reported as done only if nobody's time was up.
#pragma once
#include <stdint.h>

#include "fq_math.h"

namespace hipie {

// what a launch tells the host in its slot's word, 0 before it
constexpr uint32_t kReportCancelled = 1, kReportLost = 2, kReportDone = 3;

// A wait whose time is up: from here on what the workgroup computes may be wrong.
template <class Workgroup>
HIPIE_HD void give_up(Workgroup& w) {
    w.tell(kReportLost);
    w.lose();
}

// Behind a step.  A workgroup that gave up its wait in front of the step does not arrive: the counters that this step completes stay
// short for good, so nobody gets past them, and the first workgroup does not come to write "done" over "lost".
template <class Workgroup>
HIPIE_HD void arrive_at(Workgroup& w) {
    const int32_t held = w.verdict();        // (on its way while the stores are acknowledged)
    w.settle();
    w.count(held != 0);                      // (by the lane that adds: the rest of the workgroup finds out beside the addition)
    w.dead = w.lost(held);
}

// Behind the wait for everybody's last arrival, by the first workgroup.
template <class Workgroup>
HIPIE_HD void report(Workgroup& w) {
    if (!w.lost(w.verdict())) w.tell(kReportDone);
}

}  // namespace hipie
