// What the waves of a solve workgroup decide together: the buffers of their reductions, and how
// they learn of a cancel.
//
// A reduction has one barrier: each wave writes its total to its slot of a buffer, a barrier
// follows, every wave adds up all slots.  A wave may still be reading after the barrier while
// another is ahead, so a buffer is written again only if a barrier lies between its last read and
// that write.  Within the step control there are paths without any barrier from one reduction to
// the next; the reductions that can meet on such a path have buffers of their own
// (tests/red_host.cpp follows the control code and checks every pair).
#pragma once
#include "bdf_core.h"

namespace ucg {

// a value a wave; the reductions of two values have two buffers, one after the other
enum { RED_TS, RED_S, RED_TOTALS, RED_TOTALS_2, RED_CHARGE, RED_EWT, RED_EWT_2, RED_ACOR, RED_CORR, RED_HIST, RED_ORDER,
       RED_NBUF };

// The integrator's reductions (bdf_core.h's Ops).
struct OpsBuffers {
    static constexpr int weights = RED_EWT;      // set_ewt
    static constexpr int correction = RED_CORR;  // apply_correction
    static constexpr int acor = RED_ACOR;        // wrms of the accumulated correction
    static constexpr int history = RED_HIST;     // wrms of a history vector
    // wrms_acor_minus: at order 1, after a corrector that took one iteration, no barrier lies
    // between apply_correction and it
    static constexpr int order = RED_ORDER;
    static constexpr int first_step = RED_HIST;  // hub_inverse
    static constexpr int ydd = RED_CORR;         // ydd_norm
};

// Whether the caller has cancelled the launch, asked every `every`-th call (a power of two).  The
// host may raise the word at any moment, so one thread asks and all take its answer behind the
// barrier: were every wave to ask, some would leave the step loop and others go on into its
// barriers.  `flag` is shared by the threads; at least one more barrier lies between two askings.
template <class Flag, class Ask, class Barrier>
BDF_HD bool cancel_poll(int &calls, int every, bool asks, Flag &flag, Ask ask, Barrier barrier)
{
    if ((calls++ & (every - 1)) != 0) return false;
    if (asks) flag = ask() ? 1.0 : 0.0;
    barrier();
    return bdf_uni(flag) != 0.0;
}

}  // namespace ucg
