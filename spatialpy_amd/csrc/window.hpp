// The event queue's time window (NRMConstant_v5): its bounds decide when the
// reference reports an empty queue, so the queue build and the event loop keep
// its scalars with the same update rules.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>
#include <cmath>

#include "engine.hpp"

namespace ssa {

// Time window (NRMConstant_v5::setBinNumberAndBounds, NRMConstant_v5.cpp:245-281).
__device__ inline bool set_bins(QueueState &q, double newL, double psum, long long active) {
    if (active == 0) return false;
    q.L = newL;
    if (q.L > q.endTime) return false;
    double w = 16.0 / psum;
    // The empty asm keeps the square root here: without it the compiler
    // hoists it out of the rarely taken window rebuild into every event of
    // the event loop, since `active` does not change inside the rebuild.
    double act = (double)(int)active;
    asm volatile("" : "+v"(act));
    unsigned long long maxb = (unsigned long long)((double)20 * sqrt(act));
    unsigned long long endb = ULLONG_MAX, nb;
    if (q.endTime < DBL_MAX) {
        endb = (unsigned long long)ceil((q.endTime - q.L) / w);
        nb = endb < maxb ? endb : maxb;
    } else {
        nb = maxb;
    }
    q.U = q.L + w * (double)nb;
    if (q.endTime < DBL_MAX) {
        if (q.U < q.endTime && ((double)(endb - maxb) / ((double)nb)) < .2) {
            nb = endb;
            q.U = q.L + w * (double)nb;
        }
    }
    q.nbins = nb;
    return true;
}

// NRMConstant_v5::rebuild (NRMConstant_v5.cpp:194-242): returns false when
// the window cannot move (selectReaction then reports an empty queue).
__device__ inline bool rebuild(QueueState &q) {
    double est;
    if (q.rxnCount > 0) est = (double)q.rxnCount / (q.U - q.L);
    else est = 1.0 / ((q.U - q.L) / (double)q.nbins);
    if (!set_bins(q, q.U, est, (long long)q.active)) return false;
    q.rxnCount = 0;
    return q.nbins > 0;
}

}  // namespace ssa
