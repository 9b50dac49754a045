// lgpu_time.h -- device-side time state and TimeIncrement (lulesh.cc:166-222)
// of the device loops (lgpu_run, lgpu_ensemble_run).
#pragma once

#include <hip/hip_runtime.h>

#include "lgpu_kernels.h"

namespace lgpu {

// TimeIncrement operands plus the loop flag the kernels test.  fresh: no cycle
// of this loop has run, so dtcourant and dthydro are the caller's.
struct DevTime {
   double time, deltatime, dtcourant, dthydro, stoptime, dtfixed, dtmax, multlb, multub;
   int32_t cycle, maxCycle, active, fresh;
};

// TimeIncrement (lulesh.cc:166-222) at the top of a cycle, given the dt
// constraints of the cycle before (used when cycle > 0); also decides whether
// the cycle runs at all (the loop test of lulesh.cc:2745; failed: an error
// flag of the cycle before ends the loop).  One thread.
__device__ inline void time_increment(DevTime *t, double dtc, double dth, bool failed)
{
   if (!t->active) return;
   if (t->cycle > 0) {
      t->dtcourant = dtc;
      t->dthydro = dth;
   }
   if (failed || !(t->time < t->stoptime && t->cycle < t->maxCycle)) {
      t->active = 0;
      return;
   }
   double targetdt = t->stoptime - t->time;
   if (t->dtfixed <= 0.0 && t->cycle != 0) {
      const double olddt = t->deltatime;
      double newdt = 1.0e+20;
      if (t->dtcourant < newdt) newdt = t->dtcourant / 2.0;
      if (t->dthydro < newdt) newdt = t->dthydro * 2.0 / 3.0;
      const double ratio = newdt / olddt;
      if (ratio >= 1.0) {
         if (ratio < t->multlb) newdt = olddt;
         else if (ratio > t->multub) newdt = olddt * t->multub;
      }
      if (newdt > t->dtmax) newdt = t->dtmax;
      t->deltatime = newdt;
   }
   if (targetdt > t->deltatime && targetdt < 4.0 * t->deltatime / 3.0)
      targetdt = 2.0 * t->deltatime / 3.0;
   if (targetdt < t->deltatime) t->deltatime = targetdt;
   t->time += t->deltatime;
   t->cycle += 1;
}

__device__ inline bool any_error(const int32_t *err)
{
   int32_t any = 0; // all flags loaded at once (tested one by one, each load waits for the
                    // last: k_dt_reduce of 64 members 5.2 us, so 4.8)
#pragma unroll
   for (int i = 0; i < kNumErrSites; ++i) any |= err[i];
   return any != 0;
}

// The same for member m of an ensemble.
__device__ inline void time_increment(const EnsTime &t, int m, double dtc, double dth, bool failed)
{
   DevTime d{t.time[m],    t.deltatime[m], t.dtcourant[m], t.dthydro[m], t.stoptime[m],
             t.dtfixed[m], t.dtmax[m],     t.multlb[m],    t.multub[m],  t.cycle[m],
             *t.maxCycle,  t.active[m],    0};
   time_increment(&d, dtc, dth, failed);
   t.time[m] = d.time;
   t.deltatime[m] = d.deltatime;
   t.dtcourant[m] = d.dtcourant;
   t.dthydro[m] = d.dthydro;
   t.cycle[m] = d.cycle;
   t.active[m] = d.active;
}

} // namespace lgpu
