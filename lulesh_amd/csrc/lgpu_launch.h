// lgpu_launch.h -- host-side launchers of the step kernels, one explicit
// instantiation per precision policy (lgpu_step_fp64.hip, lgpu_step_mixed.hip,
// lgpu_step_fp64fma.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "lgpu_kernels.h"
#include "lgpu_time.h"

namespace lgpu {

constexpr int kEosBlock = 256;
// Slot pairs of the one-problem dt minima (k_eos atomics, k_dt_slots); a
// power of two
constexpr int kDtSlots = 256;

// A run of the EOS work list: the elements of one repeat count (of one
// problem), largest count first.
struct EosGroup {
   int64_t pos, count;
   int32_t rep;
};

// Threads that share an element's repeats in slots that share them.
constexpr int kEosShare = 4;

// Whether the threads of a group's slots share its elements' repeats: a wave's
// 10 to 50 repeats in a row are a good part of a short launch, but each sharing
// thread loads the operands again.  So only counts well above the mean of the
// problem (`repeats` in all), and the larger the launch, within which such
// waves run beside the others, the more repeats the group has to hold: one per
// element of the problem for 365,000 elements of the launch (mixed 150,000).
// One thread / shared, us: FP64, 11 regions, s=30 of 10 repeats 12.9 / 10.0, s=101 of
// 10 38.9 / 42.4 and of 50 93.8 / 73.1; mixed, 16 regions, s=63 of 50 28.2 / 21.9, near
// the mean 30.0 / 38.4.
inline bool eos_shares(int64_t launchElems, int64_t numElem, const EosGroup &g, double repeats,
                       bool mixed)
{
   return g.rep >= 8 && (double)g.rep * (double)numElem >= 2.0 * repeats &&
          (double)g.rep * (double)g.count * (mixed ? 150e3 : 365e3) >= (double)launchElems * (double)numElem;
}

// The workgroups of one group.
inline void add_eos_slots(std::vector<EosSlot> &slots, const EosGroup &g, bool shared)
{
   const int share = shared ? kEosShare : 1, per = kEosBlock / share;
   for (int64_t at = 0; at < g.count; at += per)
      slots.push_back(EosSlot{(int32_t)(g.pos + at), (int32_t)std::min<int64_t>(per, g.count - at),
                              g.rep, share});
}

// Whether a device-loop cycle begins in its first kernel (k_nodal_block or
// k_force, of `blocks` workgroups on `slots` resident ones) instead of
// k_begin_cycle, a launch of 3.0 to 4.7 us.  Each workgroup then starts up to 1
// us later, so the gain is gone after a few rounds (4 of k_nodal_block in FP64,
// otherwise 2).  Launch / first kernel, us a cycle: FP64 s=8 24.6 / 21.5, s=64 (3.6
// rounds) 64.6 / 63.8; mixed s=63 (2.4) 44.5 / 44.9; gathers s=64 (2) 82.2 / 81.2.
inline bool fold_start(int64_t blocks, int64_t slots, bool fp64Block)
{
   return blocks <= (fp64Block ? 4 : 2) * slots;
}

// EOS repeat count of region r (0-based), lulesh.cc:2390-2400.
inline int32_t region_rep(int32_t r, int32_t numReg, int32_t cost)
{
   if (r < numReg / 2) return 1;
   if (r < numReg - (numReg + 15) / 20) return 1 + cost;
   return 10 * (1 + cost);
}

template <class P>
struct Launch {
   static void force(const DevState &s, const Consts &k, int64_t planeStride, int block,
                     hipStream_t st);
   static void node(const DevState &s, const Consts &k, int64_t planeStride, double dt, int block,
                    hipStream_t st);
   static void nodal_brick(const DevState &s, const Consts &k, double dt, hipStream_t st);
   // resident k_nodal_brick workgroups per CU (0 if the query fails)
   static int nodal_brick_blocks_per_cu();
   static void kin(const DevState &s, const Consts &k, double dt, int block, hipStream_t st);
   static void kin_brick(const DevState &s, const Consts &k, double dt, hipStream_t st);
   // resident k_kin_brick workgroups per CU (0 if the query fails)
   static int kin_brick_blocks_per_cu();
   // ensemble on the brick path: one launch over every member's workgroups
   // (16x16-thread tiles), the grid sizes from the member tables
   static void nodal_brick_members(const DevState &s, const Consts &k, unsigned grid,
                                   hipStream_t st);
   static void kin_brick_members(const DevState &s, const Consts &k, unsigned grid, hipStream_t st);
   static void eos(const DevState &s, const Consts &k, hipStream_t st);
   static void dt_reduce(const DevState &s, hipStream_t st);
   // start of a device-loop cycle as a launch of its own (k_begin_cycle)
   static void begin(const DevState &s, hipStream_t st);
   // start and end of a device loop (k_run_start, k_run_end)
   static void run_start(const DevTime &t, DevTime *time, double *dtOut, hipStream_t st);
   static void run_end(const DevState &s, double *slots0, int32_t *err0, DevTime *hostTime,
                       hipStream_t st);
};

extern template struct Launch<PolicyFp64>;
extern template struct Launch<PolicyMixed>;
extern template struct Launch<PolicyFp64Fma>;

} // namespace lgpu
