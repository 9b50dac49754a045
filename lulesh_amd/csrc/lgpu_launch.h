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

// Threads that share an element's repeats, and the repeat count from which
// they do, in launches that split (eos_split).
constexpr int kEosShare = 4;
constexpr int kEosSplitReps = 8;

// Whether k_eos shares the repeats of the heaviest elements between threads:
// up to 2^20 elements, where a wave's 20 to 50 repeats in a row are a good part
// of the launch.  One thread / shared: s=8 13.7 / 7.4 us, s=30 14.8 / 8.1, s=45
// 15.6 / 11.6, s=63 mixed (50 repeats) 25.6 / 20.3, s=64 22.1 / 21.2, s=96 FMA
// 44.7 / 43.0, s=101 50.6 / 49.9; above: 64 members, 6.0 M elements, 268 / 291,
// s=192 299 / 341 (each sharing thread loads the operands again).
inline bool eos_split(int64_t numElem) { return numElem <= (1 << 20); }

// The workgroups of one group.
inline void add_eos_slots(std::vector<EosSlot> &slots, const EosGroup &g, bool split)
{
   const int share = split && g.rep >= kEosSplitReps ? kEosShare : 1, per = kEosBlock / share;
   for (int64_t at = 0; at < g.count; at += per)
      slots.push_back(EosSlot{(int32_t)(g.pos + at), (int32_t)std::min<int64_t>(per, g.count - at),
                              g.rep, share});
}

// Whether a device-loop cycle begins in its first kernel (k_nodal_block or
// k_force, of `blocks` workgroups on `slots` resident ones) instead of
// k_begin_cycle, a launch of 3.0 to 4.7 us.  Each workgroup then starts about
// 1 us later, so the gain is gone after a few rounds.  Launch / first kernel,
// us a cycle, FP64: s=8 24.6 / 21.5, s=30 25.8 / 24.1, s=45 40.1 / 39.1, s=64
// gathers (2 rounds) 68.8 / 68.8; k_nodal_brick s=101 4.7 less and 5.5 more.
inline bool fold_start(int64_t blocks, int64_t slots) { return blocks <= 2 * slots; }

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
