// lgpu_kernels.h -- device kernels of the Lagrange leapfrog step.
//
// The passes of a cycle, each a single launch over its whole index space:
//
//   k_force  (elements)  stress integration + Flanagan-Belytschko hourglass,
//                        per-corner forces to corner planes
//   k_node   (nodes)     deterministic corner gather in nodeElemCornerList
//                        order, acceleration, symmetry BCs, velocity, position
//   k_kin    (elements)  volume, vnew, characteristic length, strain rate,
//                        monotonic-Q gradients
//   k_eos    (region-ordered elements)  qstop check, monotonic-Q limiter,
//                        delv = vnew - v, EOS with its region repeat count,
//                        sound speed, volume update, Courant/hydro block minima
//                        (one problem: by atomic minima into 256 slot pairs)
//   k_dt_slots           host-driven cycles: Courant/hydro minima of the slots
//   k_begin_cycle        device loop: the same, and TimeIncrement, as the next
//                        cycle begins; in short cycles in its first kernel
//   k_dt_reduce          ensembles: each member's minima and TimeIncrement
//
// On the structured brick k_nodal_brick (column walks) or k_nodal_block (small
// bricks) take the place of k_force and k_node, and k_kin_brick (column walks) or
// k_kin_flat (bricks of up to kKinFlatMax elements an edge) that of k_kin.
//
// The Policy template parameter selects the arithmetic of each part:
// PolicyFp64 keeps everything in FP64 with the reference's association order,
// PolicyMixed runs force integration (corner forces and their node sums),
// Q gradients/limiter and EOS pressure and sound speed in FP32 on
// element-local coordinates; node accelerations, velocities and positions,
// element volume, delv, strain rate, characteristic length, the energy
// update and the dt candidates stay FP64.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <type_traits>

#include "lgpu_geom.h"

namespace lgpu {

// Error sites, in the order the reference checks them within one cycle.
enum ErrSite {
   kErrForceDeterm = 0, // lulesh.cc:1082-1091  determ <= 0       -> VolumeError
   kErrHourglassV = 1,  // lulesh.cc:1033-1040  v <= 0            -> VolumeError
   kErrKinVnew = 2,     // lulesh.cc:1597-1605  vnew <= 0         -> VolumeError
   kErrQStop = 3,       // lulesh.cc:1993-2008  q > qstop         -> QStopError
   kErrMaterialV = 4,   // lulesh.cc:2366-2384  clamped v <= 0    -> VolumeError
   kNumErrSites = 8
};

// One k_eos workgroup: `count` elements from position `pos` of the work list,
// all with `rep` repeats, each of them shared by `share` threads (1, or
// kEosShare in launches with k_eos's kSplit).
struct EosSlot {
   int32_t pos, count, rep, share;
};

struct Consts {
   double e_cut, p_cut, q_cut, v_cut, u_cut;
   double hgcoef, ss4o3, qstop, monoq_max_slope, monoq_limiter_mult;
   double qlc_monoq, qqc_monoq, qqc, eosvmax, eosvmin, pmin, emin, dvovmax, refdens;
   int32_t fastEos; // fast_eos_consts(*this), set by the host
};

// The constants k_eos's fast EOS repeats assume (both arithmetics): e_cut and p_cut
// positive (the values then clamped below by emin and pmin are never -0),
// emin and pmin not -0 and of magnitude <= 2^100, refdens in [2^-64, 2^64].
inline bool fast_eos_consts(const Consts &k)
{
   const double big = 0x1p100;
   return k.e_cut > 0. && k.p_cut > 0. && std::fabs(k.emin) <= big && std::fabs(k.pmin) <= big &&
          !(k.emin == 0. && std::signbit(k.emin)) && !(k.pmin == 0. && std::signbit(k.pmin)) &&
          k.refdens >= 0x1p-64 && k.refdens <= 0x1p64;
}

struct PolicyFp64 {
   using force_t = double;  // force integration arithmetic
   using corner_t = double; // stored per-corner force
   using grad_t = double;   // Q gradients + limiter arithmetic and storage
   using eos_t = double;    // EOS pressure / sound-speed arithmetic
   using nodesum_t = double; // per-node sums of the corner forces
   using pqs_t = double;     // stored p, q, ss
   static constexpr bool kLocalCoords = false;
   // geometry in the compact regrouped forms (different roundings) instead
   // of the reference's association order
   static constexpr bool kCompact = false;
   // waves per SIMD (min, max) for the nodal brick kernel's register
   // allocation and scheduling; (1, 8) leaves it to the compiler
   static constexpr int kNodalWavesMin = 1, kNodalWavesMax = 8;
   // the ensemble form takes a register or two more for its members' tiles, and
   // FP64_FMA then has 258, for one wave per SIMD: held to two waves, 64 members
   // of 16..64 602 -> 470 us.  The single problem's form has 256 by itself
   // (held to them it spills 3, s=96 63.9 -> 64.9 us)
   static constexpr int kMemberWavesMin = 2;
   // brick kernel: load the node update's operands before the element work
   static constexpr bool kPrefetchNode = true;
   // brick kernel: 32-bit byte offsets from scalar bases (at32) instead of
   // 64-bit per-lane addresses; FP64 runs 1.4% slower with them (more VGPRs)
   static constexpr bool kOffset32 = false;
   // brick kernel: issue the first hourglass velocity gather before the
   // hourglass modes (true) or after them; the later components are always
   // loaded one component ahead.  FP64 s=192: after, 598 us against 748 (256
   // VGPRs before); FMA and mixed: before, 1.4% and 0.5% faster
   static constexpr bool kHgVelEarly = false;
   // brick kernel: a scheduling barrier after the element-field loads (p, q,
   // v, volo, ss, elemMass), so that none is sunk to its use.  Mixed s=192:
   // 416 -> 411 us; FP64 582 -> 600 us, FMA 505 -> 534 us (the stress work
   // then waits for every load at once)
   static constexpr bool kPinElemFields = false;
   // brick kernel: carry an element's upper corners to the next plane in
   // registers, and load the next plane's other corners and fields in the
   // node phase of the current one.  s=192: FP64 555 -> 507 us, FP64_FMA 473 ->
   // 438 (all eight corners loaded there instead, the FMA form's way before:
   // FP64 534), s=101 FP64 90.4 -> 85.8; mixed spills 12 registers at 3
   // waves/SIMD (s=192 410 -> 527 us)
   static constexpr bool kCarryPlane = true;
   // k_eos waves per SIMD: FP64 at 7 (at most 72 VGPRs); 8 (64 VGPRs, four
   // spilled) ran 326 -> 332 us at s=192
   static constexpr int kEosWaves = 7;
   // brick kernel: the node phase at raised wave priority (s_setprio 2).
   // s=192, every kernel timed: FP64 576.4 -> 568.9 us, FP64_FMA 489 ->
   // 476.5 us (device loop: FP64 unchanged, FP64_FMA 484 -> 472 us); mixed
   // 417.5 -> 420.4 us
   static constexpr bool kNodePhasePrio = true;
   // k_nodal_block waves per SIMD
   static constexpr int kBlockWaves = 2;
};

// The FP64 policy compiled with multiply-add contraction (its own
// translation unit); the types are those of PolicyFp64.
struct PolicyFp64Fma : PolicyFp64 {
   static constexpr bool kHgVelEarly = true;
};

struct PolicyMixed {
   using force_t = float;
   using corner_t = float;
   using grad_t = float;
   using eos_t = float;
   using nodesum_t = float;
   using pqs_t = float;
   static constexpr bool kLocalCoords = true;
   static constexpr bool kCompact = true;
   // exactly 3: aiming for 4 (128 VGPRs) makes the scheduler issue the
   // hourglass velocity loads one at a time, each waited on at once
   static constexpr int kNodalWavesMin = 3, kNodalWavesMax = 3;
   static constexpr int kMemberWavesMin = 3;
   static constexpr bool kPrefetchNode = true;
   static constexpr bool kOffset32 = true;
   static constexpr bool kHgVelEarly = true;
   static constexpr bool kPinElemFields = true;
   static constexpr bool kCarryPlane = false;
   // k_eos at 8 waves per SIMD (at most 64 VGPRs): 214 -> 211 us at s=192
   static constexpr int kEosWaves = 8;
   static constexpr bool kNodePhasePrio = false;
   static constexpr int kBlockWaves = 3;
};

// Element i of a device array through a 32-bit byte offset: the access
// compiles to the scalar-base + 32-bit vector-offset form of the global
// load/store instead of per-lane 64-bit address arithmetic.  The caller
// guarantees i * sizeof(T) < 2^32 (the brick kernels: lgpu_create admits at
// most 2^28 elements, so a brick has fewer than 2^28.1 nodes).
template <typename T>
__device__ __forceinline__ T &at32(T *base, uint32_t i)
{
   using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
   return *reinterpret_cast<T *>(reinterpret_cast<B *>(base) + i * (uint32_t)sizeof(T));
}

// Division by a run-time constant d (< 2^32) as a 64-bit multiply-high:
// q = hi64(n * m) with m = floor((2^64 - 1) / d) + 1 is exact for n < 2^32.
struct FastDiv {
   uint64_t m;
   uint32_t d;
};

// Structured-brick description: s elements per edge, lattice node/element
// numbering of lulesh-init.cc:217-267.  Set when the mesh is the reference's
// brick, which lets the nodal pass run as one fused kernel.  The k_kin_brick
// tiles of one problem are 16 x 16.
struct Brick {
   int32_t s, en;          // elements and nodes per edge
   int32_t tilesX, tilesY; // k_nodal_brick column tiles of (tileW-1) x (rows-1) nodes
   int32_t chunkZ, chunks; // node planes per z-chunk, number of chunks
   int32_t rows;           // thread rows per k_nodal_brick workgroup: 16 or 8 of 16 threads,
                           // or 256 / tileW (ensemble members, pick_brick_walk)
   int32_t tileW;          // threads per k_nodal_brick row (4..64)
   FastDiv divS, divS2;    // element index -> (a, b, c)
   // k_kin_brick: 16x16-element column tiles per edge, element planes per z-chunk
   int32_t kinTiles, kinChunk, kinChunks;
   // ensemble members: kinW x kinH element tiles, kinTilesX x kinTilesY per plane
   int32_t kinW, kinH, kinTilesX, kinTilesY;
   // k_nodal_block: blkW x blkH x blkD elements per workgroup, blkX x blkY x
   // blkZ workgroups
   int32_t blkW, blkH, blkD, blkX, blkY, blkZ;
};

// One ensemble member on the brick path: its brick, where its nodes and
// elements start in the concatenated arrays.
struct MemberBrick {
   Brick g;
   int32_t nodeOff, elemOff;
};

// A k_eos workgroup's member in an ensemble, and its dt partial, which are by
// member whatever the order of the workgroups.
struct EosBlock {
   int32_t member, partial;
};

// One workgroup of a brick kernel in an ensemble.
struct MemberBlock {
   int32_t member;
   uint32_t wg; // within the member's grid
};

// Per-member time state of an ensemble, struct of arrays (the kernels read
// deltatime and active as plain arrays).
struct EnsTime {
   double *time, *deltatime, *dtcourant, *dthydro, *stoptime, *dtfixed, *dtmax, *multlb, *multub;
   int32_t *cycle, *active;
   // the run's cycle limit, one value in device memory: set by each
   // lgpu_ensemble_run, so that the cycle graphs do not depend on it
   int32_t *maxCycle;
};

// What the host polls, in pinned host memory: results of k_dt_slots or
// k_run_end, with the launch's count seq stored after them, and of a device
// loop the count of the last cycle begun and whether the loop has ended.
struct HostOut {
   double dt[2];
   int32_t err[kNumErrSites];
   uint32_t seq, started, ended;
};

// Everything a cycle touches on the device.
struct DevState {
   int32_t numElem, numNode;
   int32_t xcdRemap; // 1: map consecutive blocks onto one XCD's L2
   // node fields (current buffer; the brick path writes the other one)
   double *x, *y, *z, *xd, *yd, *zd, *nodalMass;
   double *xo, *yo, *zo, *xdo, *ydo, *zdo; // second node buffer (brick path)
   double *fx, *fy, *fz, *xdd, *ydd, *zdd; // diagnostics (may be null)
   const uint8_t *nodeBC;                  // bit0 symmX, bit1 symmY, bit2 symmZ
   const int32_t *nodeElemStart, *cornerList;
   // element fields
   const int32_t *nodelist;
   const int32_t *lxim, *lxip, *letam, *letap, *lzetam, *lzetap, *elemBC;
   double *e, *v, *volo;
   // P::pqs_t (FP64, or FP32 in the mixed form): p, q, ss
   void *p, *q, *ss;
   double *elemMass;
   double *vnew, *delv;
   double *arealg, *vdov;
   double *ql, *qq; // diagnostics (may be null)
   double *delvOut; // diagnostics: delv = vnew - v, stored by k_eos (may be null)
   void *delx_xi, *delx_eta, *delx_zeta, *delv_xi, *delv_eta, *delv_zeta; // grad_t
   // corner planes: [(component*2 + kind)*8 + corner][elem], kind 0 stress, 1 hourglass
   void *corner;
   // region order
   const int32_t *perm;     // elements grouped by EOS repeat count
   const struct EosSlot *eosSlot; // what each k_eos workgroup works on
   int32_t eosBlocks;       // k_eos workgroups
   int32_t eosSplit;        // some slots share elements between threads
   // control
   int32_t *err;            // kNumErrSites flags
   double *dtPartial;       // one problem: kDtSlots pairs of min_key values; ensemble: 2 per
                            // k_eos block
   double *dtOut;           // [0] dtcourant, [1] dthydro
   // Device loop (null otherwise): a cycle begins with timeOut made from
   // timeIn, the error flags and the dt slots of the cycle before (begin_cycle
   // in lgpu_step.inc), and sets err and dtPartial itself.
   int32_t startFold; // by the cycle's first kernel, not a launch of its own
   const struct DevTime *timeIn;
   struct DevTime *timeOut;
   const int32_t *errPrev;
   double *dtPartialPrev;
   HostOut *hostOut;        // one problem (null: ensembles)
   uint32_t hostSeq;        // what this launch stores in hostOut->seq or started
   const double *dtDevice;  // device-side deltatime (null: use argument)
   const int32_t *active;   // device-side loop flag (null: always active)
   Brick brick;             // valid when isBrick
   int32_t isBrick;
   int32_t nodalBlock; // nodal pass by k_nodal_block instead of k_nodal_brick
   int32_t kinFlat;    // kinematics by k_kin_flat instead of k_kin_brick
   int32_t brickFaces; // k_eos computes face neighbours and BC masks from the brick (or each member's)
   // Ensemble of independent problems (nMembers > 0): members are
   // concatenated; each has its own dt, loop flag and error flags.
   int32_t nMembers;
   const int32_t *memberNodeStart; // nMembers+1
   const int32_t *memberElemStart; // nMembers+1
   const double *memberDt;         // per-member deltatime
   const int32_t *memberActive;    // per-member loop flag
   int32_t *memberErr;             // nMembers x kNumErrSites
   const EosBlock *eosBlock;       // k_eos block -> member and dt partial
   const int32_t *memberBlockStart; // nMembers+1: k_eos blocks of each member
   double *memberDtOut;            // 2 per member: dtcourant, dthydro
   EnsTime ensTime;                // the members' next TimeIncrement
   // ensemble on the brick path (memberBrick non-null)
   const MemberBrick *memberBrick;
   const MemberBlock *nodalBlocks; // the nodal brick kernels' workgroups
   const MemberBlock *kinBlocks;   // the kinematics brick kernels' workgroups
   // the first ones, whole chunks, are mapped to XCDs; those after them are
   // shorter and dealt out longest first
   int32_t nodalWhole, kinWhole;
};

} // namespace lgpu
