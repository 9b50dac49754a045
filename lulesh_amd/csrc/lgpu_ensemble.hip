// lgpu_ensemble.hip -- a batch of independent Sedov problems advanced
// together: one launch per kernel covers every member, each member keeps its
// own dt (TimeIncrement, lulesh.cc:166-222, evaluated per member on the
// device), and one cycle is captured once as a hipGraph and replayed.
//
// Members are concatenated in one device arena: node arrays, element arrays
// and node-to-corner lists are offset per member, and the region-ordered EOS
// list is padded per member to whole k_eos blocks so that every block (and
// so every dt partial) belongs to exactly one member.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <functional>
#include <new>
#include <string>
#include <vector>

#include "lgpu_brick.h"
#include "lgpu_convert.h"
#include "lgpu_kernels.h"
#include "lgpu_launch.h"
#include "lgpu_time.h"
#include "lulesh_gpu.h"

using namespace lgpu;

namespace {

enum EnsKernel {
   kEForce = 0, kENode, kEKin, kEEos, kEDt, kETime, kENodalBrick, kEKinBrick, kENumKernels
};
const char *const kEnsKernelNames[kENumKernels] = {"k_force", "k_node", "k_kin", "k_eos",
                                                   "k_dt_reduce", "k_time_increment",
                                                   "k_nodal_brick", "k_kin_brick"};

constexpr size_t kAlign = 256;
inline size_t align_up(size_t v) { return (v + kAlign - 1) & ~(kAlign - 1); }

// TimeIncrement per member (lulesh.cc:166-222) of a run's first cycle; later
// ones run at the end of the cycle before (k_dt_reduce).
__global__ void k_time_increment_ens(EnsTime t, const double *dtOut, const int32_t *err,
                                     int nMembers)
{
   const int m = blockIdx.x * blockDim.x + threadIdx.x;
   if (m >= nMembers) return;
   time_increment(t, m, dtOut[2 * m], dtOut[2 * m + 1], any_error(err + m * kNumErrSites));
}

// The brick path's kernels (1: k_nodal_block, k_kin_flat) and the z-chunks of
// those that walk up columns.  blockChunk, flatChunk: the chunk that stood there
// when k_nodal_block or k_kin_flat was chosen (0: they were not), so that a
// chunk option set to what it reads keeps, or brings back, that kernel.
struct BrickChoice {
   int nodalChunk = 8, kinChunk = 12;
   int32_t nodalBlock = 0, kinFlat = 0;
   int blockChunk = 0, flatChunk = 0;

   void choose_nodal(bool block)
   {
      nodalBlock = block;
      blockChunk = block ? nodalChunk : 0;
   }
   void choose_kin(bool flat)
   {
      kinFlat = flat;
      flatChunk = flat ? kinChunk : 0;
   }
};

} // namespace

struct lgpu_ensemble {
   hipStream_t stream = nullptr;
   int32_t nMembers = 0, precision = 0;
   Consts k{};
   DevState s{};
   int64_t planeStride = 0;
   char *arena = nullptr;
   size_t arenaBytes = 0;
   size_t stateBytes = 0; // leading part of the arena holding the state (for snapshots)
   std::vector<int32_t> nodeStart, elemStart, nodeCount, elemCount;
   EnsTime t{};
   int block[3] = {256, 256, 256}; // force, node, kin
   bool useGraph = true;
   bool timing = false;
   hipGraph_t graph = nullptr;
   hipGraphExec_t exec = nullptr;
   // Brick path: every member is a reference brick; the fused nodal and
   // kinematics kernels run over all members' workgroups, node state
   // ping-pongs between two buffers (parity = which one is current), and a
   // cycle graph is captured for each parity.
   bool brick = false;
   int parity = 0;
   hipGraph_t graph2 = nullptr;
   hipGraphExec_t exec2 = nullptr;
   std::vector<int32_t> memberSize;
   BrickChoice choice; // what s and the tables are made for
   unsigned nodalBlocks = 0, kinBlocks = 0;
   char *tables = nullptr;
   int64_t kLaunches[kENumKernels] = {};
   double kMs[kENumKernels] = {};
   std::string lastError;
   // pinned: SmallCopy, host mirror of the time state
   char *host = nullptr;
   SmallCopy small;
};

namespace {

int fail_hip(lgpu_ensemble *e, hipError_t err, const char *what)
{
   if (err == hipSuccess) return LGPU_OK;
   if (e) e->lastError = std::string(what) + ": " + hipGetErrorString(err);
   return err == hipErrorOutOfMemory ? LGPU_ENOMEM : LGPU_EDEVICE;
}

#define ENS_HIP(e, call)                                            \
   do {                                                             \
      const hipError_t err_ = (call);                               \
      if (err_ != hipSuccess) return fail_hip((e), err_, #call);    \
   } while (0)

void swap_nodes(lgpu_ensemble *e)
{
   DevState &s = e->s;
   std::swap(s.x, s.xo);
   std::swap(s.y, s.yo);
   std::swap(s.z, s.zo);
   std::swap(s.xd, s.xdo);
   std::swap(s.yd, s.ydo);
   std::swap(s.zd, s.zdo);
   e->parity ^= 1;
}

template <class P>
void launch_cycle(lgpu_ensemble *e)
{
   if (e->brick) {
      Launch<P>::nodal_brick_members(e->s, e->k, e->nodalBlocks, e->stream);
      swap_nodes(e);
      Launch<P>::kin_brick_members(e->s, e->k, e->kinBlocks, e->stream);
   } else {
      Launch<P>::force(e->s, e->k, e->planeStride, e->block[0], e->stream);
      Launch<P>::node(e->s, e->k, e->planeStride, 0.0, e->block[1], e->stream);
      Launch<P>::kin(e->s, e->k, 0.0, e->block[2], e->stream);
   }
   Launch<P>::eos(e->s, e->k, e->stream);
   Launch<P>::dt_reduce(e->s, e->stream);
}

void enqueue_cycle(lgpu_ensemble *e)
{
   switch (e->precision) {
   case LGPU_MIXED: launch_cycle<PolicyMixed>(e); break;
   case LGPU_FP64_FMA: launch_cycle<PolicyFp64Fma>(e); break;
   default: launch_cycle<PolicyFp64>(e); break;
   }
}

// Events around launches; the stream is waited for before they are read.
template <int N>
struct Events {
   hipEvent_t ev[N] = {};
   ~Events()
   {
      for (hipEvent_t x : ev)
         if (x) (void)hipEventDestroy(x);
   }
};

void count_launch(lgpu_ensemble *e, int kernel, float ms)
{
   e->kLaunches[kernel] += 1;
   e->kMs[kernel] += ms;
}

// One cycle with every kernel timed (the timing option; the autotuner).
template <class P>
int timed_cycle(lgpu_ensemble *e)
{
   std::vector<int> kernels{kEForce, kENode, kEKin, kEEos, kEDt};
   if (e->brick) kernels = {kENodalBrick, kEKinBrick, kEEos, kEDt};
   Events<6> events;
   for (auto &x : events.ev) ENS_HIP(e, hipEventCreate(&x));
   hipEvent_t *next = events.ev;
   ENS_HIP(e, hipEventRecord(*next++, e->stream));
   for (int kernel : kernels) {
      switch (kernel) {
      case kENodalBrick:
         Launch<P>::nodal_brick_members(e->s, e->k, e->nodalBlocks, e->stream);
         swap_nodes(e);
         break;
      case kEKinBrick: Launch<P>::kin_brick_members(e->s, e->k, e->kinBlocks, e->stream); break;
      case kEForce: Launch<P>::force(e->s, e->k, e->planeStride, e->block[0], e->stream); break;
      case kENode: Launch<P>::node(e->s, e->k, e->planeStride, 0.0, e->block[1], e->stream); break;
      case kEKin: Launch<P>::kin(e->s, e->k, 0.0, e->block[2], e->stream); break;
      case kEEos: Launch<P>::eos(e->s, e->k, e->stream); break;
      default: Launch<P>::dt_reduce(e->s, e->stream);
      }
      ENS_HIP(e, hipEventRecord(*next++, e->stream));
   }
   ENS_HIP(e, hipGetLastError());
   ENS_HIP(e, hipStreamSynchronize(e->stream));
   for (size_t i = 0; i < kernels.size(); ++i) {
      float ms = 0.f;
      ENS_HIP(e, hipEventElapsedTime(&ms, events.ev[i], events.ev[i + 1]));
      count_launch(e, kernels[i], ms);
   }
   return LGPU_OK;
}

int timed_cycle_any(lgpu_ensemble *e)
{
   switch (e->precision) {
   case LGPU_MIXED: return timed_cycle<PolicyMixed>(e);
   case LGPU_FP64_FMA: return timed_cycle<PolicyFp64Fma>(e);
   default: return timed_cycle<PolicyFp64>(e);
   }
}

void drop_graph(lgpu_ensemble *e)
{
   if (e->exec) (void)hipGraphExecDestroy(e->exec);
   if (e->graph) (void)hipGraphDestroy(e->graph);
   if (e->exec2) (void)hipGraphExecDestroy(e->exec2);
   if (e->graph2) (void)hipGraphDestroy(e->graph2);
   e->exec = e->exec2 = nullptr;
   e->graph = e->graph2 = nullptr;
}

int capture_cycle(lgpu_ensemble *e, hipGraph_t &g, hipGraphExec_t &x)
{
   ENS_HIP(e, hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
   enqueue_cycle(e);
   const hipError_t endErr = hipStreamEndCapture(e->stream, &g);
   ENS_HIP(e, endErr);
   ENS_HIP(e, hipGraphInstantiate(&x, g, nullptr, nullptr, 0));
   return LGPU_OK;
}

// One cycle graph; on the brick path a second one for the other node-buffer
// parity (exec: captured at parity 0, exec2: at parity 1).  Capturing
// advances the host's parity; it is put back afterwards.
int build_graph(lgpu_ensemble *e)
{
   drop_graph(e);
   if (e->brick) {
      const int p0 = e->parity;
      if (p0) swap_nodes(e);
      int r = capture_cycle(e, e->graph, e->exec);
      if (!r) r = capture_cycle(e, e->graph2, e->exec2);
      if (e->parity != p0) swap_nodes(e);
      if (r) return r;
   } else {
      const int r = capture_cycle(e, e->graph, e->exec);
      if (r) return r;
   }
   return LGPU_OK;
}

// Replays one cycle: the graph of the current parity (the host mirrors the
// pointer swap the graph's nodal launch implies).
int launch_graph(lgpu_ensemble *e)
{
   if (e->brick) {
      ENS_HIP(e, hipGraphLaunch(e->parity ? e->exec2 : e->exec, e->stream));
      swap_nodes(e);
   } else {
      ENS_HIP(e, hipGraphLaunch(e->exec, e->stream));
   }
   return LGPU_OK;
}

// The brick path's default kernels and nodal chunk.  A walk's cost is taken
// over all members' workgroups.  30 members of 10..40: a walk, 68.7 us
// (k_nodal_block 84.8); 24 of 5..24: k_nodal_block, FP64 18.6 and mixed 13.6
// us (best walk 24.1 and 18.5).
BrickChoice pick_brick_kernels(const lgpu_ensemble *e)
{
   BrickChoice pick;
   int dev = 0, cus = 0, perCu = 0, largest = 0;
   if (hipGetDevice(&dev) != hipSuccess ||
       hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      cus = 0;
   switch (e->precision) {
   case LGPU_MIXED: perCu = Launch<PolicyMixed>::nodal_brick_blocks_per_cu(); break;
   case LGPU_FP64_FMA: perCu = Launch<PolicyFp64Fma>::nodal_brick_blocks_per_cu(); break;
   default: perCu = Launch<PolicyFp64>::nodal_brick_blocks_per_cu(); break;
   }
   const int slots = cus * perCu;
   std::vector<Brick> bricks;
   int64_t blocks = 0;
   for (int32_t sz : e->memberSize) {
      Brick g{};
      init_brick(g, sz);
      pick_member_tile(g);
      blocks += block_blocks(g);
      largest = std::max(largest, sz);
      bricks.push_back(g);
   }
   pick.choose_kin(largest <= kKinFlatMax);
   if (slots < 1) return pick;
   std::vector<int64_t> columns;
   std::vector<int> planes;
   for (const Brick &g : bricks) {
      columns.push_back((int64_t)g.tilesX * g.tilesY);
      planes.push_back(g.en);
   }
   pick.nodalChunk = pick_tail_chunk(columns, planes, slots, 0.25, pick.nodalChunk);
   double least = 1e300;
   for (int ch = 1; ch <= 22; ++ch) {
      int64_t walks = 0;
      for (const Brick &g : bricks) walks += (int64_t)g.tilesX * g.tilesY * ((g.en + ch - 1) / ch);
      least = std::min(least, (double)((walks + slots - 1) / slots * (ch + 1)));
   }
   pick.choose_nodal(block_is_faster(blocks, slots, least));
   return pick;
}

// The workgroups of a walking kernel over all members: those of whole z-chunks
// by member, then the members' last, shorter chunks, longest first, so that
// the launch does not end on a long walk.  Members: `columns` column tiles of
// `planes` planes each; returns the number of the first.  64 members of
// 16..64, FP64 nodal, by member throughout / so: chunk 10 522 / 485 us, 16 531 /
// 482; mixed chunk 9 399 / 378.
int32_t walk_blocks(const std::vector<int64_t> &columns, const std::vector<int> &planes, int chunk,
                    std::vector<MemberBlock> &blocks)
{
   std::vector<std::vector<MemberBlock>> last((size_t)chunk); // by length
   for (size_t m = 0; m < columns.size(); ++m) {
      const uint32_t n = (uint32_t)(columns[m] * (planes[m] / chunk));
      for (uint32_t w = 0; w < n; ++w) blocks.push_back(MemberBlock{(int32_t)m, w});
      const int rest = planes[m] % chunk;
      for (uint32_t w = 0; rest && w < (uint32_t)columns[m]; ++w)
         last[(size_t)rest].push_back(MemberBlock{(int32_t)m, n + w});
   }
   const int32_t whole = (int32_t)blocks.size();
   for (int rest = chunk - 1; rest > 0; --rest)
      blocks.insert(blocks.end(), last[(size_t)rest].begin(), last[(size_t)rest].end());
   return whole;
}

// The same for kernels of equal workgroups, blocks[m] of member m.
int32_t equal_blocks(const std::vector<int64_t> &counts, std::vector<MemberBlock> &blocks)
{
   for (size_t m = 0; m < counts.size(); ++m)
      for (uint32_t w = 0; w < (uint32_t)counts[m]; ++w) blocks.push_back(MemberBlock{(int32_t)m, w});
   return (int32_t)blocks.size();
}

// k_eos's dispatch order over all members: heavy workgroups (kEosHeavyReps
// repeats on) first where all are resident at once, and otherwise one of them
// every 3 dispatches, so that they have started well before the end; both kinds
// by member.  By member throughout, each one's heavy ones first / every 3 / every
// 5 / heavy first, us: 64 members of 16..64, FP64, 267 / 262 / 274 / 293; 16 of
// 40..90, FP64_FMA, 284 / 281 / 272 / 312; mixed 40 of 20..50 87 / 78 / 88 / 84; 24
// of 5..24 (resident) 17.0 / 18.2 / 17.3 / 16.2.
constexpr int kEosHeavyReps = 8;

void order_eos_blocks(std::vector<EosSlot> &slots, std::vector<EosBlock> &blocks, int64_t resident)
{
   std::vector<size_t> heavy, rest, order;
   for (size_t b = 0; b < slots.size(); ++b)
      (slots[b].rep >= kEosHeavyReps ? heavy : rest).push_back(b);
   const size_t between = (int64_t)slots.size() <= resident ? 0 : 2;
   size_t r = 0;
   for (size_t b : heavy) {
      order.push_back(b);
      for (size_t j = 0; j < between && r < rest.size(); ++j) order.push_back(rest[r++]);
   }
   order.insert(order.end(), rest.begin() + (std::ptrdiff_t)r, rest.end());
   std::vector<EosSlot> s2;
   std::vector<EosBlock> b2;
   for (size_t b : order) {
      s2.push_back(slots[b]);
      b2.push_back(blocks[b]);
   }
   slots.swap(s2);
   blocks.swap(b2);
}

// Takes the kernels and chunks of `want`, with the member tables for them:
// per-member bricks with offsets, and the kernels' workgroups.  Where it fails,
// the ensemble keeps those it has.
int set_brick_choice(lgpu_ensemble *e, const BrickChoice &want)
{
   const int M = e->nMembers;
   std::vector<MemberBrick> mb((size_t)M);
   std::vector<MemberBlock> nodal, kin;
   std::vector<int64_t> nodalCount, kinCount; // workgroups, or column tiles of the walks
   std::vector<int> nodePlanes, elemPlanes;
   for (int m = 0; m < M; ++m) {
      Brick g{};
      init_brick(g, e->memberSize[(size_t)m]);
      pick_member_tile(g);
      pick_member_kin_tile(g);
      set_brick_chunk(g, want.nodalChunk);
      set_kin_chunk(g, want.kinChunk);
      mb[(size_t)m].g = g;
      mb[(size_t)m].nodeOff = e->nodeStart[(size_t)m];
      mb[(size_t)m].elemOff = e->elemStart[(size_t)m];
      nodalCount.push_back(want.nodalBlock ? block_blocks(g) : (int64_t)g.tilesX * g.tilesY);
      kinCount.push_back(want.kinFlat ? flat_blocks(g) : (int64_t)g.kinTilesX * g.kinTilesY);
      nodePlanes.push_back(g.en);
      elemPlanes.push_back(g.s);
   }
   const int32_t nodalWhole = want.nodalBlock ? equal_blocks(nodalCount, nodal)
                                              : walk_blocks(nodalCount, nodePlanes, want.nodalChunk, nodal);
   const int32_t kinWhole = want.kinFlat ? equal_blocks(kinCount, kin)
                                         : walk_blocks(kinCount, elemPlanes, want.kinChunk, kin);
   const size_t nb = nodal.size(), kb = kin.size();
   const size_t b0 = align_up(sizeof(MemberBrick) * (size_t)M);
   const size_t b1 = align_up(sizeof(MemberBlock) * nb), b2 = align_up(sizeof(MemberBlock) * kb);
   char *tables = nullptr;
   ENS_HIP(e, hipMalloc((void **)&tables, b0 + b1 + b2));
   hipError_t err = hipMemcpy(tables, mb.data(), sizeof(MemberBrick) * (size_t)M, hipMemcpyHostToDevice);
   if (err == hipSuccess)
      err = hipMemcpy(tables + b0, nodal.data(), sizeof(MemberBlock) * nb, hipMemcpyHostToDevice);
   if (err == hipSuccess)
      err = hipMemcpy(tables + b0 + b1, kin.data(), sizeof(MemberBlock) * kb, hipMemcpyHostToDevice);
   if (err == hipSuccess) err = hipStreamSynchronize(e->stream); // nothing reads the old ones any more
   if (err != hipSuccess) {
      (void)hipFree(tables);
      return fail_hip(e, err, "brick tables");
   }
   drop_graph(e);
   if (e->tables) (void)hipFree(e->tables);
   e->tables = tables;
   e->choice = want;
   e->s.nodalBlock = want.nodalBlock;
   e->s.kinFlat = want.kinFlat;
   e->s.nodalWhole = nodalWhole;
   e->s.kinWhole = kinWhole;
   e->s.memberBrick = reinterpret_cast<const MemberBrick *>(tables);
   e->s.nodalBlocks = reinterpret_cast<const MemberBlock *>(tables + b0);
   e->s.kinBlocks = reinterpret_cast<const MemberBlock *>(tables + b0 + b1);
   e->nodalBlocks = (unsigned)nb;
   e->kinBlocks = (unsigned)kb;
   return LGPU_OK;
}

// Device array of a field.  `narrow`: stored as FP32 in the mixed form (the
// Q gradients, p, q and ss).
double *field_base(lgpu_ensemble *e, int f, bool &isElem, bool &narrow)
{
   isElem = f >= LGPU_E;
   narrow = e->precision == LGPU_MIXED &&
            (f >= LGPU_DELX_XI || f == LGPU_P || f == LGPU_Q || f == LGPU_SS);
   DevState &s = e->s;
   switch (f) {
   case LGPU_X: return s.x;
   case LGPU_Y: return s.y;
   case LGPU_Z: return s.z;
   case LGPU_XD: return s.xd;
   case LGPU_YD: return s.yd;
   case LGPU_ZD: return s.zd;
   case LGPU_NODALMASS: return s.nodalMass;
   case LGPU_E: return s.e;
   case LGPU_P: return static_cast<double *>(s.p);
   case LGPU_Q: return static_cast<double *>(s.q);
   case LGPU_V: return s.v;
   case LGPU_VOLO: return s.volo;
   case LGPU_VNEW: return s.vnew;
   case LGPU_DELV: return s.delv;
   case LGPU_VDOV: return s.vdov;
   case LGPU_AREALG: return s.arealg;
   case LGPU_SS: return static_cast<double *>(s.ss);
   case LGPU_ELEMMASS: return s.elemMass;
   case LGPU_DELX_XI: return static_cast<double *>(s.delx_xi);
   case LGPU_DELX_ETA: return static_cast<double *>(s.delx_eta);
   case LGPU_DELX_ZETA: return static_cast<double *>(s.delx_zeta);
   case LGPU_DELV_XI: return static_cast<double *>(s.delv_xi);
   case LGPU_DELV_ETA: return static_cast<double *>(s.delv_eta);
   case LGPU_DELV_ZETA: return static_cast<double *>(s.delv_zeta);
   default: return nullptr;
   }
}

// Device scratch of a member's elements in doubles that nothing holds between
// cycles, as for a single problem.
double *scratch_doubles(lgpu_ensemble *e)
{
   return e->brick ? e->s.xo : static_cast<double *>(e->s.corner);
}

} // namespace

extern "C" {

int lgpu_ensemble_create(const lgpu_mesh_desc *members, int32_t nMembers, lgpu_ensemble **out)
{
   if (!members || nMembers < 1 || !out) return LGPU_EINVAL;
   *out = nullptr;
   const int32_t prec = members[0].precision;
   if (prec != LGPU_FP64 && prec != LGPU_MIXED && prec != LGPU_FP64_FMA) return LGPU_EINVAL;
   for (int32_t m = 0; m < nMembers; ++m) {
      const lgpu_mesh_desc &d = members[m];
      if (d.precision != prec || memcmp(&d.k, &members[0].k, sizeof(lgpu_constants)) != 0) {
         fprintf(stderr, "lgpu_ensemble_create: members must share precision and constants\n");
         return LGPU_EINVAL;
      }
      // Validate each member on its own (connectivity ranges, regions); the
      // size limit is lgpu_create's (8 corners per element index in int32).
      if (d.numElem < 1 || d.numNode < 1 || d.numElem > INT32_MAX / 8 || !d.nodelist ||
          !d.nodeElemStart || !d.nodeElemCornerList || d.numReg < 1 || d.cost < 0)
         return LGPU_EINVAL;
      for (int64_t i = 0; i < 8 * (int64_t)d.numElem; ++i)
         if (d.nodelist[i] < 0 || d.nodelist[i] >= d.numNode) return LGPU_EINVAL;
      const int32_t *nb[6] = {d.lxim, d.lxip, d.letam, d.letap, d.lzetam, d.lzetap};
      for (const int32_t *a : nb) {
         if (!a) return LGPU_EINVAL;
         for (int32_t i = 0; i < d.numElem; ++i)
            if (a[i] < 0 || a[i] >= d.numElem) return LGPU_EINVAL;
      }
      for (int32_t n = 0; n < d.numNode; ++n)
         if (d.nodeElemStart[n + 1] < d.nodeElemStart[n]) return LGPU_EINVAL;
      if (d.nodeElemStart[0] != 0 || d.nodeElemStart[d.numNode] > 8 * d.numElem) return LGPU_EINVAL;
      for (int32_t c = 0; c < d.nodeElemStart[d.numNode]; ++c)
         if (d.nodeElemCornerList[c] < 0 || d.nodeElemCornerList[c] >= 8 * d.numElem) return LGPU_EINVAL;
      int64_t tot = 0;
      std::vector<uint8_t> seen((size_t)d.numElem, 0);
      for (int32_t r = 0; r < d.numReg; ++r)
         for (int32_t i = 0; i < d.regElemSize[r]; ++i) {
            const int32_t el = d.regElemlist[r][i];
            if (el < 0 || el >= d.numElem || seen[(size_t)el]) return LGPU_EINVAL;
            seen[(size_t)el] = 1;
            ++tot;
         }
      if (tot != d.numElem) return LGPU_EINVAL;
      const int32_t *sy[3] = {d.symmX, d.symmY, d.symmZ};
      const int32_t ns[3] = {d.numSymmX, d.numSymmY, d.numSymmZ};
      for (int a = 0; a < 3; ++a)
         for (int32_t i = 0; i < ns[a]; ++i)
            if (!sy[a] || sy[a][i] < 0 || sy[a][i] >= d.numNode) return LGPU_EINVAL;
   }

   lgpu_ensemble *e = new (std::nothrow) lgpu_ensemble();
   if (!e) return LGPU_ENOMEM;
   auto bail = [&](int code) {
      lgpu_ensemble_destroy(e);
      return code;
   };
   e->nMembers = nMembers;
   e->precision = prec;
   // Brick path when every member is the reference's brick (and the generic
   // kernels are not asked for).
   e->brick = !(members[0].flags & LGPU_FLAG_GENERIC);
   for (int32_t m = 0; m < nMembers && e->brick; ++m) e->brick = is_reference_brick(&members[m]);
   e->s.brickFaces = e->brick ? 1 : 0;
   for (int32_t m = 0; m < nMembers && e->s.brickFaces; ++m)
      e->s.brickFaces = brick_faces_computable(&members[m]) ? 1 : 0;
   for (int32_t m = 0; m < nMembers; ++m) e->memberSize.push_back(members[m].sizeX);
   const lgpu_constants &kk = members[0].k;
   e->k = Consts{kk.e_cut, kk.p_cut, kk.q_cut, kk.v_cut, kk.u_cut, kk.hgcoef, kk.ss4o3,
                 kk.qstop, kk.monoq_max_slope, kk.monoq_limiter_mult, kk.qlc_monoq,
                 kk.qqc_monoq, kk.qqc, kk.eosvmax, kk.eosvmin, kk.pmin, kk.emin, kk.dvovmax,
                 kk.refdens};
   e->k.fastEos = fast_eos_consts(e->k);
   if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess)
      return bail(LGPU_EDEVICE);

   // The concatenated arrays are indexed with int32 (corners: 8 per element).
   {
      int64_t totE = 0, totN = 0;
      for (int32_t m = 0; m < nMembers; ++m) {
         totE += members[m].numElem;
         totN += members[m].numNode;
      }
      if (totE > INT32_MAX / 8 || totN > INT32_MAX) {
         fprintf(stderr, "lgpu_ensemble_create: %lld elements / %lld nodes in all: too many\n",
                 (long long)totE, (long long)totN);
         return bail(LGPU_EINVAL);
      }
   }
   // Offsets.
   DevState &s = e->s;
   int64_t totE = 0;
   for (int32_t m = 0; m < nMembers; ++m) totE += members[m].numElem;
   e->nodeStart.assign((size_t)nMembers + 1, 0);
   e->elemStart.assign((size_t)nMembers + 1, 0);
   std::vector<int64_t> cornerStart((size_t)nMembers + 1, 0);
   // The EOS work list, as for a single domain: each member's elements grouped
   // by EOS repeat count, largest first, in mesh order within a group.
   std::vector<int32_t> perm, blockStart(1, 0);
   perm.reserve((size_t)totE);
   std::vector<EosBlock> eosBlock;
   std::vector<EosSlot> eosSlots;
   for (int32_t m = 0; m < nMembers; ++m) {
      const lgpu_mesh_desc &d = members[m];
      e->nodeStart[m + 1] = e->nodeStart[m] + d.numNode;
      e->elemStart[m + 1] = e->elemStart[m] + d.numElem;
      cornerStart[m + 1] = cornerStart[m] + d.nodeElemStart[d.numNode];
      e->nodeCount.push_back(d.numNode);
      e->elemCount.push_back(d.numElem);
      const int32_t e0 = e->elemStart[m];
      std::vector<int32_t> repOf((size_t)d.numElem, 1), reps;
      double repeats = 0.;
      for (int32_t r = 0; r < d.numReg; ++r) {
         const int32_t rep = region_rep(r, d.numReg, d.cost);
         repeats += (double)rep * d.regElemSize[r];
         if (d.regElemSize[r] > 0 && std::find(reps.begin(), reps.end(), rep) == reps.end())
            reps.push_back(rep);
         for (int32_t i = 0; i < d.regElemSize[r]; ++i) repOf[(size_t)d.regElemlist[r][i]] = rep;
      }
      std::sort(reps.begin(), reps.end(), std::greater<int32_t>());
      for (int32_t rep : reps) {
         const int64_t pos = (int64_t)perm.size();
         for (int32_t el = 0; el < d.numElem; ++el)
            if (repOf[(size_t)el] == rep) perm.push_back(el + e0);
         const EosGroup group{pos, (int64_t)perm.size() - pos, rep};
         const bool shared = eos_shares(totE, d.numElem, group, repeats, prec == LGPU_MIXED);
         if (shared) s.eosSplit = 1;
         add_eos_slots(eosSlots, group, shared);
      }
      for (size_t b = eosBlock.size(); b < eosSlots.size(); ++b)
         eosBlock.push_back(EosBlock{m, (int32_t)b});
      blockStart.push_back((int32_t)eosSlots.size());
   }
   {
      int dev = 0, cus = 0;
      if (hipGetDevice(&dev) != hipSuccess ||
          hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
         cus = 0;
      order_eos_blocks(eosSlots, eosBlock,
                       (int64_t)cus * (prec == LGPU_MIXED ? PolicyMixed::kEosWaves : PolicyFp64::kEosWaves));
   }
   const size_t E = (size_t)e->elemStart[nMembers], N = (size_t)e->nodeStart[nMembers];
   const size_t nCorner = (size_t)cornerStart[nMembers];
   const size_t cb = prec == LGPU_MIXED ? 4 : 8, gb = cb;
   const int64_t plane = (int64_t)(align_up(E * cb) / cb);
   e->planeStride = plane;

   // Arena: state first (snapshot-able), then connectivity and scratch.
   struct Slot { void **dst; size_t bytes; };
   std::vector<Slot> slots;
   auto add = [&](void **dst, size_t bytes) { slots.push_back({dst, align_up(bytes)}); };
   double **stateNode[] = {&s.x, &s.y, &s.z, &s.xd, &s.yd, &s.zd};
   // two doubles of padding, which the kinematics kernel's pair copies may
   // read past the last node
   for (double **p : stateNode) add((void **)p, 8 * (N + 2));
   if (e->brick) {
      // the second node buffer is state too: either may be current
      double **second[] = {&s.xo, &s.yo, &s.zo, &s.xdo, &s.ydo, &s.zdo};
      for (double **p : second) add((void **)p, 8 * (N + 2));
   }
   double **stateElem[] = {&s.e, &s.v};
   for (double **p : stateElem) add((void **)p, 8 * E);
   void **statePqs[] = {&s.p, &s.q, &s.ss};
   for (void **p : statePqs) add(p, gb * E);
   EnsTime &t = e->t;
   double **tf[] = {&t.time, &t.deltatime, &t.dtcourant, &t.dthydro, &t.stoptime, &t.dtfixed,
                    &t.dtmax, &t.multlb, &t.multub};
   for (double **p : tf) add((void **)p, 8 * (size_t)nMembers);
   add((void **)&t.cycle, 4 * (size_t)nMembers);
   add((void **)&t.active, 4 * (size_t)nMembers);
   add((void **)&t.maxCycle, 4);
   add((void **)&s.memberErr, 4 * (size_t)nMembers * kNumErrSites);
   add((void **)&s.memberDtOut, 16 * (size_t)nMembers);
   const size_t stateSlots = slots.size();
   add((void **)&s.nodalMass, 8 * N);
   double **elemFix[] = {&s.volo, &s.vnew, &s.delv, &s.elemMass, &s.arealg, &s.vdov};
   for (double **p : elemFix) add((void **)p, 8 * E);
   void **grads[] = {&s.delx_xi, &s.delx_eta, &s.delx_zeta, &s.delv_xi, &s.delv_eta, &s.delv_zeta};
   for (void **p : grads) add(p, gb * E);
   add((void **)&s.nodeBC, N);
   add((void **)&s.nodeElemStart, 4 * (N + 1));
   add((void **)&s.cornerList, 4 * std::max<size_t>(nCorner, 1));
   add((void **)&s.nodelist, 32 * E);
   const int32_t **nbr[] = {&s.lxim, &s.lxip, &s.letam, &s.letap, &s.lzetam, &s.lzetap, &s.elemBC};
   for (const int32_t **p : nbr) add((void **)p, 4 * E);
   if (!e->brick) add(&s.corner, cb * (size_t)plane * 48);
   add((void **)&s.perm, 4 * E);
   add((void **)&s.err, 4 * kNumErrSites);
   add((void **)&s.dtPartial, 16 * (size_t)blockStart[nMembers]);
   add((void **)&s.dtOut, 16);
   add((void **)&s.memberNodeStart, 4 * ((size_t)nMembers + 1));
   add((void **)&s.memberElemStart, 4 * ((size_t)nMembers + 1));
   add((void **)&s.eosBlock, sizeof(EosBlock) * (size_t)blockStart[nMembers]);
   add((void **)&s.eosSlot, sizeof(EosSlot) * (size_t)blockStart[nMembers]);
   add((void **)&s.memberBlockStart, 4 * ((size_t)nMembers + 1));
   size_t total = 0, stateBytes = 0;
   for (size_t i = 0; i < slots.size(); ++i) {
      if (i == stateSlots) stateBytes = total;
      total += slots[i].bytes;
   }
   if (hipMalloc((void **)&e->arena, total) != hipSuccess) {
      (void)hipGetLastError();
      return bail(LGPU_ENOMEM);
   }
   e->arenaBytes = total;
   e->stateBytes = stateBytes;
   if (hipMemset(e->arena, 0, total) != hipSuccess) return bail(LGPU_EDEVICE);
   size_t off = 0;
   for (const Slot &sl : slots) {
      *sl.dst = e->arena + off;
      off += sl.bytes;
   }
   s.numElem = (int32_t)E;
   s.numNode = (int32_t)N;
   s.eosBlocks = blockStart[nMembers];
   s.xcdRemap = 1;
   s.isBrick = 0;
   s.nMembers = nMembers;
   s.memberDt = t.deltatime;
   s.memberActive = t.active;
   s.ensTime = t;

   // Concatenated connectivity.
   std::vector<int32_t> nodelist(8 * E), nbrs[7], nodeElemStart(N + 1), corner(nCorner);
   for (auto &v : nbrs) v.assign(E, 0);
   std::vector<uint8_t> bc(N, 0);
   for (int32_t m = 0; m < nMembers; ++m) {
      const lgpu_mesh_desc &d = members[m];
      const int32_t n0 = e->nodeStart[m], e0 = e->elemStart[m];
      for (int64_t i = 0; i < 8 * (int64_t)d.numElem; ++i) nodelist[8 * (size_t)e0 + i] = d.nodelist[i] + n0;
      const int32_t *src[7] = {d.lxim, d.lxip, d.letam, d.letap, d.lzetam, d.lzetap, d.elemBC};
      for (int a = 0; a < 7; ++a)
         for (int32_t i = 0; i < d.numElem; ++i)
            nbrs[a][(size_t)(e0 + i)] = (a < 6) ? src[a][i] + e0 : src[a][i];
      for (int32_t n = 0; n <= d.numNode; ++n)
         nodeElemStart[(size_t)(n0 + n)] = (int32_t)(cornerStart[m] + d.nodeElemStart[n]);
      for (int32_t c = 0; c < d.nodeElemStart[d.numNode]; ++c)
         corner[(size_t)(cornerStart[m] + c)] = d.nodeElemCornerList[c] + 8 * e0;
      const int32_t *sy[3] = {d.symmX, d.symmY, d.symmZ};
      const int32_t ns[3] = {d.numSymmX, d.numSymmY, d.numSymmZ};
      for (int a = 0; a < 3; ++a)
         for (int32_t i = 0; i < ns[a]; ++i) bc[(size_t)(n0 + sy[a][i])] |= (uint8_t)(1u << a);
   }
   auto h2d = [&](void *dst, const void *src, size_t bytes) {
      return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
   };
   std::vector<double> ones(E, 1.0);
   bool ok = h2d((void *)s.nodelist, nodelist.data(), 4 * nodelist.size()) &&
             h2d((void *)s.lxim, nbrs[0].data(), 4 * E) && h2d((void *)s.lxip, nbrs[1].data(), 4 * E) &&
             h2d((void *)s.letam, nbrs[2].data(), 4 * E) && h2d((void *)s.letap, nbrs[3].data(), 4 * E) &&
             h2d((void *)s.lzetam, nbrs[4].data(), 4 * E) && h2d((void *)s.lzetap, nbrs[5].data(), 4 * E) &&
             h2d((void *)s.elemBC, nbrs[6].data(), 4 * E) &&
             h2d((void *)s.nodeElemStart, nodeElemStart.data(), 4 * (N + 1)) &&
             (nCorner == 0 || h2d((void *)s.cornerList, corner.data(), 4 * nCorner)) &&
             h2d((void *)s.perm, perm.data(), 4 * E) &&
             h2d((void *)s.nodeBC, bc.data(), N) &&
             h2d((void *)s.memberNodeStart, e->nodeStart.data(), 4 * e->nodeStart.size()) &&
             h2d((void *)s.memberElemStart, e->elemStart.data(), 4 * e->elemStart.size()) &&
             h2d((void *)s.eosBlock, eosBlock.data(), sizeof(EosBlock) * eosBlock.size()) &&
             h2d((void *)s.eosSlot, eosSlots.data(), sizeof(EosSlot) * eosSlots.size()) &&
             h2d((void *)s.memberBlockStart, blockStart.data(), 4 * blockStart.size()) &&
             h2d(s.v, ones.data(), 8 * E);
   if (!ok) return bail(LGPU_EDEVICE);
   if (e->brick && set_brick_choice(e, pick_brick_kernels(e)) != LGPU_OK) return bail(LGPU_EDEVICE);
   if (copies_by_kernel(e->nodeCount, e->elemCount, kSmallMembers, prec == LGPU_MIXED))
      e->small.limit = kSmallMembers;
   if (hipHostMalloc((void **)&e->host, small_copy_bytes(e->small.limit) + (size_t)nMembers * (9 * 8 + 8) + 64 +
                                            (size_t)nMembers * kNumErrSites * 4,
                     hipHostMallocDefault) != hipSuccess)
      return bail(LGPU_ENOMEM);
   e->small.init(e->host);
   *out = e;
   return LGPU_OK;
}

void lgpu_ensemble_destroy(lgpu_ensemble *e)
{
   if (!e) return;
   if (e->stream) (void)hipStreamSynchronize(e->stream);
   drop_graph(e);
   if (e->arena) (void)hipFree(e->arena);
   if (e->tables) (void)hipFree(e->tables);
   if (e->host) (void)hipHostFree(e->host);
   if (e->stream) (void)hipStreamDestroy(e->stream);
   delete e;
}

int lgpu_ensemble_upload(lgpu_ensemble *e, int32_t member, int field, const double *host)
{
   if (!e || !host || member < 0 || member >= e->nMembers) return LGPU_EINVAL;
   bool isElem, narrow;
   double *base = field_base(e, field, isElem, narrow);
   if (!base) return LGPU_EINVAL;
   const size_t n = isElem ? (size_t)e->elemCount[member] : (size_t)e->nodeCount[member];
   const size_t off = isElem ? (size_t)e->elemStart[member] : (size_t)e->nodeStart[member];
   void *dst = narrow ? (void *)(reinterpret_cast<float *>(base) + off) : (void *)(base + off);
   if (e->small.takes(n)) {
      ENS_HIP(e, e->small.upload(host, dst, narrow, (int)n, e->stream));
      return LGPU_OK;
   }
   ENS_HIP(e, hipStreamSynchronize(e->stream));
   if (narrow && converts_on_device(host, (int64_t)n, true)) {
      double *wide = scratch_doubles(e);
      ENS_HIP(e, hipMemcpy(wide, host, 8 * n, hipMemcpyHostToDevice));
      ENS_HIP(e, launch_narrow(wide, static_cast<float *>(dst), (int64_t)n, e->stream));
      ENS_HIP(e, hipStreamSynchronize(e->stream));
   } else if (narrow) {
      std::vector<float> tmp(n);
      for (size_t i = 0; i < n; ++i) tmp[i] = (float)host[i];
      ENS_HIP(e, hipMemcpy(dst, tmp.data(), 4 * n, hipMemcpyHostToDevice));
   } else {
      ENS_HIP(e, hipMemcpy(dst, host, 8 * n, hipMemcpyHostToDevice));
   }
   return LGPU_OK;
}

int lgpu_ensemble_download(lgpu_ensemble *e, int32_t member, int field, double *host)
{
   if (!e || !host || member < 0 || member >= e->nMembers) return LGPU_EINVAL;
   bool isElem, narrow;
   double *base = field_base(e, field, isElem, narrow);
   if (!base) return LGPU_EINVAL;
   const size_t n = isElem ? (size_t)e->elemCount[member] : (size_t)e->nodeCount[member];
   const size_t off = isElem ? (size_t)e->elemStart[member] : (size_t)e->nodeStart[member];
   void *src = narrow ? (void *)(reinterpret_cast<float *>(base) + off) : (void *)(base + off);
   if (e->small.takes(n)) {
      ENS_HIP(e, e->small.download(src, host, narrow, (int)n, e->stream));
      return LGPU_OK;
   }
   ENS_HIP(e, hipStreamSynchronize(e->stream));
   if (narrow && converts_on_device(host, (int64_t)n, false)) {
      double *wide = scratch_doubles(e);
      ENS_HIP(e, launch_widen(static_cast<float *>(src), wide, (int64_t)n, e->stream));
      ENS_HIP(e, hipStreamSynchronize(e->stream));
      ENS_HIP(e, hipMemcpy(host, wide, 8 * n, hipMemcpyDeviceToHost));
   } else if (narrow) {
      std::vector<float> tmp(n);
      ENS_HIP(e, hipMemcpy(tmp.data(), src, 4 * n, hipMemcpyDeviceToHost));
      for (size_t i = 0; i < n; ++i) host[i] = tmp[i];
   } else {
      ENS_HIP(e, hipMemcpy(host, src, 8 * n, hipMemcpyDeviceToHost));
   }
   return LGPU_OK;
}

int lgpu_ensemble_run(lgpu_ensemble *e, lgpu_time_state *ts, int32_t maxCycle, int32_t *status)
{
   if (!e || !ts) return LGPU_EINVAL;
   const int M = e->nMembers;
   // Pinned staging: 9 double arrays, cycle, active, err.
   double *hd = reinterpret_cast<double *>(e->host + small_copy_bytes(e->small.limit));
   int32_t *hcyc = reinterpret_cast<int32_t *>(hd + 9 * (size_t)M);
   int32_t *hact = hcyc + M;
   int32_t *herr = hact + M;
   double *cols[9];
   for (int i = 0; i < 9; ++i) cols[i] = hd + (size_t)i * M;
   for (int m = 0; m < M; ++m) {
      cols[0][m] = ts[m].time;
      cols[1][m] = ts[m].deltatime;
      cols[2][m] = ts[m].dtcourant;
      cols[3][m] = ts[m].dthydro;
      cols[4][m] = ts[m].stoptime;
      cols[5][m] = ts[m].dtfixed;
      cols[6][m] = ts[m].dtmax;
      cols[7][m] = ts[m].deltatimemultlb;
      cols[8][m] = ts[m].deltatimemultub;
      hcyc[m] = ts[m].cycle;
      hact[m] = 1;
   }
   EnsTime &t = e->t;
   double *dcols[9] = {t.time, t.deltatime, t.dtcourant, t.dthydro, t.stoptime, t.dtfixed,
                       t.dtmax, t.multlb, t.multub};
   for (int i = 0; i < 9; ++i)
      ENS_HIP(e, hipMemcpyAsync(dcols[i], cols[i], 8 * (size_t)M, hipMemcpyHostToDevice, e->stream));
   ENS_HIP(e, hipMemcpyAsync(t.cycle, hcyc, 4 * (size_t)M, hipMemcpyHostToDevice, e->stream));
   ENS_HIP(e, hipMemcpyAsync(t.active, hact, 4 * (size_t)M, hipMemcpyHostToDevice, e->stream));
   // dt results feed the first TimeIncrement of members past cycle 0.
   {
      std::vector<double> dtout(2 * (size_t)M);
      for (int m = 0; m < M; ++m) {
         dtout[2 * (size_t)m] = ts[m].dtcourant;
         dtout[2 * (size_t)m + 1] = ts[m].dthydro;
      }
      ENS_HIP(e, hipMemcpyAsync(e->s.memberDtOut, dtout.data(), 16 * (size_t)M,
                                hipMemcpyHostToDevice, e->stream));
      ENS_HIP(e, hipMemcpyAsync(t.maxCycle, &maxCycle, 4, hipMemcpyHostToDevice, e->stream));
      ENS_HIP(e, hipStreamSynchronize(e->stream));
   }
   if (e->useGraph && !e->timing && !e->exec) {
      const int r = build_graph(e);
      if (r) return r;
   }
   Events<2> start;
   if (e->timing) {
      for (auto &x : start.ev) ENS_HIP(e, hipEventCreate(&x));
      ENS_HIP(e, hipEventRecord(start.ev[0], e->stream));
   }
   hipLaunchKernelGGL(k_time_increment_ens, dim3((unsigned)((M + 63) / 64)), dim3(64), 0, e->stream,
                      e->t, e->s.memberDtOut, e->s.memberErr, M);
   ENS_HIP(e, hipGetLastError());
   if (e->timing) {
      float ms = 0.f;
      ENS_HIP(e, hipEventRecord(start.ev[1], e->stream));
      ENS_HIP(e, hipStreamSynchronize(e->stream));
      ENS_HIP(e, hipEventElapsedTime(&ms, start.ev[0], start.ev[1]));
      count_launch(e, kETime, ms);
   }
   // Cycles are enqueued in batches between host checks of the loop flags, and
   // no more of them than the member with the most cycles left can run: only
   // a run that ends at stoptime (or on an error) enqueues no-op cycles.
   int64_t remaining = 0;
   for (int m = 0; m < M; ++m)
      remaining = std::max<int64_t>(remaining, (int64_t)maxCycle - ts[m].cycle);
   while (remaining > 0) {
      const int batch = (int)std::min<int64_t>(8, remaining);
      remaining -= batch;
      for (int b = 0; b < batch; ++b) {
         if (e->timing) {
            const int r = timed_cycle_any(e);
            if (r) return r;
         } else if (e->useGraph) {
            const int r = launch_graph(e);
            if (r) return r;
         } else {
            enqueue_cycle(e);
            ENS_HIP(e, hipGetLastError());
         }
      }
      ENS_HIP(e, hipMemcpyAsync(hact, t.active, 4 * (size_t)M, hipMemcpyDeviceToHost, e->stream));
      ENS_HIP(e, hipStreamSynchronize(e->stream));
      bool any = false;
      for (int m = 0; m < M; ++m) any = any || hact[m] != 0;
      if (!any) break;
   }
   // Read back the time state; a member's last dt results are in
   // memberDtOut (inactive members leave them untouched).
   for (int i = 0; i < 9; ++i)
      ENS_HIP(e, hipMemcpyAsync(cols[i], dcols[i], 8 * (size_t)M, hipMemcpyDeviceToHost, e->stream));
   ENS_HIP(e, hipMemcpyAsync(hcyc, t.cycle, 4 * (size_t)M, hipMemcpyDeviceToHost, e->stream));
   ENS_HIP(e, hipMemcpyAsync(herr, e->s.memberErr, 4 * (size_t)M * kNumErrSites,
                             hipMemcpyDeviceToHost, e->stream));
   std::vector<double> dtout(2 * (size_t)M);
   ENS_HIP(e, hipMemcpyAsync(dtout.data(), e->s.memberDtOut, 16 * (size_t)M, hipMemcpyDeviceToHost,
                             e->stream));
   ENS_HIP(e, hipStreamSynchronize(e->stream));
   int worst = LGPU_OK;
   for (int m = 0; m < M; ++m) {
      ts[m].time = cols[0][m];
      ts[m].deltatime = cols[1][m];
      ts[m].cycle = hcyc[m];
      if (hcyc[m] > 0) {
         ts[m].dtcourant = dtout[2 * (size_t)m];
         ts[m].dthydro = dtout[2 * (size_t)m + 1];
      }
      const int32_t *er = herr + (size_t)m * kNumErrSites;
      int st = LGPU_OK;
      if (er[kErrForceDeterm] || er[kErrHourglassV] || er[kErrKinVnew]) st = LGPU_VOLUME_ERROR;
      else if (er[kErrQStop]) st = LGPU_QSTOP_ERROR;
      else if (er[kErrMaterialV]) st = LGPU_VOLUME_ERROR;
      if (status) status[m] = st;
      if (st != LGPU_OK && worst == LGPU_OK) worst = st;
   }
   return worst;
}

int lgpu_ensemble_set_option(lgpu_ensemble *e, int option, int64_t value)
{
   if (!e) return LGPU_EINVAL;
   switch (option) {
   case LGPU_ENS_OPT_GRAPH:
      e->useGraph = value != 0;
      drop_graph(e);
      return LGPU_OK;
   case LGPU_ENS_OPT_TIMING:
      e->timing = value != 0;
      return LGPU_OK;
   case LGPU_ENS_OPT_BLOCK_FORCE:
   case LGPU_ENS_OPT_BLOCK_NODE:
   case LGPU_ENS_OPT_BLOCK_KIN:
      if (value != 64 && value != 128 && value != 256) return LGPU_EINVAL;
      e->block[option - LGPU_ENS_OPT_BLOCK_FORCE] = (int)value;
      drop_graph(e);
      return LGPU_OK;
   case LGPU_ENS_OPT_XCD_REMAP:
      e->s.xcdRemap = value ? 1 : 0;
      drop_graph(e);
      return LGPU_OK;
   case LGPU_ENS_OPT_BRICK_CHUNK:
   case LGPU_ENS_OPT_KIN_CHUNK: {
      if (!e->brick || value < 1 || value > 1024) return LGPU_EINVAL;
      BrickChoice want = e->choice;
      if (option == LGPU_ENS_OPT_BRICK_CHUNK) {
         want.nodalChunk = (int)value;
         want.nodalBlock = want.nodalChunk == want.blockChunk;
      } else {
         want.kinChunk = (int)value;
         want.kinFlat = want.kinChunk == want.flatChunk;
      }
      return set_brick_choice(e, want);
   }
   case LGPU_ENS_OPT_NODAL_KERNEL:
   case LGPU_ENS_OPT_KIN_KERNEL: {
      if (!e->brick || (value != 0 && value != 1)) return LGPU_EINVAL;
      BrickChoice want = e->choice;
      if (option == LGPU_ENS_OPT_NODAL_KERNEL) want.choose_nodal(value == 1);
      else want.choose_kin(value == 1);
      return set_brick_choice(e, want);
   }
   default:
      return LGPU_EINVAL;
   }
}

int lgpu_ensemble_get_option(lgpu_ensemble *e, int option, int64_t *value)
{
   if (!e || !value) return LGPU_EINVAL;
   switch (option) {
   case LGPU_ENS_OPT_GRAPH: *value = e->useGraph; return LGPU_OK;
   case LGPU_ENS_OPT_TIMING: *value = e->timing; return LGPU_OK;
   case LGPU_ENS_OPT_BLOCK_FORCE:
   case LGPU_ENS_OPT_BLOCK_NODE:
   case LGPU_ENS_OPT_BLOCK_KIN: *value = e->block[option - LGPU_ENS_OPT_BLOCK_FORCE]; return LGPU_OK;
   case LGPU_ENS_OPT_XCD_REMAP: *value = e->s.xcdRemap; return LGPU_OK;
   case LGPU_ENS_OPT_BRICK_CHUNK:
      if (!e->brick) return LGPU_EINVAL;
      *value = e->choice.nodalChunk;
      return LGPU_OK;
   case LGPU_ENS_OPT_KIN_CHUNK:
      if (!e->brick) return LGPU_EINVAL;
      *value = e->choice.kinChunk;
      return LGPU_OK;
   case LGPU_ENS_OPT_PATH: *value = e->brick ? 1 : 0; return LGPU_OK;
   case LGPU_ENS_OPT_NODAL_KERNEL:
   case LGPU_ENS_OPT_KIN_KERNEL:
      if (!e->brick) return LGPU_EINVAL;
      *value = option == LGPU_ENS_OPT_NODAL_KERNEL ? e->choice.nodalBlock : e->choice.kinFlat;
      return LGPU_OK;
   default: return LGPU_EINVAL;
   }
}

int lgpu_ensemble_autotune(lgpu_ensemble *e, const lgpu_time_state *ts, int32_t trialCycles)
{
   if (!e || !ts || trialCycles < 1) return LGPU_EINVAL;
   // The trials advance the state: snapshot the state part of the arena (on
   // the brick path both node buffers) and restore it, and the node-buffer
   // parity, after every trial.
   char *snap = nullptr;
   ENS_HIP(e, hipMalloc((void **)&snap, e->stateBytes));
   ENS_HIP(e, hipMemcpyAsync(snap, e->arena, e->stateBytes, hipMemcpyDeviceToDevice, e->stream));
   const int M = e->nMembers;
   const int parity0 = e->parity;
   std::vector<lgpu_time_state> tsv(ts, ts + M);
   const bool savedTiming = e->timing, savedGraph = e->useGraph;
   e->timing = true;
   auto trial = [&](float ms[kENumKernels]) -> int {
      for (int i = 0; i < kENumKernels; ++i) ms[i] = 0.f;
      for (int i = 0; i < kENumKernels; ++i) {
         e->kLaunches[i] = 0;
         e->kMs[i] = 0.0;
      }
      std::vector<lgpu_time_state> t2 = tsv;
      const int r = lgpu_ensemble_run(e, t2.data(), t2[0].cycle + trialCycles, nullptr);
      if (r <= -100) return r;
      for (int i = 0; i < kENumKernels; ++i)
         ms[i] = e->kLaunches[i] ? (float)(e->kMs[i] / e->kLaunches[i]) : 0.f;
      ENS_HIP(e, hipMemcpyAsync(e->arena, snap, e->stateBytes, hipMemcpyDeviceToDevice, e->stream));
      ENS_HIP(e, hipStreamSynchronize(e->stream));
      if (e->parity != parity0) swap_nodes(e);
      return LGPU_OK;
   };
   int r = LGPU_OK;
   if (e->brick) {
      // The chunks of the walking kernels, with k_nodal_block and k_kin_flat
      // against the best of them, then the XCD mapping.
      const int nodalCands[] = {4, 6, 8, 11, 16, 22}, kinCands[] = {4, 6, 8, 12, 16};
      const BrickChoice before = e->choice;
      BrickChoice best = before;
      auto time_choice = [&](const BrickChoice &want, int kernel, float &t) {
         float ms[kENumKernels];
         int st = set_brick_choice(e, want);
         if (!st) st = trial(ms);
         t = st ? 1e30f : ms[kernel];
         return st;
      };
      float bestMs = 1e30f, t = 0.f;
      for (int c : nodalCands) {
         if (r) break;
         BrickChoice want = best;
         want.nodalChunk = c;
         want.choose_nodal(false);
         r = time_choice(want, kENodalBrick, t);
         if (!r && t < bestMs) {
            bestMs = t;
            best.nodalChunk = c;
         }
      }
      best.choose_nodal(true);
      if (!r) r = time_choice(best, kENodalBrick, t);
      best.choose_nodal(t <= bestMs);
      bestMs = 1e30f;
      for (int c : kinCands) {
         if (r) break;
         BrickChoice want = best;
         want.kinChunk = c;
         want.choose_kin(false);
         r = time_choice(want, kEKinBrick, t);
         if (!r && t < bestMs) {
            bestMs = t;
            best.kinChunk = c;
         }
      }
      best.choose_kin(true);
      if (!r) r = time_choice(best, kEKinBrick, t);
      best.choose_kin(t <= bestMs);
      if (!r) r = set_brick_choice(e, best);
      else (void)set_brick_choice(e, before);
   } else {
      // Each of the three launch-shape-sensitive kernels is tuned over the
      // block sizes.
      const int cands[3] = {64, 128, 256};
      const int kern[3] = {kEForce, kENode, kEKin};
      for (int which = 0; which < 3 && !r; ++which) {
         float best = 1e30f;
         int bestB = e->block[which];
         for (int b : cands) {
            e->block[which] = b;
            float ms[kENumKernels];
            r = trial(ms);
            if (r) break;
            if (ms[kern[which]] < best) {
               best = ms[kern[which]];
               bestB = b;
            }
         }
         e->block[which] = bestB;
      }
   }
   if (!r) {
      float tot[2];
      for (int remap = 0; remap < 2 && !r; ++remap) {
         e->s.xcdRemap = remap;
         float ms[kENumKernels];
         r = trial(ms);
         tot[remap] = 0.f;
         for (int i = 0; i < kENumKernels; ++i)
            if (i != kETime && i != kEDt) tot[remap] += ms[i];
      }
      if (!r) e->s.xcdRemap = (tot[1] <= tot[0]) ? 1 : 0;
   }
   e->timing = savedTiming;
   e->useGraph = savedGraph;
   for (int i = 0; i < kENumKernels; ++i) {
      e->kLaunches[i] = 0;
      e->kMs[i] = 0.0;
   }
   // the cycle graphs of the chosen configuration, built here rather than
   // in the first run
   drop_graph(e);
   if (!r && e->useGraph && !e->timing) r = build_graph(e);
   (void)hipFree(snap);
   return r;
}

int lgpu_ensemble_kernel_stats(lgpu_ensemble *e, int kernel, int64_t *launches, double *total_ms)
{
   if (!e || kernel < 0 || kernel >= kENumKernels) return LGPU_EINVAL;
   if (launches) *launches = e->kLaunches[kernel];
   if (total_ms) *total_ms = e->kMs[kernel];
   return LGPU_OK;
}

const char *lgpu_ensemble_kernel_name(int kernel)
{
   return (kernel >= 0 && kernel < kENumKernels) ? kEnsKernelNames[kernel] : "";
}

int lgpu_ensemble_num_kernels(void) { return kENumKernels; }

int64_t lgpu_ensemble_num_elem(lgpu_ensemble *e) { return e ? e->s.numElem : 0; }

const char *lgpu_ensemble_last_error(lgpu_ensemble *e) { return e ? e->lastError.c_str() : ""; }

} // extern "C"
