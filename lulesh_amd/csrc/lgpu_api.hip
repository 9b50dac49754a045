// lgpu_api.hip -- device context and C ABI (include/lulesh_gpu.h).
//
// One context owns one HIP stream and one device arena holding every array
// the step touches, laid out SoA with 256-byte aligned planes.  All
// connectivity is validated on the host before the first launch, so no
// kernel ever indexes outside the arena.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <new>
#include <string>
#include <vector>

#include "lgpu_brick.h"
#include "lgpu_convert.h"
#include "lgpu_kernels.h"
#include "lgpu_launch.h"
#include "lgpu_setup.h"
#include "lgpu_time.h"
#include "lgpu_wait.h"
#include "lulesh_gpu.h"

using namespace lgpu;

namespace {

enum KernelId {
   kKForce = 0, kKNode, kKKin, kKEos, kKDtReduce, kKTimeIncrement, kKNodalBrick, kKKinBrick,
   kNumKernels
};
const char *const kKernelNames[kNumKernels] = {"k_force", "k_node", "k_kin", "k_eos",
                                               "k_dt_reduce", "k_time_increment",
                                               "k_nodal_brick", "k_kin_brick"};

constexpr size_t kAlign = 256;

inline size_t align_up(size_t v) { return (v + kAlign - 1) & ~(kAlign - 1); }

// A k_eos slot and its first element.
struct PlacedSlot {
   EosSlot slot;
   int32_t elem;
};

struct TimedLaunch {
   int kernel;
   hipEvent_t start, stop;
};

} // namespace

struct lgpu_ctx {
   int device = 0;
   hipStream_t stream = nullptr;
   int32_t numElem = 0, numNode = 0, numReg = 0, cost = 0, precision = 0;
   int32_t sizeX = 0;
   int block = 256;
   bool keepDiag = false;
   std::vector<PlacedSlot> eosSlots; // in work-list order, by place within a repeat count
   int eosInterleave = 0;
   int32_t brickPerCu = 0;
   // the default tile, and the chunks that the options read while k_nodal_block
   // and k_kin_flat are in use (0: not the default kernels of this size)
   int tileW = 16, tileRows = 16, blockChunk = 0, flatChunk = 0;
   // resident workgroups: nodal brick kernels, k_force, k_eos
   int64_t brickSlots = 0, genericSlots = 0, eosResident = 0;
   bool timing = false;
   uint32_t timingMask = 0xffffffffu;
   Consts k{};
   char *arena = nullptr;
   size_t arenaBytes = 0;
   int64_t planeStride = 0; // corner plane length (elements, padded)
   DevState s{};
   // pinned: HostOut (dt[2], err[kNumErrSites], counts), time state, SmallCopy
   double *hostDt = nullptr;
   int32_t *hostErr = nullptr;
   bool hostOutFresh = false; // the last launch leaves its results in s.hostOut
   uint32_t hostSeq = 0, cycleSeq = 0; // last seq and started of s.hostOut asked for
   SmallCopy small;
   DevTime *devTime = nullptr;
   DevTime *hostTime = nullptr;
   // diagnostics storage (allocated on first use)
   double *diag = nullptr;
   std::vector<TimedLaunch> pending;
   std::vector<hipEvent_t> eventPool;
   int64_t kLaunches[kNumKernels] = {};
   double kMs[kNumKernels] = {};
   std::string lastError;
};

namespace {

int set_hip_error(lgpu_ctx *c, hipError_t e, const char *what)
{
   if (e == hipSuccess) return LGPU_OK;
   if (c) c->lastError = std::string(what) + ": " + hipGetErrorString(e);
   return (e == hipErrorOutOfMemory) ? LGPU_ENOMEM : LGPU_EDEVICE;
}

#define HIP_OR_RETURN(c, call)                                   \
   do {                                                          \
      const hipError_t e_ = (call);                              \
      if (e_ != hipSuccess) return set_hip_error((c), e_, #call); \
   } while (0)

hipEvent_t take_event(lgpu_ctx *c)
{
   if (!c->eventPool.empty()) {
      hipEvent_t e = c->eventPool.back();
      c->eventPool.pop_back();
      return e;
   }
   hipEvent_t e = nullptr;
   if (hipEventCreate(&e) != hipSuccess) return nullptr;
   return e;
}

// Folds finished timed launches into the per-kernel totals.  Call only after
// the stream has been synchronized.
void harvest_timing(lgpu_ctx *c)
{
   for (TimedLaunch &t : c->pending) {
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, t.start, t.stop) == hipSuccess) {
         c->kLaunches[t.kernel] += 1;
         c->kMs[t.kernel] += ms;
      }
      c->eventPool.push_back(t.start);
      c->eventPool.push_back(t.stop);
   }
   c->pending.clear();
}

template <class F>
int timed(lgpu_ctx *c, int kernel, F &&launch)
{
   TimedLaunch t{kernel, nullptr, nullptr};
   const bool on = c->timing && ((c->timingMask >> kernel) & 1u);
   if (on) {
      t.start = take_event(c);
      t.stop = take_event(c);
      if (t.start && t.stop) HIP_OR_RETURN(c, hipEventRecord(t.start, c->stream));
   }
   launch();
   HIP_OR_RETURN(c, hipGetLastError());
   if (on && t.start && t.stop) {
      HIP_OR_RETURN(c, hipEventRecord(t.stop, c->stream));
      c->pending.push_back(t);
   }
   return LGPU_OK;
}

bool in_range(const int32_t *a, int64_t n, int32_t lo, int32_t hi)
{
   for (int64_t i = 0; i < n; ++i)
      if (a[i] < lo || a[i] >= hi) return false;
   return true;
}

int validate(const lgpu_mesh_desc *d, std::string &why)
{
   if (!d) { why = "null description"; return LGPU_EINVAL; }
   const int64_t E = d->numElem, N = d->numNode;
   if (E < 1 || N < 1 || E > (INT32_MAX / 8)) { why = "numElem/numNode out of range"; return LGPU_EINVAL; }
   if (!d->nodelist || !d->lxim || !d->lxip || !d->letam || !d->letap || !d->lzetam ||
       !d->lzetap || !d->elemBC || !d->nodeElemStart || !d->nodeElemCornerList ||
       !d->regElemSize || !d->regElemlist) {
      why = "missing array";
      return LGPU_EINVAL;
   }
   if (d->precision != LGPU_FP64 && d->precision != LGPU_MIXED && d->precision != LGPU_FP64_FMA) {
      why = "precision";
      return LGPU_EINVAL;
   }
   if (d->numReg < 1 || d->cost < 0) { why = "numReg/cost"; return LGPU_EINVAL; }
   if (!in_range(d->nodelist, 8 * E, 0, (int32_t)N)) { why = "nodelist index out of range"; return LGPU_EINVAL; }
   const int32_t *nb[6] = {d->lxim, d->lxip, d->letam, d->letap, d->lzetam, d->lzetap};
   for (const int32_t *a : nb)
      if (!in_range(a, E, 0, (int32_t)E)) { why = "face neighbour out of range"; return LGPU_EINVAL; }
   if (d->nodeElemStart[0] != 0) { why = "nodeElemStart[0] != 0"; return LGPU_EINVAL; }
   for (int64_t n = 0; n < N; ++n)
      if (d->nodeElemStart[n + 1] < d->nodeElemStart[n]) { why = "nodeElemStart not monotone"; return LGPU_EINVAL; }
   const int64_t nc = d->nodeElemStart[N];
   if (nc > 8 * E) { why = "corner list too long"; return LGPU_EINVAL; }
   if (!in_range(d->nodeElemCornerList, nc, 0, (int32_t)(8 * E))) { why = "corner index out of range"; return LGPU_EINVAL; }
   const int32_t *sy[3] = {d->symmX, d->symmY, d->symmZ};
   const int32_t ns[3] = {d->numSymmX, d->numSymmY, d->numSymmZ};
   for (int a = 0; a < 3; ++a) {
      if (ns[a] < 0 || (ns[a] > 0 && !sy[a])) { why = "symmetry set"; return LGPU_EINVAL; }
      if (ns[a] > 0 && !in_range(sy[a], ns[a], 0, (int32_t)N)) { why = "symmetry node out of range"; return LGPU_EINVAL; }
   }
   // regions must partition the elements
   std::vector<uint8_t> seen((size_t)E, 0);
   int64_t total = 0;
   for (int r = 0; r < d->numReg; ++r) {
      const int32_t len = d->regElemSize[r];
      if (len < 0 || (len > 0 && !d->regElemlist[r])) { why = "region list"; return LGPU_EINVAL; }
      for (int32_t i = 0; i < len; ++i) {
         const int32_t e = d->regElemlist[r][i];
         if (e < 0 || e >= E || seen[(size_t)e]) { why = "regions do not partition the elements"; return LGPU_EINVAL; }
         seen[(size_t)e] = 1;
      }
      total += len;
   }
   if (total != E) { why = "regions do not cover every element"; return LGPU_EINVAL; }
   return LGPU_OK;
}

// k_eos dispatch order.  k = 0: work-list order (largest repeat count
// first).  k > 0: the workgroups of the largest repeat count are spread out,
// one every k + 1 dispatches, with the others between them, so that
// compute-bound and memory-bound workgroups share the CUs.  The others come in
// the order of their place in the mesh, whatever their repeat count, so that
// the neighbour gradients and partly used lines of one part of the mesh are
// fetched while they are in the caches (s=192, k = 4: FP64 r21 299.6 -> 291.3
// us, mixed r11 207 -> 190.8 us against one repeat count after the other; the
// heavy workgroups in mesh order too: 302-323 and 193-203 us).  The
// dispatcher deals workgroups to the 8 XCDs in turn, so an even period would
// put every heavy workgroup on the same few XCDs (measured: period 4 nearly
// doubles the EOS time); an even k + 1 is raised to the next odd period.
int set_eos_order(lgpu_ctx *c, int k)
{
   if (k > 0 && (k + 1) % 2 == 0) ++k;
   std::vector<EosSlot> slots;
   if (k <= 0) {
      for (const PlacedSlot &p : c->eosSlots) slots.push_back(p.slot);
   } else {
      const std::vector<PlacedSlot> &all = c->eosSlots;
      auto group_end = [&](size_t from) {
         while (from < all.size() && all[from].slot.rep == all[from - 1].slot.rep) ++from;
         return from;
      };
      size_t end = all.empty() ? 0 : group_end(1);
      std::vector<PlacedSlot> heavy(all.begin(), all.begin() + (std::ptrdiff_t)end), rest;
      while (end < all.size()) { // the other groups merged, each in the order of the mesh
         const size_t from = end;
         end = group_end(from + 1);
         std::vector<PlacedSlot> merged(rest.size() + (end - from));
         std::merge(rest.begin(), rest.end(), all.begin() + (std::ptrdiff_t)from, all.begin() + (std::ptrdiff_t)end,
                    merged.begin(), [](const PlacedSlot &a, const PlacedSlot &b) { return a.elem < b.elem; });
         rest.swap(merged);
      }
      // The FP64 forms walk the mesh from the top down: the kinematics pass
      // before k_eos sweeps it bottom to top, so its last outputs are still
      // in the caches when k_eos starts (s=192, 21 regions: k_eos 367 -> 357
      // us; the mixed form gains nothing and its next nodal pass loses 2 us,
      // so it keeps the ascending walk).
      if (c->precision != LGPU_MIXED) {
         std::reverse(heavy.begin(), heavy.end());
         std::reverse(rest.begin(), rest.end());
      }
      size_t h = 0, r = 0;
      while (h < heavy.size() || r < rest.size()) {
         if (h < heavy.size()) slots.push_back(heavy[h++].slot);
         for (int j = 0; j < k && r < rest.size(); ++j) slots.push_back(rest[r++].slot);
      }
   }
   c->s.eosBlocks = (int32_t)slots.size();
   HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   HIP_OR_RETURN(c, hipMemcpy(const_cast<EosSlot *>(c->s.eosSlot), slots.data(),
                              sizeof(EosSlot) * slots.size(), hipMemcpyHostToDevice));
   c->eosInterleave = std::max(0, k);
   return LGPU_OK;
}

// The default order: work-list order where all workgroups are resident at once,
// the longest started first; otherwise one workgroup of the largest repeat
// count every 5 dispatches, or every 3 where these are more than a fifth of
// all, so that they have started well before the end.  Every 5 / every 3 /
// work-list order, us: s=45 14.5 / 14.0 / 13.3; s=63 mixed (16 regions, 50
// repeats) 22.0 / 22.1 / 19.5; s=101 of 5 regions 51.1 / 50.2 / 51.4, of 11, shared
// between threads, 50.6 / 47.7 / 49.8; s=192 of 5 281 / 253 / 295 (20 repeats 322 /
// 299 / 390), of 11 262 / 272 / 340, of 21 287 / 296 / 346; mixed of 5 220 / 204 / 246,
// of 11 190 / 194 / 228.
int default_interleave(const lgpu_ctx *c)
{
   const int64_t all = (int64_t)c->eosSlots.size();
   if (all == 0 || all <= c->eosResident) return 0;
   int64_t heavy = 0;
   while (heavy < all && c->eosSlots[(size_t)heavy].slot.rep == c->eosSlots[0].slot.rep) ++heavy;
   return 5 * heavy > all ? 2 : 4;
}

// The kernels that the brick options ask for.  The default number of rows
// stands for the default tile, and the default chunk, where that is a small
// brick's, for its kernel: an option set to what it reads changes nothing.
void set_nodal_kernel(lgpu_ctx *c, int rows)
{
   Brick &g = c->s.brick;
   if (rows == 8) set_brick_tile(g, 16, 8);
   else set_brick_tile(g, c->tileW, c->tileRows);
   c->s.nodalBlock = rows == 16 && g.chunkZ == c->blockChunk;
}

// Thread rows as the option gives them: 16 for every tile of 256 threads.
int option_rows(const lgpu_ctx *c) { return other_tile(c->s.brick) ? 16 : c->s.brick.rows; }

// Device array of a field.  `narrow`: stored as FP32 in the mixed form (the
// Q gradients, p, q and ss).
double *real_field_ptr(lgpu_ctx *c, int f, bool &isElem, bool &narrow)
{
   isElem = f >= LGPU_E;
   narrow = c->precision == LGPU_MIXED &&
            (f >= LGPU_DELX_XI || f == LGPU_P || f == LGPU_Q || f == LGPU_SS);
   DevState &s = c->s;
   switch (f) {
   case LGPU_X: return s.x;
   case LGPU_Y: return s.y;
   case LGPU_Z: return s.z;
   case LGPU_XD: return s.xd;
   case LGPU_YD: return s.yd;
   case LGPU_ZD: return s.zd;
   case LGPU_XDD: return s.xdd;
   case LGPU_YDD: return s.ydd;
   case LGPU_ZDD: return s.zdd;
   case LGPU_FX: return s.fx;
   case LGPU_FY: return s.fy;
   case LGPU_FZ: return s.fz;
   case LGPU_NODALMASS: return s.nodalMass;
   case LGPU_E: return s.e;
   case LGPU_P: return static_cast<double *>(s.p);
   case LGPU_Q: return static_cast<double *>(s.q);
   case LGPU_QL: return s.ql;
   case LGPU_QQ: return s.qq;
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

// Device scratch of numElem doubles that nothing holds between cycles: the
// node buffer the next cycle writes (brick), or the corner planes.
double *scratch_doubles(lgpu_ctx *c)
{
   return c->s.isBrick ? c->s.xo : static_cast<double *>(c->s.corner);
}

int enable_diagnostics(lgpu_ctx *c)
{
   if (c->diag) return LGPU_OK;
   const size_t nn = align_up(sizeof(double) * (size_t)c->numNode);
   const size_t ne = align_up(sizeof(double) * (size_t)c->numElem);
   char *p = nullptr;
   HIP_OR_RETURN(c, hipMalloc((void **)&p, 6 * nn + 2 * ne));
   HIP_OR_RETURN(c, hipMemset(p, 0, 6 * nn + 2 * ne));
   c->diag = reinterpret_cast<double *>(p);
   double **node[6] = {&c->s.fx, &c->s.fy, &c->s.fz, &c->s.xdd, &c->s.ydd, &c->s.zdd};
   for (int i = 0; i < 6; ++i) *node[i] = reinterpret_cast<double *>(p + i * nn);
   c->s.ql = reinterpret_cast<double *>(p + 6 * nn);
   c->s.qq = reinterpret_cast<double *>(p + 6 * nn + ne);
   c->s.delvOut = c->s.delv;
   return LGPU_OK;
}

template <class P>
int launch_nodal(lgpu_ctx *c, double dt)
{
   c->hostOutFresh = false;
   if (c->s.isBrick) {
      const int r = timed(c, kKNodalBrick, [&] { Launch<P>::nodal_brick(c->s, c->k, dt, c->stream); });
      if (r) return r;
      // The new node state is in the second buffer: make it current.
      DevState &s = c->s;
      std::swap(s.x, s.xo);
      std::swap(s.y, s.yo);
      std::swap(s.z, s.zo);
      std::swap(s.xd, s.xdo);
      std::swap(s.yd, s.ydo);
      std::swap(s.zd, s.zdo);
      return LGPU_OK;
   }
   int r = timed(c, kKForce, [&] { Launch<P>::force(c->s, c->k, c->planeStride, c->block, c->stream); });
   if (r) return r;
   return timed(c, kKNode, [&] { Launch<P>::node(c->s, c->k, c->planeStride, dt, c->block, c->stream); });
}

template <class P>
int launch_elements(lgpu_ctx *c, double dt)
{
   int r = c->s.isBrick
              ? timed(c, kKKinBrick, [&] { Launch<P>::kin_brick(c->s, c->k, dt, c->stream); })
              : timed(c, kKKin, [&] { Launch<P>::kin(c->s, c->k, dt, c->block, c->stream); });
   if (r) return r;
   r = timed(c, kKEos, [&] { Launch<P>::eos(c->s, c->k, c->stream); });
   if (r) return r;
   c->hostOutFresh = !c->s.timeIn;
   if (c->s.timeIn) return LGPU_OK; // the dt slots are folded as the next cycle begins
   c->s.hostSeq = ++c->hostSeq;
   return timed(c, kKDtReduce, [&] { Launch<P>::dt_reduce(c->s, c->stream); });
}

int resolve_status(const int32_t *err)
{
   if (err[kErrForceDeterm] || err[kErrHourglassV] || err[kErrKinVnew]) return LGPU_VOLUME_ERROR;
   if (err[kErrQStop]) return LGPU_QSTOP_ERROR;
   if (err[kErrMaterialV]) return LGPU_VOLUME_ERROR;
   return LGPU_OK;
}

// What the context's arena and kernel path depend on.
struct CtxSpec {
   int32_t numElem = 0, numNode = 0, sizeX = 0, numReg = 0, cost = 0, precision = 0;
   bool brick = false, brickFaces = false;
   int64_t nCorner = 0; // length of the node-to-corner list
   lgpu_constants k{};
};

// Builds the context: stream, one zeroed arena with every array of the step,
// the brick tiling.  Tables and state are filled by the caller.
int alloc_context(const CtxSpec &sp, lgpu_ctx **out)
{
   lgpu_ctx *c = new (std::nothrow) lgpu_ctx();
   if (!c) return LGPU_ENOMEM;
   auto fail = [&](int code) {
      lgpu_destroy(c);
      return code;
   };
   int dev = 0;
   if (hipGetDevice(&dev) != hipSuccess) return fail(LGPU_EDEVICE);
   c->device = dev;
   c->numElem = sp.numElem;
   c->numNode = sp.numNode;
   c->numReg = sp.numReg;
   c->cost = sp.cost;
   c->precision = sp.precision;
   c->sizeX = sp.sizeX;
   const lgpu_constants &kk = sp.k;
   c->k = Consts{kk.e_cut, kk.p_cut, kk.q_cut, kk.v_cut, kk.u_cut, kk.hgcoef, kk.ss4o3,
                 kk.qstop, kk.monoq_max_slope, kk.monoq_limiter_mult, kk.qlc_monoq,
                 kk.qqc_monoq, kk.qqc, kk.eosvmax, kk.eosvmin, kk.pmin, kk.emin, kk.dvovmax,
                 kk.refdens};
   c->k.fastEos = fast_eos_consts(c->k);
   if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
      return fail(LGPU_EDEVICE);

   const bool brick = sp.brick;
   const size_t E = (size_t)sp.numElem, N = (size_t)sp.numNode;
   const size_t gradBytes = (sp.precision == LGPU_MIXED) ? 4 : 8;
   const size_t cornerBytes = (sp.precision == LGPU_MIXED) ? 4 : 8;
   const int64_t plane = (int64_t)(align_up(E * cornerBytes) / cornerBytes);
   c->planeStride = plane;
   const int64_t nCorner = sp.nCorner;
   int cus = 0;
   if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
   // every group may end in a partly filled workgroup
   const size_t eosBlocks = E / (size_t)(kEosBlock / kEosShare) + 4;

   // Arena layout.
   struct Slot { void **dst; size_t bytes; };
   std::vector<Slot> slots;
   DevState &s = c->s;
   auto add = [&](void **dst, size_t bytes) { slots.push_back({dst, align_up(bytes)}); };
   // node arrays: two doubles of padding, which the kinematics kernel's
   // pair copies may read past the last node
   double **nodeReal[] = {&s.x, &s.y, &s.z, &s.xd, &s.yd, &s.zd, &s.nodalMass};
   for (double **p : nodeReal) add((void **)p, sizeof(double) * (N + 2));
   if (brick) {
      double **second[] = {&s.xo, &s.yo, &s.zo, &s.xdo, &s.ydo, &s.zdo};
      for (double **p : second) add((void **)p, sizeof(double) * (N + 2));
   }
   add((void **)&s.nodeBC, N);
   add((void **)&s.nodeElemStart, sizeof(int32_t) * (N + 1));
   add((void **)&s.cornerList, sizeof(int32_t) * (size_t)std::max<int64_t>(nCorner, 1));
   add((void **)&s.nodelist, sizeof(int32_t) * 8 * E);
   const int32_t **nbr[] = {&s.lxim, &s.lxip, &s.letam, &s.letap, &s.lzetam, &s.lzetap, &s.elemBC};
   for (const int32_t **p : nbr) add((void **)p, sizeof(int32_t) * E);
   void **pqsArrays[] = {&s.p, &s.q, &s.ss};
   for (void **p : pqsArrays) add(p, gradBytes * E);
   double **elemReal[] = {&s.e, &s.v, &s.volo, &s.vnew, &s.delv, &s.elemMass, &s.arealg, &s.vdov};
   for (double **p : elemReal) add((void **)p, sizeof(double) * E);
   void **grads[] = {&s.delx_xi, &s.delx_eta, &s.delx_zeta, &s.delv_xi, &s.delv_eta, &s.delv_zeta};
   for (void **p : grads) add(p, gradBytes * E);
   if (!brick) add(&s.corner, cornerBytes * (size_t)plane * 48);
   add((void **)&s.perm, sizeof(int32_t) * E);
   add((void **)&s.eosSlot, sizeof(EosSlot) * eosBlocks);
   // two sets each, which the cycles of a device loop use in turn (set 0 by
   // host-driven cycles)
   add((void **)&s.err, 2 * sizeof(int32_t) * kNumErrSites);
   add((void **)&s.dtPartial, 2 * sizeof(double) * 2 * kDtSlots);
   add((void **)&s.dtOut, sizeof(double) * 2);
   add((void **)&c->devTime, 2 * sizeof(DevTime));
   size_t total = 0;
   for (const Slot &sl : slots) total += sl.bytes;
   if (hipMalloc((void **)&c->arena, total) != hipSuccess) {
      (void)hipGetLastError();
      fprintf(stderr, "lgpu_create: device arena of %zu bytes failed\n", total);
      return fail(LGPU_ENOMEM);
   }
   c->arenaBytes = total;
   if (hipMemset(c->arena, 0, total) != hipSuccess) return fail(LGPU_EDEVICE);
   size_t off = 0;
   for (const Slot &sl : slots) {
      *sl.dst = c->arena + off;
      off += sl.bytes;
   }
   // the dt slot pairs start at the key of 1.0e+20 (they go back to it after
   // every read): sign bit set on the value's bits
   {
      const double big = 1.0e+20;
      uint64_t key = 0;
      std::memcpy(&key, &big, sizeof key);
      key |= 0x8000000000000000ull;
      const std::vector<uint64_t> init(4 * (size_t)kDtSlots, key);
      if (hipMemcpy(s.dtPartial, init.data(), sizeof(uint64_t) * init.size(), hipMemcpyHostToDevice) !=
          hipSuccess)
         return fail(LGPU_EDEVICE);
   }
   s.numElem = sp.numElem;
   s.numNode = sp.numNode;
   s.xcdRemap = 1;
   s.isBrick = brick ? 1 : 0;
   c->genericSlots = (int64_t)cus * 2;
   c->eosResident = (int64_t)cus * (sp.precision == LGPU_MIXED ? PolicyMixed::kEosWaves : PolicyFp64::kEosWaves);
   s.brickFaces = (brick && sp.brickFaces) ? 1 : 0;
   if (brick) {
      Brick &g = s.brick;
      init_brick(g, sp.sizeX);
      int perCu = 0;
      switch (sp.precision) {
      case LGPU_MIXED: perCu = Launch<PolicyMixed>::nodal_brick_blocks_per_cu(); break;
      case LGPU_FP64_FMA: perCu = Launch<PolicyFp64Fma>::nodal_brick_blocks_per_cu(); break;
      default: perCu = Launch<PolicyFp64>::nodal_brick_blocks_per_cu(); break;
      }
      c->brickPerCu = perCu;
      c->brickSlots = (int64_t)cus * perCu;
      const int slots = cus * perCu; // k_nodal_block has the walk's occupancy
      pick_brick_walk(g, slots);
      // (mixed s=75: k_nodal_block 27.9 us, 28 columns in chunks of 3 29.7)
      const double tilePart = sp.precision == LGPU_MIXED && other_tile(g) ? 1.1 : 1.0;
      s.nodalBlock = block_is_faster(block_blocks(g), slots, tilePart * brick_walk_cost(g, slots));
      if (s.nodalBlock) // the chunk the walk would start from, should an option select it
         set_brick_chunk(g, pick_brick_chunk(g, slots, 4));
      else if (sp.precision == LGPU_MIXED)
         set_brick_chunk(g, pick_tail_chunk({(int64_t)g.tilesX * g.tilesY}, {g.en}, slots, 0.5, g.chunkZ));
      s.kinFlat = g.s <= kKinFlatMax;
      int kinPerCu = 0;
      switch (sp.precision) {
      case LGPU_MIXED: kinPerCu = Launch<PolicyMixed>::kin_brick_blocks_per_cu(); break;
      case LGPU_FP64_FMA: kinPerCu = Launch<PolicyFp64Fma>::kin_brick_blocks_per_cu(); break;
      default: kinPerCu = Launch<PolicyFp64>::kin_brick_blocks_per_cu(); break;
      }
      set_kin_chunk(g, pick_kin_chunk(g, cus * kinPerCu));
      c->tileW = g.tileW;
      c->tileRows = g.rows;
      c->blockChunk = s.nodalBlock ? g.chunkZ : 0;
      c->flatChunk = s.kinFlat ? g.kinChunk : 0;
   }
   *out = c;
   return LGPU_OK;
}

// The EOS work list's slots, from its groups (one per distinct repeat count,
// largest first, in the order of perm).  The caller sets their elements.
void set_groups(lgpu_ctx *c, const std::vector<int32_t> &reps, const std::vector<int64_t> &sizes)
{
   std::vector<EosSlot> slots;
   double repeats = 0.;
   for (size_t g = 0; g < reps.size(); ++g) repeats += (double)reps[g] * (double)sizes[g];
   int64_t at = 0;
   for (size_t g = 0; g < reps.size(); ++g) {
      const EosGroup group{at, sizes[g], reps[g]};
      const bool shared = eos_shares(c->numElem, c->numElem, group, repeats, c->precision == LGPU_MIXED);
      if (shared) c->s.eosSplit = 1;
      add_eos_slots(slots, group, shared);
      at += sizes[g];
   }
   c->eosSlots.clear();
   c->eosSlots.reserve(slots.size());
   for (const EosSlot &sl : slots) c->eosSlots.push_back(PlacedSlot{sl, 0});
}

// Last steps of both constructors: the EOS dispatch order and the pinned
// read-back buffers.
int finish_context(lgpu_ctx *c)
{
   const int st = set_eos_order(c, default_interleave(c));
   if (st != LGPU_OK) return st;
   constexpr size_t kSmallAt = (64 + sizeof(DevTime) + 63) / 64 * 64;
   if (copies_by_kernel({c->numNode}, {c->numElem}, kSmallProblem, c->precision == LGPU_MIXED))
      c->small.limit = kSmallProblem;
   if (hipHostMalloc((void **)&c->hostDt, kSmallAt + small_copy_bytes(c->small.limit), hipHostMallocDefault) !=
       hipSuccess)
      return LGPU_ENOMEM;
   c->hostErr = reinterpret_cast<int32_t *>(c->hostDt + 2);
   static_assert(sizeof(HostOut) <= 64, "hostTime follows at 64 bytes");
   c->s.hostOut = reinterpret_cast<HostOut *>(c->hostDt);
   *c->s.hostOut = HostOut{};
   c->hostTime = reinterpret_cast<DevTime *>(reinterpret_cast<char *>(c->hostDt) + 64);
   c->small.init(reinterpret_cast<char *>(c->hostDt) + kSmallAt);
   return LGPU_OK;
}

// The EOS's FP64 reciprocal and square root on caller data (lgpu_fp64_routines).
__global__ void __launch_bounds__(256)
k_fp64_routines(const double *__restrict__ x, int64_t n, double *__restrict__ rc,
                double *__restrict__ rt)
{
   const int64_t stride = (int64_t)gridDim.x * 256;
   for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
      const double v = x[i];
      if (rc) rc[i] = recip_rn_normal(v);
      if (rt) rt[i] = sqrt_rn_normal(v);
   }
}

} // namespace

extern "C" {

int lgpu_fp64_routines(const double *x, int64_t n, double *recip, double *root, void *stream)
{
   if (!x || n < 0) return LGPU_EINVAL;
   if (n == 0) return LGPU_OK;
   const int64_t want = (n + 255) / 256;
   const int grid = (int)(want < 4096 ? want : 4096);
   hipLaunchKernelGGL(k_fp64_routines, dim3(grid), dim3(256), 0, static_cast<hipStream_t>(stream),
                      x, n, recip, root);
   if (hipGetLastError() != hipSuccess) return LGPU_EDEVICE;
   return LGPU_OK;
}

void lgpu_default_constants(lgpu_constants *k)
{
   if (!k) return;
   k->e_cut = 1.0e-7;
   k->p_cut = 1.0e-7;
   k->q_cut = 1.0e-7;
   k->v_cut = 1.0e-10;
   k->u_cut = 1.0e-7;
   k->hgcoef = 3.0;
   k->ss4o3 = 4.0 / 3.0;
   k->qstop = 1.0e+12;
   k->monoq_max_slope = 1.0;
   k->monoq_limiter_mult = 2.0;
   k->qlc_monoq = 0.5;
   k->qqc_monoq = 2.0 / 3.0;
   k->qqc = 2.0;
   k->eosvmax = 1.0e+9;
   k->eosvmin = 1.0e-9;
   k->pmin = 0.0;
   k->emin = -1.0e+15;
   k->dvovmax = 0.1;
   k->refdens = 1.0;
}

int lgpu_create(const lgpu_mesh_desc *d, lgpu_ctx **out)
{
   if (!out) return LGPU_EINVAL;
   *out = nullptr;
   std::string why;
   if (validate(d, why) != LGPU_OK) {
      fprintf(stderr, "lgpu_create: invalid mesh description: %s\n", why.c_str());
      return LGPU_EINVAL;
   }
   CtxSpec sp;
   sp.numElem = d->numElem;
   sp.numNode = d->numNode;
   sp.sizeX = d->sizeX;
   sp.numReg = d->numReg;
   sp.cost = d->cost;
   sp.precision = d->precision;
   sp.brick = !(d->flags & LGPU_FLAG_GENERIC) && is_reference_brick(d);
   sp.brickFaces = sp.brick && brick_faces_computable(d);
   sp.nCorner = d->nodeElemStart[d->numNode];
   sp.k = d->k;
   lgpu_ctx *c = nullptr;
   int st = alloc_context(sp, &c);
   if (st != LGPU_OK) return st;
   auto fail = [&](int code) {
      lgpu_destroy(c);
      return code;
   };
   DevState &s = c->s;
   const size_t E = (size_t)d->numElem, N = (size_t)d->numNode;
   const int64_t nCorner = sp.nCorner;

   // Host-built tables.
   std::vector<uint8_t> bc(N, 0);
   const int32_t *sy[3] = {d->symmX, d->symmY, d->symmZ};
   const int32_t ns[3] = {d->numSymmX, d->numSymmY, d->numSymmZ};
   for (int a = 0; a < 3; ++a)
      for (int32_t i = 0; i < ns[a]; ++i) bc[(size_t)sy[a][i]] |= (uint8_t)(1u << a);
   // The EOS work list: elements grouped by their region's EOS repeat count,
   // largest first, and in mesh order within a group.  An element's EOS
   // depends only on the element and its repeat count (lulesh.cc:2387-2401
   // runs the same code for every region), so merging the regions of equal
   // count into one ascending list is exact; it turns the regions' short runs
   // (~38 elements on average) into long ones, so k_eos reads whole cache
   // lines.
   std::vector<int32_t> perm;
   perm.reserve(E);
   std::vector<int32_t> repOf(E, 1);
   std::vector<int32_t> reps;
   for (int r = 0; r < d->numReg; ++r) {
      const int32_t rep = region_rep(r, d->numReg, d->cost);
      if (d->regElemSize[r] > 0 && std::find(reps.begin(), reps.end(), rep) == reps.end())
         reps.push_back(rep);
      for (int32_t i = 0; i < d->regElemSize[r]; ++i) repOf[(size_t)d->regElemlist[r][i]] = rep;
   }
   std::sort(reps.begin(), reps.end(), std::greater<int32_t>());
   std::vector<int64_t> sizes;
   for (int32_t rep : reps) {
      const size_t before = perm.size();
      for (size_t el = 0; el < E; ++el)
         if (repOf[el] == rep) perm.push_back((int32_t)el);
      sizes.push_back((int64_t)(perm.size() - before));
   }
   std::vector<double> ones(E, 1.0);

   auto h2d = [&](const void *dst, const void *src, size_t bytes) {
      return hipMemcpy(const_cast<void *>(dst), src, bytes, hipMemcpyHostToDevice) == hipSuccess;
   };
   bool ok = h2d(s.nodeBC, bc.data(), N) &&
             h2d(s.nodeElemStart, d->nodeElemStart, sizeof(int32_t) * (N + 1)) &&
             (nCorner == 0 || h2d(s.cornerList, d->nodeElemCornerList, sizeof(int32_t) * (size_t)nCorner)) &&
             h2d(s.nodelist, d->nodelist, sizeof(int32_t) * 8 * E) &&
             h2d(s.lxim, d->lxim, sizeof(int32_t) * E) && h2d(s.lxip, d->lxip, sizeof(int32_t) * E) &&
             h2d(s.letam, d->letam, sizeof(int32_t) * E) && h2d(s.letap, d->letap, sizeof(int32_t) * E) &&
             h2d(s.lzetam, d->lzetam, sizeof(int32_t) * E) && h2d(s.lzetap, d->lzetap, sizeof(int32_t) * E) &&
             h2d(s.elemBC, d->elemBC, sizeof(int32_t) * E) &&
             h2d(s.perm, perm.data(), sizeof(int32_t) * E) &&
             h2d(s.v, ones.data(), sizeof(double) * E);
   if (!ok) return fail(LGPU_EDEVICE);
   set_groups(c, reps, sizes);
   for (PlacedSlot &p : c->eosSlots) p.elem = perm[(size_t)p.slot.pos];
   if ((st = finish_context(c)) != LGPU_OK) return fail(st);
   *out = c;
   return LGPU_OK;
}

int lgpu_create_sedov(const lgpu_sedov_desc *d, lgpu_ctx **out, lgpu_time_state *ts)
{
   if (!out) return LGPU_EINVAL;
   *out = nullptr;
   auto invalid = [](const char *why) {
      fprintf(stderr, "lgpu_create_sedov: invalid description: %s\n", why);
      return LGPU_EINVAL;
   };
   if (!d || !ts) return invalid("null argument");
   // 8 s^3 corner indices must fit int32 (s <= 645); the bound is tested
   // before any product is formed
   if (d->size < 1 || d->size > 645) return invalid("size out of range");
   const int64_t sz = d->size, E = sz * sz * sz, N = (sz + 1) * (sz + 1) * (sz + 1);
   if (d->precision != LGPU_FP64 && d->precision != LGPU_MIXED && d->precision != LGPU_FP64_FMA)
      return invalid("precision");
   if (d->numReg < 1 || d->cost < 0 || d->balance < 0) return invalid("numReg/balance/cost");
   if (!(d->emult > 0.0)) return invalid("emult");
   if (d->numRuns < 1 || !d->runReg || !d->runLen) return invalid("region runs");
   // Runs: region of each, start of each, and the groups of equal repeat count.
   std::vector<int32_t> runStart((size_t)d->numRuns + 1, 0);
   std::vector<int64_t> regSize((size_t)d->numReg, 0);
   int64_t at = 0;
   for (int32_t r = 0; r < d->numRuns; ++r) {
      if (d->runReg[r] < 1 || d->runReg[r] > d->numReg || d->runLen[r] < 1)
         return invalid("region run");
      runStart[(size_t)r] = (int32_t)at;
      at += d->runLen[r];
      if (at > E) return invalid("region runs exceed the element count");
      regSize[(size_t)(d->runReg[r] - 1)] += d->runLen[r];
   }
   if (at != E) return invalid("region runs do not cover every element");
   runStart[(size_t)d->numRuns] = (int32_t)E;
   std::vector<int32_t> reps;
   for (int r = 0; r < d->numReg; ++r) {
      const int32_t rep = region_rep(r, d->numReg, d->cost);
      if (regSize[(size_t)r] > 0 && std::find(reps.begin(), reps.end(), rep) == reps.end())
         reps.push_back(rep);
   }
   std::sort(reps.begin(), reps.end(), std::greater<int32_t>());
   std::vector<int64_t> groupSize(reps.size(), 0), groupAt(reps.size(), 0);
   std::vector<size_t> groupOf((size_t)d->numReg, 0); // of the regions that have elements
   for (int r = 0; r < d->numReg; ++r) {
      if (regSize[(size_t)r] == 0) continue;
      const int32_t rep = region_rep(r, d->numReg, d->cost);
      groupOf[(size_t)r] = (size_t)(std::find(reps.begin(), reps.end(), rep) - reps.begin());
      groupSize[groupOf[(size_t)r]] += regSize[(size_t)r];
   }
   for (size_t g = 1; g < reps.size(); ++g) groupAt[g] = groupAt[g - 1] + groupSize[g - 1];
   std::vector<int32_t> runDest((size_t)d->numRuns);
   for (int32_t r = 0; r < d->numRuns; ++r) {
      const size_t g = groupOf[(size_t)(d->runReg[r] - 1)];
      runDest[(size_t)r] = (int32_t)groupAt[g];
      groupAt[g] += d->runLen[r];
   }

   CtxSpec sp;
   sp.numElem = (int32_t)E;
   sp.numNode = (int32_t)N;
   sp.sizeX = (int32_t)sz;
   sp.numReg = d->numReg;
   sp.cost = d->cost;
   sp.precision = d->precision;
   sp.brick = !(d->flags & LGPU_FLAG_GENERIC);
   sp.brickFaces = sp.brick;
   sp.nCorner = 8 * E;
   sp.k = d->k;
   lgpu_ctx *c = nullptr;
   int st = alloc_context(sp, &c);
   if (st != LGPU_OK) return st;
   int32_t *runTables = nullptr;
   auto fail = [&](int code) {
      if (runTables) (void)hipFree(runTables);
      lgpu_destroy(c);
      return code;
   };
   const size_t runBytes = sizeof(int32_t) * ((size_t)d->numRuns + 1);
   if (hipMalloc((void **)&runTables, 2 * runBytes) != hipSuccess) {
      (void)hipGetLastError();
      return fail(LGPU_ENOMEM);
   }
   int32_t *dStart = runTables, *dDest = runTables + d->numRuns + 1;
   if (hipMemcpy(dStart, runStart.data(), runBytes, hipMemcpyHostToDevice) != hipSuccess ||
       hipMemcpy(dDest, runDest.data(), sizeof(int32_t) * (size_t)d->numRuns,
                 hipMemcpyHostToDevice) != hipSuccess)
      return fail(LGPU_EDEVICE);
   SedovSetup t;
   t.size = (int32_t)sz;
   t.runStart = dStart;
   t.runDest = dDest;
   t.numRuns = d->numRuns;
   if (launch_sedov_setup(c->s, t, c->stream) != hipSuccess) return fail(LGPU_EDEVICE);
   if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(LGPU_EDEVICE);
   (void)hipFree(runTables);
   runTables = nullptr;
   set_groups(c, reps, groupSize);
   // The element that each slot begins with, from the run that holds its
   // position: a group's slots and runs are both in the order of the mesh (the
   // runs kept, searched and the slots sorted afterwards: s=192 3.5 ms a context
   // instead of 2.2).
   std::vector<PlacedSlot> &slots = c->eosSlots;
   std::vector<size_t> next; // each group's first slot without an element
   for (size_t i = 0; i < slots.size(); ++i)
      if (i == 0 || slots[i].slot.rep != slots[i - 1].slot.rep) next.push_back(i);
   for (int32_t r = 0; r < d->numRuns; ++r) {
      const size_t g = groupOf[(size_t)(d->runReg[r] - 1)];
      const int64_t at = runDest[(size_t)r], end = at + d->runLen[r];
      for (size_t &i = next[g]; i < slots.size() && slots[i].slot.rep == reps[g] && slots[i].slot.pos < end; ++i)
         slots[i].elem = (int32_t)(runStart[(size_t)r] + (slots[i].slot.pos - at));
   }
   if ((st = finish_context(c)) != LGPU_OK) return fail(st);

   // Energy deposit and first dt (lulesh-init.cc:180-192).
   const double ebase = 3.948746e+7;
   const double scale = (double)sz / 45.0;
   double einit = ebase * scale * scale * scale;
   if (d->emult != 1.0) einit = einit * d->emult;
   double volo0 = 0.0;
   if (hipMemcpy(c->s.e, &einit, sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
       hipMemcpy(&volo0, c->s.volo, sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
      return fail(LGPU_EDEVICE);
   // Time controls, lulesh-init.cc:146-156.
   ts->time = 0.0;
   ts->deltatime = (0.5 * cbrt(volo0)) / sqrt(2.0 * einit);
   ts->dtcourant = 1.0e+20;
   ts->dthydro = 1.0e+20;
   ts->stoptime = 1.0e-2;
   ts->dtfixed = -1.0e-6;
   ts->dtmax = 1.0e-2;
   ts->deltatimemultlb = 1.1;
   ts->deltatimemultub = 1.2;
   ts->cycle = 0;
   *out = c;
   return LGPU_OK;
}

void lgpu_destroy(lgpu_ctx *c)
{
   if (!c) return;
   if (c->stream) (void)hipStreamSynchronize(c->stream);
   for (TimedLaunch &t : c->pending) {
      (void)hipEventDestroy(t.start);
      (void)hipEventDestroy(t.stop);
   }
   for (hipEvent_t e : c->eventPool) (void)hipEventDestroy(e);
   if (c->diag) (void)hipFree(c->diag);
   if (c->arena) (void)hipFree(c->arena);
   if (c->hostDt) (void)hipHostFree(c->hostDt);
   if (c->stream) (void)hipStreamDestroy(c->stream);
   delete c;
}

int lgpu_upload(lgpu_ctx *c, int field, const double *host)
{
   if (!c || !host || field < 0 || field >= LGPU_NUM_FIELDS) return LGPU_EINVAL;
   bool isElem, narrow;
   if ((field >= LGPU_XDD && field <= LGPU_FZ) || field == LGPU_QL || field == LGPU_QQ) {
      int r = enable_diagnostics(c);
      if (r) return r;
   }
   double *dst = real_field_ptr(c, field, isElem, narrow);
   if (!dst) return LGPU_EINVAL;
   const size_t n = isElem ? (size_t)c->numElem : (size_t)c->numNode;
   if (c->small.takes(n)) {
      HIP_OR_RETURN(c, c->small.upload(host, dst, narrow, (int)n, c->stream));
      return LGPU_OK;
   }
   HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   if (narrow && converts_on_device(host, (int64_t)n, true)) {
      double *wide = scratch_doubles(c);
      HIP_OR_RETURN(c, hipMemcpy(wide, host, sizeof(double) * n, hipMemcpyHostToDevice));
      HIP_OR_RETURN(c, launch_narrow(wide, reinterpret_cast<float *>(dst), (int64_t)n, c->stream));
      HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   } else if (narrow) {
      std::vector<float> tmp(n);
      for (size_t i = 0; i < n; ++i) tmp[i] = (float)host[i];
      HIP_OR_RETURN(c, hipMemcpy(dst, tmp.data(), sizeof(float) * n, hipMemcpyHostToDevice));
   } else {
      HIP_OR_RETURN(c, hipMemcpy(dst, host, sizeof(double) * n, hipMemcpyHostToDevice));
   }
   return LGPU_OK;
}

int lgpu_download(lgpu_ctx *c, int field, double *host)
{
   if (!c || !host || field < 0 || field >= LGPU_NUM_FIELDS) return LGPU_EINVAL;
   bool isElem, narrow;
   double *src = real_field_ptr(c, field, isElem, narrow);
   const size_t n = isElem ? (size_t)c->numElem : (size_t)c->numNode;
   if (src && c->small.takes(n)) {
      HIP_OR_RETURN(c, c->small.download(src, host, narrow, (int)n, c->stream));
      return LGPU_OK;
   }
   HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   if (!src) {
      std::fill(host, host + n, 0.0);
      return LGPU_OK;
   }
   if (narrow && converts_on_device(host, (int64_t)n, false)) {
      double *wide = scratch_doubles(c);
      HIP_OR_RETURN(c, launch_widen(reinterpret_cast<const float *>(src), wide, (int64_t)n, c->stream));
      HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
      HIP_OR_RETURN(c, hipMemcpy(host, wide, sizeof(double) * n, hipMemcpyDeviceToHost));
   } else if (narrow) {
      std::vector<float> tmp(n);
      HIP_OR_RETURN(c, hipMemcpy(tmp.data(), src, sizeof(float) * n, hipMemcpyDeviceToHost));
      for (size_t i = 0; i < n; ++i) host[i] = (double)tmp[i];
   } else {
      HIP_OR_RETURN(c, hipMemcpy(host, src, sizeof(double) * n, hipMemcpyDeviceToHost));
   }
   return LGPU_OK;
}

int lgpu_lagrange_nodal(lgpu_ctx *c, double dt)
{
   if (!c) return LGPU_EINVAL;
   switch (c->precision) {
   case LGPU_MIXED: return launch_nodal<PolicyMixed>(c, dt);
   case LGPU_FP64_FMA: return launch_nodal<PolicyFp64Fma>(c, dt);
   default: return launch_nodal<PolicyFp64>(c, dt);
   }
}

int lgpu_lagrange_elements(lgpu_ctx *c, double dt)
{
   if (!c) return LGPU_EINVAL;
   switch (c->precision) {
   case LGPU_MIXED: return launch_elements<PolicyMixed>(c, dt);
   case LGPU_FP64_FMA: return launch_elements<PolicyFp64Fma>(c, dt);
   default: return launch_elements<PolicyFp64>(c, dt);
   }
}

int lgpu_time_constraints(lgpu_ctx *c, double *dtcourant, double *dthydro)
{
   if (!c) return LGPU_EINVAL;
   // After lgpu_lagrange_elements k_dt_slots has written them to host memory
   // itself (s=45, host loop, us a cycle: 62.7 -> 59 without the two copies,
   // 57.7 -> 54.3 without the wait for the stream).
   if (!c->hostOutFresh) {
      HIP_OR_RETURN(c, hipMemcpyAsync(c->hostDt, c->s.dtOut, sizeof(double) * 2,
                                      hipMemcpyDeviceToHost, c->stream));
      HIP_OR_RETURN(c, hipMemcpyAsync(c->hostErr, c->s.err, sizeof(int32_t) * kNumErrSites,
                                      hipMemcpyDeviceToHost, c->stream));
   }
   if (!c->hostOutFresh || c->timing || !host_reached(&c->s.hostOut->seq, c->hostSeq))
      HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   if (c->timing) harvest_timing(c);
   const int st = resolve_status(c->hostErr);
   if (st == LGPU_OK) {
      if (dtcourant) *dtcourant = c->hostDt[0];
      if (dthydro) *dthydro = c->hostDt[1];
   }
   return st;
}

int lgpu_run(lgpu_ctx *c, lgpu_time_state *ts, int32_t maxCycle)
{
   if (!c || !ts) return LGPU_EINVAL;
   DevTime *const h = c->hostTime;
   h->time = ts->time;
   h->deltatime = ts->deltatime;
   h->dtcourant = ts->dtcourant;
   h->dthydro = ts->dthydro;
   h->stoptime = ts->stoptime;
   h->dtfixed = ts->dtfixed;
   h->dtmax = ts->dtmax;
   h->multlb = ts->deltatimemultlb;
   h->multub = ts->deltatimemultub;
   h->cycle = ts->cycle;
   h->maxCycle = maxCycle;
   h->active = 1;
   h->fresh = 1;
   DevTime *const times = c->devTime;
   double *const slots = c->s.dtPartial;
   int32_t *const errs = c->s.err;
   c->hostOutFresh = false;
   Launch<PolicyFp64>::run_start(*h, times, c->s.dtOut, c->stream);
   HIP_OR_RETURN(c, hipGetLastError());

   const bool fold = c->s.isBrick
                        ? c->s.nodalBlock && fold_start(block_blocks(c->s.brick), c->brickSlots,
                                                      c->precision != LGPU_MIXED)
                        : fold_start((c->numElem + c->block - 1) / c->block, c->genericSlots, false);
   // Cycle j reads the time state, error flags and dt slots of set j mod 2 and
   // writes the other set.
   auto use_sets = [&](int j) {
      const int in = j & 1, out = in ^ 1;
      DevState &s = c->s;
      s.timeIn = times + in;
      s.timeOut = times + out;
      s.errPrev = errs + in * kNumErrSites;
      s.err = errs + out * kNumErrSites;
      s.dtPartialPrev = slots + in * 2 * kDtSlots;
      s.dtPartial = slots + out * 2 * kDtSlots;
      s.startFold = fold ? 1 : 0;
      s.dtDevice = &s.timeOut->deltatime;
      s.active = &s.timeOut->active;
   };
   // The host runs at most kAhead cycles ahead of the last one it has seen
   // begin, so that the device does not wait for it where cycles take less than
   // the 2 ms that host_reached polls (a check after every 16 cycles left it
   // idle for 13 us; longer cycles still have one, as the stream is then waited
   // for).  No more cycles are enqueued than the
   // cycle limit allows, so only a run that ends at stoptime (or on an error)
   // enqueues no-op cycles, at most kAhead.
   constexpr uint32_t kAhead = 16;
   const int64_t cycles = std::max<int64_t>(1, (int64_t)maxCycle - (int64_t)ts->cycle);
   HostOut *const out = c->s.hostOut;
   __atomic_store_n(&out->ended, 0u, __ATOMIC_RELAXED);
   int st = LGPU_OK;
   for (int64_t n = 0; n < cycles && !st; ++n) {
      if (n >= kAhead && !host_reached(&out->started, c->cycleSeq + 1 - kAhead))
         st = set_hip_error(c, hipStreamSynchronize(c->stream), "hipStreamSynchronize");
      if (st || __atomic_load_n(&out->ended, __ATOMIC_RELAXED)) break;
      use_sets((int)(n & 1));
      c->s.hostSeq = ++c->cycleSeq;
      if (!fold) st = timed(c, kKTimeIncrement, [&] { Launch<PolicyFp64>::begin(c->s, c->stream); });
      if (!st) st = lgpu_lagrange_nodal(c, 0.0);
      if (!st) st = lgpu_lagrange_elements(c, 0.0);
      if (c->timing && (n + 1) % kAhead == 0 && !st) {
         st = set_hip_error(c, hipStreamSynchronize(c->stream), "hipStreamSynchronize");
         harvest_timing(c);
      }
   }
   if (!st) {
      c->s.hostSeq = ++c->hostSeq;
      Launch<PolicyFp64>::run_end(c->s, slots, errs, h, c->stream);
      st = set_hip_error(c, hipGetLastError(), "k_run_end");
   }
   // Back to host-driven dt (the node buffers keep whatever swaps happened).
   c->s.timeIn = nullptr;
   c->s.startFold = 0;
   c->s.timeOut = nullptr;
   c->s.errPrev = nullptr;
   c->s.dtPartialPrev = nullptr;
   c->s.err = errs;
   c->s.dtPartial = slots;
   c->s.dtDevice = nullptr;
   c->s.active = nullptr;
   if (st) return st;
   if (c->timing || !host_reached(&out->seq, c->hostSeq))
      HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   if (c->timing) harvest_timing(c);
   ts->time = h->time;
   ts->deltatime = h->deltatime;
   ts->dtcourant = h->dtcourant;
   ts->dthydro = h->dthydro;
   ts->cycle = h->cycle;
   return resolve_status(c->hostErr);
}

int lgpu_set_option(lgpu_ctx *c, int option, int64_t value)
{
   if (!c) return LGPU_EINVAL;
   switch (option) {
   case LGPU_OPT_KEEP_DIAGNOSTICS:
      if (value) {
         const int r = enable_diagnostics(c);
         if (r) return r;
      } else {
         c->s.fx = c->s.fy = c->s.fz = c->s.xdd = c->s.ydd = c->s.zdd = nullptr;
         c->s.ql = c->s.qq = c->s.delvOut = nullptr;
         HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
         if (c->diag) (void)hipFree(c->diag);
         c->diag = nullptr;
      }
      c->keepDiag = value != 0;
      return LGPU_OK;
   case LGPU_OPT_KERNEL_TIMING:
      c->timing = value != 0;
      return LGPU_OK;
   case LGPU_OPT_BLOCK_SIZE:
      if (value != 64 && value != 128 && value != 256) return LGPU_EINVAL;
      c->block = (int)value;
      return LGPU_OK;
   case LGPU_OPT_BRICK_CHUNK:
      if (!c->s.isBrick || value < 1) return LGPU_EINVAL;
      set_brick_chunk(c->s.brick, (int)std::min<int64_t>(value, 1 << 20));
      set_nodal_kernel(c, option_rows(c));
      return LGPU_OK;
   case LGPU_OPT_XCD_REMAP:
      c->s.xcdRemap = value ? 1 : 0;
      return LGPU_OK;
   case LGPU_OPT_KIN_CHUNK:
      if (!c->s.isBrick || value < 1) return LGPU_EINVAL;
      set_kin_chunk(c->s.brick, (int)std::min<int64_t>(value, 1 << 20));
      c->s.kinFlat = c->s.brick.kinChunk == c->flatChunk;
      return LGPU_OK;
   case LGPU_OPT_BRICK_ROWS:
      if (!c->s.isBrick || (value != 8 && value != 16)) return LGPU_EINVAL;
      set_nodal_kernel(c, (int)value);
      return LGPU_OK;
   case LGPU_OPT_EOS_INTERLEAVE:
      if (value < 0 || value > 1024) return LGPU_EINVAL;
      return set_eos_order(c, (int)value);
   case LGPU_OPT_KERNEL_TIMING_MASK:
      c->timingMask = (uint32_t)value;
      return LGPU_OK;
   default:
      return LGPU_EINVAL;
   }
}

int lgpu_get_option(lgpu_ctx *c, int option, int64_t *value)
{
   if (!c || !value) return LGPU_EINVAL;
   switch (option) {
   case LGPU_OPT_KEEP_DIAGNOSTICS: *value = c->keepDiag ? 1 : 0; return LGPU_OK;
   case LGPU_OPT_KERNEL_TIMING: *value = c->timing ? 1 : 0; return LGPU_OK;
   case LGPU_OPT_BLOCK_SIZE: *value = c->block; return LGPU_OK;
   case LGPU_OPT_BRICK_CHUNK:
      if (!c->s.isBrick) return LGPU_EINVAL;
      *value = c->s.brick.chunkZ;
      return LGPU_OK;
   case LGPU_OPT_XCD_REMAP: *value = c->s.xcdRemap; return LGPU_OK;
   case LGPU_OPT_KERNEL_TIMING_MASK: *value = c->timingMask; return LGPU_OK;
   case LGPU_OPT_KIN_CHUNK:
      if (!c->s.isBrick) return LGPU_EINVAL;
      *value = c->s.brick.kinChunk;
      return LGPU_OK;
   case LGPU_OPT_BRICK_ROWS:
      if (!c->s.isBrick) return LGPU_EINVAL;
      *value = option_rows(c);
      return LGPU_OK;
   case LGPU_OPT_EOS_INTERLEAVE: *value = c->eosInterleave; return LGPU_OK;
   default: return LGPU_EINVAL;
   }
}

int lgpu_num_kernels(void) { return kNumKernels; }

const char *lgpu_kernel_name(int kernel)
{
   return (kernel >= 0 && kernel < kNumKernels) ? kKernelNames[kernel] : "";
}

int lgpu_kernel_stats(lgpu_ctx *c, int kernel, int64_t *launches, double *total_ms)
{
   if (!c || kernel < 0 || kernel >= kNumKernels) return LGPU_EINVAL;
   HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   harvest_timing(c);
   if (launches) *launches = c->kLaunches[kernel];
   if (total_ms) *total_ms = c->kMs[kernel];
   return LGPU_OK;
}

int lgpu_reset_kernel_stats(lgpu_ctx *c)
{
   if (!c) return LGPU_EINVAL;
   HIP_OR_RETURN(c, hipStreamSynchronize(c->stream));
   harvest_timing(c);
   for (int i = 0; i < kNumKernels; ++i) {
      c->kLaunches[i] = 0;
      c->kMs[i] = 0.0;
   }
   return LGPU_OK;
}

int lgpu_get_info(lgpu_ctx *c, lgpu_info *info)
{
   if (!c || !info) return LGPU_EINVAL;
   info->path = c->s.isBrick ? 1 : 0;
   info->precision = c->precision;
   info->numElem = c->numElem;
   info->numNode = c->numNode;
   info->numReg = c->numReg;
   info->block = c->block;
   info->arena_bytes = (int64_t)c->arenaBytes;
   info->brick_faces = c->s.brickFaces;
   info->brick_blocks_per_cu = c->brickPerCu;
   return LGPU_OK;
}

const char *lgpu_last_error(lgpu_ctx *c) { return c ? c->lastError.c_str() : ""; }

} // extern "C"
