// lgpu_brick.h -- host-side set-up of the structured-brick path: recognising
// the reference's brick and boundary set-up in a mesh description, and the
// brick's tiling (workgroup tiles and z-chunks of the fused kernels).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstdint>
#include <vector>

#include "lgpu_kernels.h"
#include "lulesh_gpu.h"

namespace lgpu {

inline FastDiv make_fastdiv(uint32_t d)
{
   FastDiv f;
   f.d = d;
   f.m = UINT64_MAX / d + 1;
   return f;
}

// True when the description is the reference's structured brick: lattice
// element-to-node map (lulesh-init.cc:245-266) and node-to-corner lists in
// ascending corner order (lulesh-init.cc:271-319).
inline bool is_reference_brick(const lgpu_mesh_desc *d)
{
   const int64_t s = d->sizeX;
   if (s < 1 || d->sizeY != s || d->sizeZ != s) return false;
   const int64_t en = s + 1;
   if (d->numElem != s * s * s || d->numNode != en * en * en) return false;
   int64_t e = 0;
   for (int64_t c = 0; c < s; ++c)
      for (int64_t b = 0; b < s; ++b)
         for (int64_t a = 0; a < s; ++a, ++e) {
            const int64_t n0 = (c * en + b) * en + a;
            const int64_t want[8] = {n0, n0 + 1, n0 + en + 1, n0 + en, n0 + en * en,
                                     n0 + en * en + 1, n0 + en * en + en + 1, n0 + en * en + en};
            for (int j = 0; j < 8; ++j)
               if (d->nodelist[8 * e + j] != want[j]) return false;
         }
   // Corner lists: every node's corners in ascending order.
   const int64_t N = d->numNode;
   std::vector<int32_t> cnt((size_t)N, 0);
   for (int64_t c = 0; c < 8 * (int64_t)d->numElem; ++c) cnt[(size_t)d->nodelist[c]]++;
   int64_t start = 0;
   for (int64_t n = 0; n < N; ++n) {
      if (d->nodeElemStart[n] != start) return false;
      start += cnt[(size_t)n];
   }
   if (d->nodeElemStart[N] != start) return false;
   std::fill(cnt.begin(), cnt.end(), 0);
   for (int64_t c = 0; c < 8 * (int64_t)d->numElem; ++c) {
      const int32_t n = d->nodelist[c];
      if (d->nodeElemCornerList[d->nodeElemStart[n] + cnt[(size_t)n]++] != (int32_t)c) return false;
   }
   return true;
}

// True when the face neighbours and boundary masks are those of the brick
// with symmetry planes on the low faces and free surfaces on the high faces
// (the reference's single-domain set-up, lulesh-init.cc:340-398, 497-573), so
// that k_eos can compute them (brick_faces in lgpu_step.inc).  A neighbour
// index has to match only where the mask lets k_eos read it (bits 0 or COMM).
inline bool brick_faces_computable(const lgpu_mesh_desc *d)
{
   const int64_t s = d->sizeX, s2 = s * s;
   const int32_t *nb[6] = {d->lxim, d->lxip, d->letam, d->letap, d->lzetam, d->lzetap};
   const int32_t field[6] = {0x00007, 0x00038, 0x001c0, 0x00e00, 0x07000, 0x38000};
   const int32_t comm[6] = {0x00004, 0x00020, 0x00100, 0x00800, 0x04000, 0x20000};
   int64_t e = 0;
   for (int64_t c = 0; c < s; ++c)
      for (int64_t b = 0; b < s; ++b)
         for (int64_t a = 0; a < s; ++a, ++e) {
            const int32_t want = (a == 0 ? 0x00001 : 0) | (a == s - 1 ? 0x00010 : 0) |
                                 (b == 0 ? 0x00040 : 0) | (b == s - 1 ? 0x00400 : 0) |
                                 (c == 0 ? 0x01000 : 0) | (c == s - 1 ? 0x10000 : 0);
            if (d->elemBC[e] != want) return false;
            const int64_t wantN[6] = {e - 1, e + 1, e - s, e + s, e - s2, e + s2};
            for (int f = 0; f < 6; ++f) {
               const int32_t bits = want & field[f];
               if ((bits == 0 || bits == comm[f]) && nb[f][e] != wantN[f]) return false;
            }
         }
   return true;
}

inline void set_brick_chunk(Brick &g, int chunk)
{
   g.chunkZ = std::max(1, std::min(chunk, g.en));
   g.chunks = (g.en + g.chunkZ - 1) / g.chunkZ;
}

// A column-walking launch: `columns` column tiles, each cut into z-chunks of
// `chunk` planes out of `planes` and, where that does not come out even, a
// shorter last one, on `slots` resident workgroups.  A walk takes its planes
// and `extra` of one more.  The whole chunks are dispatched first and the
// last ones (logical_block's second part) into the slots that these leave.
struct WalkTime {
   double whole; // end of the whole chunks, in planes
   double end;   // end of the launch
   double work;  // planes walked per slot
};

inline WalkTime walk_time(int64_t columns, int planes, int slots, int chunk, double extra)
{
   const int64_t wholes = columns * (planes / chunk), last = planes % chunk ? columns : 0;
   const double walk = chunk + extra, lastWalk = planes % chunk + extra;
   const int64_t rounds = wholes / slots, left = wholes % slots, open = slots - left;
   WalkTime t;
   t.whole = t.end = walk * (double)(rounds + (left ? 1 : 0));
   t.work = ((double)wholes * walk + (double)last * lastWalk) / slots;
   if (last) {
      // back to back in the slots that the last round of whole chunks leaves
      // open, begun while that round lasts, and in all of them after it
      const int64_t turns = left ? (int64_t)std::ceil(walk / lastWalk) : last;
      const int64_t early = std::min(last, turns * open), late = last - early;
      t.end = std::max({t.whole, walk * (double)rounds + lastWalk * (double)((early + open - 1) / open),
                        t.whole + lastWalk * (double)((late + slots - 1) / slots)});
   }
   return t;
}

// Time of the fused nodal kernel's walk in planes.  The last chunks that run
// beyond the others have a CU's units to themselves and count half; those of at
// most a quarter of a walk fit into the spread of the others' ends and count a
// quarter (FP64 s=192, last walks at half / short ones at a quarter: 505 / 488 us;
// chunks of equal rounds 511).
inline double walk_cost(int64_t columns, int planes, int slots, int chunk)
{
   const WalkTime t = walk_time(columns, planes, slots, chunk, 1.0);
   const bool shortLast = 4 * (planes % chunk + 1) <= chunk + 1;
   return t.whole + (shortLast ? 0.25 : 0.5) * (t.end - t.whole);
}

// Default node planes per workgroup of the fused nodal kernel (at least
// `least`): the smallest walk_cost, redundant planes against idle slots.  Long
// walks drift apart and lose their neighbours' planes in L2, so more than 40
// planes are walked only in a single round, and never more than 66: FP64 s=210
// chunk 94 759 us, 47 777, 23 714; s=220 99 800, 49 816, 24 751.
inline int pick_brick_chunk(const Brick &g, int slots, int least)
{
   int best = 8;
   double bestCost = 1e300;
   const int64_t columns = (int64_t)g.tilesX * g.tilesY;
   for (int ch = least; slots > 0 && ch <= std::min(g.en, 66); ++ch) {
      if (ch > 40 && columns * (g.en / ch) > slots) continue;
      const double cost = walk_cost(columns, g.en, slots, ch);
      if (cost < bestCost) {
         bestCost = cost;
         best = ch;
      }
   }
   return best;
}

// The chunk for launches of several rounds whose workgroups end at different
// times (the mixed form, 3 a CU; ensembles): least work per resident workgroup,
// plus a part of a walk for the end of the launch, a quarter in an ensemble,
// whose many short last chunks fill it.  columns[i] column tiles of planes[i]
// planes each.  Fewest rounds / this, mixed: s=192 chunk 22 / 9, 405 / 395 us;
// s=160 22 / 7, 276 / 241; s=128 14 / 5, 129 / 125.  Half / quarter, FP64: 64
// members of 16..64 11 / 16, 486 / 482; 30 of 10..40 5 / 7, 98 / 92; 16 of 40..90
// 12 / 18, 530 / 529; mixed 40 of 20..50 6 / 8, 164 / 159.
inline int pick_tail_chunk(const std::vector<int64_t> &columns, const std::vector<int> &planes,
                           int slots, double part, int fallback)
{
   if (slots < 1) return fallback;
   int best = fallback;
   double bestWork = 1e300;
   for (int ch = 1; ch <= 64; ++ch) {
      double walked = 0.;
      for (size_t i = 0; i < columns.size(); ++i)
         walked += (double)columns[i] * (planes[i] + (planes[i] + ch - 1) / ch);
      const double work = std::max(walked / slots + part * (ch + 1), ch + 1.0);
      if (work < bestWork) {
         bestWork = work;
         best = ch;
      }
   }
   return best;
}

inline void set_kin_chunk(Brick &g, int chunk)
{
   g.kinChunk = std::max(1, std::min(chunk, g.s));
   g.kinChunks = (g.s + g.kinChunk - 1) / g.kinChunk;
}

// Default element planes per workgroup of the kinematics kernel: 4 to 12 (long
// walks drift apart and lose their neighbours' planes in L2), by the end of
// the launch, the work per slot and a fifth of a walk.  Its extra plane is
// only copied, which counts as 0.3.  By rounds of equal chunks / by this, us,
// FP64: s=160 7 / 7, 124 / 123; s=175 30 / 7, 185 / 168; s=185 37 / 7, 221 / 207;
// s=192 12 / 12, 200 / 200; s=200 23 / 9, 255 / 250; s=220 20 / 7, 361 / 338;
// mixed s=175 30 / 7, 155 / 132; s=192 12 / 9, 154 / 155.
inline int pick_kin_chunk(const Brick &g, int slots)
{
   int best = 12;
   double bestCost = 1e300;
   for (int ch = 4; slots > 0 && ch <= std::min(12, g.s); ++ch) {
      const WalkTime t = walk_time((int64_t)g.kinTiles * g.kinTiles, g.s, slots, ch, 0.3);
      const double cost = t.end + t.work + 0.2 * (ch + 0.3);
      if (cost < bestCost) {
         bestCost = cost;
         best = ch;
      }
   }
   return best;
}

// Fused nodal kernel tiles of w threads by h rows: (w-1) x (h-1) nodes each.
inline void set_brick_tile(Brick &g, int w, int h)
{
   g.tileW = w;
   g.rows = h;
   g.tilesX = (g.en + w - 2) / (w - 1);
   g.tilesY = (g.en + h - 2) / (h - 1);
}

// The tile of an ensemble member's nodal workgroups (256 threads): the
// width w (rows 256 / w) that needs the fewest tiles per plane, so that few
// lanes fall outside a small mesh (s=16: 18 x 14 threads, 2 tiles instead of
// 4 of 16 x 16); ties go to the width nearest 16.
inline void pick_member_tile(Brick &g)
{
   int bestW = 16;
   int64_t best = INT64_MAX;
   for (int w = 4; w <= 64; ++w) {
      const int h = 256 / w;
      if (h < 3) break;
      const int64_t tiles = (int64_t)((g.en + w - 2) / (w - 1)) * ((g.en + h - 2) / (h - 1));
      if (tiles < best || (tiles == best && std::abs(w - 16) < std::abs(bestW - 16))) {
         best = tiles;
         bestW = w;
      }
   }
   set_brick_tile(g, bestW, 256 / bestW);
}

// One problem's walk takes other tiles than 16 x 16 threads.
inline bool other_tile(const Brick &g) { return g.tileW != 16 || (g.rows != 16 && g.rows != 8); }

// walk_cost of the tile and chunk chosen; a plane takes 7% longer where the
// tile's width is read at run time.
inline double brick_walk_cost(const Brick &g, int slots)
{
   if (slots < 1) return 0.;
   const double cost = walk_cost((int64_t)g.tilesX * g.tilesY, g.en, slots, g.chunkZ);
   return other_tile(g) ? 1.07 * cost : cost;
}

// The fused nodal kernel's tile and chunk for one problem: 16 x 16 threads, or
// the tile that an ensemble's member of this size would have where that needs
// 7% fewer columns and the walk is 7% shorter by more than its planes cost.
// 16 x 16 / that, us: FP64 s=90 75.5 / 65.0, s=125 171 / 155; not taken: FP64 s=110
// 111.7 / 111.9, FP64_FMA s=140 187 / 196.
inline void pick_brick_walk(Brick &g, int slots)
{
   set_brick_chunk(g, pick_brick_chunk(g, slots, 1));
   Brick other = g;
   pick_member_tile(other);
   set_brick_chunk(other, pick_brick_chunk(other, slots, 1));
   const double columns = (double)g.tilesX * g.tilesY, fewer = (double)other.tilesX * other.tilesY;
   if (fewer <= 0.93 * columns && brick_walk_cost(other, slots) < brick_walk_cost(g, slots)) g = other;
}

// Kinematics tiles of w x h elements (one per thread of a 256-thread
// workgroup), kept within the LDS of the 16 x 16 tile: (h+1) node rows of
// 2 ceil((w+1)/2) values, at most 17 x 18.
inline bool kin_tile_fits(int w, int h)
{
   return w >= 1 && h >= 1 && w * h <= 256 && (h + 1) * 2 * ((w + 2) / 2) <= 17 * 18;
}

inline void set_kin_tile(Brick &g, int w, int h)
{
   g.kinW = w;
   g.kinH = h;
   g.kinTilesX = (g.s + w - 1) / w;
   g.kinTilesY = (g.s + h - 1) / h;
}

// An ensemble member's kinematics tile: the width (rows 256 / width) with
// the fewest tiles per plane that fits the LDS; ties go to the width
// nearest 16.
inline void pick_member_kin_tile(Brick &g)
{
   int bestW = 16;
   int64_t best = INT64_MAX;
   for (int w = 4; w <= 64; ++w) {
      const int h = 256 / w;
      if (!kin_tile_fits(w, h)) continue;
      const int64_t tiles = (int64_t)((g.s + w - 1) / w) * ((g.s + h - 1) / h);
      if (tiles < best || (tiles == best && std::abs(w - 16) < std::abs(bestW - 16))) {
         best = tiles;
         bestW = w;
      }
   }
   set_kin_tile(g, bestW, 256 / bestW);
}

// k_nodal_block: the block of at most 256 elements that covers the nodes with
// the fewest workgroups; ties go to the widest (rows of 16-byte loads).
inline void pick_nodal_block(Brick &g)
{
   auto tiles = [&](int n) { return (g.en + n - 2) / (n - 1); };
   int64_t best = INT64_MAX;
   for (int w = 3; w <= 18; ++w)
      for (int h = 3; w * h * 3 <= 256; ++h) {
         const int d = 256 / (w * h);
         const int64_t n = (int64_t)tiles(w) * tiles(h) * tiles(d);
         if (n <= best) {
            best = n;
            g.blkW = w;
            g.blkH = h;
            g.blkD = d;
         }
      }
   g.blkX = tiles(g.blkW);
   g.blkY = tiles(g.blkH);
   g.blkZ = tiles(g.blkD);
}

inline int64_t block_blocks(const Brick &g) { return (int64_t)g.blkX * g.blkY * g.blkZ; }

// True when k_nodal_block is the faster nodal kernel: `blocks` workgroups of
// it on `slots` resident ones take about 1 + blocks / slots planes of the
// walking kernel's time (8.3 us a plane in FP64), and the walk its `cost` and,
// with its start and end, 0.4 more.  Block / the fastest walk, us: FP64 s=30 8.6 /
// 20.3, s=45 17.1 / 31.3, s=60 31.6 / 31.8, s=64 34.0 / 31.8 (whose cycle begins
// in a launch of 3 us, the block's in the block kernel for 1.6); walk taken: FP64
// s=101 119.8 / 92.3.
inline bool block_is_faster(int64_t blocks, int slots, double cost)
{
   return slots > 0 && (double)blocks < (cost - 0.6) * slots;
}

// The largest brick of k_kin_flat.  Flat / best walk: FP64 s=30 8.5 / 9.0 us
// (14.9 at the walk's own choice), s=64 14.3 / 16.0, s=101 34.2 / 43.2, s=115
// 56.0 / 61.3, s=118 62.0 / 62.2, s=120 64.2 / 63.4, s=128 76.3 / 66.0, s=192
// 248 / 198; mixed s=105 26.3 / 30.6, s=115 41.5 / 44.1, s=120 50.5 / 47.1.
// Above it the elements in flight on an XCD, and the planes they read, no
// longer stay in its L2.  Ensembles: each member's own size counts (64 of
// 16..64, 6.0 M elements: FP64 179.5 / 203, mixed 140 / 146).
constexpr int kKinFlatMax = 117; // elements per edge

// Workgroups of k_kin_flat: 256 elements each.
inline int64_t flat_blocks(const Brick &g) { return ((int64_t)g.s * g.s * g.s + 255) / 256; }

// Tiling of an s^3 brick with the default chunks (the caller may pick
// others): 15x15-node tiles of the fused nodal kernel, 16x16-element tiles
// of the kinematics kernel.
inline void init_brick(Brick &g, int s)
{
   g.s = s;
   g.en = s + 1;
   set_brick_tile(g, 16, 16);
   g.divS = make_fastdiv((uint32_t)g.s);
   g.divS2 = make_fastdiv((uint32_t)(g.s * g.s));
   g.kinTiles = (g.s + 15) / 16;
   set_kin_tile(g, 16, 16);
   set_brick_chunk(g, 8);
   set_kin_chunk(g, 12);
   pick_nodal_block(g);
}

} // namespace lgpu
