// Which kernel and tile shape a time step runs on.  Plain C++ without device
// code, so that it can also be built and checked on its own.
#pragma once
#include <algorithm>
#include <string>

namespace brtm {

// Storage format of a source-wavefield snapshot.
enum SnapFmt { FMT_NONE = 0, FMT_F32 = 1, FMT_BF16 = 2, FMT_F16 = 3 };
// Step form: VL = V.L(p) (Born/wave_fkernel.3d8o.cu:31), LV = L(V.p) (:109).
enum StepForm { FORM_VL = 0, FORM_LV = 1 };
// What the step does with the snapshot s besides the update:
//   ACT_IMG  img += cimg . s . p_new        (zero-lag imaging, VL only)
//   ACT_BORN p_new += cimg . s . m          (Born secondary source)
enum StepAct { ACT_NONE = 0, ACT_IMG = 1, ACT_BORN = 2 };
// Receivers handled inside the step (the four-cell ring kernel, the kernel
// without LDS, and the one-cell kernel's 8-row shape):
//   REC_INJECT   pn += sum_k rsinc[k] rtr(r, rid+k) before imaging and the store
//   REC_EXTRACT  rtr(r, rid+k) += rsinc[k] . pn . (rscale[r] or 1)
// for the cells of plane rz whose rmap entry is a receiver index r >= 0.
enum RecMode { REC_NONE = 0, REC_INJECT = 1, REC_EXTRACT = 2 };

enum StepKernel {
  STEP_TILES = 0,  // k_step: one cell per lane, two-plane LDS (both forms)
  STEP_RING,       // k_step_ring: one cell per lane, six-plane halo ring
  STEP_X2,         // k_step_x2: two cells per lane
  STEP_X4,         // k_step_x4: four cells per lane, two-plane LDS
  STEP_X4R,        // k_step_x4r: four cells per lane, six-plane halo ring
  STEP_DIRECT,     // k_step_direct: four cells per lane, no LDS
};

// The grid and the context's settings (0 or -1: automatic).
struct StepSetting {
  int n1, n2, n3, ncu;
  int ty_tile, target_blocks, x_per_lane, halo_ring;
};

struct StepChoice {
  StepKernel kernel;
  int tw, ty;              // cells and rows of a tile
  int zc;                  // slices of a z chunk
  int ntx, nty, ntz;       // tiles
  int rec;                 // the receivers' mode inside the step, or REC_NONE
};

// Largest grids of the VL step without LDS, whose taps go through L1 and L2,
// which pays while the fields stay in the Infinity Cache.  Plain / FP32
// imaging / FP16 imaging / FP16 Born steps in us, in the tiled kernels and
// without LDS: 48^3 8.8 / 9.6 / 11.6 / 11.5 and 3.2 / 3.6 / 3.6 / 3.5; 128^3
// 10.6 / 11.9 / 16.3 / 15.8 and 8.4 / 11.1 / 10.6 / 9.8.  Where n1 % 4 == 0 the
// ring's tiles come near it from 7 M cells on.  There a million (2^20) cells
// take 3.1 / 4.7 / 4.35 / 3.85 us without LDS, about 3.74 (plain) or 3.44 of the
// slices that the ring's tiles are counted in (choose_ring_tiles): the ring
// is taken where it costs less, and from 10 M cells to 12.6 M, where the caches
// begin to overflow, unless it costs a tenth more.  224 x 256 x 160 (8.8 M) 25.9 /
// 38.4 / 35.7 / 31.9 and in 256 x 8 tiles 25.6 / 36.2 / 36.4 / 29.8; 272 x 541 x 86
// (12.1 M) 32.9 / 46.2 / 43.5 / 39.9 and in 64 x 16 tiles 33.6 / 62.8 / 58.9 / 41.5
// (60 in the two-cell kernel, FP32 imaging); 288 x 240 x 208 (13.7 M) 41 / 78 /
// 63 / 54 and 36 / 63 / 59 / 47.  Where n1 is no multiple of 4 the alternative is
// the one- or two-cell kernel: 257 x 201 x 233 (12 M) 41 / 66 / 60 / 52 against
// 36 / 54 / 51 / 44, 301^3 (27 M) 100 / 173 / 172 / 150 against 113 / 178 / 174 /
// 149.
constexpr long kDirectCells = 7L << 20, kDirectEven = 10L << 20,
               kDirectMaxCells = 126L * (1 << 20) / 10, kDirectMaxCellsOdd = 16L << 20;

// z chunks of tiles tw x ty: about target_blocks workgroups in all, at least
// 8 slices each.
inline void plan_tiles(StepChoice &c, const StepSetting &s, int tw, int ty, int target_blocks) {
  c.tw = tw;
  c.ty = ty;
  c.ntx = (s.n1 + tw - 1) / tw;
  c.nty = (s.n2 + ty - 1) / ty;
  const int nz = s.n3 - 8;
  const long tiles = (long)c.ntx * c.nty;
  c.zc = (int)std::min<long>(
      std::max(8L, (tiles * nz + target_blocks - 1) / target_blocks), nz);
  c.ntz = (nz + c.zc - 1) / c.zc;
}

// z chunks of a ring step whose workgroups run `capacity` at a time: a round
// of workgroups takes a chunk's slices plus about nine for its prologue, so
// the chunk count that fills one to four rounds with the fewest slices wins.
// Returns the slices all rounds take together.
inline long plan_rounds(StepChoice &c, const StepSetting &s, int tw, int ty, int capacity) {
  c.tw = tw;
  c.ty = ty;
  c.ntx = (s.n1 + tw - 1) / tw;
  c.nty = (s.n2 + ty - 1) / ty;
  const int nz = s.n3 - 8;
  const long tiles = (long)c.ntx * c.nty;
  long best = -1;
  for (int r = 1; r <= 4; ++r) {
    const long want = std::max(1L, std::min((long)nz, capacity * (long)r / tiles));
    const int zc = (int)((nz + want - 1) / want), ntz = (nz + zc - 1) / zc;
    const long rounds = (tiles * ntz + capacity - 1) / capacity;
    const long cost = rounds * (zc + 9);
    if (best < 0 || cost < best) {
      best = cost;
      c.zc = zc;
      c.ntz = ntz;
    }
  }
  return best;
}

// The four-cell ring's automatic tile shape: the one whose rounds of workgroups
// cost least, in slices of one round of 256 x 8 tiles.  What a slice of the
// others costs next to that:
//   256 x 8    1.00  one 8-wave workgroup per CU
//   256 x 16   1.50  the same with two rows per thread, plain steps only (in
//                    the others its second row costs twice: FP16 imaging at
//                    512^3 630 us against 590 us in 256 x 8); 1.66 where planes
//                    are multiples of 256 KB, whose z taps meet in the same
//                    cache sets (256^3: 42.0 us against 38.8 in 256 x 8; 240^3:
//                    35.1 against 36.2; 204 x 248 x 235: 31.2 against 35.4)
//   128 x 24   1.33  one 12-wave workgroup per CU
//   64 x 16    1.38  three 4-wave workgroups per CU
// The narrow tiles win where 256-wide ones fit the rows badly: 384^3 plain 146
// us in 128 x 24 (193 in 256 x 16), 320^3 102 and 288 x 240 x 208 36 us in 64 x 16
// (120 and 46 us in the two-cell kernel).  Imaging and Born steps move more per
// slice, which the narrow tiles' finer halos cost more (1.45, 1.60: FP32
// imaging at 512^3 617 us in 256 x 8, 754 in 64 x 16); imaging takes 1.50 and 2.00
// where rows start anywhere in a cache line, so that a tile's pieces of them
// share their first and last line with the neighbours': 164 x 544 x 393 FP32 187
// us in 256 x 8, 240 in 128 x 24, 254 in 64 x 16, 225 in the one-cell kernel.
// On 1595 steps timed on about 300 grids of 5 to 105 million cells it is 2.3 %
// slower than the best of these kernels on average.
// Steps that extract receivers (Born modelling) take 256 x 16 earlier: where
// several contexts model by turns, which overlaps their steps, the 256 x 8 tiles'
// twofold y halo costs more than the second round that 256 x 16 may leave, and
// alone the two are even.  A modelling of two shots at 256^3 (FP16 snapshots
// every 4 of 120 steps), three contexts by turns / one alone: 13.07 / 11.53 ms
// in 256 x 8, 12.65 / 11.75 in 256 x 16 (12.68 / 12.40 before 256 x 8 was
// introduced); one shot of 100 steps at 240^3 4.85 / 4.46 against 4.70 / 4.38,
// at 256 x 224 x 288 5.88 / 5.02 against 5.78 / 5.02, at 512 x 160 x 208 6.00 /
// 5.29 against 5.95 / 5.29.  Steps that inject keep the line above (adjoint at
// 256^3 12.83 / 12.05 in 256 x 8, 12.72 / 12.50 in 256 x 16).
// Returns what the choice costs.
inline double choose_ring_tiles(StepChoice &c, const StepSetting &s, int act, int rec) {
  const bool plain = act == ACT_NONE;
  const bool sets = (long)s.n1 * s.n2 % 65536 == 0;
  const double w16 = !plain               ? 1e30
                     : rec == REC_EXTRACT ? (sets ? 1.55 : 1.45)
                                          : (sets ? 1.66 : 1.50);
  const bool split = act == ACT_IMG && s.n1 % 16 != 0;
  const double w128 = plain ? 1.33 : split ? 1.50 : 1.45;
  const double w64 = plain ? 1.38 : split ? 2.00 : 1.60;
  StepChoice q[4] = {c, c, c, c};
  const double cost[4] = {1.00 * plan_rounds(q[0], s, 256, 8, s.ncu),
                          w16 * plan_rounds(q[1], s, 256, 16, s.ncu),
                          w128 * plan_rounds(q[2], s, 128, 24, s.ncu),
                          w64 * plan_rounds(q[3], s, 64, 16, 3 * s.ncu)};
  const double *best = std::min_element(cost, cost + 4);
  c = q[best - cost];
  return *best;
}

// Whether the ring's own streams are read with nontemporal loads when left
// automatic.  They pay off once a step's working set (16 B per cell: p, p_old,
// V, p_new) is well beyond the 256 MB Infinity Cache: 6 % faster at 512^3.
// Below that the fields stay cache-resident between launches, which the hint
// would forfeit: 11 % slower at 256^3.  Nor where 64-wide tiles of rows that
// start anywhere share the lines at their ends with their neighbours, which
// then read them again: plain / FP32 imaging at 164 x 544 x 393 133 / 254 us with
// it, 119 / 233 without (but 119 / 221 without at 400 x 208 x 432, whose rows
// start on half lines, 115 / 213 with it).
constexpr double kStreamMinStepBytes = 512.0 * 1024 * 1024;

inline bool choose_streaming(const StepSetting &s, const StepChoice &c) {
  return 16.0 * s.n1 * s.n2 * s.n3 > kStreamMinStepBytes && (c.tw > 64 || s.n1 % 16 == 0);
}

// rec: the receivers' mode that the caller would have inside the step.
inline StepChoice choose_step(const StepSetting &s, int form, int act, int fmt, int rec) {
  StepChoice c{};
  // The automatic choice: the kernel without LDS while the fields stay in the
  // caches, the four-cell ring where n1 allows it, else tiles as below.
  const bool autosel =
      form == FORM_VL && s.ty_tile == 0 && s.x_per_lane == 0 && s.halo_ring < 0;
  const bool quad = s.n1 % 4 == 0;
  const long ncell = (long)s.n1 * s.n2 * s.n3;
  double ring_cost = 1e30;
  if (autosel && quad && ncell > kDirectCells) {
    c.kernel = STEP_X4R;
    c.rec = rec;
    ring_cost = choose_ring_tiles(c, s, act, rec);
  }
  const double direct_cost =
      (act == ACT_NONE ? 3.74 : 3.44) * (ncell <= kDirectEven ? 1.0 : 1.1) * ncell / (1 << 20);
  if (autosel && (quad ? ncell <= kDirectMaxCells && direct_cost < ring_cost
                       : ncell <= kDirectMaxCellsOdd)) {
    // lanes run over the (group of four cells, row) pairs of the update set;
    // two slices per thread once that still leaves 12 waves per compute unit
    const long groups = (s.n1 - 5L) / 4 * (s.n2 - 8);
    c.kernel = STEP_DIRECT;
    c.tw = 1024;
    c.ty = c.nty = 1;
    c.zc = groups * ((s.n3 - 7) / 2) / 64 >= 12L * s.ncu ? 2 : 1;
    c.ntx = (int)((groups + 255) / 256);
    c.ntz = (s.n3 - 8 + c.zc - 1) / c.zc;
    c.rec = rec;
    return c;
  }
  if (autosel && quad) return c;
  // cells per lane: 4 or 2 where asked for and n1 allows, else 1; automatic
  // (0): the widest whose tiles keep at least 3/4 of the lanes busy
  int xl = 1;
  if (form == FORM_VL) {
    int want = s.x_per_lane;
    if (want == 0) {
      want = 1;
      for (int k : {4, 2}) {
        const int w = 64 * k, used = ((s.n1 + w - 1) / w) * w;
        if (s.n1 % k == 0 && 4 * s.n1 >= 3 * used) { want = k; break; }
      }
    }
    if (want == 4 && s.n1 % 4 == 0) xl = 4;
    else if (want >= 2 && s.n1 % 2 == 0) xl = 2;
  }
  // halo ring: automatic (-1) means on for the 4-cell kernel
  const bool ring = s.halo_ring < 0 ? xl == 4 : s.halo_ring != 0;
  // Tile rows / workgroup target per variant (measured on MI355X at 512^3):
  // plain steps prefer tall tiles, 16-bit snapshot variants short ones.
  int ty = s.ty_tile, tb = s.target_blocks;
  if (ty == 0) {
    if (xl == 4) { ty = (ring && act == ACT_IMG && fmt == FMT_F32) ? 8 : 16; tb = 256; }
    else if (xl == 2) { ty = 16; tb = 2048; }
    else if (act == ACT_NONE) { ty = 32; tb = 1024; }
    else if (fmt == FMT_F32) { ty = 16; tb = 8192; }
    else { ty = 8; tb = 8192; }
  }
  if (xl == 4 && ty == 32) ty = 16;  // the 4-cell kernel's tiles are 8 or 16 rows
  c.kernel = xl == 4 ? (ring ? STEP_X4R : STEP_X4)
             : xl == 2 ? STEP_X2
             : ring && form == FORM_VL ? STEP_RING : STEP_TILES;
  plan_tiles(c, s, 64 * xl, ty, tb);
  if (form == FORM_VL &&
      (c.kernel == STEP_X4R || (c.kernel == STEP_TILES && !ring && ty == 8)))
    c.rec = rec;
  return c;
}

inline std::string step_kernel_name(const StepChoice &c) {
  const std::string tiles = std::to_string(c.tw) + "x" + std::to_string(c.ty) + " tiles";
  switch (c.kernel) {
    case STEP_TILES: return "k_step, " + tiles;
    case STEP_RING: return "k_step_ring (six-plane halo ring), " + tiles;
    case STEP_X2: return "k_step_x2 (2 cells/lane), " + tiles;
    case STEP_X4: return "k_step_x4 (4 cells/lane), " + tiles;
    case STEP_X4R: return "k_step_x4r (4 cells/lane, six-plane halo ring), " + tiles;
    default: return "k_step_direct (4 cells/lane, no LDS), " + std::to_string(c.zc) +
                    (c.zc == 1 ? " slice" : " slices") + " per thread";
  }
}

}  // namespace brtm
