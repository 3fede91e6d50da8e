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

// Largest grids of the VL step without LDS.  Its taps go through L1 and L2,
// which pays while the fields stay in the Infinity Cache.  Plain / FP32
// imaging / FP16 imaging / FP16 Born steps in us, before and with it: 48^3 8.8
// / 9.6 / 11.6 / 11.5 and 3.2 / 3.6 / 3.6 / 3.5; 128^3 10.6 / 11.9 / 16.3 / 15.8
// and 8.4 / 11.1 / 10.6 / 9.8; 208^3 (9.0 M cells) 31 / 63 / 47 / 45 and 26 / 40
// / 37 / 33.  At 288 x 240 x 208 (14.4 M) it takes 41 / 77 / 61 / 57, the ring's
// 64 x 16 tiles 36 / 62 / 63 / 55.  Where n1 is no multiple of 4 the
// alternative is the one- or two-cell kernel: 257 x 201 x 233 (12 M) 41 / 66 /
// 60 / 52 against 36 / 54 / 51 / 44, 301^3 (27 M) 100 / 173 / 172 / 150 against
// 113 / 178 / 174 / 149.
constexpr long kDirectMaxCells = 10L << 20, kDirectMaxCellsOdd = 16L << 20;

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

// The four-cell ring's automatic tile shape, and what a slice of one round of
// workgroups costs next to a slice of 256 x 8 tiles (plain steps at 256^3 to
// 512^3):
//   256 x 8   1.00  one 8-wave workgroup per CU
//   256 x 16  1.66  the same with two rows per thread, plain steps only (in
//                   the others its second row costs twice: FP16 imaging at
//                   512^3 630 us against 590 us in 256 x 8); 1.55 where the
//                   step extracts receivers
//   128 x 24  1.33  one 12-wave workgroup per CU
//   64 x 16   1.38  three 4-wave workgroups per CU
// The shape whose rounds cost least is taken: where 256-wide tiles fit the
// rows they win (256^3: plain 38.6 us against 39.9 us in 128 x 24 and 42.0
// us in the 256 x 16 tiles used there before; 512^3 256 x 16), elsewhere the
// narrow ones: 384^3 149 us in 128 x 24 (287-323 us in 256 x 16 with a
// second round of 32 workgroups before), 320^3 101 us and 288 x 240 x 208 36
// us in 64 x 16 (120 and 46 us in the two-cell kernel before).
// (imaging and Born steps move more per slice, which the narrow shapes' finer
// halos cost more: FP32 imaging at 512^3 640 us in 256 x 8, 750 us in 64 x 16)
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
inline void choose_ring_tiles(StepChoice &c, const StepSetting &s, int act, int rec) {
  const bool plain = act == ACT_NONE;
  StepChoice q[4] = {c, c, c, c};
  const double cost[4] = {
      1.00 * plan_rounds(q[0], s, 256, 8, s.ncu),
      plain ? (rec == REC_EXTRACT ? 1.55 : 1.66) * plan_rounds(q[1], s, 256, 16, s.ncu) : 1e30,
      (plain ? 1.33 : 1.45) * plan_rounds(q[2], s, 128, 24, s.ncu),
      (plain ? 1.38 : 1.60) * plan_rounds(q[3], s, 64, 16, 3 * s.ncu)};
  c = q[std::min_element(cost, cost + 4) - cost];
}

// rec: the receivers' mode that the caller would have inside the step.
inline StepChoice choose_step(const StepSetting &s, int form, int act, int fmt, int rec) {
  StepChoice c{};
  // The automatic choice: the kernel without LDS while the fields stay in the
  // caches, the four-cell ring where n1 allows it, else tiles as below.
  const bool autosel =
      form == FORM_VL && s.ty_tile == 0 && s.x_per_lane == 0 && s.halo_ring < 0;
  const long ncell = (long)s.n1 * s.n2 * s.n3;
  if (autosel && ncell <= (s.n1 % 4 == 0 ? kDirectMaxCells : kDirectMaxCellsOdd)) {
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
  if (autosel && s.n1 % 4 == 0) {
    c.kernel = STEP_X4R;
    c.rec = rec;
    choose_ring_tiles(c, s, act, rec);
    return c;
  }
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
