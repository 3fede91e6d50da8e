// 3-D convolutions of the learned preconditioner on gfx950 MFMA.
//
// Forward (and input-gradient) convolutions are implicit GEMMs (k_conv): M =
// output channels, N = 16 consecutive x positions per row, K = the 27
// taps x input channels, one v_mfma_f32_16x16x32_bf16 per (16-channel output
// tile, row, tap, 32-channel chunk) and one v_mfma_f32_16x16x16_bf16 per
// 16-channel remainder.  Operand lanes: lane l holds A[l%16][8(l/16)+i] and
// B[8(l/16)+i][l%16] (i < 8; K = 16: 4(l/16)+i, i < 4), and receives
// D[4(l/16)+j][l%16] (j < 4) (checked on the device against a host product).  In channels-last layout
// the 8 K values of a lane are 8 consecutive channels of one position: one
// 16-byte load.  The weight gradient is a GEMM over positions (K) whose
// operands are read from LDS with the transposing read (k_wgrad).
#include "conv3d.h"

#include "conv_plan.h"

#include <algorithm>
#include <utility>

namespace brtm {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ uint16_t f2bf(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
// two of them in one conversion (round to nearest even, as f2bf)
__device__ __forceinline__ uint32_t f2bf2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

__device__ __forceinline__ bf16x8 ld8(const uint16_t *p) {
  const uint4 u = *reinterpret_cast<const uint4 *>(p);
  return __builtin_bit_cast(bf16x8, u);
}
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0)); }

// four bf16 values (8 bytes) as the K = 16 MFMA's operand type
typedef short i16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i16x4 ld4h(const uint16_t *p) {
  const uint2 u = *reinterpret_cast<const uint2 *>(p);
  return __builtin_bit_cast(i16x4, u);
}
__device__ __forceinline__ i16x4 zero4h() { return __builtin_bit_cast(i16x4, make_uint2(0, 0)); }

// v, in a form that the compiler cannot move out of a loop.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

__host__ __device__ inline int cpad(int c) { return (c + 31) / 32 * 32; }
int grid1(long n, int bs = 256) {
  long g = (n + bs - 1) / bs;
  return (int)(g < 1 ? 1 : (g > 65535 * 4 ? 65535 * 4 : g));
}

// ------------------------------------------------------------- forward GEMM
// Elements between two positions (or two weight rows) in LDS.  Sixteen rows
// are read at once, 16 bytes (or, for 16 channels, 8) of each by the four lane
// groups: free of bank conflicts where the stride is an odd multiple of 32
// bytes (of 16 for 16 channels), measured 4.1 clocks for a 16-byte read of a
// wave against 8.2 at 64 bytes and 16 at 128.
__host__ __device__ constexpr int pos_stride(int c) {
  return c == 16 ? 24 : c / 16 % 2 ? c : c + 16;
}

// Where lane group kq finds its 4 channels of the 16-channel remainder behind
// 32 channels: the two 16-byte halves change places every four positions,
// which keeps the 8-byte reads at that stride free of bank conflicts.
__device__ __forceinline__ int remainder_at(int kq, int pos) {
  return ((kq >> 1) ^ (pos >> 2 & 1)) * 8 + (kq & 1) * 4;
}

template <int V>
struct Int {
  static constexpr int value = V;
};

// f(Int<0>()), f(Int<1>()), ...: a loop unrolled whatever its length
template <class F, int... K>
__device__ __forceinline__ void unrolled(F &&f, std::integer_sequence<int, K...>) {
  (f(Int<K>()), ...);
}

// Two gradients through the ReLU of two BF16 activations, as BF16.
__device__ __forceinline__ uint32_t masked2(uint32_t act, float g0, float g1) {
  g0 = __uint_as_float(act << 16) > 0.f ? g0 : 0.f;
  g1 = __uint_as_float(act & 0xffff0000u) > 0.f ? g1 : 0.f;
  return f2bf2(g0, g1);
}

// What happens to a finished output tile.
// OUT_ACT: bias and ReLU, BF16.  OUT_GRAD: FP32 as it is.  OUT_MASK: an input
// gradient through the ReLU that made that input, BF16 (zero where the
// activation aux is not positive).
enum { OUT_ACT = 0, OUT_GRAD = 1, OUT_MASK = 2 };

// A workgroup sweeps z over zl output planes of a tile of 16 WX positions by
// YT WY rows.  Each input plane of the tile (with its halo, zeros outside the
// volume) is staged in LDS once and serves all 27 taps of the three output
// planes around it, whose sums wait in registers; the next plane is loaded
// into registers meanwhile.  A wave computes 16 positions of YT rows and MTW
// 16-channel output tiles: for a (dx, 32-channel chunk) the YT + 2 row
// fragments are read once for the nine (dz, dy) taps, and a weight fragment
// once for the YT rows.  Weights wait in LDS (WL) where they fit beside the
// plane, else they come through the vector cache.  A 16-channel remainder
// (CIN = 16, 48) runs on the K = 16 MFMA.  Every output's sum runs over
// (dz, dx, chunk, dy) in this order, whatever the tile.
//
// The first CU input channels are a tensor of half the resolution, read
// through the nearest-neighbour upsampling as it is staged (the concatenated
// tensor is never stored: 28 us a layer for writing it, and its reads).
//
// What bounds it: the matrix unit (46 us for 48->16 at 8 x 64^3, the K = 16
// products at half rate) and what it waits for between planes: a workgroup's
// waves write, wait and finish outputs together.  A wave that loaded its rows
// from the vector cache for each dz, dx and chunk moved three times the
// fragments through a 64-byte-per-clock cache: 48->16 at 8 x 64^3 took 219 us,
// now 90; 16->16 93, now 44; 96->32 (32^3) 108, now 54; 32->32 41, now 21;
// 64->64 (16^3) 62, now 20; 32->64 21, now 11; and 16->48 at 4 x 64^3 106 with
// 12 sums of 16 x 16 outputs a wave and output plane, now 71 with six.  A wave
// has few sums (MTW YT is 4 to 6) so that more waves than two are resident on
// a matrix unit and no register is spilled: eight sums took 97 us for 48->16
// and 81 for 96->32.
template <int CIN, int CU, int COUT, int MTW, int YT, int WX, int WY, bool WL, int OUT>
__global__ void __launch_bounds__(64 * WX * WY * (COUT / 16 / MTW), 2)
k_conv(const uint16_t *__restrict__ x, int xcs, const uint16_t *__restrict__ up,
       const uint16_t *__restrict__ W, const void *__restrict__ aux, void *y, int ycs, int zl,
       int D, int H, int Wd) {
  constexpr int CIN_P = (CIN + 31) / 32 * 32;
  constexpr int NT = 64 * WX * WY * (COUT / 16 / MTW);
  constexpr int NC = CIN / 32;          // 32-channel chunks
  constexpr bool R16 = CIN % 32 == 16;  // and a 16-channel remainder
  constexpr int R = YT * WY, X = 16 * WX, PS = pos_stride(CIN), RS = (X + 2) * PS;
  constexpr int WS = WL ? PS : CIN_P;
  constexpr bool SWZ = R16 && NC > 0;  // the remainder's halves are swapped (remainder_at)
  static_assert(!SWZ || (CU == NC * 32 && WL), "the remainder is its own source");
  __shared__ __attribute__((aligned(16))) uint16_t Xs[(R + 2) * RS];
  __shared__ __attribute__((aligned(16))) uint16_t Ws[WL ? 27 * COUT * PS : 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, kq = lane >> 4;
  const int wx = wave % WX, wy = (wave / WX) % WY, wm = wave / (WX * WY);
  // XCD-aware order: workgroup b runs on XCD b % 8, so XCD k takes a
  // contiguous run of tiles and neighbouring tiles' halos meet in its L2.
  const int nb = gridDim.x, q8 = nb >> 3, r8 = nb & 7;
  const int xcd = blockIdx.x & 7, jj = blockIdx.x >> 3;
  int r = (xcd < r8) ? xcd * (q8 + 1) + jj : r8 * (q8 + 1) + (xcd - r8) * q8 + jj;
  const int x0 = r % (Wd / X) * X;
  r /= Wd / X;
  const int y0 = r % (H / R) * R;
  r /= H / R;
  const int z0 = r % (D / zl) * zl;
  const long n0 = (long)(r / (D / zl)) * D;  // plane 0 of this batch item

  // 16-byte chunks of a plane: the upsampled channels first, then the others
  constexpr int UC = CU / 8, XC = CIN / 8 - UC, NP = (R + 2) * (X + 2);
  constexpr int NU = NP * UC, NX = NP * XC, PU = (NU + NT - 1) / NT, PT = (NX + NT - 1) / NT;
  uint4 preu[PU + 1], pre[PT];
  const long plane = (long)H * Wd * xcs, uplane = (long)(H / 2) * (Wd / 2) * CU;
  const uint32_t bytes = ((uint32_t)(H * Wd - 1) * xcs + 8 * XC) * 2;
  auto fetch = [&](int z) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(x + (n0 + z) * plane), 0, bytes, 0x00020000);
    // the chunks' places are recomputed for each plane: kept over the plane
    // loop they took registers that the sums need
    const int t_ = opaque(tid);
    if constexpr (CU > 0) {
      const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint16_t *>(up + ((n0 + z) >> 1) * uplane), 0, (uint32_t)uplane * 2,
          0x00020000);
#pragma unroll
      for (int i = 0; i < PU; ++i) {
        const int e = t_ + i * NT;
        const int c = e % UC, p = (e / UC) % (X + 2), rr = e / (UC * (X + 2));
        const int yy = y0 + rr - 1, xx = x0 + p - 1;
        const bool ok = ((i + 1) * NT <= NU || e < NU) & ((unsigned)yy < (unsigned)H) & ((unsigned)xx < (unsigned)Wd);
        const uint32_t off =
            ok ? (uint32_t)((yy >> 1) * (Wd >> 1) + (xx >> 1)) * CU * 2 + 16 * c : 0x80000000u;
        preu[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ru, off, 0, 0));
      }
    }
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e = t_ + i * NT;
      const int c = e % XC, p = (e / XC) % (X + 2), rr = e / (XC * (X + 2));
      const int yy = y0 + rr - 1, xx = x0 + p - 1;
      const bool ok = ((i + 1) * NT <= NX || e < NX) & ((unsigned)yy < (unsigned)H) & ((unsigned)xx < (unsigned)Wd);
      const uint32_t off = ok ? (uint32_t)(yy * Wd + xx) * xcs * 2 + 16 * c : 0x80000000u;
      pre[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
    }
  };

  const int zf = z0 > 0 ? z0 - 1 : 0, ze = z0 + zl < D ? z0 + zl : D - 1;
  fetch(zf);
  if constexpr (WL) {
    constexpr int WC = CIN / 8;
    for (int i = tid; i < 27 * COUT * WC; i += NT) {
      const int r = i / WC, c = i % WC, sw = SWZ && c >= NC * 4 ? r >> 2 & 1 : 0;
      *reinterpret_cast<uint4 *>(&Ws[r * PS + (c ^ sw) * 8]) =
          *reinterpret_cast<const uint4 *>(W + (long)r * CIN_P + c * 8);
    }
  }
  static_assert(WL || !R16, "a remainder's weights wait in LDS");
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(W), 0, 27 * COUT * CIN_P * 2, 0x00020000);
  const int wrem = SWZ ? remainder_at(kq, col) : 4 * kq;
  const uint16_t *xb = Xs + (wy * YT) * RS + (wx * 16 + col) * PS;

  f32x4 acc[3][MTW][YT];  // outputs zp + 1, zp, zp - 1 of input plane zp
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int m = 0; m < MTW; ++m)
#pragma unroll
      for (int t = 0; t < YT; ++t) acc[d][m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto store = [&](int z) {
    // a lane's four channels 4kq .. 4kq+3 of an output tile are adjacent: one
    // 8-byte (BF16) or 16-byte (FP32) store
#pragma unroll
    for (int t = 0; t < YT; ++t) {
      const long o = (((n0 + z) * H + y0 + wy * YT + t) * Wd + x0 + wx * 16 + col) * ycs;
#pragma unroll
      for (int m = 0; m < MTW; ++m) {
        const int c0 = (wm * MTW + m) * 16 + 4 * kq;
        const f32x4 v = acc[2][m][t];
        if constexpr (OUT == OUT_GRAD) {
          *reinterpret_cast<f32x4 *>(static_cast<float *>(y) + o + c0) = v;
        } else if constexpr (OUT == OUT_MASK) {
          const uint2 a = *reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(aux) + o + c0);
          *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(y) + o + c0) =
              make_uint2(masked2(a.x, v[0], v[1]), masked2(a.y, v[2], v[3]));
        } else {
          const float4 b = *reinterpret_cast<const float4 *>(static_cast<const float *>(aux) + c0);
          const float v0 = fmaxf(v[0] + b.x, 0.f), v1 = fmaxf(v[1] + b.y, 0.f);
          const float v2 = fmaxf(v[2] + b.z, 0.f), v3 = fmaxf(v[3] + b.w, 0.f);
          *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(y) + o + c0) =
              make_uint2(f2bf2(v0, v1), f2bf2(v2, v3));
        }
      }
    }
  };

  // Products of the staged plane for the outputs zp + 1 - dz whose bit of MASK
  // is set, in steps of one weight fragment per output tile; the fragments are
  // read AHEAD steps before their products, which the compiler left next to
  // them.
  constexpr int NPC = NC + R16, AHEAD = WL ? 1 : 3;
  auto products = [&](auto mask) {
    constexpr int MASK = decltype(mask)::value;
    constexpr int ND = (MASK & 1) + (MASK >> 1 & 1) + (MASK >> 2), K = 9 * NPC * ND;
    // no weights kept over the plane loop
    const uint16_t *wq = Ws + ((wm * MTW * 16 + col) * WS + opaque(0)) * WL;
    const int wlane = ((wm * MTW * 16 + col) * WS + 8 * kq + opaque(0)) * 2;
    bf16x8 b[YT + 2], a[AHEAD + 1][MTW];
    i16x4 bh[YT + 2], ah[AHEAD + 1][MTW];
    // step k: x tap, chunk, z tap, y tap
    auto tap = [](int k) constexpr {
      const int d = k / 3 % ND, lo = MASK & 1 ? 0 : MASK & 2 ? 1 : 2;
      return (lo + d) * 9 + k % 3 * 3 + k / (3 * ND * NPC);
    };
    auto weights = [&](int k) __attribute__((always_inline)) {
      const int pc = k / (3 * ND) % NPC, o = tap(k) * COUT;
#pragma unroll
      for (int m = 0; m < MTW; ++m) {
        if (!WL)  // one register of lane offsets, the rest in the scalar offset
          a[k % (AHEAD + 1)][m] = __builtin_bit_cast(
              bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                          wrs, wlane, ((o + m * 16) * WS + pc * 32) * 2, 0));
        else if (pc < NC)
          a[k % (AHEAD + 1)][m] = ld8(wq + (o + m * 16) * WS + pc * 32 + 8 * kq);
        else
          ah[k % (AHEAD + 1)][m] = ld4h(wq + (o + m * 16) * WS + NC * 32 + wrem);
      }
    };
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) weights(k);
    auto step = [&](auto kk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      constexpr int pc = k / (3 * ND) % NPC, dx = k / (3 * ND * NPC), t9 = tap(k);
      if (k % (3 * ND) == 0) {
        const uint16_t *xr = xb + dx * PS;
        const int rem = NC * 32 + (SWZ ? remainder_at(kq, col + dx) : 4 * kq);
#pragma unroll
        for (int i = 0; i < YT + 2; ++i) {
          if (pc < NC) b[i] = ld8(xr + i * RS + pc * 32 + 8 * kq);
          else bh[i] = ld4h(xr + i * RS + rem);
        }
      }
      if (k + AHEAD < K) weights(k + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      constexpr int dz = t9 / 9, dy = t9 / 3 % 3;
#pragma unroll
      for (int m = 0; m < MTW; ++m)
#pragma unroll
        for (int t = 0; t < YT; ++t) {
          if (pc < NC)
            acc[dz][m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a[k % (AHEAD + 1)][m], b[t + dy], acc[dz][m][t], 0, 0, 0);
          else
            acc[dz][m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                ah[k % (AHEAD + 1)][m], bh[t + dy], acc[dz][m][t], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    };
    unrolled(step, std::make_integer_sequence<int, K>());
  };

  for (int zp = zf; zp <= ze; ++zp) {
    __syncthreads();  // the previous plane has been read
    const int t_ = opaque(tid);
    if constexpr (CU > 0) {
#pragma unroll
      for (int i = 0; i < PU; ++i) {
        const int e = t_ + i * NT;
        if ((i + 1) * NT <= NU || e < NU) *reinterpret_cast<uint4 *>(&Xs[e / UC * PS + e % UC * 8]) = preu[i];
      }
    }
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e = t_ + i * NT;
      if ((i + 1) * NT <= NX || e < NX) {
        const int p = e / XC, sw = SWZ ? p % (X + 2) >> 2 & 1 : 0;
        *reinterpret_cast<uint4 *>(&Xs[p * PS + ((e % XC) ^ sw) * 8 + CU]) = pre[i];
      }
    }
    __syncthreads();
    if (WL && zp < ze) fetch(zp + 1);
    const bool on0 = zp + 1 < z0 + zl, on1 = zp >= z0 && zp < z0 + zl, on2 = zp > z0;
    if (on0 && on1 && on2) products(Int<7>());
    else if (on0 && on1) products(Int<3>());
    else if (on1 && on2) products(Int<6>());
    else if (on0) products(Int<1>());
    else if (on1) products(Int<2>());
    else products(Int<4>());
    // where the weights come through the vector cache the next plane is loaded
    // behind them (loads return in order), while the other workgroup computes
    if (!WL && zp < ze) fetch(zp + 1);
    if (on2) store(zp - 1);
#pragma unroll
    for (int m = 0; m < MTW; ++m)
#pragma unroll
      for (int t = 0; t < YT; ++t) {
        acc[2][m][t] = acc[1][m][t];
        acc[1][m][t] = acc[0][m][t];
        acc[0][m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  if (z0 + zl == D) store(D - 1);  // no plane follows
}

// ------------------------------------------------------------- weight GEMM
// dW[tap][co][ci] = sum_p dy[p][co] x[p + tap][ci]: for each tap a GEMM whose
// K runs over positions, so both operands are channels-last tiles read with
// K along the slow index.  ds_read_b64_tr_b16 reads them transposed: a
// 16-lane group takes a 4-position x 16-channel block and lane j gets channel
// j's four positions, at any position offset, so a tap's x shift costs
// nothing.
//
// A workgroup stages R rows of dy (SEG positions) and the R + 2 input rows
// around them of plane z + dz - 1 (SEG + 2 positions) once and uses them for
// nine taps: wave dx (three waves) owns the taps (dz, *, dx), a fragment of
// an input row serves the three dy taps, whose dy rows wait in registers.
// The workgroup strides over the units of the volume with its sums in
// registers and writes one partial sum per element; k_grad_sum adds the
// partials in order (no atomics: the gradient is the same in every run).  The
// bias gradient is one more product, dy by ones, on the wave of the centre
// tap.  Before this a workgroup per tap re-read both tensors 27 times and
// transposed them with 2-byte LDS stores: 2.00 ms for 16->16 and 3.79 ms for
// 48->16 at 4 x 64^3, now 0.035 and 0.082 ms.  The next unit is loaded into
// registers while a unit's products run (loading it only when they were done,
// 0.055 and 0.20 ms: the loads' latency was most of the time), and WGS
// workgroups per compute unit are launched, all resident at once (a third
// part more of them than fit 48->16: another 9 %).  What bounds it now: LDS
// reads and writes of the staged tile, and three waves on four matrix units.
//
// SEG positions per K run: 64 on the full-resolution level, 32 and 16 on the
// coarser ones (their row lengths are multiples of these for every patch).
// LDS rows are an odd multiple of 32 bytes, which spreads the eight rows two
// lane groups read together over all banks.
__host__ __device__ constexpr int lds_row(int c) { return (c / 16) % 2 ? c : c + 16; }

typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
__device__ __forceinline__ i16x4 ld_tr(const uint16_t *p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)p);
}

template <int K32>  // 1: 32 positions per product, 0: 16
struct GradFrag {
  i16x4 v[K32 + 1];
  // positions 4g .. 4g+3 (and 16 + 4g ..) of the row at p, this lane's channel
  __device__ __forceinline__ void load(const uint16_t *p, int stride) {
    v[0] = ld_tr(p);
    if constexpr (K32) v[1] = ld_tr(p + 16 * stride);
  }
  __device__ __forceinline__ void ones() {
    for (int h = 0; h < K32 + 1; ++h) v[h] = i16x4{0x3f80, 0x3f80, 0x3f80, 0x3f80};
  }
  __device__ __forceinline__ static f32x4 mul(const GradFrag &a, const GradFrag &b, f32x4 c) {
    if constexpr (K32)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a.v),
                                                     __builtin_bit_cast(bf16x8, b.v), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.v[0], b.v[0], c, 0, 0, 0);
  }
};

template <int CIN, int CU, int COUT, int SEG, int R, int WGS>
__global__ void __launch_bounds__(192, WGS * 3 >= 5 ? 2 : 1)
k_wgrad(const uint16_t *__restrict__ x, int xcs, const uint16_t *__restrict__ up,
        const uint16_t *__restrict__ dy, int dycs,
        float *__restrict__ part, int D, int H, int Wd, long units) {
  constexpr int MT = COUT / 16, NT = CIN / 16, KS = SEG >= 32 ? SEG / 32 : 1;
  constexpr int XS = lds_row(CIN), DS = lds_row(COUT), XP = SEG + 2;
  typedef GradFrag<(SEG >= 32)> Frag;
  __shared__ __attribute__((aligned(16))) uint16_t Xs[R + 2][XP][XS];
  __shared__ __attribute__((aligned(16))) uint16_t Ds[R][SEG][DS];
  const int tid = threadIdx.x, lane = tid & 63, dx = tid >> 6, dz = blockIdx.y;
  const int g = lane >> 4, j = lane & 15;
  const int xo = (4 * g + (j >> 2) + dx) * XS + 4 * (j & 3);
  const int ao = (4 * g + (j >> 2)) * DS + 4 * (j & 3);
  const bool bias = dz == 1 && dx == 1;
  f32x4 acc[3][MT][NT], accb[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    accb[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[t][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  Frag one;
  one.ones();
  const int nseg = Wd / SEG, nyc = H / R;
  // 16-byte chunks of a unit: upsampled channels, the others, dy
  constexpr int UC = CU / 8, XC = CIN / 8 - UC, DC = COUT / 8;
  constexpr int NU = (R + 2) * XP * UC, NX = (R + 2) * XP * XC, ND = R * SEG * DC;
  constexpr int PU = (NU + 191) / 192, PX = (NX + 191) / 192, PD = (ND + 191) / 192;
  uint4 pu[PU + 1], px[PX], pd[PD];
  const uint32_t xbytes = ((uint32_t)(H * Wd - 1) * xcs + 8 * XC) * 2;
  const uint32_t ubytes = (uint32_t)(H / 2) * (Wd / 2) * CU * 2;
  const uint32_t dbytes = ((uint32_t)(R * Wd - 1) * dycs + COUT) * 2;
  // the first unit from u on whose input plane is inside the volume
  auto valid = [&](long u) {
    for (; u < units; u += gridDim.x) {
      const int z2 = (int)(u / ((long)nseg * nyc) % D) + dz - 1;
      if (z2 >= 0 && z2 < D) break;
    }
    return u;
  };
  auto fetch = [&](long u) {
    const int xs = (int)(u % nseg) * SEG;
    long r = u / nseg;
    const int y0 = (int)(r % nyc) * R;
    r /= nyc;
    const long z = r, z2 = r + dz - 1;  // planes of the batch
    const int t_ = opaque(tid);
    auto load = [&](const uint16_t *base, uint32_t bytes, uint32_t off) {
      return __builtin_bit_cast(
          uint4, __builtin_amdgcn_raw_buffer_load_b128(
                     __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(base), 0, bytes,
                                                       0x00020000),
                     off, 0, 0));
    };
    if constexpr (CU > 0) {
#pragma unroll
      for (int i = 0; i < PU; ++i) {
        const int e = t_ + i * 192, c = e % UC, p = (e / UC) % XP, rr = e / (UC * XP);
        const int yy = y0 + rr - 1, xx = xs + p - 1;
        const bool ok = ((i + 1) * 192 <= NU || e < NU) & ((unsigned)yy < (unsigned)H) & ((unsigned)xx < (unsigned)Wd);
        pu[i] = load(up + (z2 >> 1) * (H / 2) * (Wd / 2) * CU, ubytes,
                     ok ? (uint32_t)((yy >> 1) * (Wd >> 1) + (xx >> 1)) * CU * 2 + 16 * c
                        : 0x80000000u);
      }
    }
#pragma unroll
    for (int i = 0; i < PX; ++i) {
      const int e = t_ + i * 192, c = e % XC, p = (e / XC) % XP, rr = e / (XC * XP);
      const int yy = y0 + rr - 1, xx = xs + p - 1;
      const bool ok = ((i + 1) * 192 <= NX || e < NX) & ((unsigned)yy < (unsigned)H) & ((unsigned)xx < (unsigned)Wd);
      px[i] = load(x + z2 * H * Wd * xcs, xbytes,
                   ok ? (uint32_t)(yy * Wd + xx) * xcs * 2 + 16 * c : 0x80000000u);
    }
#pragma unroll
    for (int i = 0; i < PD; ++i) {
      const int e = t_ + i * 192, c = e % DC, p = (e / DC) % SEG, rr = e / (DC * SEG);
      pd[i] = load(dy + (z * H + y0) * Wd * dycs, dbytes,
                   (i + 1) * 192 <= ND || e < ND ? (uint32_t)(rr * Wd + xs + p) * dycs * 2 + 16 * c : 0x80000000u);
    }
  };
  long u = valid(blockIdx.x);
  if (u < units) fetch(u);
  while (u < units) {
    __syncthreads();                  // the previous unit has been read
    {
      const int t_ = opaque(tid);
      if constexpr (CU > 0) {
#pragma unroll
        for (int i = 0; i < PU; ++i) {
          const int e = t_ + i * 192;
          if ((i + 1) * 192 <= NU || e < NU)
            *reinterpret_cast<uint4 *>(&Xs[0][0][0] + e / UC * XS + e % UC * 8) = pu[i];
        }
      }
#pragma unroll
      for (int i = 0; i < PX; ++i) {
        const int e = t_ + i * 192;
        if ((i + 1) * 192 <= NX || e < NX)
          *reinterpret_cast<uint4 *>(&Xs[0][0][0] + e / XC * XS + e % XC * 8 + CU) = px[i];
      }
#pragma unroll
      for (int i = 0; i < PD; ++i) {
        const int e = t_ + i * 192;
        if ((i + 1) * 192 <= ND || e < ND) *reinterpret_cast<uint4 *>(&Ds[0][0][0] + e / DC * DS + e % DC * 8) = pd[i];
      }
    }
    __syncthreads();
    u = valid(u + gridDim.x);
    if (u < units) fetch(u);  // while this one's products run
    Frag a[3][KS][MT];
#pragma unroll
    for (int xr = 0; xr < R + 2; ++xr) {
      if (xr < R) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            a[xr % 3][ks][m].load(&Ds[xr][ks * 32][16 * m] + ao, DS);
            if (bias) accb[m] = Frag::mul(a[xr % 3][ks][m], one, accb[m]);
          }
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          Frag b;
          b.load(&Xs[xr][ks * 32][16 * n] + xo, XS);
#pragma unroll
          for (int t = 0; t < 3; ++t) {
            if (xr - t < 0 || xr - t >= R) continue;
#pragma unroll
            for (int m = 0; m < MT; ++m)
              acc[t][m][n] = Frag::mul(a[(xr - t + 3) % 3][ks][m], b, acc[t][m][n]);
          }
        }
    }
  }
  constexpr int NW = 27 * CIN * COUT;
  float *o = part + (long)blockIdx.x * (NW + COUT);
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          o[((dz * 9 + t * 3 + dx) * COUT + 16 * m + 4 * g + k) * CIN + 16 * n + j] =
              acc[t][m][n][k];
  if (bias && j == 0) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int k = 0; k < 4; ++k) o[NW + 16 * m + 4 * g + k] = accb[m][k];
  }
}

// out[e] = sum of the S partials part[s][e] (e < nw into dW, the rest into
// db): 64 elements by 4 runs of s per workgroup.
__global__ void __launch_bounds__(256)
k_grad_sum(const float *__restrict__ part, int S, int nw, int nb, float *dW, float *db) {
  __shared__ float red[4][64];
  const int q = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int e = blockIdx.x * 64 + l, n = nw + nb;
  float s = 0.f;
  if (e < n) {
#pragma unroll 8
    for (int k = q; k < S; k += 4) s += part[(long)k * n + e];
  }
  red[q][l] = s;
  __syncthreads();
  if (q == 0 && e < n) {
    s = (red[0][l] + red[1][l]) + (red[2][l] + red[3][l]);
    if (e < nw) dW[e] = s;
    else db[e - nw] = s;
  }
}

// BF16 weights of every layer, forward [27][cout][cin_p] and transposed
// [27][cin][cout_p], from the FP32 parameters: one launch (two for each layer
// before, 47 us of a training step).
__global__ void __launch_bounds__(256) k_pack(PackTable t) {
  const PackLayer l = t.l[blockIdx.y];
  const int cin_p = cpad(l.cin), cout_p = cpad(l.cout);
  const int n = 27 * l.cout * cin_p, nt = 27 * l.cin * cout_p;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n + nt; i += gridDim.x * 256) {
    if (i < n) {
      const int ci = i % cin_p, r = i / cin_p;  // r = tap * cout + co
      l.W[i] = ci < l.cin ? f2bf(l.w[(long)r * l.cin + ci]) : (uint16_t)0;
    } else {
      const int j = i - n, co = j % cout_p, ci = j / cout_p % l.cin, tap = j / (cout_p * l.cin);
      l.Wt[j] = co < l.cout ? f2bf(l.w[((long)(26 - tap) * l.cout + co) * l.cin + ci])
                            : (uint16_t)0;
    }
  }
}

// ------------------------------------------------------------- first layer
__global__ void k_first_fwd(const float *__restrict__ x, const float *__restrict__ W,
                            const float *__restrict__ b, uint16_t *y, int ycs, int cout, int N,
                            int D, int H, int Wd) {
  const long npos = (long)N * D * H * Wd;
  for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < npos;
       p += (long)gridDim.x * blockDim.x) {
    const int xx = (int)(p % Wd);
    long r = p / Wd;
    const int yv = (int)(r % H);
    r /= H;
    const int zv = (int)(r % D);
    float nb[27];
#pragma unroll
    for (int tap = 0; tap < 27; ++tap) {
      const int z2 = zv + tap / 9 - 1, y2 = yv + (tap / 3) % 3 - 1, x2 = xx + tap % 3 - 1;
      const bool ok = z2 >= 0 && z2 < D && y2 >= 0 && y2 < H && x2 >= 0 && x2 < Wd;
      nb[tap] = ok ? x[p + ((long)(tap / 9 - 1) * H + (tap / 3) % 3 - 1) * Wd + tap % 3 - 1] : 0.f;
    }
    if (cout % 8 == 0 && ycs % 8 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0) {
      // 8 channels per 16-byte store
      for (int c0 = 0; c0 < cout; c0 += 8) {
        uint32_t w[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          float s0 = b[c0 + 2 * h], s1 = b[c0 + 2 * h + 1];
#pragma unroll
          for (int tap = 0; tap < 27; ++tap) {
            s0 = fmaf(W[tap * cout + c0 + 2 * h], nb[tap], s0);
            s1 = fmaf(W[tap * cout + c0 + 2 * h + 1], nb[tap], s1);
          }
          w[h] = (uint32_t)f2bf(fmaxf(s0, 0.f)) | ((uint32_t)f2bf(fmaxf(s1, 0.f)) << 16);
        }
        *reinterpret_cast<uint4 *>(y + p * ycs + c0) = make_uint4(w[0], w[1], w[2], w[3]);
      }
    } else {
      for (int co = 0; co < cout; ++co) {
        float s = b[co];
#pragma unroll
        for (int tap = 0; tap < 27; ++tap) s = fmaf(W[tap * cout + co], nb[tap], s);
        y[p * ycs + co] = f2bf(fmaxf(s, 0.f));
      }
    }
  }
}

// Four consecutive x positions per thread (Wd % 4 == 0, 16-byte aligned x and
// y, cout % 8 == 0): each of the nine (z, y) rows of the 3x3x3 neighbourhood
// is one 16-byte load plus its two end cells, and a weight, which all lanes
// share, is loaded once for the four positions (once for each of them, with
// the loads in the way of the products, took 85.6 us at 8 x 64^3 x 16, now
// 38.2; the products alone are 23 us of the vector unit).  The taps and their
// order are k_first_fwd's: the same arithmetic for every output.
__global__ void __launch_bounds__(256)
k_first_fwd4(const float *__restrict__ x, const float *__restrict__ W,
             const float *__restrict__ b, uint16_t *__restrict__ y, int ycs, int cout, int D,
             int H, int Wd, long nq) {
  const int wq = Wd >> 2;
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  if (q >= nq) return;
  const int x0 = (int)(q % wq) * 4;
  long r = q / wq;
  const int yv = (int)(r % H);
  r /= H;
  const int zv = (int)(r % D);
  const long nn = r / D;
  // nb[dz * 3 + dy][k]: the input at (zv + dz - 1, yv + dy - 1, x0 + k - 1)
  float nb[9][6];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int z2 = zv + t / 3 - 1, y2 = yv + t % 3 - 1;
    float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
    float lo = 0.f, hi = 0.f;
    if (z2 >= 0 && z2 < D && y2 >= 0 && y2 < H) {
      const float *row = x + ((nn * D + z2) * H + y2) * Wd;
      c = *reinterpret_cast<const float4 *>(row + x0);
      if (x0 > 0) lo = row[x0 - 1];
      if (x0 + 4 < Wd) hi = row[x0 + 4];
    }
    nb[t][0] = lo;
    nb[t][1] = c.x;
    nb[t][2] = c.y;
    nb[t][3] = c.z;
    nb[t][4] = c.w;
    nb[t][5] = hi;
  }
  uint16_t *o = y + 4 * q * ycs;
  for (int c0 = 0; c0 < cout; c0 += 8) {
    float s[4][8];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int h = 0; h < 8; ++h) s[j][h] = b[c0 + h];
#pragma unroll
    for (int tap = 0; tap < 27; ++tap)
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        const float w = W[tap * cout + c0 + h];
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j][h] = fmaf(w, nb[tap / 3][j + tap % 3], s[j][h]);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t w[4];
#pragma unroll
      for (int h = 0; h < 4; ++h)
        w[h] = f2bf2(fmaxf(s[j][2 * h], 0.f), fmaxf(s[j][2 * h + 1], 0.f));
      *reinterpret_cast<uint4 *>(o + j * ycs + c0) = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
}

// First layer's weight and bias gradient: dW[tap][co] = sum_p x[p + tap]
// dy[p][co] on the FP32 matrix unit (v_mfma_f32_16x16x4_f32, K = 4 positions:
// the input stays FP32): 16 channels by 27 taps, the 28th column is ones and
// gives the bias.  Lane l holds A[l%16][l/16] and B[l/16][l%16].  A workgroup
// stages 8 rows of 64 positions and the input around them, keeps its sums in
// registers over its units and writes one partial (k_grad_sum adds them).
// One tap per workgroup and 64 accumulators per thread took 1.06 ms at 4 x
// 64^3, this 0.036 ms.
__global__ void __launch_bounds__(256)
k_first_wgrad(const float *__restrict__ x, const uint16_t *__restrict__ dy, int dycs,
              float *__restrict__ part, int D, int H, int Wd, long units) {
  constexpr int R = 8, SEG = 64, XP = 68;
  __shared__ float Xs[3][R + 2][XP];
  __shared__ __attribute__((aligned(16))) uint16_t Ds[R][SEG][16];
  __shared__ float red[4][28 * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, j = lane & 15;
  const int t1 = 16 + j;
  // offsets of taps j and 16 + j from the position's cell in Xs
  auto off = [](int t) { return ((t / 9) * (R + 2) + (t / 3) % 3) * XP + t % 3; };
  const int o0 = off(j), o1 = t1 < 27 ? off(t1) : 0;
  f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  const int nseg = Wd / SEG, nyc = H / R;
  for (long u = blockIdx.x; u < units; u += gridDim.x) {
    const int xs = (int)(u % nseg) * SEG;
    long r = u / nseg;
    const int y0 = (int)(r % nyc) * R;
    r /= nyc;
    const int z = (int)(r % D);
    const long nn = r / D;
    __syncthreads();
#pragma unroll 4
    for (int i = tid; i < 3 * (R + 2) * (SEG + 2); i += 256) {
      const int p = i % (SEG + 2), rr = (i / (SEG + 2)) % (R + 2), pz = i / ((SEG + 2) * (R + 2));
      const int zz = z + pz - 1, yy = y0 + rr - 1, xx = xs + p - 1;
      const bool ok = zz >= 0 && zz < D && yy >= 0 && yy < H && xx >= 0 && xx < Wd;
      Xs[pz][rr][p] = ok ? x[((nn * D + zz) * H + yy) * Wd + xx] : 0.f;
    }
    const uint16_t *dp = dy + (((nn * D + z) * H + y0) * Wd + xs) * dycs;
#pragma unroll
    for (int i = tid; i < R * SEG * 2; i += 256) {
      const int c = i & 1, p = (i >> 1) % SEG, rr = i / (2 * SEG);
      *reinterpret_cast<uint4 *>(&Ds[rr][p][8 * c]) =
          *reinterpret_cast<const uint4 *>(dp + ((long)rr * Wd + p) * dycs + 8 * c);
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < R / 4; ++h) {
      const int row = wave * (R / 4) + h;
      const float *xr = &Xs[0][row][0] + g;
#pragma unroll 4
      for (int p = 0; p < SEG; p += 4) {
        const float a = bf2f(Ds[row][p + g][j]);
        const float b0 = xr[p + o0];
        float b1 = xr[p + o1];
        b1 = t1 < 27 ? b1 : (t1 == 27 ? 1.f : 0.f);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b0, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b1, acc1, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    red[wave][j * 16 + 4 * g + k] = acc0[k];
    if (t1 < 28) red[wave][t1 * 16 + 4 * g + k] = acc1[k];
  }
  __syncthreads();
  for (int e = tid; e < 28 * 16; e += 256)
    part[(long)blockIdx.x * (28 * 16) + e] = (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
}

// -------------------------------------------------------------------- head
__global__ void k_head_fwd(const uint16_t *__restrict__ y, int ycs, int c,
                           const float *__restrict__ W, const float *__restrict__ b,
                           const float *__restrict__ x0, float *out, long npos) {
  for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < npos;
       p += (long)gridDim.x * blockDim.x) {
    float s = b[0] + x0[p];
    if (c % 8 == 0 && ycs % 8 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0) {
      // 8 channels per 16-byte load
      for (int k0 = 0; k0 < c; k0 += 8) {
        const uint4 u = *reinterpret_cast<const uint4 *>(y + p * ycs + k0);
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          s = fmaf(W[k0 + 2 * h], __uint_as_float(w[h] << 16), s);
          s = fmaf(W[k0 + 2 * h + 1], __uint_as_float(w[h] & 0xffff0000u), s);
        }
      }
    } else {
      for (int k = 0; k < c; ++k) s = fmaf(W[k], bf2f(y[p * ycs + k]), s);
    }
    out[p] = s;
  }
}

// Head backward: the gradient g W of the last activation y through its ReLU,
// and the head's own gradient (16 channels and the bias) as one partial sum
// per workgroup.  One position of 16 channels per thread in 16-byte moves;
// writing the gradient in FP32 one channel at a time, to be masked in another
// pass, took 181 + 35 us at 4 x 64^3, now 16.
__global__ void __launch_bounds__(256)
k_head_bwd(const uint16_t *__restrict__ y, const float *__restrict__ W,
           const float *__restrict__ g, uint16_t *__restrict__ dpre, float *__restrict__ part,
           long npos) {
  float acc[17] = {};
  for (long p = (long)blockIdx.x * 256 + threadIdx.x; p < npos; p += (long)gridDim.x * 256) {
    const float gv = g[p];
    const uint4 *src = reinterpret_cast<const uint4 *>(y + p * 16);
    const uint4 u[2] = {src[0], src[1]};
    uint32_t o[8];
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      const uint4 q = u[h / 4];
      const uint32_t a = h % 4 == 0 ? q.x : h % 4 == 1 ? q.y : h % 4 == 2 ? q.z : q.w;
      o[h] = masked2(a, gv * W[2 * h], gv * W[2 * h + 1]);
      acc[2 * h] = fmaf(gv, __uint_as_float(a << 16), acc[2 * h]);
      acc[2 * h + 1] = fmaf(gv, __uint_as_float(a & 0xffff0000u), acc[2 * h + 1]);
    }
    uint4 *dst = reinterpret_cast<uint4 *>(dpre + p * 16);
    dst[0] = make_uint4(o[0], o[1], o[2], o[3]);
    dst[1] = make_uint4(o[4], o[5], o[6], o[7]);
    acc[16] += gv;
  }
  __shared__ float red[4][17];
#pragma unroll
  for (int k = 0; k < 17; ++k) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) acc[k] += __shfl_xor(acc[k], m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x < 17)
    part[blockIdx.x * 17 + threadIdx.x] = (red[0][threadIdx.x] + red[1][threadIdx.x]) +
                                          (red[2][threadIdx.x] + red[3][threadIdx.x]);
}

// ----------------------------------------------------------- elementwise
// 2x2x2 average of 8 channels of one coarse position per thread, 16 bytes a
// load (memory bound: 28.7 us with one channel per thread at 8 x 64^3 x 16,
// now 9.4).
__global__ void __launch_bounds__(256)
k_pool_fwd(const uint16_t *__restrict__ x, int xcs, uint16_t *__restrict__ y, int ycs, int c8,
           long n, int H, int Wd) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int h2 = H / 2, w2 = Wd / 2;
  const int k = (int)(i % c8) * 8;
  const long p = i / c8;
  const int xx = (int)(p % w2);
  long r = p / w2;
  const int yv = (int)(r % h2);
  r /= h2;  // coarse plane of the batch: 2 r, 2 r + 1 are its fine planes
  uint4 v[8];
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    const long q = ((2 * r + (o >> 2)) * H + 2 * yv + ((o >> 1) & 1)) * Wd + 2 * xx + (o & 1);
    v[o] = *reinterpret_cast<const uint4 *>(x + q * xcs + k);
  }
  uint32_t w[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    float lo = 0.f, hi = 0.f;
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const uint32_t u = h == 0 ? v[o].x : h == 1 ? v[o].y : h == 2 ? v[o].z : v[o].w;
      lo += __uint_as_float(u << 16);
      hi += __uint_as_float(u & 0xffff0000u);
    }
    w[h] = f2bf2(0.125f * lo, 0.125f * hi);
  }
  *reinterpret_cast<uint4 *>(y + p * ycs + k) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Gradient of a skip activation y: that of the decoder (FP32, stride dycs)
// plus a 1/8 of the pooled one's, through the ReLU that made y, as BF16.
// Four channels of a fine position per thread (memory bound; adding the
// pooled gradient in place and masking in a second pass took 46 + 26 us on
// average of the two levels at 4 x 64^3, now 23).
__global__ void __launch_bounds__(256)
k_pool_bwd(const float *__restrict__ dskip, int dscs, const float *__restrict__ dpool,
           const uint16_t *__restrict__ y, uint16_t *__restrict__ dpre, int c4, long n, int H,
           int Wd) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int k = (int)(i % c4) * 4;
  const long p = i / c4;
  const int xx = (int)(p % Wd);
  long r = p / Wd;
  const int yv = (int)(r % H);
  r /= H;  // fine plane of the batch
  const long q = ((r >> 1) * (H / 2) + yv / 2) * (Wd / 2) + xx / 2;
  const float4 s = *reinterpret_cast<const float4 *>(dskip + p * dscs + k);
  const float4 d = *reinterpret_cast<const float4 *>(dpool + q * 4 * c4 + k);
  const uint2 a = *reinterpret_cast<const uint2 *>(y + p * 4 * c4 + k);
  *reinterpret_cast<uint2 *>(dpre + p * 4 * c4 + k) =
      make_uint2(masked2(a.x, s.x + 0.125f * d.x, s.y + 0.125f * d.y),
                 masked2(a.y, s.z + 0.125f * d.z, s.w + 0.125f * d.w));
}

// Gradient of an upsampled activation y: the sum over its eight fine
// positions, through the ReLU that made y, as BF16 (27 us on average of the
// two levels at 4 x 64^3 with one channel per thread, the mask and the
// clearing of the sums in other passes, now 20).
__global__ void __launch_bounds__(256)
k_up_bwd(const float *__restrict__ dy, int dycs, const uint16_t *__restrict__ y,
         uint16_t *__restrict__ dpre, int c4, long n, int H, int Wd) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int k = (int)(i % c4) * 4;
  const long p = i / c4;
  const int xx = (int)(p % Wd);
  long r = p / Wd;
  const int yv = (int)(r % H);
  r /= H;  // coarse plane of the batch
  float4 v[8];
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    const long q =
        ((2 * r + (o >> 2)) * 2 * H + 2 * yv + ((o >> 1) & 1)) * 2 * Wd + 2 * xx + (o & 1);
    v[o] = *reinterpret_cast<const float4 *>(dy + q * dycs + k);
  }
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    s.x += v[o].x;
    s.y += v[o].y;
    s.z += v[o].z;
    s.w += v[o].w;
  }
  const uint2 a = *reinterpret_cast<const uint2 *>(y + p * 4 * c4 + k);
  *reinterpret_cast<uint2 *>(dpre + p * 4 * c4 + k) =
      make_uint2(masked2(a.x, s.x, s.y), masked2(a.y, s.z, s.w));
}

__global__ void k_adam(float *p, const float *__restrict__ g, float *m, float *v, long n,
                       float lr, float b1, float b2, float eps, float bc1, float bc2, float wd) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * ((mi / bc1) / (sqrtf(vi / bc2) + eps) + wd * p[i]);
  }
}

template <int OUT, int CIN, int CU, int COUT, int MTW, int YT, int WX, int WY, bool WL>
hipError_t conv_t(const Act &x, const uint16_t *up, const uint16_t *W, const void *aux, Act y, Vol v,
                  int ncu, hipStream_t st) {
  if (v.w % (16 * WX) || v.h % (YT * WY)) return hipErrorInvalidValue;
  constexpr int NT = 64 * WX * WY * (COUT / 16 / MTW);
  const long tiles = (long)v.n * (v.h / (YT * WY)) * (v.w / (16 * WX));
  const int zl = sweep_planes(tiles, v.d, NT, ncu);
  const int grid = (int)(tiles * (v.d / zl));
  k_conv<CIN, CU, COUT, MTW, YT, WX, WY, WL, OUT><<<grid, NT, 0, st>>>(
      (const uint16_t *)x.p, x.cs, up, W, aux, y.p, y.cs, zl, v.d, v.h, v.w);
  return hipGetLastError();
}

template <int CIN, int CU, int COUT, int SEG, int R, int WGS>
hipError_t wgrad_t(const Act &x, const uint16_t *up, const Act &dy, float *dW, float *db, Vol v,
                   float *scratch, int ncu, hipStream_t st) {
  constexpr int NW = 27 * CIN * COUT;
  if (v.w % SEG || v.h % R) return hipErrorInvalidValue;
  const long units = (long)v.n * v.d * (v.h / R) * (v.w / SEG);
  const int S = grad_groups(units, ncu, WGS, kGradScratch / (NW + COUT));
  k_wgrad<CIN, CU, COUT, SEG, R, WGS><<<dim3(S, 3), 192, 0, st>>>(
      (const uint16_t *)x.p, x.cs, up, (const uint16_t *)dy.p, dy.cs, scratch, v.d, v.h, v.w, units);
  k_grad_sum<<<(NW + COUT + 63) / 64, 256, 0, st>>>(scratch, S, NW, COUT, dW, db);
  return hipGetLastError();
}

}  // namespace

// The weight gradients of the network: (cin, of these upsampled, cout,
// positions per K run, rows per unit, workgroups per CU).  The level fixes the
// run; 96 input channels take four rows so that two workgroups fit a CU's LDS;
// 64->64 has 228 sums in registers and is alone on its CU (24 us at 4 x 16^3;
// two of them, with spills, 54).
#define BRTM_WGRAD_SHAPES(X)                                                               \
  X(16, 0, 16, 64, 8, 3) X(48, 32, 16, 64, 8, 2) X(16, 0, 32, 32, 8, 3) X(32, 0, 32, 32, 8, 2) \
  X(96, 64, 32, 32, 4, 2) X(32, 0, 64, 16, 8, 2) X(64, 0, 64, 16, 8, 1)

// The forward convolutions (ACT) and the transposed ones (MASK, GRAD): (out,
// cin, of these upsampled, cout, output tiles and rows per wave, waves in x
// and y, weights in LDS).
#define BRTM_CONV_SHAPES(X)                                                          \
  X(ACT, 16, 0, 16, 1, 4, 4, 1, true) X(ACT, 48, 32, 16, 1, 4, 4, 2, true)           \
  X(ACT, 16, 0, 32, 1, 4, 2, 2, true) X(ACT, 32, 0, 32, 1, 4, 2, 2, true)            \
  X(ACT, 96, 64, 32, 1, 4, 2, 2, false) X(ACT, 32, 0, 64, 1, 4, 1, 2, false)         \
  X(ACT, 64, 0, 64, 1, 4, 1, 2, false) X(MASK, 16, 0, 16, 1, 4, 4, 1, true)          \
  X(MASK, 32, 0, 32, 1, 4, 2, 2, true) X(MASK, 64, 0, 64, 1, 4, 1, 2, false)         \
  X(GRAD, 16, 0, 48, 3, 2, 4, 2, true) X(GRAD, 32, 0, 96, 3, 2, 2, 2, false)         \
  X(GRAD, 32, 0, 16, 1, 4, 2, 4, true) X(GRAD, 64, 0, 32, 1, 4, 1, 1, false)

// Whether (x, up) are CI input channels of which the first CU are upsampled.
static bool is_input(const Act &x, const Act &up, int ci, int cu) {
  return up.c == cu && x.c == ci - cu && (cu == 0 || up.cs == cu);
}

static hipError_t conv(const Act &x, const Act &up, const uint16_t *W, const void *aux, Act y,
                       Vol v, int out, int ncu, hipStream_t st) {
  if (x.cs % 8 || y.cs % 4) return hipErrorInvalidValue;
#define X(O, CI, CU, CO, MTW, YT, WX, WY, WL)                                               \
  if (out == OUT_##O && is_input(x, up, CI, CU) && y.c == CO)                               \
    return conv_t<OUT_##O, CI, CU, CO, MTW, YT, WX, WY, WL>(x, (const uint16_t *)up.p, W, aux, y, \
                                                            v, ncu, st);
  BRTM_CONV_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t conv3d_fwd(const Act &x, const Act &up, const uint16_t *W, const float *bias, Act y,
                      Vol v, int ncu, hipStream_t st) {
  return conv(x, up, W, bias, y, v, OUT_ACT, ncu, st);
}

hipError_t conv3d_bwd(const Act &dy, const uint16_t *Wt, const Act &act, Act dx, Vol v, int ncu,
                      hipStream_t st) {
  if (act.p && act.cs != dx.cs) return hipErrorInvalidValue;
  return conv(dy, Act{nullptr, 0, 0}, Wt, act.p, dx, v, act.p ? OUT_MASK : OUT_GRAD, ncu, st);
}

hipError_t conv3d_wgrad(const Act &x, const Act &up, const Act &dy, float *dW, float *db, Vol v,
                        float *scratch, int ncu, hipStream_t st) {
  if (x.cs % 8 || dy.cs % 8) return hipErrorInvalidValue;
#define X(CI, CU, CO, SEG, R, WGS)                                                            \
  if (is_input(x, up, CI, CU) && dy.c == CO)                                                 \
    return wgrad_t<CI, CU, CO, SEG, R, WGS>(x, (const uint16_t *)up.p, dy, dW, db, v, scratch, ncu, \
                                         st);
  BRTM_WGRAD_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t pack_weights(const PackTable &t, int layers, hipStream_t st) {
  k_pack<<<dim3(64, layers), 256, 0, st>>>(t);
  return hipGetLastError();
}

hipError_t conv3d_first_fwd(const float *x, const float *W, const float *b, Act y, Vol v,
                            hipStream_t st) {
  const bool quad = v.w % 4 == 0 && y.c % 8 == 0 && y.cs % 8 == 0 &&
                    reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(y.p) % 16 == 0;
  const long nq = (long)v.n * v.spatial() / 4;
  if (quad)
    k_first_fwd4<<<(int)((nq + 255) / 256), 256, 0, st>>>(x, W, b, (uint16_t *)y.p, y.cs, y.c,
                                                          v.d, v.h, v.w, nq);
  else
    k_first_fwd<<<grid1((long)v.n * v.spatial()), 256, 0, st>>>(x, W, b, (uint16_t *)y.p, y.cs,
                                                                 y.c, v.n, v.d, v.h, v.w);
  return hipGetLastError();
}

hipError_t conv3d_first_wgrad(const float *x, const Act &dy, float *dW, float *db, Vol v,
                              float *scratch, int ncu, hipStream_t st) {
  if (dy.c != 16 || dy.cs % 8 || v.w % 64 || v.h % 8) return hipErrorInvalidValue;
  const long units = (long)v.n * v.d * (v.h / 8) * (v.w / 64);
  const int S = (int)std::min(units, 2L * ncu);
  k_first_wgrad<<<S, 256, 0, st>>>(x, (const uint16_t *)dy.p, dy.cs, scratch, v.d, v.h, v.w,
                                   units);
  k_grad_sum<<<7, 256, 0, st>>>(scratch, S, 27 * 16, 16, dW, db);
  return hipGetLastError();
}

hipError_t head_fwd(const Act &y, const float *W, const float *b, const float *x0, float *out,
                    Vol v, hipStream_t st) {
  const long npos = (long)v.n * v.spatial();
  k_head_fwd<<<grid1(npos), 256, 0, st>>>((const uint16_t *)y.p, y.cs, y.c, W, b, x0, out, npos);
  return hipGetLastError();
}

hipError_t head_bwd(const Act &y, const float *W, const float *g, Act dpre, float *dW, float *db,
                    Vol v, float *scratch, hipStream_t st) {
  if (y.c != 16 || y.cs != 16 || dpre.cs != 16) return hipErrorInvalidValue;
  const long npos = (long)v.n * v.spatial();
  k_head_bwd<<<1024, 256, 0, st>>>((const uint16_t *)y.p, W, g, (uint16_t *)dpre.p, scratch, npos);
  k_grad_sum<<<1, 256, 0, st>>>(scratch, 1024, 16, 1, dW, db);
  return hipGetLastError();
}

hipError_t avgpool_fwd(const Act &x, Act y, Vol v, hipStream_t st) {
  if (x.c % 8 || x.cs % 8 || y.cs % 8 || v.d % 2 || v.h % 2 || v.w % 2)
    return hipErrorInvalidValue;
  const long n = (long)v.n * (v.d / 2) * (v.h / 2) * (v.w / 2) * (x.c / 8);
  k_pool_fwd<<<(int)((n + 255) / 256), 256, 0, st>>>((const uint16_t *)x.p, x.cs,
                                                     (uint16_t *)y.p, y.cs, x.c / 8, n, v.h, v.w);
  return hipGetLastError();
}

hipError_t avgpool_bwd(const float *dskip, int dskip_cs, const float *dpool, const Act &y,
                       Act dpre, Vol v, hipStream_t st) {
  if (y.c % 4 || y.cs != y.c || dpre.cs != y.c || dskip_cs % 4) return hipErrorInvalidValue;
  const long n = (long)v.n * v.spatial() * (y.c / 4);
  k_pool_bwd<<<(int)((n + 255) / 256), 256, 0, st>>>(dskip, dskip_cs, dpool,
                                                     (const uint16_t *)y.p, (uint16_t *)dpre.p,
                                                     y.c / 4, n, v.h, v.w);
  return hipGetLastError();
}

hipError_t upsample_bwd(const float *dy, int dy_cs, const Act &y, Act dpre, Vol v,
                        hipStream_t st) {
  if (y.c % 4 || y.cs != y.c || dpre.cs != y.c || dy_cs % 4) return hipErrorInvalidValue;
  const long n = (long)v.n * v.spatial() * (y.c / 4);
  k_up_bwd<<<(int)((n + 255) / 256), 256, 0, st>>>(dy, dy_cs, (const uint16_t *)y.p,
                                                   (uint16_t *)dpre.p, y.c / 4, n, v.h, v.w);
  return hipGetLastError();
}

hipError_t adam_step(float *p, const float *g, float *m, float *v, long n, float lr, float b1,
                     float b2, float eps, float bc1, float bc2, float wd, hipStream_t st) {
  k_adam<<<grid1(n), 256, 0, st>>>(p, g, m, v, n, lr, b1, b2, eps, bc1, bc2, wd);
  return hipGetLastError();
}

}  // namespace brtm
