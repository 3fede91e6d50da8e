// 3-D convolution kernels of the learned image-domain preconditioner
// (gfx950).  Activations are channels-last [n][z][y][x][c] BF16 with an
// explicit channel stride (so a layer can read or write a channel slice of a
// buffer); weights are [27 taps][cout][cin_pad] BF16 with
// cin_pad = cin rounded up to 32; accumulation is FP32 on MFMA.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace brtm {

struct Act {          // a channel slice of an activation buffer
  void *p;            // element (0,0,0,0,c0) of the slice
  int c;              // channels in the slice
  int cs;             // channel stride of the buffer (elements)
};

struct Vol {          // spatial shape (per batch item)
  int n, d, h, w;
  long spatial() const { return (long)d * h * w; }
};

// y = ReLU(conv3x3x3(x, W) + b), zero padding 1.
// up: the first input channels when they come from a volume of half the size
// through nearest-neighbour upsampling (channels contiguous), or no channels.
// ncu (here and below): compute units of the device.
hipError_t conv3d_fwd(const Act &x, const Act &up, const uint16_t *W, const float *bias, Act y,
                      Vol v, int ncu, hipStream_t st);
// Input gradient: the convolution of dy with the transposed weights, FP32
// into dx; with act (the input itself, an activation), through its ReLU
// (dx = 0 where act <= 0) as BF16.
hipError_t conv3d_bwd(const Act &dy, const uint16_t *Wt, const Act &act, Act dx, Vol v, int ncu,
                      hipStream_t st);
// dW[tap][co][ci] = sum_p dy[p][co] x[p + tap][ci] (FP32, [27][cout][cin]);
// db[co] = sum_p dy[p][co].  scratch holds kGradScratch floats.
constexpr long kGradScratch = 8L << 20;
hipError_t conv3d_wgrad(const Act &x, const Act &up, const Act &dy, float *dW, float *db, Vol v,
                        float *scratch, int ncu, hipStream_t st);
// BF16 weights of a layer from the FP32 masters w [27][cout][cin]: W
// [27][cout][cin_pad], and those of the transposed convolution Wt[tap][ci][co]
// = W[26-tap][co][ci] (channels padded to 32).
struct PackLayer {
  const float *w;
  uint16_t *W, *Wt;
  int cin, cout;
};
struct PackTable {
  PackLayer l[9];
};
hipError_t pack_weights(const PackTable &t, int layers, hipStream_t st);

// First layer: 1 FP32 input channel -> cout BF16 channels, ReLU.
hipError_t conv3d_first_fwd(const float *x, const float *W, const float *b, Act y, Vol v,
                            hipStream_t st);
// Its weight and bias gradient (16 channels; overwrites dW [27][16] and db).
hipError_t conv3d_first_wgrad(const float *x, const Act &dy, float *dW, float *db, Vol v,
                              float *scratch, int ncu, hipStream_t st);
// Head: 1x1x1 conv cin -> 1 FP32 plus the residual input: out = x0 + W.y + b.
hipError_t head_fwd(const Act &y, const float *W, const float *b, const float *x0, float *out,
                    Vol v, hipStream_t st);
// Head backward: dpre = g W through the ReLU of y (BF16), dW and db.
hipError_t head_bwd(const Act &y, const float *W, const float *g, Act dpre, float *dW, float *db,
                    Vol v, float *scratch, hipStream_t st);

// 2x2x2 average pool (v is the input shape).
hipError_t avgpool_fwd(const Act &x, Act y, Vol v, hipStream_t st);
// Gradient of a pooled activation y that also is a skip connection: dskip
// plus the pool's adjoint of dpool, through y's ReLU.
hipError_t avgpool_bwd(const float *dskip, int dskip_cs, const float *dpool, const Act &y,
                       Act dpre, Vol v, hipStream_t st);
// Gradient of an activation y (of shape v) that was upsampled x2: the adjoint
// of the upsampling, through y's ReLU.
hipError_t upsample_bwd(const float *dy, int dy_cs, const Act &y, Act dpre, Vol v,
                        hipStream_t st);
// Adam step on FP32 parameters.
hipError_t adam_step(float *p, const float *g, float *m, float *v, long n, float lr, float b1,
                     float b2, float eps, float bc1, float bc2, float wd, hipStream_t st);

}  // namespace brtm
