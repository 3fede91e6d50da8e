// How the network's convolutions and weight gradients are cut for a device of
// ncu compute units.  Plain C++, so that it can also be checked on its own.
#pragma once
#include <algorithm>

namespace brtm {

// Output planes per sweep of a forward convolution (a power of two up to 16
// that divides the depth): as many as leave two workgroups of four waves, or
// one of eight, for a compute unit.  Each sweep stages two planes more than it
// writes: with 1024 workgroups on 256 compute units 16->16 took 48.4 us at 8 x
// 64^3, 44.5 with 512.
inline int sweep_planes(long tiles, int depth, int threads, int ncu) {
  const long want = threads > 256 ? ncu : 2L * ncu;
  int zl = 16;
  while (zl > 1 && (depth % zl || tiles * (depth / zl) < want)) zl /= 2;
  return zl;
}

// Workgroups of a weight gradient for each of its three dz: together up to wgs
// per compute unit, fewer where the volume has fewer units or where the
// partial sums, of which `most` fit their scratch, would be more.
inline int grad_groups(long units, int ncu, int wgs, long most) {
  return (int)std::max(1L, std::min({units, (long)ncu * wgs / 3, most}));
}

}  // namespace brtm
