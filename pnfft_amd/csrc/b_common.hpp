// b_common.hpp -- per-node stencil geometry shared by the B kernels and the binning.
#pragma once

#include "device_common.hpp"

namespace pnfft_amd {

// Natural grid index of stencil point s = 0 on one axis, (floor(n x) - m) mod n
// (kernel/ndft-parallel.c:2165-2174), and the FP64 fractional part of n x.
template <class R>
struct NodeAxis {
  int start;  // natural index of stencil point s = 0
  R frac;     // n x - floor(n x)
};

// n is a power of two (plans reject other oversampled lengths): floor(n x) mod n
// is fl - n floor(fl / n), exact in FP64 for |n x| < 2^53 (the scaling by 1/n is
// an exponent shift), and the shift by -m wraps with a mask.  sh (0 or 1/2, the
// interlaced pass) is added to n x in FP64, where both are exact.
template <class R>
__device__ inline NodeAxis<R> node_axis(R xv, int n, int m, double sh) {
  const double nx = (double)n * (double)xv + sh;
  const double fl = floor(nx);
  NodeAxis<R> a;
  a.frac = (R)(nx - fl);
  const double q = floor(ldexp(fl, -__builtin_ctz((unsigned)n)));
  const int r = (int)fma(-q, (double)n, fl);
  a.start = (r - m) & (n - 1);
  return a;
}

// Ranges of a tile of cnt nodes for the matrix-core gather with tables (gather_mm.hip) and
// the nodes of one: 512 each, or about `item` < 512 in whole groups of 16 (a tile of up to 1.25
// `item` is one; the last ranges may be short or empty).
__host__ __device__ inline int tile_ranges(int cnt, int item) {
  if (item >= 512) return (cnt + item - 1) / item;
  return cnt <= 0 ? 0 : (cnt + item * 3 / 4 < 2 * item ? 1 : (cnt + item * 3 / 4) / item);
}
__host__ __device__ inline int range_len(int cnt, int item) {
  if (item >= 512) return item;
  const int k = tile_ranges(cnt, item);
  return k <= 1 ? cnt : ((cnt + k - 1) / k + 15) / 16 * 16;
}

}  // namespace pnfft_amd
