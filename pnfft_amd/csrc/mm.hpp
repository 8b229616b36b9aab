// mm.hpp -- helpers shared by the matrix-core kernels that take every window from
// tables (gather_mm.hip, scatter_mm.hip): FP64 at m = 2..6, FP32 at m = 7, 8.
#pragma once

#include "b_device.hpp"

namespace pnfft_amd {
namespace mm {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
template <class R>
struct Vec;
template <>
struct Vec<double> {
  using V4 = d4;
  using V2 = double2;
};
template <>
struct Vec<float> {
  using V4 = f4;
  using V2 = float2;
};

// 16 x 4 times 4 x 16 added to c: lane (j = lane & 15, k = lane >> 4) gives A[j][k]
// and B[k][j] and holds four rows of column j (acc_row)
__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// row of element r of a lane's accumulator, k = lane >> 4
template <class R>
__device__ __forceinline__ constexpr int acc_row(int k, int r) {
  return sizeof(R) == 8 ? k + 4 * r : 4 * k + r;
}

constexpr size_t kLdsPerCu = 160 * 1024;  // gfx950

// LDS writes of one lane become visible to the other lanes of its wave
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Windows of one axis evaluated straight into LDS rows (psi and, if WD, psi'),
// for nodes whose coordinates are no longer those of the tables: the formulas
// and operation order of window_axis_s with rolled loops, the B-spline recursion
// in the rows themselves, so that no register array is needed.
template <class R, int CM, bool WD>
__device__ inline void eval_rows(int win, R frac, R nR, R b, R ws, R* psi, R* dpsi) {
  constexpr int m = (CM - 1) / 2;
  const R pi = pi_v(R(0));
  if (win == WIN_BSPLINE) {
    const R u = R(1) - frac;
    psi[1] = R(1);  // M_r values at psi[1 ..], psi[0] = 0 as the window's left edge
    for (int r = 2; r <= 2 * m; r++) {
      if (WD && r == 2 * m)  // the order 2m - 1 values give the derivative
        for (int s = 0; s < CM; s++)
          dpsi[s] = -nR * ((s >= 1 && s < 2 * m ? psi[s] : R(0)) - (s >= 2 ? psi[s - 1] : R(0))) * ws;
      const R inv = R(1) / R(r - 1);
      psi[r] = R(0);
      for (int d = r - 1; d >= 0; d--) {
        const R left = d > 0 ? psi[d] : R(0);
        psi[d + 1] = ((u + R(d)) * psi[d + 1] + (R(r) - u - R(d)) * left) * inv;
      }
    }
    psi[0] = R(0);
    for (int s = 1; s < CM; s++) psi[s] *= ws;
    return;
  }
  const R norm = R(1) / m_sqrt(pi * b);
  for (int s = 0; s < CM; s++) {
    const R u = R(s - m) - frac, xn = frac + R(m - s);
    R p, d = R(0);
    if (win == WIN_GAUSS) {
      p = m_exp(-(u * u) / b) * norm;
      if (WD) d = R(-2) * nR / b * xn * p;
    } else if (win == WIN_SINCPOW) {
      p = ipow(sinc_ref<R>(pi * u / b), 2 * m) / b;
      const R y = pi * xn / b;
      if (WD && m_fabs(y) > Consts<R>::eps) d = R(2 * m) * pi * nR / b * sincpow_c1(y) * p;
    } else {
      p = kb_psi<R>(u, b, m);
      if (WD) d = kb_dpsi<R>(xn, nR, b, m, p);
    }
    psi[s] = p * ws;
    if (WD) dpsi[s] = d * ws;
  }
}

}  // namespace mm
}  // namespace pnfft_amd
