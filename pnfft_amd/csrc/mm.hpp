// mm64.hpp -- shapes and LDS layout shared by the FP64 matrix-core kernels
// (gather_mm64.hip, scatter_mm64.hip).
#pragma once

#include "b_device.hpp"

namespace pnfft_amd {
namespace mm64 {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr size_t kLdsPerCu = 160 * 1024;  // gfx950

// LDS writes of one lane become visible to the other lanes of its wave
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// OR of v over each row of 16 lanes (DPP row shifts); lane 15 of a row holds it
__device__ __forceinline__ unsigned row_or16(unsigned v) {
  v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
  return v;
}

// Windows of one axis evaluated straight into LDS rows (psi and, if WD, psi'),
// for nodes whose coordinates are no longer those of the tables: the formulas
// and operation order of window_axis_s with rolled loops, the B-spline recursion
// in the rows themselves, so that no register array is needed.
template <int CM, bool WD>
__device__ inline void eval_rows(int win, double frac, double nR, double b, double ws, double* psi, double* dpsi) {
  constexpr int m = (CM - 1) / 2;
  const double pi = pi_v(0.);
  if (win == WIN_BSPLINE) {
    const double u = 1. - frac;
    psi[1] = 1.;  // M_r values at psi[1 ..], psi[0] = 0 as the window's left edge
    for (int r = 2; r <= 2 * m; r++) {
      if (WD && r == 2 * m)  // the order 2m - 1 values give the derivative
        for (int s = 0; s < CM; s++)
          dpsi[s] = -nR * ((s >= 1 && s < 2 * m ? psi[s] : 0.) - (s >= 2 ? psi[s - 1] : 0.)) * ws;
      const double inv = 1. / (double)(r - 1);
      psi[r] = 0.;
      for (int d = r - 1; d >= 0; d--) {
        const double left = d > 0 ? psi[d] : 0.;
        psi[d + 1] = ((u + (double)d) * psi[d + 1] + ((double)r - u - (double)d) * left) * inv;
      }
    }
    psi[0] = 0.;
    for (int s = 1; s < CM; s++) psi[s] *= ws;
    return;
  }
  const double norm = 1. / m_sqrt(pi * b);
  for (int s = 0; s < CM; s++) {
    const double u = (double)(s - m) - frac, xn = frac + (double)(m - s);
    double p, d = 0.;
    if (win == WIN_GAUSS) {
      p = m_exp(-(u * u) / b) * norm;
      if (WD) d = -2. * nR / b * xn * p;
    } else if (win == WIN_SINCPOW) {
      p = ipow(sinc_ref<double>(pi * u / b), 2 * m) / b;
      const double y = pi * xn / b;
      if (WD && m_fabs(y) > Consts<double>::eps) d = (double)(2 * m) * pi * nR / b * sincpow_c1(y) * p;
    } else {
      p = kb_psi<double>(u, b, m);
      if (WD) d = kb_dpsi<double>(xn, nR, b, m, p);
    }
    psi[s] = p * ws;
    if (WD) dpsi[s] = d * ws;
  }
}

}  // namespace mm64
}  // namespace pnfft_amd
