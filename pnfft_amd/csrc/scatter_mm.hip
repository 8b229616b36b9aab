// scatter_mm.hip -- adjoint window scatter B^T on the matrix cores with windows from
// tables: FP64 at m = 2..6 (tiles of 8 cells), FP32 at m = 7, 8 (tiles of 4).
//
// This file is compiled once per (precision, mode); the build passes PNFFT_B_REAL
// (float|double) and PNFFT_B_MODE (B_F, B_GRAD or B_FGRAD).
//
// Reference: the scatter node loop of kernel/ndft-parallel.c:2890-3009 with the
// stencil kernels spread_f_c2c / spread_grad_f_c2c of kernel/assign.c:478-640
// (cutoff 2m+1, kernel/ndft-parallel.c:910).
//
// One block per nonempty tile, tiles with more nodes first.  The tile's padded
// subgrid (P = TS + 2m cells per axis) is accumulated in registers: for a plane a
// and four nodes v,
//   G[a][b][c] += sum_v (X_v[a] Y_v[b]) (W_v Z_v[c])
// is one 16x16x4 MFMA per real and imaginary part.  Gradient values add
//   X Y (x) (f Z + g2 Z') + (g0 X'Y + g1 X Y') (x) Z,
// four products instead of the six of three rank-one terms, as the weights g0
// and g1 go into the (complex) left operand.  The eight waves own the planes a =
// w + 8 p: over the eight offsets of a tile every wave meets the stencil equally
// often.  On tiles of 8 cells subgrids of more than 16 columns are taken in two
// phases, the nodes that start in the lower half of axis 2 (columns 0 .. 15) and then the upper
// half (columns 4 .. P - 1): column n of an accumulator holds cell n, and cell
// 16 + n for n < 4 in the second phase, so only those four are written out
// between the phases.  Rows past the sixteenth (XR = P - 16) of PB = 16 / XR
// planes share one accumulator block.  FP32 stencils of 15 and 17 points on tiles
// of 4 cells also have blocks of the columns past the sixteenth (the PB planes on
// the column side) and of the rows and columns past it.
// The subgrid goes to the tile's slot; the fold sums the slots in a fixed order.
//
// What it is bound by: at m = 6 on uniform nodes (N = 128^3, M = 2^22, 128 nodes
// per tile) a launch takes 3.2 ms, against 10.2 ms of the vector column kernel,
// in which each node was applied by the 169 of 400 threads whose column it
// meets.  1.5 ms are the products (timing copies without the one or the other
// part), 1.1 ms the 4.2 GB of slots, the rest the window rows; f takes 128 VGPRs,
// so two blocks share a CU and the rows of one overlap the products of the other
// (256 VGPRs and one block: the same time).  The gradient modes replace kernels
// that added every stencil cell by FP64 LDS atomics: charges and dipoles at m =
// 4, M = 2^19 2.86 -> 0.27 ms per launch.  At m = 2 (25 of the 144 cells of a plane) f is still
// faster than on the column kernel (adjoint, n = 128^3, 6 10^5 uniform nodes 653 -> 252 us)
// and f with gradients than with atomics (552 -> 330).  Gradients alone are 0.5 to 1.0 of the
// atomics' time on most sets (n = 256^3, 10^6 nodes 1682 -> 1103 us) and up to 1.5 where a few
// dense tiles keep the atomics in LDS (n = 32^3, 3 10^5 nodes 188 -> 282); they stay here, where
// the sums repeat bit for bit.
#include "mm.hpp"

namespace pnfft_amd {

namespace {

using namespace bdev;
using namespace mm;

template <class R, int MT, int MODE>
struct ScatterShape {
  static constexpr int CM = 2 * MT + 1, TS = std_tile(MT, sizeof(R) == 8), P = TS + 2 * MT;
  static constexpr bool WF = (MODE == B_F || MODE == B_FGRAD);
  static constexpr bool WG = (MODE == B_GRAD || MODE == B_FGRAD);
  static constexpr int XR = P > 16 ? P - 16 : 0;  // rows past the sixteenth
  static constexpr int PB = XR ? 16 / XR : 1;     // planes whose extra rows fill one block
  static constexpr bool PHASES = XR > 0 && TS == 8, WIDE = XR > 0 && TS == 4;
  static constexpr int NXB = (P + PB - 1) / PB;   // blocks of extra rows (WIDE: of each of three kinds)
  static constexpr int NX = WIDE ? 2 : 1;         // of them per wave at most
  static constexpr int E = P > 16 ? P : 16;      // entries of a window row (zero outside the stencil)
  static constexpr int PITCH = E | 1;            // odd: the 64 rows of a batch start in distinct banks
  static constexpr int NW = 8, NT = 64 * NW, NB = 64;  // waves, threads, nodes per batch
  static constexpr int NP = (P + NW - 1) / NW;   // planes per wave
};

// one thread's share of a node's data: half of the windows of one axis (psi at
// v[0 .. NH), psi' at v[NH .. 2 NH)), or two of its weights (v[0 .. 3])
template <class R, int NH, bool WG>
struct RowLoad {
  int j;  // node id, -1: no node
  R x;    // coordinate now ...
  R px;   // ... and when the tables were made
  R v[(WG ? 2 * NH : NH) > 4 ? (WG ? 2 * NH : NH) : 4];
};

// the it-th batch of NB nodes of the positions [beg, mid) and [mid, end), nlow
// batches in the first part
struct Batch {
  int first, end;
};
template <int NB>
__device__ __forceinline__ Batch batch_at(int it, int beg, int mid, int end, int nlow) {
  Batch b;
  if (it < nlow) {
    b.first = beg + NB * it;
    b.end = mid;
  } else {
    b.first = mid + NB * (it - nlow);
    b.end = end;
  }
  return b;
}

// RG: the real grid of a c2r plan (real node values: the imaginary products are left out).
// ONE: compiled for one block per CU (256 VGPRs) where two are the rule (light_tiles).
template <class R, int MT, int MODE, bool RG, bool ONE>
__global__ __launch_bounds__((ScatterShape<R, MT, MODE>::NT),
                             (ONE || ((sizeof(R) == 8 || !RG) && ScatterShape<R, MT, MODE>::WG) ? 2 : 4)) void scatter_mm_k(
    BArgs<R> A) {
  using S = ScatterShape<R, MT, MODE>;
  using V2 = typename Vec<R>::V2;
  // FP64 sums for FP32 plans as well, as the column and LDS-atomic kernels have: FP32 sums
  // took 757 us instead of 849 (m = 8, M = 2^20, N = 64^3 real; column kernel 3431) but
  // f_hat of clustered nodes was 2.7 times further from an FP64 plan's
  using V4 = d4;
  // Operands of the products.  In the gradient modes they hold sums of a node's terms (f Z +
  // g2 Z', g0 X' Y + g1 X Y'): formed in FP64 as well, so that no term is rounded to 2^-24 of a
  // larger one.
  using Q = std::conditional_t<S::WG, double, R>;
  constexpr int CM = S::CM, TS = S::TS, P = S::P, XR = S::XR, PB = S::PB, E = S::E, PITCH = S::PITCH;
  constexpr int NW = S::NW, NB = S::NB, NP = S::NP, NX = S::NX, NXB = S::NXB;
  constexpr int XD = XR ? XR : 1;  // divisor where there are no extra rows
  constexpr bool WF = S::WF, WG = S::WG;
  constexpr int H0 = (CM + 1) / 2;  // window entries 0 .. H0 - 1 and H0 .. CM - 1 are two threads' share
  __shared__ R s_row[3 * (WG ? 2 : 1)][NB * PITCH];  // X, Y, Z (and X', Y', Z') rows
  __shared__ V2 s_w[WG ? 4 : 1][NB];                 // f, g0, g1, g2
  __shared__ unsigned s_km[NB / 4];                       // per four nodes: planes reached
  __shared__ unsigned char s_bad[3][NB];

  const int4 range = A.oranges[blockIdx.x];
  const int tile = range.x, beg = range.y, end = range.w;
  const int mid = S::PHASES ? range.z : end;
  const int t2 = tile % A.ntile[2];
  const int t1 = (tile / A.ntile[2]) % A.ntile[1];
  const int t0 = tile / (A.ntile[2] * A.ntile[1]);
  const int o0 = t0 * TS, o1 = t1 * TS, o2 = t2 * TS;
  const int n0 = A.g.n[0], n1 = A.g.n[1], n2 = A.g.n[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const long M = A.M;

  // rows phase: waves 0 .. 5 take (axis, half) of node `lane` of the batch, wave
  // 6 the weights f, g0, wave 7 the weights g1, g2
  const int ax = wave < 6 ? wave >> 1 : 0, half = wave & 1;
  const int nt = ax == 0 ? n0 : (ax == 1 ? n1 : n2);
  const int ot = ax == 0 ? o0 : (ax == 1 ? o1 : o2);
  const R bt = (R)(ax == 0 ? A.g.b[0] : (ax == 1 ? A.g.b[1] : A.g.b[2]));
  const R wst = (R)(ax == 0 ? A.g.ws[0] : (ax == 1 ? A.g.ws[1] : A.g.ws[2]));

  const int nlow = (mid - beg + NB - 1) / NB, nbat = nlow + (end - mid + NB - 1) / NB;
  // unconditional loads from clamped positions (discarded where no node exists)
  auto load = [&](int it, RowLoad<R, H0, WG>& L) __attribute__((always_inline)) {
    const Batch b = batch_at<NB>(min(it, nbat - 1), beg, mid, end, nlow);
    const long q = min(b.first + lane, b.end - 1);
    const long j = A.perm[q];
    L.j = b.first + lane < b.end ? (int)j : -1;
    // values go through locals: stores to L on both sides of a branch would be
    // merged into one with a selected address, which puts L in scratch memory
    constexpr int NV = (int)(sizeof(L.v) / sizeof(R));
    R x = R(0), px = R(0), t[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) t[k] = R(0);
    if (wave < 6) {
      x = A.x[3 * j + ax];
      px = A.pre_x[(long)ax * M + q];
#pragma unroll
      for (int s = 0; s < H0; s++) {
        const long at = ((long)ax * CM + min(half * H0 + s, CM - 1)) * M + q;
        t[s] = A.pre_psi[at];
        if (WG) t[H0 + s] = A.pre_dpsi[at];
      }
    } else if (wave == 6) {
      if (WF) {
        const Cplx<R> f = load_f(A, j);
        t[0] = f.x;
        t[1] = f.y;
      }
      if (WG) {
        const Cplx<R> g = load_g(A, j, 0);
        t[2] = g.x;
        t[3] = g.y;
      }
    } else if (WG) {
      const Cplx<R> g = load_g(A, j, 1), h = load_g(A, j, 2);
      t[0] = g.x;
      t[1] = g.y;
      t[2] = h.x;
      t[3] = h.y;
    }
    L.x = x;
    L.px = px;
#pragma unroll
    for (int k = 0; k < NV; k++) L.v[k] = t[k];
  };

  // plane wave + 8 p: G[b = acc_row(lk, r)][column li] in re[p][r], im[p][r]
  const V4 zero4 = {0.0, 0.0, 0.0, 0.0};
  V4 re[NP], im[NP], xre[NX], xim[NX];
#pragma unroll
  for (int p = 0; p < NP; p++) re[p] = im[p] = zero4;
#pragma unroll
  for (int u = 0; u < NX; u++) xre[u] = xim[u] = zero4;
  // this wave's blocks of rows or columns past the sixteenth (planes PB xb .. PB xb +
  // PB - 1; -1: none), kind 0: rows, 1: columns, 2: both.  In two phases the five (m =
  // 6) or three (m = 5) blocks of rows are spread over the SIMDs
  int xb[NX], xk[NX];
  if constexpr (S::WIDE) {
#pragma unroll
    for (int u = 0; u < NX; u++) {
      const int id = wave + NW * u;
      xb[u] = id < 3 * NXB ? id % NXB : -1;
      xk[u] = id / NXB;
    }
  } else {
    xk[0] = 0;
    xb[0] = XR == 4 ? (wave == 3 ? 4 : (wave == 7 ? 0 : (wave >= 4 ? wave - 3 : -1)))
                    : (XR == 2 ? (wave >= 4 && wave < 7 ? wave - 4 : -1) : -1);
  }

  Cplx<R>* const slot = A.slots + (size_t)blockIdx.x * (size_t)(P * P * P);
  // writes the accumulated columns: the four (first phase) or all of them at cells `c`
  auto put = [&](int c, bool on) __attribute__((always_inline)) {
    if (!on) return;
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const int a = wave + NW * p;
      if (a < P) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int b = acc_row<double>(lk, r);
          if (b < P) slot[(a * P + b) * P + c] = cmk<R>((R)re[p][r], (R)im[p][r]);
        }
      }
    }
    if constexpr (XR > 0) {
#pragma unroll
      for (int u = 0; u < NX; u++) {
        if (xb[u] < 0) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int i = acc_row<double>(lk, r);
          int a = PB * xb[u] + i / XD, b = 16 + i % XD, cc = c;
          bool ok = true;
          if (S::WIDE && xk[u] == 1) {
            a = PB * xb[u] + li / XD;
            b = i;
            cc = 16 + li % XD;
          } else if (S::WIDE && xk[u] == 2) {
            ok = li < XD;
            cc = 16 + li;
          }
          if (ok && a < P) slot[(a * P + b) * P + cc] = cmk<R>((R)xre[u][r], (R)xim[u][r]);
        }
      }
    }
  };

  RowLoad<R, H0, WG> L;
  load(0, L);
  int c = li;  // cell of this lane's column
  for (int it = 0; it < nbat || it == nlow; it++) {
    if (S::PHASES && it == nlow) {  // second phase: columns 0 .. 3 become cells 16 .. 19
      put(li, li < 4);
      if (li < 4) {
#pragma unroll
        for (int p = 0; p < NP; p++) re[p] = im[p] = zero4;
        xre[0] = xim[0] = zero4;
        c = 16 + li;
      }
      if (it == nbat) break;
    }
    if (it >= nbat) break;
    const Batch batch = batch_at<NB>(it, beg, mid, end, nlow);
    const int nb = min(NB, batch.end - batch.first);
    // window rows and weights of the batch
    if (wave < 6) {
      int l = 0;
      bool bad = true, moved = false;
      R frac = R(0);
      if (L.j >= 0) {
        const NodeAxis<R> na = node_axis<R>(L.x, nt, MT, A.g.shift);
        const int lo = local_off(na.start, ot, TS, nt);
        // outside the tile, or (moved since binning) in the other half of axis 2
        // than its phase: a zero row, so that the node adds nothing here
        bad = lo < 0 || (S::PHASES && ax == 2 && (lo >= 4) != (it >= nlow));
        l = bad ? 0 : lo;
        frac = na.frac;
        moved = !(L.x == L.px);
      }
      R* const row = s_row[ax] + lane * PITCH;
      R* const drow = s_row[WG ? 3 + ax : ax] + lane * PITCH;
      if (!moved || bad) {
#pragma unroll
        for (int s = 0; s < H0; s++) {
          if (s < CM - H0 || !half) {
            const int i = l + (half ? H0 : 0) + s;
            row[i] = bad ? R(0) : L.v[s];
            if (WG) drow[i] = bad ? R(0) : L.v[H0 + s];
          }
        }
      } else if (!half) {  // its coordinates changed since the tables were made
        eval_rows<R, CM, WG>(A.g.win, frac, (R)nt, bt, wst, row + l, drow + l);
      }
      // zeros at the entries outside the stencil, split between the two threads
#pragma unroll
      for (int s = 0; s < (E - CM + 1) / 2; s++) {
        const int k = 2 * s + half;
        if (k < E - CM) {
          int i = l + CM + k;
          if (i >= E) i -= E;
          row[i] = R(0);
          if (WG) drow[i] = R(0);
        }
      }
      if (!half) {
        s_bad[ax][lane] = (bad && L.j >= 0) ? 1 : 0;
        if (ax == 0) {
          unsigned pm = bad ? 0u : ((1u << CM) - 1u) << l;
          pm |= (unsigned)__shfl_xor((int)pm, 1);
          pm |= (unsigned)__shfl_xor((int)pm, 2);
          if ((lane & 3) == 0) s_km[lane >> 2] = pm;
        }
      }
    } else if (WG || wave == 6) {
      const bool on = L.j >= 0;
      V2 a, b;
      a.x = on ? L.v[0] : R(0);
      a.y = on ? L.v[1] : R(0);
      b.x = on ? L.v[2] : R(0);
      b.y = on ? L.v[3] : R(0);
      if (wave == 6) {
        if (WF) s_w[0][lane] = a;
        if (WG) s_w[WG ? 1 : 0][lane] = b;
      } else {
        s_w[WG ? 2 : 0][lane] = a;
        s_w[WG ? 3 : 0][lane] = b;
      }
    }
    __syncthreads();
    if (wave == 7 && lane < nb && (s_bad[0][lane] | s_bad[1][lane] | s_bad[2][lane]))
      A.stale_list[atomicAdd(A.stale_count, 1u)] = batch.first + lane;  // added by scatter_stale_mm_k
    load(it + 1, L);  // in flight during the products
    const int nq = (nb + 3) >> 2;
    const int ce = min(c, E - 1);
#pragma unroll 1
    for (int q = 0; q < nq; q++) {
      const int v = 4 * q + lk, o = v * PITCH;
      const unsigned km = (unsigned)__builtin_amdgcn_readfirstlane((int)s_km[q]);
      // the B operands of column cell cc (weights times Z): f Z + g2 Z' and, with gradients, Z
      struct Weight {
        Q x, y;
      };
      auto weight = [&](int k) __attribute__((always_inline)) {
        const V2 w = s_w[k][v];
        return Weight{(Q)w.x, (Q)w.y};
      };
      Weight f = {Q(0), Q(0)}, g0 = f, g1 = f, g2 = f;
      if (WF) f = weight(0);
      if constexpr (WG) {
        g0 = weight(1);
        g1 = weight(2);
        g2 = weight(3);
      }
      struct ColOp {
        Q z, re, im;
      };
      auto col = [&](int cc) __attribute__((always_inline)) {
        ColOp q;
        q.z = s_row[2][o + cc];
        q.re = f.x * q.z;
        q.im = f.y * q.z;
        if constexpr (WG) {
          const Q dz = s_row[WG ? 5 : 2][o + cc];
          q.re = fma(g2.x, dz, q.re);
          q.im = fma(g2.y, dz, q.im);
        }
        return q;
      };
      // plane cell a and row b of the A operand against column operand q
      auto mm = [&](int a, int b, const ColOp& q, V4& cr, V4& ci) __attribute__((always_inline)) {
        const Q x = s_row[0][o + a], y = s_row[1][o + b], xy = x * y;
        cr = mfma(xy, q.re, cr);
        if constexpr (!RG) ci = mfma(xy, q.im, ci);
        if constexpr (WG) {
          const Q u = s_row[WG ? 3 : 0][o + a] * y, t = x * s_row[WG ? 4 : 1][o + b];
          cr = mfma(fma(g0.x, u, g1.x * t), q.z, cr);
          if constexpr (!RG) ci = mfma(fma(g0.y, u, g1.y * t), q.z, ci);
        }
      };
      const ColOp main = col(ce);
#pragma unroll
      for (int p = 0; p < NP; p++) {
        const int a = wave + NW * p;
        if (a < P && ((km >> a) & 1u)) mm(a, li, main, re[p], im[p]);
      }
      if constexpr (XR > 0) {
#pragma unroll
        for (int u = 0; u < NX; u++) {
          if (xb[u] < 0 || !((km >> (PB * xb[u])) & ((1u << PB) - 1u))) continue;
          const int a = min(PB * xb[u] + li / XD, P - 1);
          if (!S::WIDE || xk[u] == 0) {
            mm(a, 16 + li % XD, main, xre[u], xim[u]);
          } else if (xk[u] == 2) {
            mm(a, 16 + li % XD, col(16 + li % XD), xre[u], xim[u]);
          } else {
            // columns past the sixteenth: the planes are on the column side, the rows alone on the other,
            //   Y (x) ((f X + g0 X') Z + g2 X Z') + Y' (x) g1 X Z
            const int cc = 16 + li % XD;
            const Q x = s_row[0][o + a], y = s_row[1][o + li], xz = x * s_row[2][o + cc];
            Q br = f.x * xz, bi = f.y * xz;
            if constexpr (WG) {
              const Q dxz = s_row[WG ? 3 : 0][o + a] * (Q)s_row[2][o + cc], xdz = x * s_row[WG ? 5 : 2][o + cc];
              br = fma(g0.x, dxz, fma(g2.x, xdz, br));
              bi = fma(g0.y, dxz, fma(g2.y, xdz, bi));
            }
            xre[u] = mfma(y, br, xre[u]);
            if constexpr (!RG) xim[u] = mfma(y, bi, xim[u]);
            if constexpr (WG) {
              const Q dy = s_row[WG ? 4 : 1][o + li];
              xre[u] = mfma(dy, g1.x * xz, xre[u]);
              if constexpr (!RG) xim[u] = mfma(dy, g1.y * xz, xim[u]);
            }
          }
        }
      }
    }
    __syncthreads();
  }
  put(c, c < P);
}

// nodes found outside the tile (or its half) they are binned to (bins older than
// x): added to the folded grid through global atomics
template <class R, int MT, int MODE>
__global__ __launch_bounds__(256) void scatter_stale_mm_k(BArgs<R> A) {
  using S = ScatterShape<R, MT, MODE>;
  const unsigned count = *A.stale_count;
  for (unsigned k = blockIdx.x * 256 + threadIdx.x; k < count; k += gridDim.x * 256) {
    const long j = A.perm[A.stale_list[k]];
    NodeWin<R, S::CM> w;
    node_windows<R, MT, S::CM, S::WG>(A, -1, j, MT, w);
    scatter_node_global<R, S::CM, MODE, true>(A, j, w, S::CM);
  }
}

// FP64 f on complex grids at m = 5, 6: most tiles hold at most one batch of nodes, so a
// block is its prologue, one batch and its slot.  The two blocks per CU of the dense case
// spill 35 of their 128 VGPRs there, and overlapping them gains nothing: m = 5, n = 256^3, M
// = 10^5 2461 us, one block per CU with 173 VGPRs 2141 (vector column kernel 2264); n =
// 128^3, M = 10^4 358 and 315 us.  From about 70 nodes per tile on two blocks are faster
// (n = 128^3, M = 3 10^5 457 and 448 us, 10^6 673 and 760), and with few tiles as well (512 tiles
// of 20 nodes 110 and 114 us).
template <class R, int MT, int MODE>
bool light_tiles(const BArgs<R>& A) {
  return sizeof(R) == 8 && MODE == B_F && MT > 4 && !A.c2r && A.n_torder >= 1024 && A.M < 64L * A.n_torder;
}

template <class R, int MT, int MODE>
int launch(const BArgs<R>& A, hipStream_t s) {
  using S = ScatterShape<R, MT, MODE>;
  constexpr bool HAS_ONE = sizeof(R) == 8 && MODE == B_F && MT > 4;
  hipLaunchKernelGGL(zero_u32_k, dim3(1), dim3(64), 0, s, A.stale_count);
  const dim3 grid((unsigned)A.n_torder), block(S::NT);
  if (A.c2r)
    hipLaunchKernelGGL((scatter_mm_k<R, MT, MODE, true, false>), grid, block, 0, s, A);
  else if (light_tiles<R, MT, MODE>(A))
    hipLaunchKernelGGL((scatter_mm_k<R, MT, MODE, false, HAS_ONE>), grid, block, 0, s, A);
  else
    hipLaunchKernelGGL((scatter_mm_k<R, MT, MODE, false, false>), grid, block, 0, s, A);
  if (A.mid) (void)hipEventRecord(A.mid, s);
  const int st = fold_slots<R>(A, s);
  if (st != kOk) return st;
  if (A.mid2) (void)hipEventRecord(A.mid2, s);
  hipLaunchKernelGGL((scatter_stale_mm_k<R, MT, MODE>), dim3(64), dim3(256), 0, s, A);
  return hipGetLastError() == hipSuccess ? kOk : kHipError;
}

}  // namespace

template <class R, int MODE>
int scatter_mm(const BArgs<R>& A, hipStream_t s) {
  const int ts = std_tile(A.g.m, sizeof(R) == 8);
  if (A.no_mfma || !A.pre_psi || !A.pre_x || (MODE != B_F && !A.pre_dpsi) || !A.oranges || !A.slots || !A.tile_slot ||
      A.n_torder <= 0 || !A.perm || !A.stale_count || !A.stale_list || A.ts[0] != ts || A.ts[1] != ts || A.ts[2] != ts)
    return kUnsupported;
  if constexpr (sizeof(R) == 8) {
    switch (A.g.m) {
      case 2: return launch<R, 2, MODE>(A, s);
      case 3: return launch<R, 3, MODE>(A, s);
      case 4: return launch<R, 4, MODE>(A, s);
      case 5: return launch<R, 5, MODE>(A, s);
      case 6: return launch<R, 6, MODE>(A, s);
      default: return kUnsupported;
    }
  } else {
    switch (A.g.m) {
      case 7: return launch<R, 7, MODE>(A, s);
      case 8: return launch<R, 8, MODE>(A, s);
      default: return kUnsupported;
    }
  }
}

template int scatter_mm<PNFFT_B_REAL, PNFFT_B_MODE>(const BArgs<PNFFT_B_REAL>&, hipStream_t);

}  // namespace pnfft_amd
