// gather_mm.hip -- gather (trafo B) on the matrix cores with windows from tables:
// FP64 at m = 3..6 (tiles of 8 cells), FP32 at m = 7, 8 (tiles of 4).
//
// This file is compiled once per (precision, mode); the build passes PNFFT_B_REAL
// (float|double) and PNFFT_B_MODE (BMode).
//
// Reference: the node loops of kernel/ndft-parallel.c:2703-3009 and the
// stencil kernels of kernel/assign.c:642-1066 (cutoff 2m+1, :910).
//
// For a plane a of a tile's padded subgrid (P = TS + 2m cells per axis) and a
// group of 16 sorted nodes,
//   T_a[b][j] = sum_c G[a][b][c] Z_j[c]      (Z_j = psi_z of node j, zero outside its stencil)
// is a product of a 16 x 4 NK and a 4 NK x 16 matrix: a 16x16x4 MFMA per
// K-block of four c, per real and imaginary part (and with psi'_z for the
// gradient).  A lane (j = lane & 15, k = lane >> 4) then holds T_a[b][j] for the
// rows b = acc_row(k, r) and forms f_j = sum_a X_j[a] sum_b Y_j[b] T_a[b][j] on the
// vector units.  Subgrids of 18 and 20 rows have XR = 2 or 4 rows past the
// sixteenth; those of 16 / XR planes make one more 16-row product.
//
// What it is bound by: at m = 6 on uniform nodes (N = 128^3, M = 2^22, 128 nodes
// per tile) a launch takes 2.49 ms, against 8.53 ms of the vector kernel, whose
// threads read every stencil cell of their own node from LDS (13^3 16-byte
// reads per node; here 16 nodes share each read).  1.15 ms are matrix-core
// cycles (64 per product, 16 nodes: 2.2 times the stencil's own multiply-adds),
// about 0.3 ms the row sums, which do not overlap with them (FP64 products and
// FP64 vector instructions share one pipe), and 1.1 ms the phases before and
// after, which one block per CU cannot hide (the 128 KB subgrid of m = 6 leaves
// no room for a second; staging alone is 0.49 ms).  Windows always come from
// tables: evaluating them here costs registers for 13 doubles per axis and
// leaves two waves per SIMD instead of three, with spills in the product loops
// (gradient modes at m = 5: 1.27 ms with, 0.90 ms without the evaluation).  Waves
// in flight decide the rest: m = 4, M = 2^20, 2048 nodes per tile, f takes 323 us
// with three waves per SIMD and 227 us with four.
#include "mm.hpp"

namespace pnfft_amd {

namespace {

using namespace bdev;
using namespace mm;

// Items of at most kFew nodes are gathered from the grid, one wave per node:
// staging a subgrid reads P^3 cells where kFew stencils read kFew (2m+1)^3.
constexpr int kFew = 3;

template <class R, int MT, int MODE, bool RG>
struct GatherShape {
  static constexpr int CM = 2 * MT + 1, TS = std_tile(MT, sizeof(R) == 8), P = TS + 2 * MT;
  static constexpr int NK = (P + 3) / 4;        // K-blocks of a subgrid row
  static constexpr int PITCH = 4 * NK;          // cells per row in LDS (columns past P are zero)
  static constexpr int XR = P > 16 ? P - 16 : 0;  // rows past the sixteenth
  static constexpr int PB = XR ? 16 / XR : 1;     // planes whose extra rows fill one product
  static constexpr bool WF = (MODE == B_F || MODE == B_FGRAD);
  static constexpr bool WG = (MODE == B_GRAD || MODE == B_FGRAD || MODE == B_VJP);
  static constexpr size_t SUB = (size_t)P * P * PITCH * sizeof(R) * (RG ? 1 : 2);
  static constexpr int AREA = 16 * CM * (WG ? 2 : 1);  // reals: one axis' windows of a wave's 16 nodes
  static constexpr size_t lds(int nw) { return SUB + (size_t)nw * AREA * sizeof(R); }
  // waves per SIMD, in as many blocks as the LDS holds: FP64 four for f up to m = 4
  // (128 VGPRs suffice) and three above, two for the gradient modes; FP32 three
  static constexpr int WAVES = sizeof(R) == 4 ? 3 : (WG ? 2 : (P <= 16 ? 4 : 3));
  static constexpr bool fits(int blocks) {
    return 4 * WAVES % blocks == 0 && 4 * WAVES / blocks >= 4 && blocks * lds(4 * WAVES / blocks) <= kLdsPerCu;
  }
  static constexpr int BLOCKS = fits(4) ? 4 : (fits(3) ? 3 : (fits(2) ? 2 : 1));
  static constexpr int NW = 4 * WAVES / BLOCKS;
  // the next group's window loads are in flight during the products, except where
  // their 4 CM registers would spill (FP64 gradient modes on complex grids at m = 5, 6)
  static constexpr bool AHEAD = !WG || MT <= 4 || RG || sizeof(R) == 4;
  static constexpr int NT = 64 * NW;
  static constexpr size_t LDS = lds(NW);
  static_assert(LDS <= kLdsPerCu, "subgrid and window rows fit the LDS");
  static_assert(NW >= kFew, "a wave for each of few nodes");
};

// Position of cell c in LDS row b.  A wave's operand read takes one cell per
// lane: 16 rows b and four consecutive c; the exclusive-or spreads rows whose
// pitch is a multiple of the bank period over distinct banks.
template <class R, int NK, bool RG>
__device__ __forceinline__ int cell_pos(int b, int c) {
  if constexpr (RG || sizeof(R) == 4)
    return c ^ (NK % 2 == 0 ? 2 * ((b >> 1) & 7) : 2 * ((b >> 3) & 1));
  else
    return c ^ (NK % 2 == 0 ? (b & 7) : ((b >> 1) & 3));
}

// one lane's share of a node's window data: axis lk of node li of a group
template <class R, int CM, bool WG>
struct AxisLoad {
  int j;  // node id, -1: no node
  R x;    // coordinate now ...
  R px;   // ... and when the tables were made
  R psi[CM];
  R dpsi[WG ? CM : 1];
};

// positions of one group of nodes
struct Group {
  int first, end;
};
// Group g of the positions [beg, mid) and [mid, end), nlow groups in the first part.
__device__ __forceinline__ Group group_at(int g, int beg, int mid, int end, int nlow) {
  Group p;
  if (g < nlow) {
    p.first = beg + 16 * g;
    p.end = mid;
  } else {
    p.first = mid + 16 * (g - nlow);
    p.end = end;
  }
  return p;
}
// Group that a wave takes in round `it`: one each, in the last round (it ==
// rounds) `whole` of them whole and the others by sp waves each.
__device__ __forceinline__ int group_of(int it, int rounds, int NW, int wave, int whole, int sp) {
  int k = wave;
  if (it == rounds && wave >= whole) k = whole + (wave - whole) / sp;
  return it * NW + k;
}

template <int N>
struct IntC {
  static constexpr int value = N;
};

template <class R, int MT, int MODE, bool RG>
__global__ __launch_bounds__((GatherShape<R, MT, MODE, RG>::NT),
                             (GatherShape<R, MT, MODE, RG>::WAVES)) void gather_mm_k(BArgs<R> A) {
  using S = GatherShape<R, MT, MODE, RG>;
  using V2 = typename Vec<R>::V2;
  using V4 = typename Vec<R>::V4;
  constexpr int CM = S::CM, TS = S::TS, P = S::P, NK = S::NK, PITCH = S::PITCH, XR = S::XR, PB = S::PB;
  constexpr int NW = S::NW, NT = S::NT;
  constexpr bool WF = S::WF, WG = S::WG;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  V2* const sub = reinterpret_cast<V2*>(smem_raw);  // [P][P][PITCH] complex cells ...
  R* const sub_r = reinterpret_cast<R*>(smem_raw);  // ... or real cells (c2r plans)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  R* const rows = reinterpret_cast<R*>(smem_raw + S::SUB) + wave * S::AREA;  // this wave's window rows

  const int4 range = A.ranges[blockIdx.x];
  const int tile = range.x, beg = range.y, end = range.w;
  const int t2 = tile % A.ntile[2];
  const int t1 = (tile / A.ntile[2]) % A.ntile[1];
  const int t0 = tile / (A.ntile[2] * A.ntile[1]);
  const int o0 = t0 * TS, o1 = t1 * TS, o2 = t2 * TS;
  const int n0 = A.g.n[0], n1 = A.g.n[1], n2 = A.g.n[2];
  const bool few = end - beg <= kFew;

  // Groups of 16 nodes, one per wave and round, formed apart for the nodes that
  // start in the lower and in the upper half of axis 2 (positions up to mid and
  // from there on): each then reaches one K-block less than a row has, and its
  // nodes, sorted by axis 0, share most of their planes.  The last round's groups are
  // taken whole by fours (one per SIMD); the up to three left over are shared by
  // `sp` of the idle waves each, which take every sp-th plane and add their sums
  // at the end: nine groups then cost a SIMD 2.25 groups instead of 3.
  const int mid = few ? end : range.z;  // few nodes: one group, every wave reads all of it
  const int nlow = (mid - beg + 15) >> 4;
  const int ngroups = nlow + ((end - mid + 15) >> 4);
  const int rounds = ngroups / NW, left = ngroups - rounds * NW;
  const int whole = few ? 0 : left & ~3, odd = left - whole;
  const int sp = few || odd == 0 ? 1 : (4 * odd <= NW - whole ? 4 : (2 * odd <= NW - whole ? 2 : 1));
  const int nit = rounds + (left > 0 ? 1 : 0);

  // this lane's axis (lane group 3 holds none)
  const int ax = lk < 3 ? lk : 0;
  const int nt = ax == 0 ? n0 : (ax == 1 ? n1 : n2);
  const int ot = ax == 0 ? o0 : (ax == 1 ? o1 : o2);
  const R bt = (R)(ax == 0 ? A.g.b[0] : (ax == 1 ? A.g.b[1] : A.g.b[2]));
  const R wst = (R)(ax == 0 ? A.g.ws[0] : (ax == 1 ? A.g.ws[1] : A.g.ws[2]));
  const long M = A.M;

  // unconditional loads from clamped positions (discarded where no node exists)
  auto pos_at = [&](int it) __attribute__((always_inline)) {
    const Group p = group_at(min(group_of(min(it, nit - 1), rounds, NW, wave, whole, sp), ngroups - 1), beg, mid, end, nlow);
    return min(p.first + li, p.end - 1);
  };
  auto load_group = [&](int it, int j, AxisLoad<R, CM, WG>& L) __attribute__((always_inline)) {
    const Group p = group_at(min(group_of(min(it, nit - 1), rounds, NW, wave, whole, sp), ngroups - 1), beg, mid, end, nlow);
    const bool ok = p.first + li < p.end;
    const long q = min(p.first + li, p.end - 1);
    L.j = ok ? j : -1;
    L.x = A.x[3 * (long)j + ax];
    L.px = A.pre_x[(long)ax * M + q];
    const R* tp = A.pre_psi + (long)ax * CM * M + q;
#pragma unroll
    for (int s = 0; s < CM; s++) L.psi[s] = tp[s * M];
    if (WG) {
      const R* td = A.pre_dpsi + (long)ax * CM * M + q;
#pragma unroll
      for (int s = 0; s < CM; s++) L.dpsi[s] = td[s * M];
    }
  };

  AxisLoad<R, CM, WG> L;
  const int j0 = A.perm[pos_at(0)];
  int jn = A.perm[pos_at(1)];

  if (!few) {
    // stage the subgrid: LDS positions in order, the cells they hold from the grid
    if constexpr (RG) {  // pairs of real cells (an even offset never straddles the wrap)
      constexpr int NQ = P * P * PITCH / 2, K = (NQ + NT - 1) / NT;
      const V2* src = reinterpret_cast<const V2*>(A.grid);
      V2 v[K];
#pragma unroll
      for (int k = 0; k < K; k++) {
        const int q = tid + NT * k;
        v[k].x = v[k].y = R(0);
        if (q < NQ) {
          const int cy = (q / (PITCH / 2)) % P, cx = q / (PITCH / 2 * P);
          const int c = cell_pos<R, NK, RG>(cy, 2 * (q % (PITCH / 2)));
          const size_t row = (size_t)((o0 + cx) & (n0 - 1)) * n1 + ((o1 + cy) & (n1 - 1));
          if (c < P) v[k] = src[(row * n2 + ((o2 + c) & (n2 - 1))) >> 1];
        }
      }
#pragma unroll
      for (int k = 0; k < K; k++)
        if (tid + NT * k < NQ) reinterpret_cast<V2*>(sub_r)[tid + NT * k] = v[k];
    } else {
      constexpr int NQ = P * P * PITCH, K = (NQ + NT - 1) / NT;
      const V2* src = reinterpret_cast<const V2*>(A.grid);
      V2 v[K];
#pragma unroll
      for (int k = 0; k < K; k++) {
        const int q = tid + NT * k;
        v[k].x = v[k].y = R(0);
        if (q < NQ) {
          const int cy = (q / PITCH) % P, cx = q / (PITCH * P);
          const int c = cell_pos<R, NK, RG>(cy, q % PITCH);
          const size_t row = (size_t)((o0 + cx) & (n0 - 1)) * n1 + ((o1 + cy) & (n1 - 1));
          if (c < P) v[k] = src[row * n2 + ((o2 + c) & (n2 - 1))];
        }
      }
#pragma unroll
      for (int k = 0; k < K; k++)
        if (tid + NT * k < NQ) sub[tid + NT * k] = v[k];
    }
  }
  __syncthreads();
  load_group(0, j0, L);

  // operand reads: this lane's row and, per K-block, its cell in it
  const int bl = min(li, P - 1);
  int off[NK];
#pragma unroll
  for (int e = 0; e < NK; e++) off[e] = bl * PITCH + cell_pos<R, NK, RG>(bl, 4 * e + lk);

  for (int it = 0; it < nit; it++) {
    const bool adds = it == rounds && sp > 1;  // uniform in the block
    const bool works = few ? wave < end - beg : (it < rounds || wave < whole + odd * sp);
    if (!works) {
      if (adds) __syncthreads();
      break;
    }
    const bool shared = adds && wave >= whole;
    const int part = shared ? (wave - whole) % sp : 0, step = shared ? sp : 1;
    const int jg = L.j, pos = pos_at(it);
    // windows of this lane's axis for node li of the group
    int l = 1 << 20, start = 0;  // l: offset of the stencil start in the tile; out of reach: no contribution
    bool bad = false;
    bool moved = false;  // coordinates changed since the tables were made
    R frac = R(0);
    if (lk < 3 && jg >= 0) {
      const NodeAxis<R> na = node_axis<R>(L.x, nt, MT, A.g.shift);
      start = na.start;
      frac = na.frac;
      const int lo = local_off(na.start, ot, TS, nt);
      bad = lo < 0;
      if (!bad) l = lo;
      moved = !(L.x == L.px);
    }
    if (__any(moved)) {
      for (int t = 0; t < 3; t++) {
        const bool mine = lk == t && moved;
        wave_sync();
        if (mine)
          eval_rows<R, CM, WG>(A.g.win, frac, (R)nt, bt, wst, rows + li * CM, rows + 16 * CM + li * CM);
        wave_sync();
        if (mine) {
#pragma unroll
          for (int s = 0; s < CM; s++) {
            L.psi[s] = rows[li * CM + s];
            if (WG) L.dpsi[s] = rows[16 * CM + li * CM + s];
          }
        }
      }
    }
    const unsigned long long badm = __ballot(bad);
    const unsigned stale = (unsigned)(badm | (badm >> 16) | (badm >> 32)) & 0xFFFFu;
    const bool ok = jg >= 0 && !((stale >> li) & 1u);
    if (!ok) l = 1 << 20;

    // A node's sums over planes and lane groups are FP64 for FP32 plans too: with FP32
    // sums f at m = 8 was up to 1.3% further from an FP64 plan's than the vector
    // kernel's.
    double fr = 0.0, fi = 0.0, g0r = 0.0, g0i = 0.0, g1r = 0.0, g1i = 0.0, g2r = 0.0, g2i = 0.0;
    if (few) {
      // this wave's node straight from the grid: windows of axis t of node li at
      // rows[(4 t + li) CM ..], lane r takes the stencil rows (a, b) = (r / CM, r % CM), r + 64, ...
      wave_sync();
      if (lk < 3 && li < kFew) {
#pragma unroll
        for (int s = 0; s < CM; s++) {
          rows[(4 * lk + li) * CM + s] = L.psi[s];
          if (WG) rows[16 * CM + (4 * lk + li) * CM + s] = L.dpsi[s];
        }
      }
      const int s0 = __shfl(start, wave), s1 = __shfl(start, 16 + wave), s2 = __shfl(start, 32 + wave);
      const int j = __shfl(jg, wave);
      wave_sync();
      const R *wx = rows + wave * CM, *wy = wx + 4 * CM, *wz = wx + 8 * CM;
      for (int r = lane; r < CM * CM; r += 64) {
        const int a = r / CM, b = r - (r / CM) * CM;
        const size_t row = ((size_t)((s0 + a) & (n0 - 1)) * n1 + ((s1 + b) & (n1 - 1))) * n2;
        R hr = R(0), hi = R(0), hzr = R(0), hzi = R(0);
#pragma unroll
        for (int s = 0; s < CM; s++) {
          const size_t i = row + ((s2 + s) & (n2 - 1));
          R gr, gi = R(0);
          if constexpr (RG) {
            gr = reinterpret_cast<const R*>(A.grid)[i];
          } else {
            const V2 v = reinterpret_cast<const V2*>(A.grid)[i];
            gr = v.x;
            gi = v.y;
          }
          hr += wz[s] * gr;
          if (!RG) hi += wz[s] * gi;
          if (WG) {
            hzr += wz[16 * CM + s] * gr;
            if (!RG) hzi += wz[16 * CM + s] * gi;
          }
        }
        const R xy = wx[a] * wy[b];
        fr = fma((double)xy, (double)hr, fr);
        fi = fma((double)xy, (double)hi, fi);
        if (WG) {
          const R dxy = wx[16 * CM + a] * wy[b], xdy = wx[a] * wy[16 * CM + b];
          g0r = fma((double)dxy, (double)hr, g0r);
          g0i = fma((double)dxy, (double)hi, g0i);
          g1r = fma((double)xdy, (double)hr, g1r);
          g1i = fma((double)xdy, (double)hi, g1i);
          g2r = fma((double)xy, (double)hzr, g2r);
          g2i = fma((double)xy, (double)hzi, g2i);
        }
      }
      auto red = [](double v) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
        return v;
      };
      Cplx<R> v[4] = {cmk<R>(red(fr), red(fi)), cmk<R>(R(0), R(0)), cmk<R>(R(0), R(0)), cmk<R>(R(0), R(0))};
      if (WG) {
        v[1] = cmk<R>(red(g0r), red(g0i));
        v[2] = cmk<R>(red(g1r), red(g1i));
        v[3] = cmk<R>(red(g2r), red(g2i));
      }
      if (lane == 0) gather_store<R, MODE>(A, j, v);
      return;
    }

    // offsets of the group's nodes per axis as bit masks (lane 15 + 16 t of axis t)
    const unsigned om = row_or16(l < TS ? (1u << l) : 0u);
    const unsigned xm = (unsigned)__builtin_amdgcn_readlane((int)om, 15);
    const unsigned ym = (unsigned)__builtin_amdgcn_readlane((int)om, 31);
    const unsigned zm = (unsigned)__builtin_amdgcn_readlane((int)om, 47);
    const int amin = xm ? __builtin_ctz(xm) : P, amax = xm ? 31 - __builtin_clz(xm) + CM - 1 : -1;
    // the nodes' offsets on each axis for this lane's node li
    const int lx = __shfl(l, li), ly = __shfl(l, 16 + li), lz = __shfl(l, 32 + li);

    // one axis' windows at a time through the wave's rows
    auto put = [&](int t) __attribute__((always_inline)) {
      wave_sync();
      if (lk == t) {
#pragma unroll
        for (int s = 0; s < CM; s++) {
          rows[li * CM + s] = L.psi[s];
          if (WG) rows[16 * CM + li * CM + s] = L.dpsi[s];
        }
      }
      wave_sync();
    };
    // window (d = 1: derivative) of node li at cell c of the axis in the rows, whose offset is lo
    auto at = [&](int d, int c, int lo) __attribute__((always_inline)) {
      const int i = c - lo;
      const bool in = (unsigned)i < (unsigned)CM;
      const R v = rows[(d ? 16 * CM : 0) + li * CM + (in ? i : 0)];
      return in ? v : R(0);
    };
    R y[4], dy[4], y16[4], dy16[4], z[NK], dz[NK];
    put(1);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int b = acc_row<R>(lk, r);
      y[r] = at(0, b, ly);
      dy[r] = WG ? at(1, b, ly) : R(0);
      if constexpr (XR > 0) {  // rows past the sixteenth: row b of their product is row 16 + b % XR
        y16[r] = at(0, 16 + b % XR, ly);
        dy16[r] = WG ? at(1, 16 + b % XR, ly) : R(0);
      }
    }
    put(2);
#pragma unroll
    for (int e = 0; e < NK; e++) {
      z[e] = at(0, 4 * e + lk, lz);
      dz[e] = WG ? at(1, 4 * e + lk, lz) : R(0);
    }
    put(0);

    // loads for the wave's next group
    if (S::AHEAD && it + 1 < nit) {
      load_group(it + 1, jn, L);
      jn = A.perm[pos_at(it + 2)];
    }

    // 16 rows of the subgrid (per lane: base address of its row) times the
    // z windows, K-blocks K0 .. K0 + N - 1
    auto sums = [&](auto k0c, auto nkc) __attribute__((always_inline)) {
      constexpr int K0 = decltype(k0c)::value, N = decltype(nkc)::value;
      struct Op {
        R re[N], im[N];
      };
      auto ld = [&](int base, const int (&of)[NK], Op& o) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < N; e++) {
          if constexpr (RG) {
            o.re[e] = sub_r[base + of[K0 + e]];
          } else {
            const V2 v = sub[base + of[K0 + e]];
            o.re[e] = v.x;
            o.im[e] = v.y;
          }
        }
      };
      auto prod = [&](const Op& o, const R (&zz)[NK], V4& tr, V4& ti) __attribute__((always_inline)) {
        tr = V4{R(0), R(0), R(0), R(0)};
        ti = tr;
#pragma unroll
        for (int e = 0; e < N; e++) {
          tr = mfma(o.re[e], zz[K0 + e], tr);
          if constexpr (!RG) ti = mfma(o.im[e], zz[K0 + e], ti);
        }
      };
      Op o;
      ld(min(amin + part, P - 1) * (P * PITCH), off, o);
      for (int a = amin + part; a <= amax; a += step) {
        Op on;
        ld(min(a + step, P - 1) * (P * PITCH), off, on);
        const R xa = at(0, a, lx);
        V4 tr, ti;
        prod(o, z, tr, ti);
        R sr = y[0] * tr[0], si = y[0] * ti[0];
#pragma unroll
        for (int r = 1; r < 4; r++) {
          sr += y[r] * tr[r];
          if constexpr (!RG) si += y[r] * ti[r];
        }
        if (WF) {
          fr = fma((double)xa, (double)sr, fr);
          if constexpr (!RG) fi = fma((double)xa, (double)si, fi);
        }
        if constexpr (WG) {
          const R da = at(1, a, lx);
          g0r = fma((double)da, (double)sr, g0r);
          if constexpr (!RG) g0i = fma((double)da, (double)si, g0i);
          sr = dy[0] * tr[0];
          si = dy[0] * ti[0];
#pragma unroll
          for (int r = 1; r < 4; r++) {
            sr += dy[r] * tr[r];
            if constexpr (!RG) si += dy[r] * ti[r];
          }
          g1r = fma((double)xa, (double)sr, g1r);
          if constexpr (!RG) g1i = fma((double)xa, (double)si, g1i);
          prod(o, dz, tr, ti);
          sr = y[0] * tr[0];
          si = y[0] * ti[0];
#pragma unroll
          for (int r = 1; r < 4; r++) {
            sr += y[r] * tr[r];
            if constexpr (!RG) si += y[r] * ti[r];
          }
          g2r = fma((double)xa, (double)sr, g2r);
          if constexpr (!RG) g2i = fma((double)xa, (double)si, g2i);
        }
        o = on;
      }
      if constexpr (XR > 0) {
        // rows 16 .. P - 1 of the planes a0 .. a0 + PB - 1: row i of the product is
        // row 16 + i % XR of plane a0 + i / XR (past amax the x windows are zero)
        if (ym >> (16 - (CM - 1) > 0 ? 16 - (CM - 1) : 0)) {
          const int b16 = 16 + li % XR;
          int of[NK];
#pragma unroll
          for (int e = 0; e < NK; e++) of[e] = b16 * PITCH + cell_pos<R, NK, RG>(b16, 4 * e + lk);
          for (int a0 = amin + PB * part; a0 <= amax; a0 += PB * step) {
            Op q;
            ld(min(a0 + li / XR, P - 1) * (P * PITCH), of, q);
            V4 tr, ti;
            prod(q, z, tr, ti);
            R xy[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const int a = a0 + acc_row<R>(lk, r) / XR;
              const R xa = at(0, a, lx);
              xy[r] = xa * y16[r];
              if (WF) {
                fr = fma((double)xy[r], (double)tr[r], fr);
                if constexpr (!RG) fi = fma((double)xy[r], (double)ti[r], fi);
              }
              if constexpr (WG) {
                const R dxy = at(1, a, lx) * y16[r], xdy = xa * dy16[r];
                g0r = fma((double)dxy, (double)tr[r], g0r);
                g1r = fma((double)xdy, (double)tr[r], g1r);
                if constexpr (!RG) {
                  g0i = fma((double)dxy, (double)ti[r], g0i);
                  g1i = fma((double)xdy, (double)ti[r], g1i);
                }
              }
            }
            if constexpr (WG) {
              prod(q, dz, tr, ti);
#pragma unroll
              for (int r = 0; r < 4; r++) {
                g2r = fma((double)xy[r], (double)tr[r], g2r);
                if constexpr (!RG) g2i = fma((double)xy[r], (double)ti[r], g2i);
              }
            }
          }
        }
      }
    };
    if (xm) {
      // a stencil of 2m+1 cells from an offset below four ends before the last
      // K-block, one from four or more starts after the first; both meet in a
      // group only where nodes moved since they were binned
      const bool lo = (zm & 0x0Fu) != 0, hi = (zm & 0xF0u) != 0;
      if constexpr (TS < 8) sums(IntC<0>{}, IntC<NK>{});  // stencils of 4 (NK - 1) - 1 cells and more
      else if (lo && hi) sums(IntC<0>{}, IntC<NK>{});
      else if (lo) sums(IntC<0>{}, IntC<NK - 1>{});
      else sums(IntC<1>{}, IntC<NK - 1>{});
    }
    // sum over the four lane groups
    auto red = [](double v) {
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      return v;
    };
    if (WF) {
      fr = red(fr);
      fi = red(fi);
    }
    if (WG) {
      g0r = red(g0r);
      g0i = red(g0i);
      g1r = red(g1r);
      g1i = red(g1i);
      g2r = red(g2r);
      g2i = red(g2i);
    }
    if (adds) {
      // the sums of the group's waves, through their window rows (read by now)
      const R part_sum[8] = {(R)fr, (R)fi, (R)g0r, (R)g0i, (R)g1r, (R)g1i, (R)g2r, (R)g2i};
      constexpr int V0 = WF ? 0 : 2, NV = (WG ? 8 : 2) - V0;
      static_assert(16 * NV <= S::AREA, "a wave's sums fit its window rows");
      wave_sync();
      if (part > 0 && lk == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) rows[k * 16 + li] = part_sum[V0 + k];
      __syncthreads();
      if (part > 0) break;
      R sum[8];
#pragma unroll
      for (int k = 0; k < NV; k++) {
        sum[V0 + k] = part_sum[V0 + k];
        for (int q = 1; q < step; q++) sum[V0 + k] += rows[q * S::AREA + k * 16 + li];
      }
      if (WF) {
        fr = sum[0];
        fi = sum[1];
      }
      if (WG) {
        g0r = sum[2];
        g0i = sum[3];
        g1r = sum[4];
        g1i = sum[5];
        g2r = sum[6];
        g2i = sum[7];
      }
    }
    if (lk == 0 && jg >= 0) {
      if (ok) {
        Cplx<R> v[4] = {cmk<R>((R)fr, (R)fi), cmk<R>((R)g0r, (R)g0i), cmk<R>((R)g1r, (R)g1i),
                        cmk<R>((R)g2r, (R)g2i)};
        gather_store<R, MODE>(A, jg, v);
      } else {
        A.stale_list[atomicAdd(A.stale_count, 1u)] = pos;  // gathered by gather_stale_mm_k
      }
    }
    if (!S::AHEAD && it + 1 < nit) {
      load_group(it + 1, jn, L);
      jn = A.perm[pos_at(it + 2)];
    }
  }
}

// nodes found outside the tile they are binned to (bins older than x): gathered
// straight from the grid
template <class R, int MT, int MODE>
__global__ __launch_bounds__(256) void gather_stale_mm_k(BArgs<R> A) {
  constexpr int CM = 2 * MT + 1;
  constexpr bool WG = (MODE == B_GRAD || MODE == B_FGRAD || MODE == B_VJP);
  const unsigned count = *A.stale_count;
  for (unsigned k = blockIdx.x * 256 + threadIdx.x; k < count; k += gridDim.x * 256) {
    const long j = A.perm[A.stale_list[k]];
    NodeWin<R, CM> w;
    node_windows<R, MT, CM, WG>(A, -1, j, MT, w);
    gather_node_global<R, CM, MODE, true>(A, j, w, CM);
  }
}

template <class R, int MT, int MODE>
void launch(const BArgs<R>& A, hipStream_t s) {
  hipLaunchKernelGGL(zero_u32_k, dim3(1), dim3(64), 0, s, A.stale_count);
  auto go = [&](auto rgc) {
    constexpr bool RG = decltype(rgc)::value;
    using S = GatherShape<R, MT, MODE, RG>;
    (void)hipFuncSetAttribute((const void*)gather_mm_k<R, MT, MODE, RG>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)S::LDS);
    hipLaunchKernelGGL((gather_mm_k<R, MT, MODE, RG>), dim3((unsigned)A.n_ranges), dim3(S::NT), S::LDS, s, A);
  };
  if (A.c2r)
    go(std::true_type{});
  else
    go(std::false_type{});
  if (A.mid) (void)hipEventRecord(A.mid, s);
  if (A.mid2) (void)hipEventRecord(A.mid2, s);
  hipLaunchKernelGGL((gather_stale_mm_k<R, MT, MODE>), dim3(64), dim3(256), 0, s, A);
}

}  // namespace

// FP64 gradient modes on complex grids whose node set the vector kernel takes faster, with
// windows from the same tables.
// m = 3: few tiles that are heavy, or so uneven that some are cut (n = 128^3, 3 10^5 nodes in
// eight clusters 183 and 219 us here; 122 uniform nodes per tile 328 and 286).
// m = 5, where registers and the 104 KB subgrid leave two waves per SIMD and nothing to overlap
// the staging: tiles that are one vector block of 512 nodes but a long range or two short ones
// here (n = 64^3, 293 per tile 184 and 216 us, n = 128^3, 488 per tile 1345 and 1462; 244 per tile
// 1016 and 806, n = 64^3, 586 per tile 331 and 297), and sets of full ranges whose waves of 256
// blocks (40 us each) cost more than those of the vector kernel (73 us; 10^5 nodes on n = 32^3
// 128 and 151 us, 5 10^4 120 and 112).
template <class R, int MODE>
bool vector_gradient(const BArgs<R>& A) {
  if (sizeof(R) != 8 || MODE == B_F || A.c2r || !A.items || A.n_items <= 0) return false;
  if (A.g.m == 3) return A.n_torder <= 4096 && (A.n_cut > 0 || A.M >= 150L * A.n_items);
  if (A.g.m != 5) return false;
  const bool one = A.n_cut == 0 && A.M > 256L * A.n_torder && A.M <= 512L * A.n_torder;
  return one || (A.M >= 65536 && 73L * ((A.n_items + 255) / 256) < 40L * ((A.n_ranges + 255) / 256));
}

template <class R, int MODE>
int gather_mm(const BArgs<R>& A, hipStream_t s) {
  const int ts = std_tile(A.g.m, sizeof(R) == 8);
  if (A.no_mfma || !A.pre_psi || !A.pre_x || (MODE != B_F && !A.pre_dpsi) || !A.ranges || A.n_ranges <= 0 ||
      !A.all_dense || !A.perm || !A.stale_count || !A.stale_list || A.ts[0] != ts || A.ts[1] != ts || A.ts[2] != ts ||
      vector_gradient<R, MODE>(A))
    return kUnsupported;
  if constexpr (sizeof(R) == 8) {
    switch (A.g.m) {
      case 3: launch<R, 3, MODE>(A, s); break;
      case 4: launch<R, 4, MODE>(A, s); break;
      case 5: launch<R, 5, MODE>(A, s); break;
      case 6: launch<R, 6, MODE>(A, s); break;
      default: return kUnsupported;
    }
  } else {
    switch (A.g.m) {
      case 7: launch<R, 7, MODE>(A, s); break;
      case 8: launch<R, 8, MODE>(A, s); break;
      default: return kUnsupported;
    }
  }
  return hipGetLastError() == hipSuccess ? kOk : kHipError;
}

template int gather_mm<PNFFT_B_REAL, PNFFT_B_MODE>(const BArgs<PNFFT_B_REAL>&, hipStream_t);

}  // namespace pnfft_amd
