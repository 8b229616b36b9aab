// nfft_b.hip -- matrix B of the NFFT (window gather for trafo, window scatter
// for adj) and the binning of nodes by grid cell.
//
// Reference: PNX(trafo_B_ad) / PNX(adjoint_B_ad) and their node loops
// (kernel/ndft-parallel.c:2521-3009) with the stencil kernels of
// kernel/assign.c:478-1066.  The reference stores the FFT output shifted and
// ghost-padded by m cells and exchanges the ghost layers (PX(exchange) /
// PX(reduce), :2558, :2679); here the grid stays in natural DFT order and the
// periodic wrap is applied to the stencil indices, so no ghost copy exists.
//
// Node n's stencil on axis t covers grid indices (floor(n_t x_t) - m + s) mod n_t,
// s = 0..2m (cutoff 2m+1, :910, :2165-2174).  floor(n x) is taken in FP64 for
// both precisions; the window is evaluated in the compute precision from the
// FP64 fractional part.
#include <algorithm>
#include <cstdio>
#include <mutex>

#include "device_common.hpp"
#include "b_common.hpp"
#include "nfft_b.hpp"
#include "window_math.hpp"

namespace pnfft_amd {

namespace {

constexpr int kB = 256;  // threads per block of the B kernels

// ---------------------------------------------------------------------------
// binning: keys, stable LSD radix sort, tile bounds
//
// Up to about 2^21 nodes it is bound by the number of dependent launches and
// host waits, not by bytes: three launches per digit pass (the first pass takes
// its counts from the key kernel), four for the tile lists, one host wait.  With
// five launches per pass, separate kernels for the items, classes and bounds and
// five waits a binning took 357 us at M = 2^19 (now 135) and 365 at 2^20 (now 148).
// ---------------------------------------------------------------------------
constexpr int kSortT = 256;
constexpr int kScanChunk = 4096;

// Items per block of the sort passes.  A block ranks its items 256 at a time, a
// chain of barriers, so small node sets take small blocks (M = 20001: 20 us per
// pass with 4096 items, 8 us with 1024); from 2^20 nodes on 4096 items fill the
// chip and keep the digit counts few.
inline int sort_ipb(long M) { return M <= (1L << 18) ? 1024 : (M <= (1L << 20) ? 2048 : 4096); }
inline long sort_blocks(long M) { return (M + sort_ipb(M) - 1) / sort_ipb(M); }

// Bin key of every node, and the counts of the keys' lowest digit per block of
// IPB items (digit-major: hist[d nblk + block]).
template <class R, int IPB>
__global__ __launch_bounds__(kSortT) void bin_keys_k(const R* __restrict__ x, long M, GridGeom g, TileLayout T,
                                                     unsigned* keys, unsigned* hist, int nblk) {
  __shared__ unsigned h[256];
  const int tid = threadIdx.x;
  h[tid] = 0;
  __syncthreads();
  // cell order inside a tile: runs of q = min(TS2, 4) cells along axis 2
  // outermost, then axis 0, axis 1 and the cell within the run, so that
  // consecutive nodes of a tile share the quarter of axis 2 their stencils start
  // in (the matrix-core gather then skips one of its four K-blocks for most
  // 16-node groups)
  const unsigned q = T.ts[2] < 4 ? (unsigned)T.ts[2] : 4u;
  const long base = (long)blockIdx.x * IPB;
#pragma unroll 4
  for (int i = 0; i < IPB / kSortT; i++) {
    const long j = base + (long)i * kSortT + tid;
    if (j < M) {
      unsigned long long tile = 0;
      unsigned l[3];
      for (int t = 0; t < 3; t++) {
        const NodeAxis<R> a = node_axis<R>(x[3 * j + t], g.n[t], g.m, g.shift);
        tile = tile * T.ntile[t] + (unsigned)(a.start / T.ts[t]);
        l[t] = (unsigned)(a.start % T.ts[t]);
      }
      const unsigned long long in =
          ((unsigned long long)(l[2] / q) * (T.ts[0] * T.ts[1]) + l[0] * T.ts[1] + l[1]) * q + l[2] % q;
      const unsigned key = (unsigned)(tile * (unsigned long long)(T.ts[0] * T.ts[1] * T.ts[2]) + in);
      keys[j] = key;
      atomicAdd(&h[key & 255u], 1u);
    }
  }
  __syncthreads();
  hist[(long)tid * nblk + blockIdx.x] = h[tid];
}

template <int IPB>
__global__ __launch_bounds__(kSortT) void sort_hist_k(const unsigned* __restrict__ keys, long M, int shift,
                                                      unsigned* hist, int nblk) {
  __shared__ unsigned h[256];
  const int tid = threadIdx.x;
  h[tid] = 0;
  __syncthreads();
  const long base = (long)blockIdx.x * IPB;
#pragma unroll 4
  for (int i = 0; i < IPB / kSortT; i++) {
    const long idx = base + (long)i * kSortT + tid;
    if (idx < M) atomicAdd(&h[(keys[idx] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[(long)tid * nblk + blockIdx.x] = h[tid];
}

// Block-wide exclusive scan of 256 values held one per thread.
__device__ inline unsigned block_exscan256(unsigned v, unsigned* tmp, unsigned* total) {
  const int tid = threadIdx.x;
  tmp[tid] = v;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    unsigned add = (tid >= off) ? tmp[tid - off] : 0u;
    __syncthreads();
    tmp[tid] += add;
    __syncthreads();
  }
  const unsigned incl = tmp[tid];
  if (total) *total = tmp[255];
  __syncthreads();
  return incl - v;
}

// exclusive scan in place of d[0, n) by one block, 16 values per thread and round
__device__ inline void block_scan(unsigned* d, long n, unsigned* tmp, unsigned* total) {
  constexpr int PER = 16;
  __shared__ unsigned tot;
  unsigned carry = 0;
  for (long base = 0; base < n; base += 256 * PER) {
    const long at = base + (long)threadIdx.x * PER;
    unsigned loc[PER], s = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      loc[i] = at + i < n ? d[at + i] : 0u;
      s += loc[i];
    }
    unsigned ex = block_exscan256(s, tmp, &tot) + carry;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      if (at + i < n) d[at + i] = ex;
      ex += loc[i];
    }
    carry += tot;
    __syncthreads();
  }
  if (total && threadIdx.x == 0) *total = carry;
}

// block d: exclusive scan of digit d's per-block counts in place; total[d] = their sum
__global__ __launch_bounds__(kSortT) void digit_scan_k(unsigned* hist, int nblk, unsigned* total) {
  __shared__ unsigned tmp[256];
  block_scan(hist + (long)blockIdx.x * nblk, nblk, tmp, total + blockIdx.x);
}

// Exclusive scans of several arrays of n values (array blockIdx.y at d +
// blockIdx.y n): one block per array, or chunk sums, their scan and its addition.
__global__ __launch_bounds__(kSortT) void scan_whole_k(unsigned* d, long n) {
  __shared__ unsigned tmp[256];
  block_scan(d + (long)blockIdx.y * n, n, tmp, nullptr);
}

__global__ __launch_bounds__(kSortT) void scan_reduce_k(const unsigned* __restrict__ d, long n, unsigned* partial) {
  __shared__ unsigned tmp[256];
  __shared__ unsigned tot;
  constexpr int PER = kScanChunk / kSortT;
  const long base = (long)blockIdx.x * kScanChunk + (long)threadIdx.x * PER;
  unsigned s = 0;
  for (int i = 0; i < PER; i++)
    if (base + i < n) s += d[(long)blockIdx.y * n + base + i];
  (void)block_exscan256(s, tmp, &tot);
  if (threadIdx.x == 0) partial[(long)blockIdx.y * gridDim.x + blockIdx.x] = tot;
}

__global__ __launch_bounds__(kSortT) void scan_partials_k(unsigned* partial, long np) {
  __shared__ unsigned tmp[256];
  block_scan(partial + (long)blockIdx.y * np, np, tmp, nullptr);
}

__global__ __launch_bounds__(kSortT) void scan_apply_k(unsigned* d, long n, const unsigned* __restrict__ partial) {
  __shared__ unsigned tmp[256];
  __shared__ unsigned tot;
  constexpr int PER = kScanChunk / kSortT;
  unsigned* const dd = d + (long)blockIdx.y * n;
  const long base = (long)blockIdx.x * kScanChunk + (long)threadIdx.x * PER;
  unsigned loc[PER];
  unsigned s = 0;
  for (int i = 0; i < PER; i++) {
    const long idx = base + i;
    loc[i] = idx < n ? dd[idx] : 0u;
    s += loc[i];
  }
  unsigned ex = block_exscan256(s, tmp, &tot) + partial[(long)blockIdx.y * gridDim.x + blockIdx.x];
  for (int i = 0; i < PER; i++) {
    const long idx = base + i;
    if (idx < n) dd[idx] = ex;
    ex += loc[i];
  }
}

// Stable scatter of one digit pass: items of a block are ranked in index order
// and placed by digit in LDS first, so that the stores to the output are runs
// of consecutive positions (one per digit present in the block) rather than
// one scattered 4-byte store per item.  offs: per digit, the exclusive scan of
// its per-block counts (digit_scan_k), total: the digits' counts, whose scan
// every block forms itself.  vin null: the first pass, item ids in order.
template <int IPB>
__global__ __launch_bounds__(kSortT) void sort_scatter_k(const unsigned* __restrict__ kin, const int* __restrict__ vin,
                                                         unsigned* kout, int* vout, long M, int shift,
                                                         const unsigned* __restrict__ offs,
                                                         const unsigned* __restrict__ total, int nblk) {
  constexpr int kSortIPB = IPB;
  __shared__ unsigned run[256];
  __shared__ unsigned wcnt[4][256];
  __shared__ unsigned loc[256];   // first LDS position of digit d
  __shared__ unsigned gdst[256];  // output position of LDS position 0 for digit d
  __shared__ unsigned tmp[256];
  __shared__ unsigned sk[kSortIPB];
  __shared__ int sv[kSortIPB];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const long base = (long)blockIdx.x * kSortIPB;
  {
    const long e = (long)tid * nblk + blockIdx.x;  // entry (digit tid, this block)
    const unsigned in = offs[e], all = total[tid];
    const unsigned c = ((int)blockIdx.x + 1 < nblk ? offs[e + 1] : all) - in;
    const unsigned o = block_exscan256(all, tmp, nullptr) + in;
    const unsigned l = block_exscan256(c, tmp, nullptr);
    loc[tid] = l;
    gdst[tid] = o - l;
    run[tid] = 0;
  }
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int r = 0; r < kSortIPB / kSortT; r++) {
    const long idx = base + (long)r * kSortT + tid;
    const bool valid = idx < M;
    unsigned key = 0;
    int val = 0;
    unsigned d = 0;
    if (valid) {
      key = kin[idx];
      val = vin ? vin[idx] : (int)idx;
      d = (key >> shift) & 255u;
    }
#pragma unroll
    for (int w = 0; w < 4; w++) wcnt[w][tid] = 0;
    __syncthreads();
    unsigned long long mask = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < 8; bit++) {
      const bool on = (d >> bit) & 1u;
      const unsigned long long bb = __ballot(valid && on);
      mask &= on ? bb : ~bb;
    }
    const unsigned rank = (unsigned)__popcll(mask & lt_mask);
    if (valid && rank == 0) wcnt[wave][d] = (unsigned)__popcll(mask);
    __syncthreads();
    if (valid) {
      unsigned pre = run[d] + rank;
      for (int w = 0; w < wave; w++) pre += wcnt[w][d];
      const unsigned at = loc[d] + pre;  // < the block's item count: the counts of all digits sum to it
      sk[at] = key;
      sv[at] = val;
    }
    __syncthreads();
    run[tid] += wcnt[0][tid] + wcnt[1][tid] + wcnt[2][tid] + wcnt[3][tid];
    __syncthreads();
  }
  const int nv = (int)min((long)kSortIPB, M - base);
  for (int i = tid; i < nv; i += kSortT) {
    const unsigned key = sk[i];
    const unsigned pos = gdst[(key >> shift) & 255u] + (unsigned)i;
    kout[pos] = key;
    vout[pos] = sv[i];
  }
}

// First sorted position of every tile by bisection (a walk over the keys would
// leave the gap before a tile to one thread: clustered nodes), and cleared
// counters and offset masks.
__global__ __launch_bounds__(kB) void tile_bounds_k(const unsigned* __restrict__ skeys, long M, unsigned vol,
                                                    long ntiles, int* tile_start, unsigned* work, unsigned* box) {
  const long t = (long)blockIdx.x * kB + threadIdx.x;
  if (t < kTileWork) work[t] = 0u;
  if (t > ntiles) return;
  long lo = 0, hi = M;
  while (lo < hi) {
    const long c = (lo + hi) >> 1;
    if ((long)(skeys[c] / vol) < t) lo = c + 1;
    else hi = c;
  }
  tile_start[t] = (int)lo;
  if (t < ntiles) box[t] = 0u;
}

// For each class of the wave's active lanes, one lane adds the class's lane
// count to ctr[class] and every lane of the class gets the old value plus its
// rank among them (lanes in order).  Neighbouring tiles mostly share a class,
// so a wave issues a few atomics instead of one per tile.
__device__ inline unsigned wave_class_add(bool act, int cls, unsigned* ctr) {
  const int lane = threadIdx.x & 63;
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  unsigned pos = 0;
  unsigned long long todo = __ballot(act);
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const int c = __shfl(cls, leader);
    const unsigned long long same = __ballot(act && cls == c);
    unsigned base = 0;
    if (lane == leader) base = atomicAdd(&ctr[c], (unsigned)__popcll(same));
    base = __shfl(base, leader);
    if (act && cls == c) pos = base + (unsigned)__popcll(same & lt_mask);
    todo &= ~same;
  }
  return pos;
}

// Tiles per block of tile_class_k and tile_place_k: the class counts are
// gathered in LDS over this many tiles, so that a block adds each class to the
// global counters once (per-wave global atomics on the 32 counters serialize).
constexpr int kClassTiles = 8 * kB;
// (one tile per thread for small grids, where eight in a row would be a chain)
inline int class_rounds(long ntiles) { return ntiles > 65536 ? kClassTiles / kB : 1; }

// Slots (order entries) of a tile: one for up to c.whole nodes, else one per c.part nodes.
__device__ inline unsigned tile_parts(int cnt, TileCut c) {
  return cnt > c.whole ? (unsigned)((cnt + c.part - 1) / c.part) : (cnt > 0 ? 1u : 0u);
}

// Work items of a tile.
__device__ inline unsigned tile_chunks(int cnt) { return (unsigned)((cnt + kTileThreads - 1) / kTileThreads); }

// Per tile: order entries by node-count class (leading zeros of the count: more
// nodes, smaller class) added to work[class], and the values whose scans place
// the tile: flag of 2..31 nodes, flag of one node, work items of the gather, ranges
// and work items of the scatter, where they differ.
__global__ __launch_bounds__(kB) void tile_class_k(const int* __restrict__ tile_start, long ntiles, int dense_min,
                                                   TileCut cut, bool two_lists, int rounds, unsigned* work,
                                                   unsigned* scan, unsigned char* dense, unsigned char* dense_s) {
  __shared__ unsigned lc[32];
  if (threadIdx.x < 32) lc[threadIdx.x] = 0;
  __syncthreads();
  for (int i = 0; i < rounds; i++) {
    const long t = ((long)blockIdx.x * rounds + i) * kB + threadIdx.x;
    const int cnt = t < ntiles ? tile_start[t + 1] - tile_start[t] : 0;
    if (t < ntiles) {
      const bool d = cnt >= dense_min && cnt > 0;
      const unsigned ch = tile_chunks(cnt);
      dense[t] = d ? 1 : 0;
      dense_s[t] = cnt > 0 ? 1 : 0;
      scan[t] = (cnt > 1 && cnt < 32) ? 1u : 0u;
      scan[ntiles + t] = cnt == 1 ? 1u : 0u;
      scan[2 * ntiles + t] = d ? ch : 0u;
      scan[3 * ntiles + t] = (unsigned)tile_ranges(cnt, cut.item);
      if (two_lists) scan[4 * ntiles + t] = ch;
    }
    const unsigned parts = tile_parts(cnt, cut);
    (void)wave_class_add(cnt > 0, cnt > 0 ? __clz(cnt) : 0, lc);
    if (parts > 1) {
      atomicAdd(&lc[__clz(cnt)], parts - 1);
      atomicAdd(&work[66], 1u);
    }
  }
  __syncthreads();
  if (threadIdx.x < 32 && lc[threadIdx.x]) atomicAdd(&work[threadIdx.x], lc[threadIdx.x]);
}

// Order entries of tiles of 32 nodes or more are placed class by class (most
// nodes first; in a class, block by block), a tile's entries together; the tiles
// of 2..31 nodes follow in tile order (scanned flags), so that neighbouring light
// tiles, whose padded subgrids overlap, are taken by neighbouring blocks, and the
// tiles of one node come last, in tile order as well.  tile_slot[t] = (first
// entry of tile t, -1: none; entries).  ranges, oranges (or null): the position
// ranges of the matrix-core gather and of the order entries; the nodes of a
// range from mid on start in the upper half of axis 2, by bisection of the keys,
// whose in-tile index counts the runs of four cells along axis 2 outermost.
__global__ __launch_bounds__(kB) void tile_place_k(const int* __restrict__ tile_start, long ntiles, int dense_min,
                                                   TileCut cut, bool two_lists, int rounds,
                                                   const unsigned* __restrict__ keys, unsigned vol, unsigned* work,
                                                   const unsigned* __restrict__ scan, int* items, int* items_s,
                                                   int* order, int2* tile_slot, int4* ranges, int4* oranges) {
  constexpr int NI = kClassTiles / kB;
  __shared__ unsigned lc[32], gb[32];
  __shared__ unsigned light0, single0;
  if (threadIdx.x < 32) lc[threadIdx.x] = 0;
  __syncthreads();
  unsigned lpos[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    if (i >= rounds) break;
    const long t = ((long)blockIdx.x * rounds + i) * kB + threadIdx.x;
    const int cnt = t < ntiles ? tile_start[t + 1] - tile_start[t] : 0;
    const unsigned parts = tile_parts(cnt, cut);
    lpos[i] = wave_class_add(cnt >= 32 && parts == 1, cnt > 0 ? __clz(cnt) : 0, lc);
    if (cnt >= 32 && parts > 1) lpos[i] = atomicAdd(&lc[__clz(cnt)], parts);
  }
  __syncthreads();
  // classes before class k: work[0 .. k); work[32 + k] counts the entries placed
  if (threadIdx.x < 32) {
    unsigned before = 0;
    for (int k = 0; k < 32; k++) {
      if (k < (int)threadIdx.x) before += work[k];
    }
    if (lc[threadIdx.x]) gb[threadIdx.x] = before + atomicAdd(&work[32 + threadIdx.x], lc[threadIdx.x]);
    if (threadIdx.x == 27) light0 = before;
    if (threadIdx.x == 31) single0 = before;
  }
  __syncthreads();
  auto mid_of = [&](int lo, int hi) {
    while (lo < hi) {
      const int c = (lo + hi) >> 1;
      if (keys[c] % vol < vol / 2) lo = c + 1;
      else hi = c;
    }
    return lo;
  };
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const long t = ((long)blockIdx.x * rounds + i) * kB + threadIdx.x;
    if (i >= rounds || t >= ntiles) continue;
    const int beg = tile_start[t], end = tile_start[t + 1], cnt = end - beg;
    const unsigned parts = tile_parts(cnt, cut);
    unsigned p = 0;
    if (cnt > 0) {
      p = cnt >= 32 ? gb[__clz(cnt)] + lpos[i] : cnt > 1 ? light0 + scan[t] : single0 + scan[ntiles + t];
      const int mid = vol == 512u ? mid_of(beg, end) : end;  // tiles of 8^3 cells
      for (unsigned k = 0; k < parts; k++) {
        order[p + k] = (int)t;
        if (oranges) {
          const int b = beg + (int)k * cut.part, e = parts > 1 ? min(end, b + cut.part) : end;
          oranges[p + k] = make_int4((int)t, b, min(max(mid, b), e), e);
        }
      }
      const unsigned o = scan[2 * ntiles + t], ch = tile_chunks(cnt);
      for (unsigned k = 0; k < ch; k++) {
        if (cnt >= dense_min) {
          items[2 * (o + k)] = (int)t;
          items[2 * (o + k) + 1] = (int)k;
        }
        if (two_lists) {
          const unsigned os = scan[4 * ntiles + t];
          items_s[2 * (os + k)] = (int)t;
          items_s[2 * (os + k) + 1] = (int)k;
        }
      }
      if (ranges) {
        const unsigned r = scan[3 * ntiles + t];
        const int nr = tile_ranges(cnt, cut.item), len = range_len(cnt, cut.item);
        for (int k = 0; k < nr; k++) {
          const int b = min(end, beg + k * len), e = min(end, b + len);
          ranges[r + k] = make_int4((int)t, b, min(max(mid, b), e), e);
        }
      }
    }
    tile_slot[t] = cnt > 0 ? make_int2((int)p, (int)parts) : make_int2(-1, 0);
    if (t == ntiles - 1) {
      const unsigned ch = tile_chunks(cnt);
      work[64] = scan[2 * ntiles + t] + (cnt >= dense_min ? ch : 0u);
      work[65] = two_lists ? scan[4 * ntiles + t] + ch : work[64];
      work[67] = scan[3 * ntiles + t] + (unsigned)tile_ranges(cnt, cut.item);
    }
  }
}

template <class R>
__global__ void fill_zero_k(Cplx<R>* p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = cmk<R>(R(0), R(0));
}

inline unsigned grid1d(long n, int t) { return (unsigned)((n + t - 1) / t); }

}  // namespace

int sort_passes(unsigned long long key_limit) {
  int bits = 0;
  while (bits < 32 && (1ull << bits) < key_limit) bits++;
  return (bits + 7) / 8;
}

// exclusive scans in place of `arrays` arrays of n values each, one after the other at d
static void scan_exclusive(unsigned* d, long n, int arrays, unsigned* partial, hipStream_t s) {
  const long nch = (n + kScanChunk - 1) / kScanChunk;
  if (nch <= 4) {  // one block per array in one launch
    hipLaunchKernelGGL(scan_whole_k, dim3(1, arrays), dim3(kSortT), 0, s, d, n);
    return;
  }
  const dim3 grid((unsigned)nch, arrays);
  hipLaunchKernelGGL(scan_reduce_k, grid, dim3(kSortT), 0, s, d, n, partial);
  hipLaunchKernelGGL(scan_partials_k, dim3(1, arrays), dim3(kSortT), 0, s, partial, nch);
  hipLaunchKernelGGL(scan_apply_k, grid, dim3(kSortT), 0, s, d, n, partial);
}

long sort_hist_words(long M) { return 256 * std::max(sort_blocks(M), 1L); }

template <class R, int IPB>
static void sort_passes_launch(const R* x, long M, const GridGeom& g, const TileLayout& T, SortWork& W, int passes,
                               int* perm_out, unsigned* keys_out, hipStream_t s) {
  const int nblk = (int)((M + IPB - 1) / IPB);
  hipLaunchKernelGGL((bin_keys_k<R, IPB>), dim3(nblk), dim3(kSortT), 0, s, x, M, g, T, W.keys[0], W.hist, nblk);
  // the last pass stores straight into the outputs (separate from the scratch)
  int cur = 0;
  for (int ps = 0; ps < passes; ps++) {
    const int shift = 8 * ps;
    const bool last = ps == passes - 1;
    if (ps > 0)
      hipLaunchKernelGGL((sort_hist_k<IPB>), dim3(nblk), dim3(kSortT), 0, s, W.keys[cur], M, shift, W.hist, nblk);
    hipLaunchKernelGGL(digit_scan_k, dim3(256), dim3(kSortT), 0, s, W.hist, nblk, W.total);
    hipLaunchKernelGGL((sort_scatter_k<IPB>), dim3(nblk), dim3(kSortT), 0, s, W.keys[cur],
                       ps > 0 ? W.vals[cur] : nullptr, last ? keys_out : W.keys[1 - cur],
                       last ? perm_out : W.vals[1 - cur], M, shift, W.hist, W.total, nblk);
    cur = 1 - cur;
  }
}

// Bin keys of the M nodes sorted stably (LSD radix, 8-bit digits) with the
// scratch of W: perm_out = node ids in key order, keys_out = the sorted keys.
template <class R>
static int sort_bins(const R* x, long M, const GridGeom& g, const TileLayout& T, SortWork& W, int* perm_out,
                     unsigned* keys_out, hipStream_t s) {
  const unsigned long long key_limit = (unsigned long long)T.ntiles() * (unsigned long long)T.tile_vol();
  if (key_limit > (1ull << 32)) return kUnsupported;
  const int passes = std::max(1, sort_passes(key_limit));  // keys below 2 take one pass as well
  switch (sort_ipb(M)) {
    case 1024: sort_passes_launch<R, 1024>(x, M, g, T, W, passes, perm_out, keys_out, s); break;
    case 2048: sort_passes_launch<R, 2048>(x, M, g, T, W, passes, perm_out, keys_out, s); break;
    default: sort_passes_launch<R, 4096>(x, M, g, T, W, passes, perm_out, keys_out, s); break;
  }
  return hipGetLastError() == hipSuccess ? kOk : kHipError;
}

template <class R>
int bin_nodes(const R* x, long M, const GridGeom& g, const TileLayout& T, SortWork& W, int* perm_out,
              unsigned* keys_out, hipStream_t s) {
  if (M == 0) return kOk;
  return sort_bins<R>(x, M, g, T, W, perm_out, keys_out, s);
}

// ---------------------------------------------------------------------------
// binning without allocation: the sort's scratch (two key and two id buffers,
// the digits' per-block counts and totals) lives in one file-scope device
// array per GPU, of kNoAllocMaxNodes nodes at most.  Its address is taken once
// per device with hipGetSymbolAddress (the host-side name is not a device
// address); every call on a GPU shares that GPU's array, so calls that overlap
// on one GPU race.  Every scratch word a call reads was written earlier by the
// same call (the digit counts are rebuilt per pass), so nothing needs clearing.
// ---------------------------------------------------------------------------
namespace {
constexpr long kNaBlocks = 512;  // sort_blocks() of up to kNoAllocMaxNodes nodes
static_assert(kNoAllocMaxNodes <= 2048 * kNaBlocks && (1L << 18) <= 1024 * kNaBlocks, "digit counts of every M fit");
constexpr long kNaHist = 256L * kNaBlocks;
constexpr long kNaWords = 4 * kNoAllocMaxNodes + kNaHist + 256;
}  // namespace

static __device__ __align__(256) unsigned scratch[kNaWords];

static constexpr int kNaMaxDevices = 64;
static std::mutex g_na_mu;
static unsigned* g_na_ptr[kNaMaxDevices] = {};

// Device address of `scratch` on the current device (resolved on the first call there).
static unsigned* noalloc_scratch() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kNaMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_na_mu);
  if (!g_na_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_na_ptr[dev] = static_cast<unsigned*>(ptr);
  }
  return g_na_ptr[dev];
}

size_t noalloc_scratch_bytes() { return sizeof(unsigned) * (size_t)kNaWords; }

template <class R>
int bin_nodes_noalloc(const R* x, long M, const GridGeom& g, const TileLayout& T, int* perm_out, unsigned* keys_out,
                      hipStream_t s) {
  if (M < 0 || M > kNoAllocMaxNodes) return kUnsupported;
  if (M == 0) return kOk;
  unsigned* base = noalloc_scratch();
  if (!base) return kHipError;
  SortWork W;
  W.keys[0] = base;
  W.keys[1] = base + kNoAllocMaxNodes;
  W.vals[0] = reinterpret_cast<int*>(base + 2 * kNoAllocMaxNodes);
  W.vals[1] = reinterpret_cast<int*>(base + 3 * kNoAllocMaxNodes);
  W.hist = base + 4 * kNoAllocMaxNodes;
  W.total = W.hist + kNaHist;
  return sort_bins<R>(x, M, g, T, W, perm_out, keys_out, s);
}

int cols_pad(int m, bool is_double, const int* ts) {
  if (m < 2 || m > 8 || (is_double && m > 6)) return 0;
  const int TS = std_tile(m, is_double);
  if (ts[0] != TS || ts[1] != TS || ts[2] != TS) return 0;
  return TS + 2 * m;
}

// Offsets of the nodes of every tile, per axis, as bit masks: the in-tile cell
// index of a sorted key (the layout of bin_keys_k: runs of q = min(TS2, 4)
// cells along axis 2 outermost, then axis 0, axis 1 and the cell within the
// run) is decoded and OR-ed into box[tile] (bits 8 t + l for offset l on axis
// t; tile sizes of at most 8).
// The keys are sorted, so the lanes of a wave that share a tile are
// consecutive: a segmented OR scan over each such run leaves the run's OR in
// its last lane, which makes the one atomic for that tile (instead of one per
// lane on the same word).
__global__ __launch_bounds__(kB) void tile_box_k(const unsigned* __restrict__ keys, long M, TileLayout T,
                                                 unsigned* box) {
  const long i = (long)blockIdx.x * kB + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool live = i < M;
  const unsigned vol = (unsigned)(T.ts[0] * T.ts[1] * T.ts[2]);
  const unsigned key = live ? keys[i] : 0u, in = key % vol;
  const unsigned tile = live ? key / vol : 0xFFFFFFFFu;  // no tile id reaches the sentinel
  const unsigned q = T.ts[2] < 4 ? (unsigned)T.ts[2] : 4u;
  const unsigned r = in % q, rest = in / q;  // rest = (l2 / q) * TS0 * TS1 + l0 * TS1 + l1
  const unsigned l1 = rest % (unsigned)T.ts[1], l0 = (rest / (unsigned)T.ts[1]) % (unsigned)T.ts[0];
  const unsigned l2 = (rest / (unsigned)(T.ts[0] * T.ts[1])) * q + r;
  unsigned m = live ? (1u << l0) | (1u << (8 + l1)) | (1u << (16 + l2)) : 0u;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned o = (unsigned)__shfl_up((int)m, d);
    const unsigned to = (unsigned)__shfl_up((int)tile, d);
    if (lane >= d && to == tile) m |= o;
  }
  const unsigned tn = (unsigned)__shfl_down((int)tile, 1);
  if (live && (lane == 63 || tn != tile)) atomicOr(box + tile, m);
}

// box_ord[p] = box_tile[order[p]] for the n order entries (n: work's class
// counts, on the device): the masks by position in the tile order
__global__ __launch_bounds__(kB) void box_order_k(const int* __restrict__ order, const unsigned* __restrict__ work,
                                                  const unsigned* __restrict__ box_tile, unsigned* box_ord) {
  const int p = blockIdx.x * kB + threadIdx.x;
  int n = 0;
  for (int k = 0; k < 32; k++) n += (int)work[k];
  if (p < n) box_ord[p] = box_tile[order[p]];
}

int build_tile_lists(const unsigned* keys, long M, const TileLayout& T, int dense_min, const TileCut& cut, bool boxes,
                     TileLists& L, TileCounts* out, hipStream_t s) {
  const long nt = T.ntiles();
  const bool two = dense_min > 1;
  hipLaunchKernelGGL(tile_bounds_k, dim3(grid1d(std::max(nt + 1, (long)kTileWork), kB)), dim3(kB), 0, s, keys, M,
                     (unsigned)T.tile_vol(), nt, L.tile_start, L.work, L.box_tile);
  const int rounds = class_rounds(nt);
  hipLaunchKernelGGL(tile_class_k, dim3(grid1d(nt, rounds * kB)), dim3(kB), 0, s, L.tile_start, nt, dense_min,
                     cut, two, rounds, L.work, L.scan, L.dense, L.dense_s);
  scan_exclusive(L.scan, nt, two ? 5 : 4, L.partial, s);
  hipLaunchKernelGGL(tile_place_k, dim3(grid1d(nt, rounds * kB)), dim3(kB), 0, s, L.tile_start, nt, dense_min,
                     cut, two, rounds, keys, (unsigned)T.tile_vol(), L.work, L.scan, L.items, L.items_s, L.order,
                     L.tile_slot, L.ranges, L.oranges);
  if (boxes && M > 0) {
    if (T.ts[0] > 8 || T.ts[1] > 8 || T.ts[2] > 8) return kUnsupported;
    hipLaunchKernelGGL(tile_box_k, dim3(grid1d(M, kB)), dim3(kB), 0, s, keys, M, T, L.box_tile);
    hipLaunchKernelGGL(box_order_k, dim3(grid1d(L.order_cap, kB)), dim3(kB), 0, s, L.order, L.work, L.box_tile,
                       L.box_ord);
  }
  unsigned w[kTileWork] = {0};
  if (hipMemcpyAsync(w, L.work, sizeof(w), hipMemcpyDeviceToHost, s) != hipSuccess) return kHipError;
  if (hipStreamSynchronize(s) != hipSuccess) return kHipError;
  out->n_order = out->n_heavy = 0;
  for (int k = 0; k < 32; k++) {
    out->n_order += (int)w[k];
    if (k <= 26) out->n_heavy += (int)w[k];
  }
  out->n_single = (int)w[31];
  out->n_items = (int)w[64];
  out->n_items_s = (int)w[65];
  out->n_cut = (int)w[66];
  out->n_ranges = (int)w[67];
  return kOk;
}

template <class R>
int gather(const BArgs<R>& A, int mode, hipStream_t s) {
  if (A.M == 0) return kOk;
  if (A.g.m < kMinPlanM || A.g.m > kMaxPlanM) return kUnsupported;
  int st = kUnsupported;
  switch (mode) {
    case B_F: st = gather_mm<R, B_F>(A, s); break;
    case B_GRAD: st = gather_mm<R, B_GRAD>(A, s); break;
    case B_FGRAD: st = gather_mm<R, B_FGRAD>(A, s); break;
    case B_VJP: st = gather_mm<R, B_VJP>(A, s); break;
    default: break;
  }
  if (st != kUnsupported) return st;  // kUnsupported: nothing was launched
  switch (mode) {
    case B_F: return b_launch<R, 0, B_F>(A, s);
    case B_GRAD: return b_launch<R, 0, B_GRAD>(A, s);
    case B_FGRAD: return b_launch<R, 0, B_FGRAD>(A, s);
    case B_VJP: return b_launch<R, 0, B_VJP>(A, s);
    default: return kUnsupported;
  }
}

template <class R>
int scatter(const BArgs<R>& A, int mode, hipStream_t s) {
  if (A.M == 0) return kOk;
  if (A.g.m < kMinPlanM || A.g.m > kMaxPlanM) return kUnsupported;
  int mst = kUnsupported;
  switch (mode) {
    case B_F: mst = scatter_mm<R, B_F>(A, s); break;
    case B_GRAD: mst = scatter_mm<R, B_GRAD>(A, s); break;
    case B_FGRAD: mst = scatter_mm<R, B_FGRAD>(A, s); break;
    default: break;
  }
  if (mst != kUnsupported) return mst;  // kUnsupported: nothing was launched
  if (A.slots) {  // column path: writes every grid cell through the fold
    int st = kUnsupported;
    switch (mode) {
      case B_F: st = cols_launch<R, B_F>(A, s); break;
      case B_GRAD: st = cols_launch<R, B_GRAD>(A, s); break;
      case B_FGRAD: st = cols_launch<R, B_FGRAD>(A, s); break;
      default: break;
    }
    if (st != kUnsupported) return st;  // kUnsupported: nothing was launched, take the LDS-atomic path
  }
  // LDS-atomic path: accumulates into the cleared grid
  const long ncell = (long)A.g.n[0] * A.g.n[1] * A.g.n[2];
  const long ntot = A.c2r ? (ncell + 1) / 2 : ncell;  // complex elements of the grid's storage (c2r: real grid)
  hipLaunchKernelGGL((fill_zero_k<R>), dim3(grid1d(ntot, 256)), dim3(256), 0, s, A.grid, (size_t)ntot);
  switch (mode) {
    case B_F: return b_launch<R, 1, B_F>(A, s);
    case B_GRAD: return b_launch<R, 1, B_GRAD>(A, s);
    case B_FGRAD: {  // both contributions add into the same grid
      const int st = b_launch<R, 1, B_F>(A, s);
      return st != kOk ? st : b_launch<R, 1, B_GRAD>(A, s);
    }
    default: return kUnsupported;
  }
}

template <class R>
int fill_zero(Cplx<R>* p, size_t n, hipStream_t s) {
  if (n == 0) return kOk;
  hipLaunchKernelGGL((fill_zero_k<R>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
  return hipGetLastError() == hipSuccess ? kOk : kHipError;
}

template int bin_nodes<float>(const float*, long, const GridGeom&, const TileLayout&, SortWork&, int*, unsigned*,
                              hipStream_t);
template int bin_nodes<double>(const double*, long, const GridGeom&, const TileLayout&, SortWork&, int*, unsigned*,
                               hipStream_t);
template int bin_nodes_noalloc<float>(const float*, long, const GridGeom&, const TileLayout&, int*, unsigned*,
                                      hipStream_t);
template int bin_nodes_noalloc<double>(const double*, long, const GridGeom&, const TileLayout&, int*, unsigned*,
                                       hipStream_t);
template int gather<float>(const BArgs<float>&, int, hipStream_t);
template int gather<double>(const BArgs<double>&, int, hipStream_t);
template int scatter<float>(const BArgs<float>&, int, hipStream_t);
template int scatter<double>(const BArgs<double>&, int, hipStream_t);
template int fill_zero<float>(Cplx<float>*, size_t, hipStream_t);
template int fill_zero<double>(Cplx<double>*, size_t, hipStream_t);

}  // namespace pnfft_amd
