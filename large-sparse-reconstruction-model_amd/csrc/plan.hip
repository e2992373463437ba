// Planning kernels: batched exclusive scans, query-tile plans, reverse (CSR)
// maps with a deterministic per-segment sort, key-chunk items, metadata
// validation and per-token block ids.
//
// The reverse map replaces the reference's _count_queries_kernel /
// _scatter_queries_kernel / host-looped segmented sort
// (sparse/ops/triton_native_sparse_attention_impl_kvcentric.py:494-684),
// all on the device and without host synchronisation: for rows that are
// queries, stable counting passes over chunks of them; for rows that are
// run tiles, count -> scan -> atomic scatter -> per-segment sort.
#include <algorithm>

#include "plan.h"

namespace lsrm {

constexpr int SCAN_T = 256;
constexpr int SCAN_PER = 16;
constexpr int SCAN_CHUNK = SCAN_T * SCAN_PER;

__device__ inline int wave_sum(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Exclusive scan of one value per thread over a 256-thread block; returns the
// exclusive prefix and writes the block total to *total.
template <class T>
__device__ inline T block_excl_scan(T v, T* total) {
  __shared__ T s_w[SCAN_T / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  T x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    T y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_w[w] = x;
  __syncthreads();
  T off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < SCAN_T / 64; ++i) {
    if (i < w) off += s_w[i];
    tot += s_w[i];
  }
  __syncthreads();
  *total = tot;
  return off + x - v;
}

// The type of a scan's values: int, or a pair of counts packed in 64 bits.
template <bool BY_WIDTH>
struct SplitF;
template <class F>
struct ScanValue {
  using type = int32_t;
};
template <>
struct ScanValue<SplitF<true>> {
  using type = int64_t;
};
template <class F>
using scan_t = typename ScanValue<F>::type;

template <class F>
__global__ __launch_bounds__(SCAN_T) void scan_reduce(F f, int64_t n,
                                                      scan_t<F>* sums,
                                                      int nchunks) {
  const int seg = blockIdx.y;
  const int64_t base = (int64_t)blockIdx.x * SCAN_CHUNK + threadIdx.x * SCAN_PER;
  const int64_t lim = f.limit(seg, n);
  scan_t<F> s = 0;
  for (int i = 0; i < SCAN_PER; ++i) {
    const int64_t idx = base + i;
    if (idx < lim) s += f(seg, idx);
  }
  scan_t<F> tot;
  block_excl_scan(s, &tot);
  if (threadIdx.x == 0) sums[(int64_t)seg * nchunks + blockIdx.x] = tot;
}

// In-place exclusive scan of each segment's chunk sums; totals[seg] = total.
template <class T>
__global__ __launch_bounds__(SCAN_T) void scan_chunks(T* sums, int nchunks, T* totals) {
  const int seg = blockIdx.x;
  T* p = sums + (int64_t)seg * nchunks;
  T carry = 0;
  for (int base = 0; base < nchunks; base += SCAN_T) {
    const int i = base + threadIdx.x;
    const T v = i < nchunks ? p[i] : T(0);
    T tot;
    const T ex = block_excl_scan(v, &tot);
    if (i < nchunks) p[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) totals[seg] = carry;
}

template <class F, class W>
__global__ __launch_bounds__(SCAN_T) void scan_apply(F f, W w, int64_t n,
                                                     const scan_t<F>* sums,
                                                     int nchunks) {
  const int seg = blockIdx.y;
  const int64_t base = (int64_t)blockIdx.x * SCAN_CHUNK + threadIdx.x * SCAN_PER;
  const int64_t lim = f.limit(seg, n);
  scan_t<F> v[SCAN_PER];
  scan_t<F> s = 0;
#pragma unroll
  for (int i = 0; i < SCAN_PER; ++i) {
    const int64_t idx = base + i;
    v[i] = idx < lim ? f(seg, idx) : scan_t<F>(0);
    s += v[i];
  }
  scan_t<F> tot;
  scan_t<F> ex = block_excl_scan(s, &tot) + sums[(int64_t)seg * nchunks + blockIdx.x];
#pragma unroll
  for (int i = 0; i < SCAN_PER; ++i) {
    const int64_t idx = base + i;
    if (idx < lim) w(seg, idx, ex, v[i], lim);
    ex += v[i];
  }
}

// Runs scan_reduce / scan_chunks / scan_apply over `nseg` segments of at
// most n elements; totals[seg] receives each segment's sum.
template <class F, class W>
int run_scan(F f, W w, int64_t n, int nseg, scan_t<F>* chunk_sums,
             scan_t<F>* totals, hipStream_t st) {
  if (n <= 0 || nseg <= 0) return LSRM_OK;
  const int nchunks = ceil_div(n, SCAN_CHUNK);
  dim3 grid(nchunks, nseg);
  hipLaunchKernelGGL((scan_reduce<F>), grid, dim3(SCAN_T), 0, st, f, n,
                     chunk_sums, nchunks);
  hipLaunchKernelGGL(scan_chunks<scan_t<F>>, dim3(nseg), dim3(SCAN_T), 0, st, chunk_sums,
                     nchunks, totals);
  hipLaunchKernelGGL((scan_apply<F, W>), grid, dim3(SCAN_T), 0, st, f, w, n,
                     chunk_sums, nchunks);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

inline int64_t scan_sums_size(int64_t n, int64_t nseg) {
  return (int64_t)ceil_div(n > 0 ? n : 1, SCAN_CHUNK) * nseg;
}

// ------------------------------------------------------------- utilities --

__global__ void zero_i32_kernel(int32_t* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}

int launch_zero_i32(int32_t* p, int64_t n, hipStream_t st) {
  if (n <= 0) return LSRM_OK;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(zero_i32_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                     p, n);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

// Number of valid (batch-local id in [0, nbb)) entries in a selection row is
// not needed; rows compare by their sequence of normalised entries.
__device__ inline int norm_entry(int v, int nbb) {
  return (v >= 0 && v < nbb) ? v : -1;
}

// --------------------------------------------------------------- tiles --

// brk[h, i] = 1 where a new run of identical (normalised) rows starts.
__global__ __launch_bounds__(256) void breaks_kernel(
    const int32_t* __restrict__ topk, int64_t nq, int k,
    const int32_t* __restrict__ cu_q, int64_t batch,
    const int32_t* __restrict__ cu_sb, uint8_t* __restrict__ brk) {
  const int h = blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nq) return;
  int b, bs, nbb;
  bool start;
  query_batch(cu_q, batch, cu_sb, i, &b, &bs, &nbb, &start);
  bool br = (i == 0) || start;
  if (!br) {
    const int32_t* r1 = topk + ((int64_t)h * nq + i) * k;
    const int32_t* r0 = r1 - k;
    for (int j = 0; j < k; ++j) {
      if (norm_entry(r1[j], nbb) != norm_entry(r0[j], nbb)) {
        br = true;
        break;
      }
    }
  }
  brk[(int64_t)h * nq + i] = br ? 1 : 0;
}

// Same as breaks_kernel for k % 4 == 0 and 16-byte-aligned rows: each
// thread reads its row with 16-byte loads (a wave reads 64 consecutive rows
// contiguously) and takes the previous row from the neighbouring lane.
__global__ __launch_bounds__(256) void breaks_vec_kernel(
    const int32_t* __restrict__ topk, int64_t nq, int k,
    const int32_t* __restrict__ cu_q, int64_t batch,
    const int32_t* __restrict__ cu_sb, uint8_t* __restrict__ brk) {
  const int h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = i < nq;
  int b = 0, bs = 0, nbb = 0;
  bool start = true;
  if (live) query_batch(cu_q, batch, cu_sb, i, &b, &bs, &nbb, &start);
  const int64_t ii = live ? i : nq - 1;
  const u32x4* r1 = reinterpret_cast<const u32x4*>(topk + ((int64_t)h * nq + ii) * k);
  const u32x4* r0 = reinterpret_cast<const u32x4*>(
      topk + ((int64_t)h * nq + (ii > 0 ? ii - 1 : 0)) * k);
  bool diff = false;
  for (int c = 0; c < k / 4; ++c) {
    const u32x4 cur = r1[c];
    u32x4 prev;
#pragma unroll
    for (int e = 0; e < 4; ++e) prev[e] = (uint32_t)__shfl_up((int)cur[e], 1);
    if (lane == 0) prev = r0[c];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      diff |= norm_entry((int)cur[e], nbb) != norm_entry((int)prev[e], nbb);
  }
  if (live) brk[(int64_t)h * nq + i] = (i == 0 || start || diff) ? 1 : 0;
}

// Row flags from lane flags where P neighbouring lanes hold one row: bit r * P
// is set when any bit of lanes r * P .. r * P + P - 1 is (scalar work).
template <int P>
constexpr uint64_t ROW_LSB = ROW_LSB<2 * P> * (1ull | (1ull << P));
template <>
constexpr uint64_t ROW_LSB<64> = 1ull;
template <int P>
__device__ inline uint64_t row_or(uint64_t m) {
#pragma unroll
  for (int o = 1; o < P; o <<= 1) m |= m >> o;
  return m & ROW_LSB<P>;
}

// Same for rows of P 16-byte pieces (k = 4 P), P a power of two <= 64: lane
// (row i, piece p) holds piece p of row i and of row i - 1, so a wave reads
// 64 / P whole rows as one contiguous run per load (the second read of a line
// is served by the cache), and the P lanes of a row are combined in scalar
// registers.  A wave covers BRK_G such groups with all their loads in flight,
// and looks its batch element up once when its rows lie inside one (else row
// by row).
constexpr int BRK_G = 8;
template <int P>
__global__ __launch_bounds__(256) void breaks_rows_kernel(
    const int32_t* __restrict__ topk, int64_t nq, const int32_t* __restrict__ cu_q,
    int64_t batch, const int32_t* __restrict__ cu_sb, uint8_t* __restrict__ brk) {
  static_assert(P >= 1 && P <= 64 && (P & (P - 1)) == 0, "rows must tile a wave");
  constexpr int RPW = 64 / P;  // rows per group
  const int h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int64_t i0 =
      ((int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6)) * (RPW * BRK_G);
  if (i0 >= nq) return;  // whole waves
  const int p = lane % P, rl = lane / P;
  const u32x4* rows = reinterpret_cast<const u32x4*>(topk + (int64_t)h * nq * (4 * P));
  u32x4 cur[BRK_G], prev[BRK_G];
#pragma unroll
  for (int g = 0; g < BRK_G; ++g) {
    const int64_t i = i0 + g * RPW + rl < nq ? i0 + g * RPW + rl : nq - 1;
    cur[g] = rows[i * P + p];
    prev[g] = rows[(i > 0 ? i - 1 : 0) * P + p];
  }
  const int64_t i_last = i0 + RPW * BRK_G - 1 < nq ? i0 + RPW * BRK_G - 1 : nq - 1;
  int b0 = 0, bs0 = 0, nbb0 = 0;
  bool st0 = true;
  query_batch(cu_q, batch, cu_sb, i0, &b0, &bs0, &nbb0, &st0);
  const int64_t qs0 = b0 >= 0 ? cu_q[b0] : 0;
  const bool one = b0 >= 0 && i_last < (int64_t)cu_q[b0 + 1];
#pragma unroll
  for (int g = 0; g < BRK_G; ++g) {
    const int64_t i = i0 + g * RPW + rl;
    int nbb = nbb0;
    bool start = i == qs0;
    if (!one && i < nq) {
      int b, bs;
      query_batch(cu_q, batch, cu_sb, i, &b, &bs, &nbb, &start);
    }
    bool diff = i == 0 || start;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      diff |= norm_entry((int)cur[g][e], nbb) != norm_entry((int)prev[g][e], nbb);
    const uint64_t brks = row_or<P>(__ballot(diff));
    if (i < nq && p == 0) brk[(int64_t)h * nq + i] = (uint8_t)((brks >> lane) & 1);
  }
}

struct BrkF {
  const uint8_t* brk;
  int64_t nq;
  __device__ int64_t limit(int, int64_t n) const { return n; }
  __device__ int operator()(int h, int64_t i) const {
    return brk[(int64_t)h * nq + i];
  }
};
struct RunStartW {
  int32_t* run_start;  // [hkv, nq + 1]
  int64_t nq;
  __device__ void operator()(int h, int64_t i, int ex, int v,
                             int64_t lim) const {
    int32_t* rs = run_start + (int64_t)h * (nq + 1);
    if (v) rs[ex] = (int32_t)i;
    if (i == lim - 1) rs[ex + v] = (int32_t)nq;
  }
};

struct RunTilesF {
  const int32_t* run_start;
  const int32_t* n_runs;  // [hkv]
  int64_t nq;
  int tq;
  __device__ int64_t limit(int h, int64_t) const { return n_runs[h]; }
  __device__ int operator()(int h, int64_t r) const {
    const int32_t* rs = run_start + (int64_t)h * (nq + 1);
    const int len = rs[r + 1] - rs[r];
    return (len + tq - 1) / tq;
  }
};
struct EmitTilesW {
  const int32_t* run_start;
  int2* tiles;
  int64_t nq;
  int tq;
  __device__ void operator()(int h, int64_t r, int ex, int v, int64_t) const {
    const int32_t* rs = run_start + (int64_t)h * (nq + 1);
    const int s = rs[r];
    const int len = rs[r + 1] - s;
    int2* out = tiles + (int64_t)h * nq + ex;
    for (int t = 0; t < v; ++t) {
      const int q0 = s + t * tq;
      const int rem = len - t * tq;
      out[t] = make_int2(q0, rem < tq ? rem : tq);
    }
  }
};


// --------------------------------------------------------- union tiles --
// Consecutive short run tiles (fewer than tq / 4 queries) of one batch
// element whose first queries fall in the same window of 3 tq / 4 queries
// form a group of at most tq - 1 queries; two neighbours of which one has 8
// or more queries join only when their rows share at least half of the
// first one's valid ids.  Per-token rows change every few queries and share
// most blocks with their neighbours; a block-row selection's short runs are
// whole small blocks whose neighbours select other blocks (config 5: 0-6 of
// 32 shared), where the union only adds masked keys to a tile that already
// runs as a whole tile of its own.  Groups of two or more run tiles
// become grouped tiles (TilePlan::gtiles): the forward runs them over the
// union of their queries' selections with a per-query mask, or run by run
// when that is cheaper.  Every other run tile is kept as it is.
constexpr int GROUP_FEW_Q = 8;

// gbrk[h, t] = 1 where run tile t starts a new group.  One thread per tile
// decides the plain cases; the tiles that need the shared-ids count (at most
// a few hundred per head) are taken one at a time by their whole wave: lane
// j holds id j of both rows (one load round for rows of <= 64 ids) and the
// other row's ids are broadcast with readlane.
__global__ __launch_bounds__(256) void group_breaks_kernel(
    const int2* __restrict__ tiles, const int32_t* __restrict__ count,
    const int32_t* __restrict__ cu_q, int64_t batch, const int32_t* __restrict__ topk,
    int64_t nq, int k, int short_q, int window_q, uint8_t* __restrict__ gbrk) {
  const int h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t cnt = count[h];
  int brk = 1;
  bool check = false;
  int qa = 0, qb = 0;
  if (t > 0 && t < cnt) {
    const int2 a = tiles[(int64_t)h * nq + t - 1], b = tiles[(int64_t)h * nq + t];
    if (a.y < short_q && b.y < short_q && a.x / window_q == b.x / window_q &&
        batch_of(cu_q, batch, a.x) == batch_of(cu_q, batch, b.x)) {
      if (a.y < GROUP_FEW_Q && b.y < GROUP_FEW_Q) {
        brk = 0;
      } else {
        // a run's rows are identical: its first query's row stands for it
        check = true;
        qa = a.x;
        qb = b.x;
      }
    }
  }
  uint64_t pend = __ballot(check);
  while (pend) {
    const int l = __builtin_ctzll(pend);
    pend &= pend - 1;
    const int64_t ra = ((int64_t)h * nq + __builtin_amdgcn_readlane(qa, l)) * k;
    const int64_t rb = ((int64_t)h * nq + __builtin_amdgcn_readlane(qb, l)) * k;
    int valid = 0, shared = 0;
    for (int c0 = 0; c0 < k; c0 += 64) {
      const int x = c0 + lane < k ? topk[ra + c0 + lane] : -1;
      bool hit = false;
      for (int d0 = 0; d0 < k; d0 += 64) {
        const int y = d0 + lane < k ? topk[rb + d0 + lane] : -1;
        const int m_end = k - d0 < 64 ? k - d0 : 64;
        for (int m = 0; m < m_end; ++m) hit |= x == __builtin_amdgcn_readlane(y, m);
      }
      valid += __popcll(__ballot(x >= 0));
      shared += __popcll(__ballot(x >= 0 && hit));
    }
    if (lane == l) brk = 2 * shared >= valid ? 0 : 1;
  }
  if (t < cnt) gbrk[(int64_t)h * nq + t] = (uint8_t)brk;
}

struct GroupF {
  const uint8_t* gbrk;
  const int32_t* count;
  int64_t nq;
  __device__ int64_t limit(int h, int64_t) const { return count[h]; }
  __device__ int operator()(int h, int64_t t) const { return gbrk[(int64_t)h * nq + t]; }
};
struct GroupW {
  int32_t* gstart;  // [hkv, nq + 1]
  int64_t nq;
  __device__ void operator()(int h, int64_t t, int ex, int v, int64_t lim) const {
    int32_t* gs = gstart + (int64_t)h * (nq + 1);
    if (v) gs[ex] = (int32_t)t;
    if (t == lim - 1) gs[ex + v] = (int32_t)lim;
  }
};
// Second pass over the groups: grouped (>= 2 run tiles) or kept, and for a list
// by width whether a kept tile is narrow; the two counts are scanned together,
// packed in 64 bits.
template <bool BY_WIDTH>
struct SplitF {
  const int2* run_tiles;
  const int32_t* gstart;
  const int32_t* n_groups;
  int64_t nq;
  int narrow_q;
  __device__ int64_t limit(int h, int64_t) const { return n_groups[h]; }
  __device__ scan_t<SplitF> operator()(int h, int64_t s) const {
    const int32_t* gs = gstart + (int64_t)h * (nq + 1);
    if (gs[s + 1] - gs[s] > 1) return 1;
    if constexpr (BY_WIDTH)
      return run_tiles[(int64_t)h * nq + gs[s]].y <= narrow_q ? int64_t{1} << 32 : 0;
    else
      return 0;
  }
};
template <bool BY_WIDTH>
struct SplitW {
  using T = scan_t<SplitF<BY_WIDTH>>;
  const int2* run_tiles;
  const int32_t* gstart;
  int64_t nq;
  int2* tiles;
  int2* gtiles;
  int2* by_width;
  __device__ void operator()(int h, int64_t s, T ex, T v, int64_t) const {
    const int32_t* gs = gstart + (int64_t)h * (nq + 1);
    const int t0 = gs[s], t1 = gs[s + 1];
    const int64_t g = (int32_t)ex;  // grouped tiles before
    const int64_t at = (int64_t)h * nq;
    const int2 first = run_tiles[at + t0];
    if (v == 1) {
      const int2 last = run_tiles[at + t1 - 1];
      gtiles[at + g] = make_int2(first.x, last.x + last.y - first.x);
      return;
    }
    tiles[at + (s - g)] = first;
    if constexpr (BY_WIDTH) {
      const int64_t nar = ex >> 32;  // narrow tiles before
      by_width[at + (v ? nq - 1 - nar : s - g - nar)] = first;
    }
  }
};

// The lists' counts per head from the groups and the split's totals, and the
// heads' offsets in every list (lane i takes list i: run tiles, grouped, wide,
// narrow).  T: the split's scan type (64 bits: with narrow tiles counted).
template <class T>
__global__ void plan_offsets_kernel(const int32_t* n_groups, const T* split, TilePlan plan,
                                    int hkv) {
  if (blockIdx.x != 0) return;
  if (threadIdx.x < 4) {
    const int i = threadIdx.x;
    int32_t* off = i == 0 ? plan.head_off
                          : (i == 1 ? plan.ghead_off : (i == 2 ? plan.wide_off : plan.narrow_off));
    int acc = 0;
    off[0] = 0;
    for (int h = 0; h < hkv; ++h) {
      int c = 0;
      if (n_groups) {
        const int g = (int32_t)split[h], kept = n_groups[h] - g;
        const int nar = sizeof(T) == 8 ? (int)((int64_t)split[h] >> 32) : 0;
        c = i == 0 ? kept : (i == 1 ? g : (i == 2 ? kept - nar : nar));
      }
      if (i == 0) plan.tile_count[h] = c;
      if (i == 1) plan.gtile_count[h] = c;
      acc += c;
      off[h + 1] = acc;
    }
  }
  int32_t* counter = plan.counter;
  if (threadIdx.x == 0) {
    for (int i = 0; i < PLAN_BWD_SLOT; ++i) counter[i] = 0;
    counter[PLAN_BWD_SLOT] = 0;  // set again by mark_backward_plan
    counter[PLAN_KC_SLOT] = 0;   // set again by the key-centric part
    counter[BY_WIDTH_SLOT] = sizeof(T) == 8 ? 1 : 0;
  }
}

__global__ void mark_backward_plan_kernel(TilePlan plan, int hkv, const int32_t* totals) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    int listed = totals ? 0 : plan.ghead_off[hkv];
    for (int h = 0; totals && h < hkv; ++h) listed |= totals[h] > 0 ? 1 : 0;
    plan.counter[PLAN_QMAP_SLOT] = listed;
    plan.counter[PLAN_BWD_SLOT] = PLAN_BWD_MAGIC;
  }
}

int mark_backward_plan(const TilePlan& plan, int64_t hkv, const int32_t* totals, hipStream_t st) {
  hipLaunchKernelGGL(mark_backward_plan_kernel, dim3(1), dim3(64), 0, st, plan, (int)hkv, totals);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

// The last scan and the lists' offsets: the grouped tiles go to their list, and
// with BY_WIDTH the others also to the one by width.
template <bool BY_WIDTH>
int split_tiles(const int2* run_tiles, const int32_t* gstart, const int32_t* n_groups, int64_t hkv,
                int64_t nq, int narrow_q, int64_t* sums, int64_t* split, const TilePlan& plan,
                hipStream_t st) {
  using T = scan_t<SplitF<BY_WIDTH>>;
  T* totals = reinterpret_cast<T*>(split);
  if (nq > 0) {
    const int rc =
        run_scan(SplitF<BY_WIDTH>{run_tiles, gstart, n_groups, nq, narrow_q},
                 SplitW<BY_WIDTH>{run_tiles, gstart, nq, plan.tiles, plan.gtiles, plan.by_width},
                 nq, (int)hkv, reinterpret_cast<T*>(sums), totals, st);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(plan_offsets_kernel<T>, dim3(1), dim3(64), 0, st,
                     nq > 0 ? n_groups : nullptr, totals, plan, (int)hkv);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

int build_tile_plan(const int32_t* topk, int64_t hkv, int64_t nq,
                    int64_t topk_n, const int32_t* cu_q, int64_t batch,
                    const int32_t* cu_sb, int tq, int narrow_q, Carver& ws, TilePlan& plan,
                    hipStream_t st) {
  uint8_t* brk = ws.take<uint8_t>((size_t)(hkv * nq));
  int32_t* run_start = ws.take<int32_t>((size_t)(hkv * (nq + 1)));
  int32_t* n_runs = ws.take<int32_t>((size_t)hkv);
  int64_t* split_sums = ws.take<int64_t>((size_t)scan_sums_size(nq, hkv));
  int32_t* sums = reinterpret_cast<int32_t*>(split_sums);  // the 32-bit scans' before
  const size_t n_tiles = (size_t)(hkv * (nq > 0 ? nq : 1));
  plan.tiles = ws.take<int2>(n_tiles);
  plan.tile_count = ws.take<int32_t>((size_t)hkv);
  plan.head_off = ws.take<int32_t>((size_t)(hkv + 1));
  plan.counter = ws.take<int32_t>(64);
  plan.gtile_count = ws.take<int32_t>((size_t)hkv);
  plan.ghead_off = ws.take<int32_t>((size_t)(hkv + 1));
  plan.wide_off = ws.take<int32_t>((size_t)(hkv + 1));
  plan.narrow_off = ws.take<int32_t>((size_t)(hkv + 1));
  plan.gtiles = ws.take<int2>(n_tiles);
  plan.by_width = ws.take<int2>(n_tiles);
  int2* run_tiles = ws.take<int2>(n_tiles);
  int32_t* run_count = ws.take<int32_t>((size_t)hkv);
  int32_t* gstart = ws.take<int32_t>((size_t)(hkv * (nq + 1)));
  int32_t* n_groups = ws.take<int32_t>((size_t)hkv);
  int64_t* split = ws.take<int64_t>((size_t)hkv);
  if (!ws.base || ws.dry) return LSRM_OK;
  if (!ws.ok()) return LSRM_ERR_WORKSPACE;

  if (nq > 0) {
    dim3 grid(ceil_div(nq, 256), (unsigned)hkv);
    const int64_t pieces = topk_n / 4;
    const bool vec = topk_n % 4 == 0 && ((uintptr_t)topk % 16) == 0;
    // Rows of 4 or more pieces: one row per lane would read 64 rows' worth
    // of lines per load and lose them between the row's loads (config 5's
    // 128-byte rows fetched 6.9x their bytes); with eight row groups per wave
    // the piece-per-lane form also beats it on 64-byte rows (top-16: 42 -> 39
    // us on average over bench.py's plans).  Shorter rows keep one per lane.
    if (vec && pieces >= 4 && pieces <= 64 && (pieces & (pieces - 1)) == 0) {
      // one wave per BRK_G groups of 64 / pieces rows, four waves per block
      const dim3 grow(ceil_div(ceil_div(nq, (64 / pieces) * BRK_G), 4), (unsigned)hkv);
#define LSRM_BRK(P)                                                                  \
  case P:                                                                            \
    hipLaunchKernelGGL(breaks_rows_kernel<P>, grow, dim3(256), 0, st, topk, nq, cu_q, \
                       batch, cu_sb, brk);                                           \
    break;
      switch (pieces) {
        LSRM_BRK(4) LSRM_BRK(8) LSRM_BRK(16) LSRM_BRK(32) LSRM_BRK(64)
      }
#undef LSRM_BRK
    } else if (vec)
      hipLaunchKernelGGL(breaks_vec_kernel, grid, dim3(256), 0, st, topk, nq,
                         (int)topk_n, cu_q, batch, cu_sb, brk);
    else
      hipLaunchKernelGGL(breaks_kernel, grid, dim3(256), 0, st, topk, nq,
                         (int)topk_n, cu_q, batch, cu_sb, brk);
    LSRM_CHECK_LAUNCH();
    int rc = run_scan(BrkF{brk, nq}, RunStartW{run_start, nq}, nq, (int)hkv,
                      sums, n_runs, st);
    if (rc) return rc;
    rc = run_scan(RunTilesF{run_start, n_runs, nq, tq},
                  EmitTilesW{run_start, run_tiles, nq, tq}, nq, (int)hkv, sums,
                  run_count, st);
    if (rc) return rc;
    const int short_q = tq / 4 > 1 ? tq / 4 : 1;
    const int window_q = (3 * tq) / 4 > 1 ? (3 * tq) / 4 : 1;
    // brk is free again: it takes the group starts
    hipLaunchKernelGGL(group_breaks_kernel, grid, dim3(256), 0, st, run_tiles, run_count,
                       cu_q, batch, topk, nq, (int)topk_n, short_q, window_q, brk);
    LSRM_CHECK_LAUNCH();
    rc = run_scan(GroupF{brk, run_count, nq}, GroupW{gstart, nq}, nq, (int)hkv, sums, n_groups,
                  st);
    if (rc) return rc;
  }
  const auto split_lists = narrow_q > 0 ? split_tiles<true> : split_tiles<false>;
  return split_lists(run_tiles, gstart, n_groups, hkv, nq, narrow_q, split_sums, split, plan, st);
}

// --------------------------------------------------------- reverse map --

// Rows that are run tiles: row r of head h reads the selection of its tile's
// first query; tiles of at most `skip_q` queries are not entered.
struct RowSrc {
  const int2* tiles;
  const int32_t* count;  // tiles per head
  int64_t nq;
  int skip_q;
  __device__ int64_t n_rows(int h) const { return (int64_t)count[h]; }
  __device__ bool skip(int h, int64_t r) const {
    return skip_q > 0 && tiles[(int64_t)h * nq + r].y <= skip_q;
  }
  __device__ int64_t query(int h, int64_t r) const {
    return (int64_t)tiles[(int64_t)h * nq + r].x;
  }
};

__global__ __launch_bounds__(256) void rev_count_kernel(
    const int32_t* __restrict__ topk, int64_t nq, int k,
    const int32_t* __restrict__ cu_q, int64_t batch,
    const int32_t* __restrict__ cu_sb, int64_t nb, RowSrc rows,
    int32_t* __restrict__ counts) {
  const int h = blockIdx.y;
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows.n_rows(h) || rows.skip(h, r)) return;
  const int64_t q = rows.query(h, r);
  int b, bs, nbb;
  bool start;
  query_batch(cu_q, batch, cu_sb, q, &b, &bs, &nbb, &start);
  const int32_t* row = topk + ((int64_t)h * nq + q) * k;
  for (int j = 0; j < k; ++j) {
    const int v = row[j];
    if (v >= 0 && v < nbb && (int64_t)bs + v < nb)
      atomicAdd(&counts[(int64_t)h * nb + bs + v], 1);
  }
}

__global__ __launch_bounds__(256) void rev_scatter_kernel(
    const int32_t* __restrict__ topk, int64_t nq, int k,
    const int32_t* __restrict__ cu_q, int64_t batch,
    const int32_t* __restrict__ cu_sb, int64_t nb, RowSrc rows,
    const int32_t* __restrict__ cu_rev, int32_t* __restrict__ fill,
    int32_t* __restrict__ rev, int64_t cap) {
  const int h = blockIdx.y;
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows.n_rows(h) || rows.skip(h, r)) return;
  const int64_t q = rows.query(h, r);
  int b, bs, nbb;
  bool start;
  query_batch(cu_q, batch, cu_sb, q, &b, &bs, &nbb, &start);
  const int32_t* row = topk + ((int64_t)h * nq + q) * k;
  for (int j = 0; j < k; ++j) {
    const int v = row[j];
    if (v >= 0 && v < nbb && (int64_t)bs + v < nb) {
      const int64_t c = bs + v;
      const int64_t pos =
          cu_rev[(int64_t)h * (nb + 1) + c] +
          atomicAdd(&fill[(int64_t)h * nb + c], 1);
      if (pos < cap) rev[(int64_t)h * cap + pos] = (int32_t)r;
    }
  }
}

// rev_count_kernel / rev_scatter_kernel with the workgroup's listings first
// gathered in LDS (nb <= REV_LDS_BINS): a block listed by many rows (the
// forced blocks, listed by every tile) takes one global atomic per
// workgroup instead of one per listing.  The scatter reserves each block's
// range for the workgroup with one atomic and places its listings in that
// range through LDS counters; the segment sort that follows fixes the order.
constexpr int REV_LDS_BINS = 8192;

__global__ __launch_bounds__(256) void rev_count_lds_kernel(
    const int32_t* __restrict__ topk, int64_t nq, int k,
    const int32_t* __restrict__ cu_q, int64_t batch,
    const int32_t* __restrict__ cu_sb, int64_t nb, RowSrc rows,
    int32_t* __restrict__ counts) {
  __shared__ int hist[REV_LDS_BINS];
  const int h = blockIdx.y;
  const int64_t r0 = (int64_t)blockIdx.x * blockDim.x;
  if (r0 >= rows.n_rows(h)) return;  // whole workgroup
  for (int i = threadIdx.x; i < nb; i += blockDim.x) hist[i] = 0;
  __syncthreads();
  const int64_t r = r0 + threadIdx.x;
  if (r < rows.n_rows(h) && !rows.skip(h, r)) {
    const int64_t q = rows.query(h, r);
    int b, bs, nbb;
    bool start;
    query_batch(cu_q, batch, cu_sb, q, &b, &bs, &nbb, &start);
    const int32_t* row = topk + ((int64_t)h * nq + q) * k;
    for (int j = 0; j < k; ++j) {
      const int v = row[j];
      if (v >= 0 && v < nbb && (int64_t)bs + v < nb) atomicAdd(&hist[bs + v], 1);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += blockDim.x)
    if (hist[i]) atomicAdd(&counts[(int64_t)h * nb + i], hist[i]);
}

__global__ __launch_bounds__(256) void rev_scatter_lds_kernel(
    const int32_t* __restrict__ topk, int64_t nq, int k,
    const int32_t* __restrict__ cu_q, int64_t batch,
    const int32_t* __restrict__ cu_sb, int64_t nb, RowSrc rows,
    const int32_t* __restrict__ cu_rev, int32_t* __restrict__ fill,
    int32_t* __restrict__ rev, int64_t cap) {
  __shared__ int cnt[REV_LDS_BINS];   // listings of the workgroup, then its base
  __shared__ int local[REV_LDS_BINS];  // placed so far
  const int h = blockIdx.y;
  const int64_t r0 = (int64_t)blockIdx.x * blockDim.x;
  if (r0 >= rows.n_rows(h)) return;  // whole workgroup
  for (int i = threadIdx.x; i < nb; i += blockDim.x) {
    cnt[i] = 0;
    local[i] = 0;
  }
  __syncthreads();
  const int64_t r = r0 + threadIdx.x;
  const bool on = r < rows.n_rows(h) && !rows.skip(h, r);
  int bs = 0, nbb = 0;
  const int32_t* row = topk;
  if (on) {
    const int64_t q = rows.query(h, r);
    int b;
    bool start;
    query_batch(cu_q, batch, cu_sb, q, &b, &bs, &nbb, &start);
    row = topk + ((int64_t)h * nq + q) * k;
    for (int j = 0; j < k; ++j) {
      const int v = row[j];
      if (v >= 0 && v < nbb && (int64_t)bs + v < nb) atomicAdd(&cnt[bs + v], 1);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += blockDim.x)
    if (cnt[i]) cnt[i] = atomicAdd(&fill[(int64_t)h * nb + i], cnt[i]);
  __syncthreads();
  if (on) {
    for (int j = 0; j < k; ++j) {
      const int v = row[j];
      if (v >= 0 && v < nbb && (int64_t)bs + v < nb) {
        const int64_t c = bs + v;
        const int64_t pos = cu_rev[(int64_t)h * (nb + 1) + c] + cnt[c] + atomicAdd(&local[c], 1);
        if (pos < cap) rev[(int64_t)h * cap + pos] = (int32_t)r;
      }
    }
  }
}

struct CountF {
  const int32_t* counts;
  int64_t nb;
  __device__ int64_t limit(int, int64_t n) const { return n; }
  __device__ int operator()(int h, int64_t c) const {
    return counts[(int64_t)h * nb + c];
  }
};
struct CuRevW {
  int32_t* cu_rev;
  int64_t nb;
  __device__ void operator()(int h, int64_t c, int ex, int v,
                             int64_t lim) const {
    int32_t* p = cu_rev + (int64_t)h * (nb + 1);
    p[c] = ex;
    if (c == lim - 1) p[c + 1] = ex + v;
  }
};

constexpr int SORT_CAP = 8192;  // segments sorted in LDS up to this length

// Sorts every segment rev[h, cu_rev[h,c] .. cu_rev[h,c+1]) ascending.  Short
// segments use an LDS bitonic sort; longer ones a windowed counting sort over
// the row-id range through `aux` (same shape as rev).
__global__ __launch_bounds__(256) void rev_sort_kernel(
    const int32_t* __restrict__ cu_rev, int32_t* __restrict__ rev,
    int32_t* __restrict__ aux, int64_t nb, int64_t cap, RowSrc rows) {
  __shared__ int s[SORT_CAP];
  const int h = blockIdx.y;
  const int64_t c = blockIdx.x;
  const int64_t s0 = cu_rev[(int64_t)h * (nb + 1) + c];
  int64_t s1 = cu_rev[(int64_t)h * (nb + 1) + c + 1];
  if (s1 > cap) s1 = cap;
  const int64_t len = s1 - s0;
  if (len <= 1) return;
  int32_t* seg = rev + (int64_t)h * cap + s0;
  if (len <= SORT_CAP) {
    int p = 1;
    while (p < len) p <<= 1;
    for (int i = threadIdx.x; i < p; i += blockDim.x)
      s[i] = i < len ? seg[i] : INT32_MAX;
    __syncthreads();
    for (int kk = 2; kk <= p; kk <<= 1) {
      for (int j = kk >> 1; j > 0; j >>= 1) {
        for (int i = threadIdx.x; i < p; i += blockDim.x) {
          const int ixj = i ^ j;
          if (ixj > i) {
            const bool up = (i & kk) == 0;
            const int a = s[i], bb = s[ixj];
            if ((a > bb) == up) {
              s[i] = bb;
              s[ixj] = a;
            }
          }
        }
        __syncthreads();
      }
    }
    for (int i = threadIdx.x; i < len; i += blockDim.x) seg[i] = s[i];
    return;
  }
  // Windowed counting sort: values are row ids in [0, n_rows).
  int32_t* out = aux + (int64_t)h * cap + s0;
  const int64_t range = rows.n_rows(h);
  __shared__ int s_base;
  if (threadIdx.x == 0) s_base = 0;
  __syncthreads();
  for (int64_t w0 = 0; w0 < range; w0 += SORT_CAP) {
    for (int i = threadIdx.x; i < SORT_CAP; i += blockDim.x) s[i] = 0;
    __syncthreads();
    for (int64_t i = threadIdx.x; i < len; i += blockDim.x) {
      const int64_t v = seg[i] - w0;
      if (v >= 0 && v < SORT_CAP) atomicAdd(&s[v], 1);
    }
    __syncthreads();
    // Exclusive scan of the window counts: 256 threads x 32 entries.
    constexpr int PER = SORT_CAP / 256;
    int loc[PER];
    int sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      loc[i] = s[threadIdx.x * PER + i];
      sum += loc[i];
    }
    int tot;
    int ex = block_excl_scan(sum, &tot) + s_base;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int n = loc[i];
      for (int m = 0; m < n; ++m)
        out[ex + m] = (int32_t)(w0 + threadIdx.x * PER + i);
      ex += n;
    }
    __syncthreads();
    if (threadIdx.x == 0) s_base += tot;
    __syncthreads();
  }
  for (int64_t i = threadIdx.x; i < len; i += blockDim.x) seg[i] = out[i];
}

// --------------------------------- query rows: stable counting passes --
// Rows that are queries (all of them, or those marked in `only`): a head's
// queries are cut into chunks, each chunk's listings counted per block in LDS,
// the counts scanned in (block, chunk) order, and each chunk's listings placed
// in (query, slot) order behind the chunk's offset in every block.  Where the
// counts would outgrow the listings (rev_one_pass) two such passes sort by the
// low and then by the high half of the block number, the first from the rows,
// the second from the first's (block, listing) pairs.  A chunk without marked
// queries costs its mask bytes and its zero counts, which are written and
// scanned like others.
//
// Bound by the vector instructions of the ranks and by the scattered writes.
// Whole maps (us), against a radix sort of (block, listing) pairs and against
// chunks placed through one 64-query mask per block:
//   2 heads x 131072 top-16 rows over 462 / 4881 / 30000 blocks:
//     136 / 137 / 138, 115 / 322 / 710, here 66 / 115 / 140
//   24 x 131072 top-16 over 462 / 4881 / 30000:
//     1246 / 1611 / 1668, 905 / 2570 / 6700, here 566 / 961 / 1417
//   rows that list a block twice: as others with the sort and here, 3 to 6
//   times as long with masks.
// Backward plan of 4 x 524288 top-32 block rows over 4881 blocks (no listing):
// 1795 with the sort, 400 here.
constexpr int REV_WIN = 8192;            // buckets per workgroup (32 KB of LDS)
// Whether one pass takes the whole block number: a second pass costs its six
// launches and another trip of every listing, one pass counts and writes that
// spread over more blocks.  One / two passes (us): 2 heads x 131072 top-16
// rows, 2048 blocks 95 / 111, 4881 blocks 147 / 115; 8 x 65536 top-32, 4881
// blocks 331 / 297; 24 x 131072 top-16, 4881 blocks 961 / 1007, 8192 blocks 848
// / 1116, 16384 blocks 1514 / 1323.
inline bool rev_one_pass(int64_t listings, int64_t nb) {
  return nb <= 2048 || (nb <= 8192 && listings >= (int64_t{1} << 25));
}
// Chunks over all heads (one wave per SIMD; of two passes, with less work in
// each, four) and chunk counts over all heads, at most (16 and 8 MB).
constexpr int64_t REV_WAVES = 1024, REV_COUNTS = 4 << 20;
constexpr int64_t REV_WAVES_2 = 4096, REV_COUNTS_2 = 2 << 20;

struct RevChunks {
  int64_t len, n;  // items per chunk (a multiple of `unit`), chunks per head
};
inline RevChunks rev_chunks(bool one, int64_t hkv, int64_t items, int64_t unit, int64_t buckets) {
  int64_t n = std::min<int64_t>(ceil_div(one ? REV_WAVES : REV_WAVES_2, hkv),
                                (one ? REV_COUNTS : REV_COUNTS_2) / (hkv * buckets));
  n = std::max<int64_t>(1, std::min<int64_t>(n, (items + unit - 1) / unit));
  RevChunks c;
  c.len = std::max<int64_t>(unit, ((items + n - 1) / n + unit - 1) / unit * unit);
  c.n = std::max<int64_t>(1, (items + c.len - 1) / c.len);
  return c;
}

struct RevQueries {
  const int32_t* topk;
  int64_t nq;
  int k;
  const int32_t* cu_q;
  int64_t batch;
  const int32_t* cu_sb;
  int64_t nb;
  const uint8_t* only;  // [hkv, nq], or null: every query
  bool encode;          // a listing stores q * k + slot, else q
};

// One pass: what it reads, and its buckets.
struct RevPass {
  RevQueries rows;      // read when pairs is null
  const int2* pairs;    // [hkv, in_cap]: the listings' blocks and what they store
  const int32_t* n_in;  // [hkv]: their number
  int64_t in_cap;
  int shift, mask;      // block c lies in bucket (c >> shift) & mask
  int64_t buckets;
  int64_t chunk_len;    // queries, or pairs, per chunk
  int n_chunks, hkv;
};

// Workgroup -> (head, chunk): each XCD takes consecutive chunks, so that the
// neighbouring counts and listings that they write meet in one L2.
struct RevItem {
  int h, chunk;
};
__device__ inline bool rev_item(const RevPass& a, RevItem* it) {
  const int item = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
  it->h = item / a.n_chunks;
  it->chunk = item - it->h * a.n_chunks;
  return it->h < a.hkv;
}

// The queries q0 .. q0 + 63 of head h that are listed (bit i: q0 + i).
__device__ inline uint64_t rev_marked(const RevQueries& a, int h, int64_t q0, int lane) {
  const int64_t q = q0 + lane;
  return __ballot(q < a.nq && (!a.only || a.only[(int64_t)h * a.nq + q]));
}

// Calls f(c) for the block c of every listing of the marked queries among
// q0 .. q0 + 63.  U ids per load (4: rows of whole, aligned 16-byte pieces).
// One wave; consecutive lanes hold consecutive ids.
template <int U, class F>
__device__ inline void rev_listings(const RevQueries& a, int h, int64_t q0, uint64_t marked,
                                    int lane, F f) {
  int b, bs0, nbb0;
  bool st;
  query_batch(a.cu_q, a.batch, a.cu_sb, q0, &b, &bs0, &nbb0, &st);
  const bool one = b >= 0 && q0 + 63 < (int64_t)a.cu_q[b + 1];  // one batch element
  const int units = a.k / U;  // per row
  const int32_t* rows = a.topk + ((int64_t)h * a.nq + q0) * a.k;
  for (int i = lane; i < 64 * units; i += 64) {
    const int r = i / units;
    if (!((marked >> r) & 1ull)) continue;
    int32_t v[U];
    if constexpr (U == 4) {
      const u32x4 x = reinterpret_cast<const u32x4*>(rows)[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (int32_t)x[e];
    } else {
      v[0] = rows[i];
    }
    int bs = bs0, nbb = nbb0;
    if (!one) query_batch(a.cu_q, a.batch, a.cu_sb, q0 + r, &b, &bs, &nbb, &st);
#pragma unroll
    for (int e = 0; e < U; ++e) {
      const int64_t c = (int64_t)bs + v[e];
      if (v[e] >= 0 && v[e] < nbb && c >= 0 && c < a.nb) f((int)c);
    }
  }
}

// U: ids per load of the rows; 0: from the pairs.
template <int U>
__global__ __launch_bounds__(256) void rev_chunk_count_kernel(RevPass a,
                                                              int32_t* __restrict__ counts) {
  extern __shared__ int hist[];
  RevItem it;
  if (!rev_item(a, &it)) return;
  const int h = it.h, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int w0 = (int)blockIdx.z * REV_WIN;
  const int nw = (int)(a.buckets - w0 < REV_WIN ? a.buckets - w0 : REV_WIN);
  for (int i = threadIdx.x; i < nw; i += blockDim.x) hist[i] = 0;
  __syncthreads();
  auto add = [&](int c) {
    const int x = ((c >> a.shift) & a.mask) - w0;
    if (x >= 0 && x < nw) atomicAdd(&hist[x], 1);
  };
  const int64_t c0 = it.chunk * a.chunk_len;
  if constexpr (U > 0) {
    const int64_t c1 = c0 + a.chunk_len < a.rows.nq ? c0 + a.chunk_len : a.rows.nq;
    for (int64_t q0 = c0 + wv * 64; q0 < c1; q0 += 256) {
      const uint64_t m = rev_marked(a.rows, h, q0, lane);
      if (m) rev_listings<U>(a.rows, h, q0, m, lane, add);
    }
  } else {
    const int64_t n = a.n_in[h], c1 = c0 + a.chunk_len < n ? c0 + a.chunk_len : n;
    const int2* pairs = a.pairs + (int64_t)h * a.in_cap;
    constexpr int G = 8;  // loads in flight
    for (int64_t i0 = c0 + threadIdx.x; i0 < c1; i0 += 256 * G) {
      int x[G];
#pragma unroll
      for (int u = 0; u < G; ++u) x[u] = i0 + 256 * u < c1 ? pairs[i0 + 256 * u].x : -1;
#pragma unroll
      for (int u = 0; u < G; ++u)
        if (x[u] >= 0) add(x[u]);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nw; i += blockDim.x)
    counts[((int64_t)h * a.buckets + w0 + i) * a.n_chunks + it.chunk] = hist[i];
}

// Chunk counts in (bucket, chunk) order -> offsets in place, and the CSR
// offsets of the buckets.
struct ChunkCountF {
  const int32_t* counts;
  int64_t per_head;  // buckets * n_chunks
  __device__ int64_t limit(int, int64_t n) const { return n; }
  __device__ int operator()(int h, int64_t i) const { return counts[(int64_t)h * per_head + i]; }
};
struct ChunkOffW {
  int32_t* counts;
  int64_t per_head;
  int n_chunks;
  int32_t* cu_rev;
  int64_t nb;
  __device__ void operator()(int h, int64_t i, int ex, int v, int64_t lim) const {
    counts[(int64_t)h * per_head + i] = ex;
    const int32_t c = (int32_t)i / n_chunks;  // i < REV_COUNTS + buckets
    int32_t* p = cu_rev + (int64_t)h * (nb + 1);
    if (c * n_chunks == (int32_t)i) p[c] = ex;
    if (i == lim - 1) p[nb] = ex + v;
  }
};

// One wave per chunk.  Its listings are taken REV_STEPS x 64 at a time in
// order; a listing's place is the bucket's offset plus the number of lower
// lanes that hold the same bucket, found from one ballot per bit of the bucket
// number, and the lowest lane of each bucket moves the offset past all of them
// (rows that list a block twice cost nothing extra).  The next listings are
// loaded before and taken in before the places of these are written, so that no
// load waits for the scattered writes.  FIRST of two passes: pairs for the
// second; the last (or only) pass: out [hkv, cap], what the listings store, and
// after a first pass their blocks in `sorted` [hkv, in_cap].
constexpr int REV_STEPS = 16;
enum RevKind { REV_ONLY, REV_FIRST, REV_SECOND };
template <RevKind KIND, int BITS>
__global__ __launch_bounds__(64) void rev_chunk_place_kernel(RevPass a,
                                                             const int32_t* __restrict__ offs,
                                                             int32_t* __restrict__ out,
                                                             int64_t cap,
                                                             int2* __restrict__ out_pairs,
                                                             int32_t* __restrict__ sorted) {
  constexpr int S = REV_STEPS;
  constexpr bool ROWS = KIND != REV_SECOND;
  extern __shared__ int next[];  // [buckets of the window]
  RevItem it;
  if (!rev_item(a, &it)) return;
  const int h = it.h, lane = threadIdx.x;
  const int w0 = (int)blockIdx.z * REV_WIN;
  const int nw = (int)(a.buckets - w0 < REV_WIN ? a.buckets - w0 : REV_WIN);
  const int64_t c0 = it.chunk * a.chunk_len;
  const RevQueries& q = a.rows;
  const int k = ROWS ? q.k : 1;
  const int64_t n_in = ROWS ? q.nq : (int64_t)a.n_in[h];
  const int64_t c1 = c0 + a.chunk_len < n_in ? c0 + a.chunk_len : n_in;
  if (c0 >= c1) return;
  if (ROWS && q.only) {
    uint64_t m = 0;
    for (int64_t q0 = c0; q0 < c1 && !m; q0 += 64) m = rev_marked(q, h, q0, lane);
    if (!m) return;
  }
  for (int i = lane; i < nw; i += 64)
    next[i] = offs[((int64_t)h * a.buckets + w0 + i) * a.n_chunks + it.chunk];
  wave_lds_order();
  const uint32_t total = (uint32_t)((c1 - c0) * k);  // listings (n_q * topk < 2^31)
  const int32_t* src = ROWS ? q.topk + ((int64_t)h * q.nq + c0) * k : nullptr;
  const int2* pairs = ROWS ? nullptr : a.pairs + (int64_t)h * a.in_cap + c0;
  const uint8_t* only = ROWS && q.only ? q.only + (int64_t)h * q.nq + c0 : nullptr;
  out += (int64_t)h * cap;
  out_pairs += (int64_t)h * a.in_cap;
  sorted += (int64_t)h * a.in_cap;
  // row and slot of a lane's listing, 64 listings further
  const int dr = 64 / k, dj = 64 - dr * k;
  auto advance = [&](int& r, int& j) __attribute__((always_inline)) {
    j += dj;
    const int over = j >= k ? 1 : 0;
    j -= over ? k : 0;
    r += dr + over;
  };
  int r_load = lane / k, j_load = lane - r_load * k, r_put = r_load, j_put = j_load;
  const int r_last = (int)(c1 - c0) - 1;
  int32_t v[S], w[S];  // ids (or blocks), and what the listings store
  uint8_t mk[S];
  auto load = [&](uint32_t base) __attribute__((always_inline)) {  // (past the end: the last one)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const uint32_t i = base + s * 64 + lane;
      if constexpr (ROWS) {
        v[s] = src[i < total ? i : total - 1];
      } else {
        const int2 p = pairs[i < total ? i : total - 1];
        v[s] = p.x;
        w[s] = p.y;
      }
      mk[s] = 1;
    }
    if (only) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        mk[s] = only[r_load < r_last ? r_load : r_last];
        advance(r_load, j_load);
      }
    }
  };
  // The batch element at hand: its listings [i_lo, i_hi) of the chunk, its blocks.
  int b = 0, bs = 0, nbb = 0;
  int64_t i_lo = 0, i_hi = 0;
  auto element = [&]() {
    i_lo = ((int64_t)q.cu_q[b] - c0) * k;
    i_hi = ((int64_t)q.cu_q[b + 1] - c0) * k;
    bs = q.cu_sb[b];
    nbb = q.cu_sb[b + 1] - bs;
  };
  if constexpr (ROWS) {
    b = batch_of(q.cu_q, q.batch, c0);
    element();
  }
  int blk[S], val[S];  // the listings' blocks (-1: none), and what they store
  auto take = [&](uint32_t base) __attribute__((always_inline)) {
    const uint32_t end = base + S * 64 < total ? base + S * 64 : total;
    if constexpr (!ROWS) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        blk[s] = base + s * 64 + lane < end ? v[s] : -1;
        val[s] = w[s];
      }
      return;
    }
#pragma unroll
    for (int s = 0; s < S; ++s) blk[s] = -1;
    for (;;) {
      const uint32_t lo = i_lo > 0 ? (uint32_t)(i_lo < end ? i_lo : end) : 0u;
      const uint32_t hi = i_hi > 0 ? (uint32_t)(i_hi < end ? i_hi : end) : 0u;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const uint32_t i = base + s * 64 + lane;
        const int64_t c = (int64_t)bs + v[s];
        if (i >= lo && i < hi && mk[s] && v[s] >= 0 && v[s] < nbb && c >= 0 && c < q.nb)
          blk[s] = (int)c;
      }
      if (i_hi >= end || b + 1 >= q.batch) break;  // the last element of these listings
      ++b;
      element();
    }
  };
  load(0);
  take(0);
  for (uint32_t base = 0; base < total; base += S * 64) {
    load(base + S * 64);
    int pos[S], key[S], put[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int x = ((blk[s] >> a.shift) & a.mask) - w0;
      const bool in = blk[s] >= 0 && x >= 0 && x < nw;
      const uint64_t same = __ballot(in);
      uint32_t lo = (uint32_t)same, hi = (uint32_t)(same >> 32);
#pragma unroll
      for (int i = 0; i < BITS; ++i) {
        const int on = (x << (31 - i)) >> 31;  // all ones where bit i is set
        const uint64_t m = __ballot(on != 0);
        lo &= ~((uint32_t)m ^ (uint32_t)on);
        hi &= ~((uint32_t)(m >> 32) ^ (uint32_t)on);
      }
      const int rank = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
      int at = 0;
      if (in) at = next[x];
      wave_lds_order();
      if (in && rank == 0) next[x] = at + __popc(lo) + __popc(hi);
      wave_lds_order();
      pos[s] = in ? at + rank : -1;
      key[s] = blk[s];
      if constexpr (ROWS) {
        put[s] = q.encode ? (int)(c0 * k + base + s * 64 + lane) : (int)(c0 + r_put);
        advance(r_put, j_put);
      } else {
        put[s] = val[s];
      }
    }
    take(base + S * 64);
    // the loads end here, ahead of the writes
#pragma unroll
    for (int s = 0; s < S; ++s) asm volatile("" : "+v"(blk[s]));
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if constexpr (KIND == REV_FIRST) {
        if (pos[s] >= 0) out_pairs[pos[s]] = make_int2(key[s], put[s]);
      } else {
        if (pos[s] >= 0 && pos[s] < cap) out[pos[s]] = put[s];
        if (KIND == REV_SECOND && pos[s] >= 0) sorted[pos[s]] = key[s];
      }
    }
  }
}

// Offsets of the blocks in each head's sorted listings: one thread per block, a
// binary search.
__global__ __launch_bounds__(256) void rev_offsets_kernel(const int32_t* __restrict__ sorted,
                                                          int64_t in_cap,
                                                          const int32_t* __restrict__ n_in,
                                                          int64_t nb, int32_t* __restrict__ cu_rev) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int h = blockIdx.y;
  if (c > nb) return;
  const int32_t* p = sorted + (int64_t)h * in_cap;
  int64_t lo = 0, hi = n_in[h];  // answer in [lo, hi]
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (p[mid] < c)
      lo = mid + 1;
    else
      hi = mid;
  }
  cu_rev[(int64_t)h * (nb + 1) + c] = (int32_t)lo;
}

// Counts, scans and places one pass (chunks as rev_chunks gives them).
template <RevKind KIND>
int run_rev_pass(RevPass a, const RevChunks& ch, int32_t* counts, int32_t* sums, int32_t* cu,
                 int32_t* totals, int32_t* out, int64_t cap, int2* out_pairs, int32_t* sorted,
                 hipStream_t st) {
  a.chunk_len = ch.len;
  a.n_chunks = (int)ch.n;
  const int64_t win = std::min<int64_t>(a.buckets, REV_WIN), per_head = a.buckets * ch.n;
  const dim3 grid((unsigned)((ch.n * a.hkv + 7) / 8 * 8), 1, (unsigned)ceil_div(a.buckets, REV_WIN));
  const size_t lds = (size_t)win * sizeof(int);
  const bool vec = a.rows.k % 4 == 0 && ((uintptr_t)a.rows.topk % 16) == 0;
  const auto count = KIND == REV_SECOND
                         ? rev_chunk_count_kernel<0>
                         : (vec ? rev_chunk_count_kernel<4> : rev_chunk_count_kernel<1>);
  hipLaunchKernelGGL(count, grid, dim3(256), lds, st, a, counts);
  LSRM_CHECK_LAUNCH();
  const int rc = run_scan(ChunkCountF{counts, per_head},
                          ChunkOffW{counts, per_head, a.n_chunks, cu, a.buckets}, per_head, a.hkv,
                          sums, totals, st);
  if (rc) return rc;
  // the instantiation for the next larger number of bits of a bucket in a window
  const auto place = win <= 16     ? rev_chunk_place_kernel<KIND, 4>
                     : win <= 64   ? rev_chunk_place_kernel<KIND, 6>
                     : win <= 128  ? rev_chunk_place_kernel<KIND, 7>
                     : win <= 256  ? rev_chunk_place_kernel<KIND, 8>
                     : win <= 512  ? rev_chunk_place_kernel<KIND, 9>
                     : win <= 1024 ? rev_chunk_place_kernel<KIND, 10>
                     : win <= 4096 ? rev_chunk_place_kernel<KIND, 12>
                                   : rev_chunk_place_kernel<KIND, 13>;
  static_assert(REV_WIN <= 1 << 13, "a bucket's number in a window has 13 bits");
  hipLaunchKernelGGL(place, grid, dim3(64), lds, st, a, counts, out, cap, out_pairs, sorted);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

int build_query_reverse_map(const int32_t* topk, int64_t hkv, int64_t nq, int64_t topk_n,
                            const int32_t* cu_q, int64_t batch, const int32_t* cu_sb,
                            int64_t nb, Carver& ws, RevMap& map, hipStream_t st,
                            const uint8_t* only, bool encode_slot) {
  const bool two = !rev_one_pass(hkv * nq * topk_n, nb);
  int shift = 0;  // bits of the first of two passes: half of the block number's
  while (two && ((int64_t)1 << (2 * shift)) < nb) ++shift;
  const int64_t n = nq * topk_n > 0 ? nq * topk_n : 1;  // listings per head, at most
  const int64_t buckets[2] = {two ? int64_t{1} << shift : (nb > 0 ? nb : 1),
                              two ? (nb + (int64_t{1} << shift) - 1) >> shift : 1};
  const RevChunks ch[2] = {rev_chunks(!two, hkv, nq, 64, buckets[0]),
                           rev_chunks(!two, hkv, two ? n : 1, REV_STEPS * 64, buckets[1])};
  const int64_t per_head = std::max(buckets[0] * ch[0].n, buckets[1] * ch[1].n);
  int32_t* counts = ws.take<int32_t>((size_t)(hkv * per_head));
  int32_t* sums = ws.take<int32_t>((size_t)scan_sums_size(per_head, hkv));
  int32_t *cu = nullptr, *n_in = nullptr, *sorted = nullptr;
  int2* pairs = nullptr;
  if (two) {
    cu = ws.take<int32_t>((size_t)(hkv * (std::max(buckets[0], buckets[1]) + 1)));
    n_in = ws.take<int32_t>((size_t)hkv);
    pairs = ws.take<int2>((size_t)(hkv * n));
    sorted = ws.take<int32_t>((size_t)(hkv * n));
  }
  if (!map.cu_rev) map.cu_rev = ws.take<int32_t>((size_t)(hkv * (nb + 1)));
  if (!map.rev) map.rev = ws.take<int32_t>((size_t)(hkv * (map.cap > 0 ? map.cap : 1)));
  if (!map.totals) map.totals = ws.take<int32_t>((size_t)hkv);
  if (!ws.base || ws.dry) return LSRM_OK;
  if (!ws.ok()) return LSRM_ERR_WORKSPACE;
  if (nb == 0 || nq == 0) {
    int rc = launch_zero_i32(map.cu_rev, hkv * (nb + 1), st);
    if (rc) return rc;
    return launch_zero_i32(map.totals, hkv, st);
  }
  RevPass a{};
  a.rows = RevQueries{topk, nq, (int)topk_n, cu_q, batch, cu_sb, nb, only, encode_slot};
  a.in_cap = n;
  a.hkv = (int)hkv;
  a.buckets = buckets[0];
  if (!two) {
    a.mask = INT32_MAX;
    return run_rev_pass<REV_ONLY>(a, ch[0], counts, sums, map.cu_rev, map.totals, map.rev, map.cap,
                                  nullptr, nullptr, st);
  }
  a.mask = (int)buckets[0] - 1;
  int rc = run_rev_pass<REV_FIRST>(a, ch[0], counts, sums, cu, n_in, nullptr, 0, pairs, nullptr, st);
  if (rc) return rc;
  a.pairs = pairs;
  a.n_in = n_in;
  a.shift = shift;
  a.mask = INT32_MAX;
  a.buckets = buckets[1];
  rc = run_rev_pass<REV_SECOND>(a, ch[1], counts, sums, cu, map.totals, map.rev, map.cap, nullptr,
                                sorted, st);
  if (rc) return rc;
  hipLaunchKernelGGL(rev_offsets_kernel, dim3(ceil_div(nb + 1, 256), (unsigned)hkv), dim3(256), 0,
                     st, sorted, n, map.totals, nb, map.cu_rev);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

int build_reverse_map(const int32_t* topk, int64_t hkv, int64_t nq,
                      int64_t topk_n, const int32_t* cu_q, int64_t batch,
                      const int32_t* cu_sb, int64_t nb, bool rows_are_tiles,
                      const TilePlan* plan, Carver& ws, RevMap& map,
                      hipStream_t st, const uint8_t* only, bool encode_slot, int skip_q) {
  if (!rows_are_tiles)
    return build_query_reverse_map(topk, hkv, nq, topk_n, cu_q, batch, cu_sb, nb, ws, map, st,
                                   only, encode_slot);
  int32_t* counts = ws.take<int32_t>((size_t)(hkv * (nb > 0 ? nb : 1)));
  int32_t* fill = ws.take<int32_t>((size_t)(hkv * (nb > 0 ? nb : 1)));
  int32_t* sums = ws.take<int32_t>((size_t)scan_sums_size(nb, hkv));
  int32_t* aux = ws.take<int32_t>((size_t)(hkv * (map.cap > 0 ? map.cap : 1)));
  if (!map.cu_rev) map.cu_rev = ws.take<int32_t>((size_t)(hkv * (nb + 1)));
  if (!map.rev) map.rev = ws.take<int32_t>((size_t)(hkv * (map.cap > 0 ? map.cap : 1)));
  if (!map.totals) map.totals = ws.take<int32_t>((size_t)hkv);
  if (!ws.base || ws.dry) return LSRM_OK;
  if (!ws.ok()) return LSRM_ERR_WORKSPACE;

  RowSrc rows{plan->tiles, plan->tile_count, nq, skip_q};
  int rc = launch_zero_i32(counts, hkv * nb, st);
  if (rc) return rc;
  rc = launch_zero_i32(fill, hkv * nb, st);
  if (rc) return rc;
  if (nb == 0) {
    rc = launch_zero_i32(map.cu_rev, hkv, st);
    if (rc) return rc;
    return launch_zero_i32(map.totals, hkv, st);
  }
  const bool lds_bins = nb <= REV_LDS_BINS;
  if (nq > 0) {
    dim3 grid(ceil_div(nq, 256), (unsigned)hkv);
    if (lds_bins)
      hipLaunchKernelGGL(rev_count_lds_kernel, grid, dim3(256), 0, st, topk, nq,
                         (int)topk_n, cu_q, batch, cu_sb, nb, rows, counts);
    else
      hipLaunchKernelGGL(rev_count_kernel, grid, dim3(256), 0, st, topk, nq,
                         (int)topk_n, cu_q, batch, cu_sb, nb, rows, counts);
    LSRM_CHECK_LAUNCH();
  }
  rc = run_scan(CountF{counts, nb}, CuRevW{map.cu_rev, nb}, nb, (int)hkv, sums,
                map.totals, st);
  if (rc) return rc;
  if (nq > 0) {
    dim3 grid(ceil_div(nq, 256), (unsigned)hkv);
    if (lds_bins)
      hipLaunchKernelGGL(rev_scatter_lds_kernel, grid, dim3(256), 0, st, topk, nq,
                         (int)topk_n, cu_q, batch, cu_sb, nb, rows, map.cu_rev,
                         fill, map.rev, map.cap);
    else
      hipLaunchKernelGGL(rev_scatter_kernel, grid, dim3(256), 0, st, topk, nq,
                         (int)topk_n, cu_q, batch, cu_sb, nb, rows, map.cu_rev,
                         fill, map.rev, map.cap);
    LSRM_CHECK_LAUNCH();
    dim3 sgrid((unsigned)nb, (unsigned)hkv);
    hipLaunchKernelGGL(rev_sort_kernel, sgrid, dim3(256), 0, st, map.cu_rev,
                       map.rev, aux, nb, map.cap, rows);
    LSRM_CHECK_LAUNCH();
  }
  return LSRM_OK;
}

__global__ __launch_bounds__(256) void mark_grouped_kernel(const int2* __restrict__ gtiles,
                                                           const int32_t* __restrict__ gcount,
                                                           int64_t nq,
                                                           uint8_t* __restrict__ flags) {
  const int h = blockIdx.y;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= gcount[h]) return;
  const int2 g = gtiles[(int64_t)h * nq + t];
  for (int i = 0; i < g.y; ++i) flags[(int64_t)h * nq + g.x + i] = 1;
}

__global__ __launch_bounds__(256) void mark_short_kernel(const int2* __restrict__ tiles,
                                                         const int32_t* __restrict__ count,
                                                         int64_t nq, int short_q,
                                                         uint8_t* __restrict__ flags) {
  const int h = blockIdx.y;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count[h]) return;
  const int2 r = tiles[(int64_t)h * nq + t];
  if (r.y > short_q) return;
  for (int i = 0; i < r.y; ++i) flags[(int64_t)h * nq + r.x + i] = 1;
}

int mark_short_tiles(const TilePlan& plan, int64_t hkv, int64_t nq, int short_q,
                     uint8_t* flags, hipStream_t st) {
  if (nq <= 0 || short_q <= 0) return LSRM_OK;
  hipLaunchKernelGGL(mark_short_kernel, dim3(ceil_div(nq, 256), (unsigned)hkv), dim3(256), 0, st,
                     plan.tiles, plan.tile_count, nq, short_q, flags);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

int mark_grouped_queries(const TilePlan& plan, int64_t hkv, int64_t nq,
                         uint8_t* flags, hipStream_t st) {
  if (nq <= 0) return LSRM_OK;
  int rc = launch_zero_i32(reinterpret_cast<int32_t*>(flags), (hkv * nq + 3) / 4, st);
  if (rc) return rc;
  if (!plan.gtiles) return LSRM_OK;
  // Grouped tiles hold >= 2 queries, so at most nq / 2 per head.
  hipLaunchKernelGGL(mark_grouped_kernel, dim3(ceil_div(nq / 2 + 1, 256), (unsigned)hkv),
                     dim3(256), 0, st, plan.gtiles, plan.gtile_count, nq, flags);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

// -------------------------------------------------- key-centric part --

// Token count of block c, clamped as the attention kernels clamp it.
__device__ inline int64_t kc_block_len(const int32_t* cu_blk, int64_t nk, int64_t c) {
  int64_t s0 = cu_blk[c], s1 = cu_blk[c + 1];
  s0 = s0 < 0 ? 0 : (s0 > nk ? nk : s0);
  s1 = s1 < s0 ? s0 : (s1 > nk ? nk : s1);
  return s1 - s0;
}

// The listings of block c of grev's segment of kv head h that belong to
// queries [p * pq, (p + 1) * pq) (pass p of pq queries): [s, e) of the
// segment, found by binary search (listings q * topk + slot ascend).
struct KcPassRange {
  const int32_t* cu_rev;
  const int32_t* rev;
  int64_t nb, cap;
  int hkv;
  int64_t pass_listings;  // query passes: pq * topk; 0 = no query cut
  int pass_heads;         // head passes: kv heads per pass; 0 = none
  __device__ void operator()(int vs, int64_t c, int64_t& s, int64_t& e) const {
    const int p = vs / hkv, h = vs - p * hkv;
    const int32_t* cr = cu_rev + (int64_t)h * (nb + 1);
    s = cr[c];
    e = cr[c + 1];
    e = e < cap ? e : cap;
    if (pass_heads > 0 && h / pass_heads != p) e = s;  // another pass's head
    if (pass_listings == 0 || e <= s) return;
    const int32_t* r = rev + (int64_t)h * cap;
    auto first_at = [&](int64_t x) {  // first i in [s, e) with r[i] >= x
      int64_t lo = s, hi = e;
      while (lo < hi) {
        const int64_t m = (lo + hi) >> 1;
        if ((int64_t)r[m] < x) lo = m + 1; else hi = m;
      }
      return lo;
    };
    const int64_t a = first_at(p * pass_listings), b = first_at((p + 1) * pass_listings);
    s = a;
    e = b;
  }
};

// Gathered tiles of block c in the segment "vs" = (pass p, kv head h):
// ceil(listings / tq) pieces of the pass's listings of the block.  With
// cu_blk set, only blocks of lo + 1 .. hi keys count (the resident forwards'
// items, lo >= 0), or with `outside` only the other blocks (the streaming
// forward's); with cu_blk null, every block counts.
struct KcItemsF {
  KcPassRange rg;
  int tq;
  const int32_t* cu_blk;
  int64_t nk;
  int lo, hi;
  bool outside;
  __device__ int64_t limit(int, int64_t n) const { return n; }
  __device__ int operator()(int vs, int64_t c) const {
    if (cu_blk) {
      const int64_t len = kc_block_len(cu_blk, nk, c);
      const bool in = len > lo && len <= hi;
      if (in == outside) return 0;
    }
    int64_t s, e;
    rg(vs, c, s, e);
    return e > s ? (int)((e - s + tq - 1) / tq) : 0;
  }
};
struct KcItemsW {
  KcPassRange rg;
  int tq;
  int4* items;
  int64_t item_cap;
  __device__ void operator()(int vs, int64_t c, int ex, int v, int64_t) const {
    if (v == 0) return;
    int64_t s, e;
    rg(vs, c, s, e);
    for (int t = 0; t < v && ex + t < item_cap; ++t) {
      const int64_t e0 = s + (int64_t)tq * t;
      const int64_t n = e - e0 < tq ? e - e0 : tq;
      items[(int64_t)vs * item_cap + ex + t] = make_int4((int)c, (int)e0, (int)n, 0);
    }
  }
};

__global__ __launch_bounds__(256) void derive_offsets_kernel(RevMap enc, RevMap plain,
                                                             int64_t hkv, int64_t nb) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < hkv * (nb + 1)) plain.cu_rev[i] = enc.cu_rev[i];
  if (i < hkv) plain.totals[i] = enc.totals[i];
}
__global__ __launch_bounds__(256) void derive_rev_kernel(RevMap enc, RevMap plain, int64_t hkv,
                                                         int k) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < hkv * enc.cap;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t h = i / enc.cap;
    if (i - h * enc.cap < enc.totals[h]) plain.rev[i] = enc.rev[i] / k;
  }
}

int derive_query_map(const RevMap& enc, const RevMap& plain, int64_t hkv, int64_t nb,
                     int64_t topk_n, hipStream_t st) {
  if (enc.cap != plain.cap || hkv <= 0 || topk_n <= 0) return LSRM_ERR_INVALID_ARG;
  hipLaunchKernelGGL(derive_offsets_kernel, dim3(ceil_div(hkv * (nb + 1) + hkv, 256)), dim3(256),
                     0, st, enc, plain, hkv, nb);
  LSRM_CHECK_LAUNCH();
  const int64_t grid = std::min<int64_t>(ceil_div(hkv * enc.cap, 256), 16384);
  hipLaunchKernelGGL(derive_rev_kernel, dim3(grid > 0 ? grid : 1), dim3(256), 0, st, enc, plain,
                     hkv, (int)topk_n);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

// Per-(pass, head) offsets of the item lists (resident, eight-wave
// resident, streaming) -- each pass's heads from 0 -- and their cleared work
// counters.
struct KcCounts {
  const int32_t* count[3];
  int32_t* off[3];
};
__global__ void kc_offsets_kernel(KcCounts c, int hkv, int n_pass, int32_t* counter,
                                  int32_t marker) {
  if (threadIdx.x < 3 && blockIdx.x == 0) {
    const int32_t* cnt = c.count[threadIdx.x];
    int32_t* off = c.off[threadIdx.x];
    for (int p = 0; p < n_pass; ++p) {
      int acc = 0;
      off[p * (hkv + 1)] = 0;
      for (int h = 0; h < hkv; ++h) {
        acc += cnt[p * hkv + h];
        off[p * (hkv + 1) + h + 1] = acc;
      }
    }
  }
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    counter[KC_QUEUE_SLOT] = 0;
    counter[KC_EXIT_SLOT] = 0;
    counter[KC_RQUEUE_SLOT] = 0;
    counter[KC_REXIT_SLOT] = 0;
    counter[KC_R2QUEUE_SLOT] = 0;
    counter[KC_R2EXIT_SLOT] = 0;
    counter[PLAN_KC_SLOT] = marker;
  }
}

void kc_passes(int64_t n_q, int64_t hkv, int64_t topk, int g, int64_t head_dim, int* n_pass,
               int* pass_heads, int64_t* q_span) {
  const int64_t nq = n_q > 0 ? n_q : 1;
  const int64_t per_row = topk * g * (2 * (head_dim > 0 ? head_dim : 1) + 4);
  const int64_t per_head = nq * per_row;
  if (per_head * hkv <= KC_PART_BUDGET || per_head <= KC_PART_BUDGET) {
    // whole kv heads per pass (one pass when everything fits)
    int64_t hp = KC_PART_BUDGET / per_head;
    hp = hp < 1 ? 1 : (hp > hkv ? hkv : hp);
    *pass_heads = hkv > 1 && hp < hkv ? (int)hp : 0;
    *q_span = nq;
    *n_pass = (int)((hkv + hp - 1) / hp);
    if (*pass_heads == 0) *n_pass = 1;
    return;
  }
  int64_t span = KC_PART_BUDGET / (hkv * per_row);
  if (span < 1) span = 1;
  if (span >= nq) span = nq;
  *pass_heads = 0;
  *q_span = span;
  *n_pass = (int)((nq + span - 1) / span);
}

int build_kc_items(const RevMap& grev, const int32_t* cu_blk, int64_t nk, int64_t hkv,
                   int64_t nb, int tq, int64_t head_dim, int64_t topk_n, Carver& ws,
                   KcPlan& kc, int32_t* counter, int32_t marker, hipStream_t st) {
  const int rq = tq * KC_RES_CHUNKS;
  const int res_max = kc_res_max((int)(head_dim > 0 ? head_dim : 1));
  const int np = kc.n_pass > 0 ? kc.n_pass : 1;
  // listings of one (pass, head): at most the pass's queries times topk
  const int64_t lst = (np > 1 && kc.pass_heads == 0) ? kc.q_span_max * topk_n : grev.cap;
  kc.ritem_cap = lst / (rq > 0 ? rq : 1) + nb + 1;
  kc.ritems = ws.take<int4>((size_t)(np * hkv * kc.ritem_cap));
  kc.ritem_count = ws.take<int32_t>((size_t)(np * hkv));
  kc.ritem_off = ws.take<int32_t>((size_t)(np * (hkv + 1)));
  kc.r2item_cap = kc.ritem_cap;
  kc.r2items = ws.take<int4>((size_t)(np * hkv * kc.r2item_cap));
  kc.r2item_count = ws.take<int32_t>((size_t)(np * hkv));
  kc.r2item_off = ws.take<int32_t>((size_t)(np * (hkv + 1)));
  kc.fitem_cap = lst / (tq > 0 ? tq : 1) + nb + 1;
  kc.fitems = ws.take<int4>((size_t)(np * hkv * kc.fitem_cap));
  kc.fitem_count = ws.take<int32_t>((size_t)(np * hkv));
  kc.fitem_off = ws.take<int32_t>((size_t)(np * (hkv + 1)));
  int32_t* sums = ws.take<int32_t>((size_t)scan_sums_size(nb, np * hkv));
  if (!ws.base || ws.dry) return LSRM_OK;
  if (!ws.ok()) return LSRM_ERR_WORKSPACE;
  for (int32_t* cnt : {kc.ritem_count, kc.r2item_count, kc.fitem_count}) {
    const int rc = launch_zero_i32(cnt, np * hkv, st);
    if (rc) return rc;
  }
  const KcPassRange rg{grev.cu_rev, grev.rev, nb, grev.cap, (int)hkv,
                       (np > 1 && kc.pass_heads == 0) ? kc.q_span_max * topk_n : 0,
                       kc.pass_heads};
  const int nseg = (int)(np * hkv);
  int rc = run_scan(KcItemsF{rg, rq, cu_blk, nk, 0, KC_RES_KEYS, false},
                    KcItemsW{rg, rq, kc.ritems, kc.ritem_cap}, nb, nseg, sums, kc.ritem_count,
                    st);
  if (rc) return rc;
  if (res_max > KC_RES_KEYS) {
    rc = run_scan(KcItemsF{rg, rq, cu_blk, nk, KC_RES_KEYS, res_max, false},
                  KcItemsW{rg, rq, kc.r2items, kc.r2item_cap}, nb, nseg, sums, kc.r2item_count,
                  st);
    if (rc) return rc;
  }
  rc = run_scan(KcItemsF{rg, tq, cu_blk, nk, 0, res_max, true},
                KcItemsW{rg, tq, kc.fitems, kc.fitem_cap}, nb, nseg, sums, kc.fitem_count, st);
  if (rc) return rc;
  const KcCounts c{{kc.ritem_count, kc.r2item_count, kc.fitem_count},
                   {kc.ritem_off, kc.r2item_off, kc.fitem_off}};
  hipLaunchKernelGGL(kc_offsets_kernel, dim3(1), dim3(64), 0, st, c, (int)hkv, np, counter,
                     marker);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

// ----------------------------------------------------------- key items --

struct KeyChunksF {
  const int32_t* cu;
  int64_t nk;
  __device__ int64_t limit(int, int64_t n) const { return n; }
  __device__ int operator()(int, int64_t c) const {
    int64_t s = cu[c], e = cu[c + 1];
    s = s < 0 ? 0 : (s > nk ? nk : s);
    e = e < 0 ? 0 : (e > nk ? nk : e);
    return e > s ? (int)((e - s + KEY_CHUNK - 1) / KEY_CHUNK) : 0;
  }
};
struct KeyChunksW {
  const int32_t* cu;
  int64_t nk;
  int4* items;
  int64_t cap;
  __device__ void operator()(int, int64_t c, int ex, int v, int64_t) const {
    int64_t s = cu[c], e = cu[c + 1];
    s = s < 0 ? 0 : (s > nk ? nk : s);
    e = e < 0 ? 0 : (e > nk ? nk : e);
    for (int t = 0; t < v && ex + t < cap; ++t) {
      const int64_t t0 = s + (int64_t)KEY_CHUNK * t;
      const int64_t len = e - t0 < KEY_CHUNK ? e - t0 : KEY_CHUNK;
      items[ex + t] = make_int4((int)c, (int)t0, (int)len, 0);
    }
  }
};

int build_key_items(const int32_t* cu_blk, int64_t nb, int64_t nk, Carver& ws,
                    KeyItems& ki, hipStream_t st) {
  const int64_t cap = nb + nk / KEY_CHUNK + 2;
  ki.items = ws.take<int4>((size_t)cap);
  ki.n_items = ws.take<int32_t>(64);
  int32_t* sums = ws.take<int32_t>((size_t)scan_sums_size(nb, 1));
  if (!ws.base || ws.dry) return LSRM_OK;
  if (!ws.ok()) return LSRM_ERR_WORKSPACE;
  int rc = launch_zero_i32(ki.n_items, 1, st);
  if (rc) return rc;
  return run_scan(KeyChunksF{cu_blk, nk}, KeyChunksW{cu_blk, nk, ki.items, cap}, nb,
                  1, sums, ki.n_items, st);
}

// ------------------------------------------------------------ validate --

__global__ __launch_bounds__(256) void validate_meta_kernel(
    const int32_t* __restrict__ cu_sb, const int32_t* __restrict__ cu_blk,
    int64_t nb, const int32_t* __restrict__ cu_q,
    const int32_t* __restrict__ cu_k, int64_t batch, int64_t nq, int64_t nk,
    int32_t* flags) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int f = 0;
  if (i < nb) {
    const int64_t s = cu_blk[i], e = cu_blk[i + 1];
    if (e < s) f |= LSRM_META_OFFSETS_NOT_MONOTONE;
    if (s < 0 || e > nk) f |= LSRM_META_BLOCK_OUT_OF_RANGE;
  }
  if (i < batch) {
    if (cu_sb[i + 1] < cu_sb[i] || cu_sb[i] < 0 || cu_sb[i + 1] > nb)
      f |= LSRM_META_SEQBLOCKS_BAD;
    if (cu_q[i + 1] < cu_q[i] || cu_k[i + 1] < cu_k[i] || cu_q[i] < 0 ||
        cu_k[i] < 0 || cu_k[i + 1] > nk)
      f |= LSRM_META_SEQLENS_BAD;
    if (i == 0 && (cu_q[0] != 0 || cu_q[batch] != nq))
      f |= LSRM_META_SEQLENS_BAD;
    const int64_t b0 = cu_sb[i], b1 = cu_sb[i + 1];
    if (b0 >= 0 && b1 <= nb && b1 > b0) {
      if (cu_blk[b0] < cu_k[i] || cu_blk[b1] > cu_k[i + 1])
        f |= LSRM_META_BLOCK_OUTSIDE_SEQ;
    }
  }
  if (f) atomicOr(flags, f);
}

// Row checks of a selection in one read of it: the metadata bits of every row
// (LSRM_META_TOPK_*) and, with `changes`, the number of rows whose entries
// differ from the previous row's of the same head (raw entries, whatever the
// batch element: what a host comparison of neighbouring rows counts).
//
// One row per thread, any k.
__global__ __launch_bounds__(256) void inspect_rows_kernel(
    const int32_t* __restrict__ topk, int64_t nq, int k,
    const int32_t* __restrict__ cu_q, int64_t batch,
    const int32_t* __restrict__ cu_sb, int32_t* flags,
    unsigned long long* __restrict__ changes) {
  __shared__ int s_changes, s_flags;
  const int h = blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (threadIdx.x == 0) s_changes = s_flags = 0;
  __syncthreads();
  if (i < nq) {
    int b, bs, nbb;
    bool start;
    query_batch(cu_q, batch, cu_sb, i, &b, &bs, &nbb, &start);
    const int32_t* row = topk + ((int64_t)h * nq + i) * k;
    const int32_t* up = i > 0 ? row - k : row;
    bool seen_invalid = false, any = false, diff = false;
    int f = 0;
    for (int j = 0; j < k; ++j) {
      const int v = row[j];
      const bool valid = norm_entry(v, nbb) >= 0;
      if (valid) {
        any = true;
        if (seen_invalid) f |= LSRM_META_TOPK_NOT_PREFIX;
      } else {
        seen_invalid = true;
      }
      if (changes) diff |= v != up[j];
    }
    if (!any) f |= LSRM_META_TOPK_EMPTY_ROW;
    if (f) atomicOr(&s_flags, f);
    if (diff) atomicAdd(&s_changes, 1);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_flags) atomicOr(flags, s_flags);
  if (changes && threadIdx.x == 0 && s_changes)
    atomicAdd(changes, (unsigned long long)s_changes);
}

// The same for rows of P 16-byte pieces (k = 4 P, P a power of two <= 64,
// 16-byte-aligned rows), in the lane layout of breaks_rows_kernel: bound by
// the one read of the rows.  One row per thread fetches a line again for each
// 16-byte column of a wave's 64 rows: 268 MB of top-32 rows took 1194 us
// without the count of changed rows (torch: another 485 us), this form takes
// 75 us with it (3.6 TB/s); 201 MB of top-16 rows 112 + 370 -> 56 us.
template <int P>
__global__ __launch_bounds__(256) void inspect_pieces_kernel(
    const int32_t* __restrict__ topk, int64_t nq, const int32_t* __restrict__ cu_q,
    int64_t batch, const int32_t* __restrict__ cu_sb, int32_t* flags,
    unsigned long long* __restrict__ changes) {
  static_assert(P >= 1 && P <= 64 && (P & (P - 1)) == 0, "rows must tile a wave");
  constexpr int RPW = 64 / P;  // rows per group
  __shared__ int s_changes, s_flags;
  const int h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int p = lane % P, rl = lane / P;
  const u32x4* rows = reinterpret_cast<const u32x4*>(topk + (int64_t)h * nq * (4 * P));
  if (threadIdx.x == 0) s_changes = s_flags = 0;
  __syncthreads();
  int f = 0, n_diff = 0;
  const int64_t step = (int64_t)gridDim.x * (blockDim.x / 64) * (RPW * BRK_G);
  for (int64_t i0 =
           ((int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6)) * (RPW * BRK_G);
       i0 < nq; i0 += step) {  // whole waves
    // the row and the row above it (the same lines, served by the cache)
    u32x4 cur[BRK_G], prev[BRK_G];
#pragma unroll
    for (int g = 0; g < BRK_G; ++g) {
      const int64_t i = i0 + g * RPW + rl < nq ? i0 + g * RPW + rl : nq - 1;
      cur[g] = rows[i * P + p];
      prev[g] = rows[(i > 0 ? i - 1 : 0) * P + p];  // row 0 compares with itself
    }
    const int64_t i_last = i0 + RPW * BRK_G - 1 < nq ? i0 + RPW * BRK_G - 1 : nq - 1;
    int b0 = 0, bs0 = 0, nbb0 = 0;
    bool st0 = true;
    query_batch(cu_q, batch, cu_sb, i0, &b0, &bs0, &nbb0, &st0);
    const bool one = b0 >= 0 && i_last < (int64_t)cu_q[b0 + 1];
#pragma unroll
    for (int g = 0; g < BRK_G; ++g) {
      const int64_t i = i0 + g * RPW + rl;
      int nbb = nbb0;
      if (!one && i < nq) {
        int b, bs;
        bool start;
        query_batch(cu_q, batch, cu_sb, i, &b, &bs, &nbb, &start);
      }
      const bool live = i < nq;  // a lane past the rows raises no flag
      bool diff = false, any = !live, valid[4], gap = false;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        diff |= cur[g][e] != prev[g][e];
        valid[e] = live && norm_entry((int)cur[g][e], nbb) >= 0;
        any |= valid[e];
        if (e > 0) gap |= valid[e] && !valid[e - 1];
      }
      n_diff += __popcll(row_or<P>(__ballot(live && diff)));
      if (row_or<P>(__ballot(any)) != ROW_LSB<P>) f |= LSRM_META_TOPK_EMPTY_ROW;
      // an entry 0 of a piece follows entry 3 of the row's piece before it
      const uint64_t before = (__ballot(valid[3]) << 1) | ROW_LSB<P>;
      if (__ballot(gap) | (__ballot(valid[0]) & ~before)) f |= LSRM_META_TOPK_NOT_PREFIX;
    }
  }
  if (lane == 0 && f) atomicOr(&s_flags, f);
  if (lane == 0 && n_diff) atomicAdd(&s_changes, n_diff);
  __syncthreads();
  if (threadIdx.x == 0 && s_flags) atomicOr(flags, s_flags);
  if (changes && threadIdx.x == 0 && s_changes)
    atomicAdd(changes, (unsigned long long)s_changes);
}

constexpr int64_t INSPECT_GROUPS = 1536;  // six workgroups per CU

// Launches the row checks: the piece form where the rows allow it (as
// build_tile_plan's row comparison), else one row per thread.
int launch_inspect_rows(const int32_t* topk, int64_t hkv, int64_t nq, int64_t topk_n,
                        const int32_t* cu_q, int64_t batch, const int32_t* cu_sb,
                        int32_t* flags, unsigned long long* changes, hipStream_t st) {
  if (nq <= 0) return LSRM_OK;
  const int64_t pieces = topk_n / 4;
  if (topk_n % 4 == 0 && ((uintptr_t)topk % 16) == 0 && pieces <= 64 &&
      (pieces & (pieces - 1)) == 0) {
    // A bounded grid: every workgroup that saw a change adds to one word
    // (about 6 ns each: 8192 of them took half of the kernel's time).
    const int64_t need = ceil_div(ceil_div(nq, (64 / pieces) * BRK_G), 4);
    const dim3 grid((unsigned)std::min<int64_t>(need, ceil_div(INSPECT_GROUPS, hkv)),
                    (unsigned)hkv);
#define LSRM_INSPECT(P)                                                                   \
  case P:                                                                                 \
    hipLaunchKernelGGL(inspect_pieces_kernel<P>, grid, dim3(256), 0, st, topk, nq, cu_q,  \
                       batch, cu_sb, flags, changes);                                     \
    break;
    switch (pieces) {
      LSRM_INSPECT(1) LSRM_INSPECT(2) LSRM_INSPECT(4) LSRM_INSPECT(8)
      LSRM_INSPECT(16) LSRM_INSPECT(32) LSRM_INSPECT(64)
    }
#undef LSRM_INSPECT
  } else {
    hipLaunchKernelGGL(inspect_rows_kernel, dim3(ceil_div(nq, 256), (unsigned)hkv), dim3(256), 0,
                       st, topk, nq, (int)topk_n, cu_q, batch, cu_sb, flags, changes);
  }
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

// ----------------------------------------------------------- block ids --

__global__ __launch_bounds__(256) void block_ids_kernel(
    const int32_t* __restrict__ cu_sb, int64_t batch,
    const int32_t* __restrict__ cu_blk, int64_t nb, int64_t n, int64_t hkv,
    int32_t* __restrict__ ids) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  int id = -1;
  const int64_t b = upper_index(cu_blk, 0, nb + 1, t);
  if (b >= 0 && b < nb && t < cu_blk[b + 1]) {
    const int64_t e = upper_index(cu_sb, 0, batch + 1, b);
    if (e >= 0 && e < batch) id = (int)(b - cu_sb[e]);
  }
  for (int64_t h = 0; h < hkv; ++h) ids[h * n + t] = id;
}

}  // namespace lsrm

using namespace lsrm;

namespace {

// lsrm_sel_attn_validate, and with `changes` lsrm_sel_attn_inspect.
int inspect_impl(const int32_t* topk_idx, int64_t hkv, int64_t n_q, int64_t topk,
                 const int32_t* cu_seqblocks, const int32_t* cu_block_tokens, int64_t n_blocks,
                 const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int64_t batch,
                 int64_t n_k, int32_t* flags, unsigned long long* changes, hipStream_t st) {
  if (hkv <= 0 || n_q < 0 || topk <= 0 || n_blocks < 0 || batch <= 0 ||
      n_k < 0 || !flags || !cu_seqblocks || !cu_block_tokens || !cu_seqlens_q ||
      !cu_seqlens_k || (n_q > 0 && !topk_idx))
    return LSRM_ERR_INVALID_ARG;
  // the count's word follows the flags' in lsrm_sel_attn_inspect's result
  int rc = launch_zero_i32(flags, changes ? 4 : 1, st);
  if (rc) return rc;
  const int64_t m = n_blocks > batch ? n_blocks : batch;
  hipLaunchKernelGGL(validate_meta_kernel, dim3(ceil_div(m > 0 ? m : 1, 256)),
                     dim3(256), 0, st, cu_seqblocks, cu_block_tokens, n_blocks,
                     cu_seqlens_q, cu_seqlens_k, batch, n_q, n_k, flags);
  LSRM_CHECK_LAUNCH();
  return launch_inspect_rows(topk_idx, hkv, n_q, topk, cu_seqlens_q, batch, cu_seqblocks, flags,
                             changes, st);
}

}  // namespace

extern "C" int lsrm_sel_attn_validate(
    const int32_t* topk_idx, int64_t hkv, int64_t n_q, int64_t topk,
    const int32_t* cu_seqblocks, const int32_t* cu_block_tokens,
    int64_t n_blocks, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
    int64_t batch, int64_t n_k, int32_t* flags, void* stream) {
  return inspect_impl(topk_idx, hkv, n_q, topk, cu_seqblocks, cu_block_tokens, n_blocks,
                      cu_seqlens_q, cu_seqlens_k, batch, n_k, flags, nullptr,
                      (hipStream_t)stream);
}

extern "C" int lsrm_sel_attn_inspect(
    const int32_t* topk_idx, int64_t hkv, int64_t n_q, int64_t topk,
    const int32_t* cu_seqblocks, const int32_t* cu_block_tokens,
    int64_t n_blocks, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
    int64_t batch, int64_t n_k, int64_t* info, void* stream) {
  if (!info) return LSRM_ERR_INVALID_ARG;
  return inspect_impl(topk_idx, hkv, n_q, topk, cu_seqblocks, cu_block_tokens, n_blocks,
                      cu_seqlens_q, cu_seqlens_k, batch, n_k, reinterpret_cast<int32_t*>(info),
                      reinterpret_cast<unsigned long long*>(info + 1), (hipStream_t)stream);
}

extern "C" size_t lsrm_reverse_query_map_workspace_size(int64_t n_q,
                                                        int64_t hkv,
                                                        int64_t topk,
                                                        int64_t n_blocks) {
  if (n_q < 0 || hkv <= 0 || topk <= 0 || n_blocks < 0) return 0;
  Carver ws{nullptr, 0, 0};
  RevMap map{};
  map.cap = n_q * topk;
  // cu_rev / rev / totals are caller outputs: mark them present.
  map.cu_rev = reinterpret_cast<int32_t*>(1);
  map.rev = reinterpret_cast<int32_t*>(1);
  map.totals = reinterpret_cast<int32_t*>(1);
  build_reverse_map(nullptr, hkv, n_q, topk, nullptr, 1, nullptr, n_blocks,
                    false, nullptr, ws, map, nullptr);
  return ws.used + 256;
}

extern "C" int lsrm_reverse_query_map(
    const int32_t* topk_idx, int64_t hkv, int64_t n_q, int64_t topk,
    const int32_t* cu_seqlens_q, const int32_t* cu_seqblocks, int64_t batch,
    int64_t n_blocks, int32_t* cu_reverse_count,
    int32_t* reverse_query_indices, int64_t capacity, int32_t* totals,
    void* workspace, size_t workspace_bytes, void* stream) {
  if (hkv <= 0 || n_q < 0 || topk <= 0 || n_blocks < 0 || batch <= 0 ||
      capacity < 0 || !cu_reverse_count || !totals || !cu_seqlens_q ||
      !cu_seqblocks || (n_q > 0 && !topk_idx) ||
      (capacity > 0 && !reverse_query_indices))
    return LSRM_ERR_INVALID_ARG;
  const size_t need =
      lsrm_reverse_query_map_workspace_size(n_q, hkv, topk, n_blocks);
  if (workspace_bytes < need || !workspace) return LSRM_ERR_WORKSPACE;
  Carver ws{reinterpret_cast<char*>(align_up((size_t)workspace, 256)), 0,
            workspace_bytes - 256};
  RevMap map{cu_reverse_count, reverse_query_indices, totals, capacity};
  // The sort's aux buffer is sized by map.cap: keep it equal to capacity.
  return build_reverse_map(topk_idx, hkv, n_q, topk, cu_seqlens_q, batch,
                           cu_seqblocks, n_blocks, false, nullptr, ws, map,
                           (hipStream_t)stream);
}

extern "C" int lsrm_block_ids(const int32_t* cu_seqblocks, int64_t batch,
                              const int32_t* cu_block_tokens, int64_t n_blocks,
                              int64_t n_tokens, int64_t hkv, int32_t* ids,
                              void* stream) {
  if (batch <= 0 || n_blocks < 0 || n_tokens < 0 || hkv <= 0 || !cu_seqblocks ||
      !cu_block_tokens || (n_tokens > 0 && !ids))
    return LSRM_ERR_INVALID_ARG;
  if (n_tokens == 0) return LSRM_OK;
  hipLaunchKernelGGL(block_ids_kernel, dim3(ceil_div(n_tokens, 256)), dim3(256),
                     0, (hipStream_t)stream, cu_seqblocks, batch,
                     cu_block_tokens, n_blocks, n_tokens, hkv, ids);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}
