// Per-query-block top-k block selection.
//
// The rule (no reference function implements it; the reference's learned
// selection is sparse/ops/block_score.py:16-98): mean-pool Q and K per block
// (fp32, the lsrm_block_mean_pool contract), score every (query block b,
// key block c) pair of a batch element as
//     s(b, c) = sum_{g in group(h)} sum_d (double)pq[b,g,d] * (double)pk[c,h,d]
// accumulated in fp64 in that order (fp32 x fp32 products are exact in fp64,
// so the sum is a fixed function of the pooled means), then take the forced
// blocks followed by the best remaining blocks under (score descending,
// block id ascending).  Selected ids are written ascending, -1 padded.
#include <type_traits>

#include "common.h"

namespace lsrm {

int launch_block_mean_pool(const void* x, int x_dtype, int64_t n, int64_t ch,
                           const int32_t* cu, int64_t nb, void* out,
                           int out_dtype, float* partial, int32_t* first,
                           hipStream_t st);
int64_t pool_partial_rows(int64_t n, int64_t nb);
int64_t pool_first_count(int64_t n);

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int SEL_MAXD = 128;
constexpr int SEL_CAND_LDS = 8192;      // candidate scores cached in LDS
constexpr int SEL_MAX_CAND = 65536;     // bitmap capacity (blocks per batch)
constexpr int SEL_MAXK = 256;

// scores[h, b, c] for b, c in [0, nb): 128 rows x 64 columns per workgroup,
// 32x64 per wave as 2x4 blocks of v_mfma_f64_16x16x4 (bound by that
// instruction's rate, the fp64 rate of the chip; a wave's 64 accumulator
// registers leave room for four waves per SIMD, which hide the short loop's
// loads -- with 64x64 per wave and two waves it was busy 47% of the time).
// The vector form with 8x8 scores per thread needed 16 LDS reads per 64 fused
// multiply-adds and reached less: 423 -> 337 us for 4 heads x 4881 x 4881
// x 64, of which 175 us at the fp64 rate.  The instruction adds its four
// products one by one in ascending order, each a fused multiply-add (checked
// bit for bit against that chain), so a score is the same fixed function of
// the pooled means: fp64 accumulation over (g, d) in order.  The pooled rows
// are staged in LDS as doubles, SCORE_DC head-dim columns at a time.
//
// With `keys`, the kernel also writes for every row and class of four columns
// (16 apart in a tile) the largest score, rounded down to fp32, as an
// order-preserving key (NaN scores left out; 0 for a class without a score):
// [hkv, nb, column tiles, 16], read by topk_bound_kernel.
constexpr int SCORE_ROWS = 128, SCORE_COLS = 64;
constexpr int SCORE_DC = 16;
constexpr int SCORE_CLASSES = 16;  // per column tile and row

// Order-preserving key of an fp32 value, and the largest fp32 value <= x.
__device__ inline uint32_t f32_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ inline float key_f32(uint32_t k) {
  return __uint_as_float(k & 0x80000000u ? k ^ 0x80000000u : ~k);
}
__device__ inline float f32_below(double x) {
  const float f = (float)x;
  if (!((double)f > x)) return f;
  const uint32_t u = __float_as_uint(f);
  return __uint_as_float((u << 1) == 0 ? 0x80000001u : (u & 0x80000000u ? u + 1 : u - 1));
}

__global__ __launch_bounds__(256) void score_kernel(
    const float* __restrict__ pq, const float* __restrict__ pk, int64_t nb,
    int hq, int hkv, int d, double* __restrict__ scores, uint32_t* __restrict__ keys) {
  // [column][row]: an operand is 16 rows of 4 columns.  Neighbouring columns lie
  // half the banks apart, so a read's two runs of 16 doubles do not meet, and
  // column pair p shifts its rows by XOR 4 p, so that the 16 columns x 4 rows
  // of a staging write spread over the banks as well.
  __shared__ double sq[SCORE_DC][SCORE_ROWS + 16];
  __shared__ double sk[SCORE_DC][SCORE_COLS + 16];
  const int h = blockIdx.z;
  const int64_t b0 = (int64_t)blockIdx.y * SCORE_ROWS;
  const int64_t c0 = (int64_t)blockIdx.x * SCORE_COLS;
  const int g_n = hq / hkv;
  const int lane = threadIdx.x & 63, r0 = (threadIdx.x >> 6) * 32;  // the wave's rows
  const int l16 = lane & 15, l4 = lane >> 4;
  f64x4 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};

  // Chunks (g, dc) in order; each thread stages column dd of PER_Q Q rows and
  // PER_K K rows, 16 apart (rows past the last block repeat it: their scores
  // are not stored).  The next chunk's global loads are issued into registers
  // before the current chunk's products, so their latency overlaps the
  // arithmetic.  A last, partial chunk is filled with zeros: fma(0, 0, s)
  // leaves s as it is, up to the sign of a zero sum.  Vector instructions do
  // not overlap the fp64 matrix ones, so the loop keeps its addresses as row
  // pointers and immediate LDS offsets.
  constexpr int PER_Q = SCORE_ROWS / 16, PER_K = SCORE_COLS / 16;
  const int n_dc = (d + SCORE_DC - 1) / SCORE_DC;
  const int n_chunk = g_n * n_dc;
  const int dd = threadIdx.x % SCORE_DC, rt = threadIdx.x / SCORE_DC;
  const float *qp[PER_Q], *kp[PER_K];
#pragma unroll
  for (int u = 0; u < PER_Q; ++u) {
    const int64_t b = b0 + rt + 16 * u < nb ? b0 + rt + 16 * u : nb - 1;
    qp[u] = pq + (b * hq + (int64_t)h * g_n) * d + dd;
  }
#pragma unroll
  for (int u = 0; u < PER_K; ++u) {
    const int64_t c = c0 + rt + 16 * u < nb ? c0 + rt + 16 * u : nb - 1;
    kp[u] = pk + (c * hkv + h) * (int64_t)d + dd;
  }
  float pq_r[PER_Q], pk_r[PER_K];
  auto fetch = [&](int g, int dc) __attribute__((always_inline)) {
    if (dc + SCORE_DC <= d) {  // workgroup-uniform: a whole chunk
#pragma unroll
      for (int u = 0; u < PER_Q; ++u) pq_r[u] = qp[u][g * d + dc];
#pragma unroll
      for (int u = 0; u < PER_K; ++u) pk_r[u] = kp[u][dc];
    } else {
      const bool in_d = dc + dd < d;
#pragma unroll
      for (int u = 0; u < PER_Q; ++u) pq_r[u] = in_d ? qp[u][g * d + dc] : 0.0f;
#pragma unroll
      for (int u = 0; u < PER_K; ++u) pk_r[u] = in_d ? kp[u][dc] : 0.0f;
    }
  };
  double* wq = &sq[dd][rt ^ (((dd >> 1) & 3) << 2)];
  double* wk = &sk[dd][rt ^ (((dd >> 1) & 3) << 2)];
  // columns s * 4 + l4 of step s: the shift of steps 0, 2 and of steps 1, 3
  const double *aq[2], *ak[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int row = l16 ^ (((2 * x + (l4 >> 1)) & 3) << 2);
    aq[x] = &sq[l4][r0 + row];
    ak[x] = &sk[l4][row];
  }
  int g = 0, dc = 0;
  fetch(0, 0);
  for (int ci = 0; ci < n_chunk; ++ci) {
#pragma unroll
    for (int u = 0; u < PER_Q; ++u) wq[16 * u] = (double)pq_r[u];
#pragma unroll
    for (int u = 0; u < PER_K; ++u) wk[16 * u] = (double)pk_r[u];
    __syncthreads();
    dc += SCORE_DC;
    if (dc >= d) {
      dc = 0;
      ++g;
    }
    if (ci + 1 < n_chunk) fetch(g, dc);
#pragma unroll
    for (int s = 0; s < SCORE_DC / 4; ++s) {
      double a[2], bv[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = aq[s & 1][s * 4 * (SCORE_ROWS + 16) + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) bv[j] = ak[s & 1][s * 4 * (SCORE_COLS + 16) + 16 * j];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], bv[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // acc[i][j][v]: row r0 + 16 i + 4 v + l4, column 16 j + l16
  const int64_t bl = b0 + r0 + l4;
  double* orow = scores + ((int64_t)h * nb + bl) * nb + c0 + l16;
  uint32_t* krow =
      keys ? keys + (((int64_t)h * nb + bl) * gridDim.x + blockIdx.x) * SCORE_CLASSES + l16
           : nullptr;
  bool in_c[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) in_c[j] = c0 + 16 * j + l16 < nb;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * i + 4 * v;
      if (bl + row < nb) {
        // (fmax leaves a NaN out; NaN only if every column is)
        double best = __builtin_nan("");
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (in_c[j]) {
            orow[16 * j] = acc[i][j][v];
            best = __builtin_fmax(best, acc[i][j][v]);
          }
        if (krow) *krow = best == best ? f32_key(f32_below(best)) : 0u;
      }
      orow += 4 * nb;
      if (krow) krow += (int64_t)4 * gridDim.x * SCORE_CLASSES;
    }
}

// dst[t * topk + j] = ord[j] for the `total` / topk token rows at dst, the
// stores spread over the calling threads (`first`, `step`).  When topk / 4
// divides `step`, a thread's 16-byte stores all carry the same four ids.
__device__ inline void fill_token_rows(int32_t* __restrict__ dst, int64_t total,
                                       const int* __restrict__ ord, int topk, int first,
                                       int step) {
  const int q4 = topk >> 2;
  if ((topk & 3) == 0 && step % q4 == 0 && ((uintptr_t)dst & 15) == 0) {
    const int j = (first % q4) * 4;
    const int4 val = make_int4(ord[j], ord[j + 1], ord[j + 2], ord[j + 3]);
    int4* d4 = reinterpret_cast<int4*>(dst);
    for (int64_t i = first; i < (total >> 2); i += step) d4[i] = val;
  } else {
    for (int64_t i = first; i < total; i += step) dst[i] = ord[i % topk];
  }
}

// A block outside every batch element selects nothing: its compact row and
// the per-token rows of its tokens (clamped to [0, n_tokens)) become -1.
// `first` / `step` spread the stores over the calling threads.
__device__ inline void clear_block_rows(const int32_t* __restrict__ cu_blk, int64_t b,
                                        int64_t n_tokens, int topk, int32_t* crow,
                                        int32_t* head_rows, int first, int step) {
  for (int j = first; j < topk; j += step) crow[j] = -1;
  int64_t t0 = cu_blk[b], t1 = cu_blk[b + 1];
  t0 = t0 < 0 ? 0 : (t0 > n_tokens ? n_tokens : t0);
  t1 = t1 < t0 ? t0 : (t1 > n_tokens ? n_tokens : t1);
  int32_t* dst = head_rows + t0 * topk;
  const int64_t total = (t1 - t0) * topk;
  for (int64_t i = first; i < total; i += step) dst[i] = -1;
}

__device__ inline bool sel_better(double s1, int i1, double s2, int i2) {
  return s1 > s2 || (s1 == s2 && i1 < i2);
}

__device__ inline double readlane_f64(double x, int j) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, j);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), j);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The best R candidates (score descending, id ascending) of those a wave
// holds -- M per lane: candidate (lane, m) has id lane + 64 m and score
// v[m], and bit m of `taken` marks it unavailable -- written to ls / li in
// that order (ls may be null: ids only); returns how many there are
// (min(R, available)).
// Threshold pass: each lane's best available candidate is its lane best;
// the lane bests of rank 0 .. R-1 are R distinct candidates no worse than
// the rank R-1 lane best T, so every member of the best R is no worse than
// T.  The candidates no worse than T (the survivors) are compacted through
// cs / ci (64 entries) and ranked among themselves.  Fallback (fewer than R
// lane bests, or more than 64 survivors): R rounds of lane-local scan plus
// wave butterfly.  Both give the same list, since the best R under a strict
// total order are unique.
template <int M>
__device__ int wave_best_r(const double (&v)[M], uint32_t taken, int R,
                           double* __restrict__ ls, int* __restrict__ li,
                           double* __restrict__ cs, int* __restrict__ ci) {
  const int lane = threadIdx.x & 63;
  if (R <= 0) return 0;
  double bs = -__builtin_inf();
  int bi = INT32_MAX;
#pragma unroll
  for (int m = 0; m < M; ++m)
    if (!((taken >> m) & 1u) && sel_better(v[m], lane + 64 * m, bs, bi)) {
      bs = v[m];
      bi = lane + 64 * m;
    }
  const int nv = __popcll(__ballot(bi != INT32_MAX));
  int S = 65;
  if (nv >= R) {
    int rank = 0;
#pragma unroll
    for (int j = 0; j < 64; ++j)
      rank += sel_better(readlane_f64(bs, j), __builtin_amdgcn_readlane(bi, j), bs, bi) ? 1 : 0;
    const unsigned long long at = __ballot(bi != INT32_MAX && rank == R - 1);
    const int tl = __builtin_amdgcn_readfirstlane(__ffsll((long long)at) - 1);
    const double ts = readlane_f64(bs, tl);
    const int ti = __builtin_amdgcn_readlane(bi, tl);
    S = 0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int id = lane + 64 * m;
      const bool p = !((taken >> m) & 1u) && !sel_better(ts, ti, v[m], id);
      const unsigned long long bm = __ballot(p);
      const int pos = S + (int)__builtin_amdgcn_mbcnt_hi(
                              (uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u));
      if (p && pos < 64) {
        cs[pos] = v[m];
        ci[pos] = id;
      }
      S += __popcll(bm);
    }
  }
  if (S <= 64) {
    // One wave's LDS accesses complete in order; the clobber keeps the
    // compiler from moving the reads above the writes.
    asm volatile("" ::: "memory");
    const double xs = lane < S ? cs[lane] : -__builtin_inf();
    const int xi = lane < S ? ci[lane] : INT32_MAX;
    int rank = 0;
    for (int j = 0; j < S; ++j)
      rank += sel_better(readlane_f64(xs, j), __builtin_amdgcn_readlane(xi, j), xs, xi) ? 1 : 0;
    const int nw = S < R ? S : R;
    if (lane < S && rank < nw) {
      if (ls) ls[rank] = xs;
      li[rank] = xi;
    }
    return nw;
  }
  uint32_t tk = taken;
  int nw = 0;
  for (int n = 0; n < R; ++n) {
    double rs = -__builtin_inf();
    int ri = INT32_MAX;
#pragma unroll
    for (int m = 0; m < M; ++m)
      if (!((tk >> m) & 1u) && sel_better(v[m], lane + 64 * m, rs, ri)) {
        rs = v[m];
        ri = lane + 64 * m;
      }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double os = __shfl_xor(rs, o);
      const int oi = __shfl_xor(ri, o);
      if (sel_better(os, oi, rs, ri)) {
        rs = os;
        ri = oi;
      }
    }
    ri = __builtin_amdgcn_readfirstlane(ri);
    if (ri == INT32_MAX) break;  // no candidate left
    if ((ri & 63) == lane) tk |= 1u << (ri >> 6);
    if (lane == 0) {
      if (ls) ls[nw] = rs;
      li[nw] = ri;
    }
    ++nw;
  }
  return nw;
}

// One workgroup per (query block b, kv head h).
__global__ __launch_bounds__(256) void topk_kernel(
    const double* __restrict__ scores, int64_t nb,
    const int32_t* __restrict__ cu_sb, int64_t batch,
    const int32_t* __restrict__ cu_blk, int64_t n_tokens, int topk,
    const int32_t* __restrict__ forced, int n_forced, int force_self,
    int32_t* __restrict__ topk_idx, int32_t* __restrict__ compact) {
  __shared__ double s_sc[SEL_CAND_LDS];
  __shared__ uint32_t s_taken[SEL_MAX_CAND / 32];
  __shared__ int s_sel[SEL_MAXK];
  __shared__ int s_out[SEL_MAXK];
  __shared__ double s_ws[4];
  __shared__ int s_wi[4];
  __shared__ int s_nsel;

  const int h = blockIdx.y;
  const int64_t b = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t e = upper_index(cu_sb, 0, batch + 1, b);
  int32_t* crow = compact + ((int64_t)h * nb + b) * topk;
  if (e < 0 || e >= batch || b >= cu_sb[e + 1]) {
    clear_block_rows(cu_blk, b, n_tokens, topk, crow, topk_idx + (int64_t)h * n_tokens * topk,
                     tid, 256);
    return;
  }
  const int64_t cs = cu_sb[e];
  const int nbb = (int)(cu_sb[e + 1] - cs);
  const bool cached = nbb <= SEL_CAND_LDS;
  const double* row = scores + ((int64_t)h * nb + b) * nb + cs;

  for (int i = tid; i < (nbb + 31) / 32; i += 256) s_taken[i] = 0u;
  if (cached) {
    for (int i = tid; i < nbb; i += 256) {
      const double v = row[i];
      s_sc[i] = (v != v) ? -__builtin_inf() : v;
    }
  }
  __syncthreads();
  const int kmax = topk < nbb ? topk : nbb;
  if (tid == 0) {
    int n = 0;
    auto add = [&](int id) {
      if (n >= kmax || id < 0 || id >= nbb) return;
      if (s_taken[id >> 5] & (1u << (id & 31))) return;
      s_taken[id >> 5] |= 1u << (id & 31);
      s_sel[n++] = id;
    };
    if (force_self) add((int)(b - cs));
    for (int f = 0; f < n_forced; ++f) add(forced[f]);
    s_nsel = n;
  }
  __syncthreads();

  for (int n = s_nsel; n < kmax; ++n) {
    double bs = -__builtin_inf();
    int bi = INT32_MAX;
    for (int i = tid; i < nbb; i += 256) {
      if (s_taken[i >> 5] & (1u << (i & 31))) continue;
      double v;
      if (cached) {
        v = s_sc[i];
      } else {
        v = row[i];
        if (v != v) v = -__builtin_inf();
      }
      if (sel_better(v, i, bs, bi)) {
        bs = v;
        bi = i;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double os = __shfl_xor(bs, o);
      const int oi = __shfl_xor(bi, o);
      if (sel_better(os, oi, bs, bi)) {
        bs = os;
        bi = oi;
      }
    }
    if (lane == 0) {
      s_ws[w] = bs;
      s_wi[w] = bi;
    }
    __syncthreads();
    if (tid == 0) {
      double fs = s_ws[0];
      int fi = s_wi[0];
      for (int i = 1; i < 4; ++i)
        if (sel_better(s_ws[i], s_wi[i], fs, fi)) {
          fs = s_ws[i];
          fi = s_wi[i];
        }
      s_sel[n] = fi;
      s_taken[fi >> 5] |= 1u << (fi & 31);
    }
    __syncthreads();
  }
  // Ascending order by rank (ids are distinct), -1 padding.
  for (int j = tid; j < topk; j += 256) s_out[j] = -1;
  __syncthreads();
  for (int j = tid; j < kmax; j += 256) {
    const int v = s_sel[j];
    int r = 0;
    for (int m = 0; m < kmax; ++m) r += s_sel[m] < v;
    s_out[r] = v;
  }
  __syncthreads();
  for (int j = tid; j < topk; j += 256) crow[j] = s_out[j];
  int64_t t0 = cu_blk[b], t1 = cu_blk[b + 1];
  t0 = t0 < 0 ? 0 : (t0 > n_tokens ? n_tokens : t0);
  t1 = t1 < t0 ? t0 : (t1 > n_tokens ? n_tokens : t1);
  int32_t* dst = topk_idx + ((int64_t)h * n_tokens + t0) * topk;
  const int64_t total = (t1 - t0) * topk;
  fill_token_rows(dst, total, s_out, topk, tid, 256);
}

// One wave per (kv head, query block) row when the candidates fit the
// registers (M per lane, blocks per batch <= 64 M): the row's scores stay in
// registers, forced blocks are taken first, then wave_best_r lists the best
// of the rest (score descending, id ascending).  No LDS candidate cache and
// no workgroup barriers.
template <int M>
__global__ __launch_bounds__(256) void topk_wave_kernel(
    const double* __restrict__ scores, int64_t nb,
    const int32_t* __restrict__ cu_sb, int64_t batch,
    const int32_t* __restrict__ cu_blk, int64_t n_tokens, int hkv, int topk,
    const int32_t* __restrict__ forced, int n_forced, int force_self,
    int32_t* __restrict__ topk_idx, int32_t* __restrict__ compact) {
  __shared__ int s_sel[4][SEL_MAXK];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t rowid = (int64_t)blockIdx.x * 4 + wv;
  if (rowid >= (int64_t)hkv * nb) return;  // whole wave
  const int h = (int)(rowid / nb);
  const int64_t b = rowid - (int64_t)h * nb;
  int* sel = s_sel[wv];
  const int64_t e = upper_index(cu_sb, 0, batch + 1, b);
  int32_t* crow = compact + ((int64_t)h * nb + b) * topk;
  if (e < 0 || e >= batch || b >= cu_sb[e + 1]) {
    clear_block_rows(cu_blk, b, n_tokens, topk, crow, topk_idx + (int64_t)h * n_tokens * topk,
                     lane, 64);
    return;
  }
  const int64_t cs = cu_sb[e];
  const int nbb = (int)(cu_sb[e + 1] - cs);
  const double* row = scores + ((int64_t)h * nb + b) * nb + cs;

  double v[M];
  uint32_t taken = 0u;  // bit m: candidate lane + 64 m is unavailable
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int i = lane + 64 * m;
    if (i < nbb) {
      const double x = row[i];
      v[m] = (x != x) ? -__builtin_inf() : x;
    } else {
      v[m] = -__builtin_inf();
      taken |= 1u << m;
    }
  }
  const int kmax = topk < nbb ? topk : nbb;
  int n = 0;
  auto take = [&](int id) {  // wave-uniform id
    if (n >= kmax || id < 0 || id >= nbb) return;
    const bool mine = (id & 63) == lane;
    const bool was = mine && ((taken >> (id >> 6)) & 1u);
    if (__builtin_amdgcn_ballot_w64(was) != 0) return;
    if (mine) taken |= 1u << (id >> 6);
    if (lane == 0) sel[n] = id;
    ++n;
  };
  if (force_self) take((int)(b - cs));
  for (int f = 0; f < n_forced; ++f) take(forced[f]);
  __shared__ double s_cs[4][64];
  __shared__ int s_ci[4][64];
  n += wave_best_r<M>(v, taken, kmax - n, nullptr, sel + n, s_cs[wv], s_ci[wv]);
  asm volatile("" ::: "memory");
  // Ascending ids (distinct), -1 padding: id -> its rank among the chosen.
  __shared__ int s_out[4][SEL_MAXK];
  int* ord = s_out[wv];
  for (int j = lane; j < topk; j += 64) ord[j] = -1;
  for (int j = lane; j < kmax; j += 64) {
    const int id = sel[j];
    int r = 0;
    for (int t = 0; t < kmax; ++t) r += sel[t] < id;
    ord[r] = id;
  }
  for (int j = lane; j < topk; j += 64) crow[j] = ord[j];
  int64_t t0 = cu_blk[b], t1 = cu_blk[b + 1];
  t0 = t0 < 0 ? 0 : (t0 > n_tokens ? n_tokens : t0);
  t1 = t1 < t0 ? t0 : (t1 > n_tokens ? n_tokens : t1);
  int32_t* dst = topk_idx + ((int64_t)h * n_tokens + t0) * topk;
  const int64_t total = (t1 - t0) * topk;
  fill_token_rows(dst, total, ord, topk, lane, 64);
}

// One wave per (query block, kv head) row of up to 64 * NM / 16 column tiles:
// the row's classes (score_kernel's keys; those of tiles inside the row's batch
// element) give a lower bound of its topk-th best score -- the largest value
// that at least topk class maxima reach, and these are distinct columns -- and
// only the columns that reach it are listed (about topk of them, at most four
// per class that reaches the bound) and ranked by wave_best_r.  The forced
// blocks are taken first and count among the topk.  More than BOUND_CAP such
// columns (ties in great number) are taken in pieces, each ranked beside the
// best so far: whole selections of 4 x 4881 rows, top-32, take 0.65 ms, 0.70
// with all scores equal or NaN (0.92 with four waves per row, 4.56 with one
// scan of the row per pick); 4 x 8192 rows, top-64, 1.38 and 1.57 (2.45, 34.8).
// Bound by reading the scores once (the row's arithmetic is a third of that):
// 4 x 4881 rows of 4881 scores, top-32, 465 us with four waves per row that
// each listed their quarter's best, 306 us here (763 MB of scores read and 268 MB of
// token rows written: 3.4 TB/s).
constexpr int BOUND_CAP = 1024;

template <int NM>
__global__ __launch_bounds__(64) void topk_bound_kernel(
    const double* __restrict__ scores, const uint32_t* __restrict__ keys, int ntile, int64_t nb,
    const int32_t* __restrict__ cu_sb, int64_t batch, const int32_t* __restrict__ cu_blk,
    int64_t n_tokens, int topk, const int32_t* __restrict__ forced, int n_forced,
    int force_self, int32_t* __restrict__ topk_idx, int32_t* __restrict__ compact) {
  __shared__ int s_id[BOUND_CAP];
  __shared__ double s_cs[64], s_ls[64];
  __shared__ int s_ci[64], s_at[64], s_sel[64], s_out[64];
  const int h = blockIdx.y;
  const int64_t b = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t e = upper_index(cu_sb, 0, batch + 1, b);
  int32_t* crow = compact + ((int64_t)h * nb + b) * topk;
  if (e < 0 || e >= batch || b >= cu_sb[e + 1]) {
    clear_block_rows(cu_blk, b, n_tokens, topk, crow, topk_idx + (int64_t)h * n_tokens * topk,
                     lane, 64);
    return;
  }
  const int64_t cs = cu_sb[e];
  const int nbb = (int)(cu_sb[e + 1] - cs);
  const double* row = scores + ((int64_t)h * nb + b) * nb + cs;
  const uint32_t* krow = keys + ((int64_t)h * nb + b) * ntile * SCORE_CLASSES;
  uint32_t key[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const int ci = lane + 64 * m, tile = ci / SCORE_CLASSES;
    const int64_t c0 = (int64_t)tile * SCORE_COLS;
    const int64_t c1 = c0 + SCORE_COLS < nb ? c0 + SCORE_COLS : nb;
    key[m] = tile < ntile && c0 >= cs && c1 <= cs + nbb ? krow[ci] : 0u;
  }
  // Forced blocks in order, distinct, valid, at most kmax.
  const int kmax = topk < nbb ? topk : nbb;
  int nf = 0;
  auto add = [&](int id) {  // wave-uniform
    if (nf >= kmax || id < 0 || id >= nbb) return;
    if (__ballot(lane < nf && s_sel[lane] == id)) return;
    if (lane == 0) s_sel[nf] = id;
    ++nf;
    __syncthreads();
  };
  if (force_self) add((int)(b - cs));
  for (int f = 0; f < n_forced; ++f) add(forced[f]);
  const int r_need = kmax - nf;
  auto is_forced = [&](int id) {
    for (int t = 0; t < nf; ++t)
      if (s_sel[t] == id) return true;
    return false;
  };
  // The bound, to 24 bits of the key.
  uint32_t kb = 0u;
  for (int bit = 31; bit >= 8; --bit) {
    const uint32_t tryk = kb | (1u << bit);
    int reach = 0;
#pragma unroll
    for (int m = 0; m < NM; ++m) reach += __popcll(__ballot(key[m] >= tryk));
    if (reach >= topk) kb = tryk;
  }
  const double bound =
      kb > f32_key(-__builtin_inff()) ? (double)key_f32(kb) : -__builtin_inf();
  // The columns that reach it, in ascending order.
  int n = 0;
  constexpr int U = 8;
  for (int base = 0; base < nbb; base += 64 * U) {
    double x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + 64 * u + lane;
      x[u] = i < nbb ? row[i] : __builtin_nan("");
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + 64 * u + lane;
      if (x[u] != x[u]) x[u] = -__builtin_inf();  // NaN ranks lowest
      const bool in = i < nbb && x[u] >= bound;
      const unsigned long long m = __ballot(in);
      if (m == 0ull) continue;
      const int pos = n + __popcll(m & ((1ull << lane) - 1ull));
      if (in && pos < BOUND_CAP) s_id[pos] = i;
      n += __popcll(m);
    }
  }
  __syncthreads();
  // wave_best_r over the listed columns: their places ascend with their ids.
  auto best = [&](auto per) {
    constexpr int M = decltype(per)::value;
    double v[M];
    uint32_t taken = 0u;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int at = lane + 64 * m;
      v[m] = -__builtin_inf();
      if (at < n) {  // (read again: a few cached lines)
        const double x = row[s_id[at]];
        if (x == x) v[m] = x;
      }
      if (at >= n || is_forced(s_id[at])) taken |= 1u << m;
    }
    const int nw = wave_best_r<M>(v, taken, r_need, nullptr, s_at, s_cs, s_ci);
    __syncthreads();
    if (lane < nw) s_sel[nf + lane] = s_id[s_at[lane]];
  };
  if (n <= 256) {
    best(std::integral_constant<int, 4>{});
  } else if (n <= BOUND_CAP) {
    best(std::integral_constant<int, BOUND_CAP / 64>{});
  } else if (r_need > 0) {
    // 960 columns at a time beside the best so far (places 0 .. 63, best
    // first).  Those have smaller ids than the columns, so places rank ties
    // as ids do, and only a column above the last of them can enter.
    constexpr int M = BOUND_CAP / 64;
    int nc = 0;
    double cv = 0.0, last = 0.0;  // this lane's score of the best so far, the last one
    for (int base = 0; base < nbb; base += 64 * (M - 1)) {
      double v[M];
      v[0] = cv;
      uint32_t taken = lane < nc ? 0u : 1u;
      bool enters = false;
#pragma unroll
      for (int m = 1; m < M; ++m) {
        const int i = base + 64 * (m - 1) + lane;
        const double x = i < nbb ? row[i] : -__builtin_inf();
        v[m] = x == x ? x : -__builtin_inf();
        if (i >= nbb || is_forced(i)) taken |= 1u << m;
        enters |= v[m] > last;
      }
      if (nc == r_need && !__ballot(enters)) continue;
      const int nw = wave_best_r<M>(v, taken, r_need, s_ls, s_at, s_cs, s_ci);
      __syncthreads();
      const int at = lane < nw ? s_at[lane] : 0;
      const int id = at < 64 ? s_id[at] : base + at - 64;
      if (lane < nw) cv = s_ls[lane];
      __syncthreads();
      if (lane < nw) s_id[lane] = id;
      nc = nw;
      last = readlane_f64(cv, nw > 0 ? nw - 1 : 0);
      __syncthreads();
    }
    if (lane < nc) s_sel[nf + lane] = s_id[lane];
  }
  __syncthreads();
  // Ascending order by rank (ids are distinct), -1 padding.
  if (lane < topk) s_out[lane] = -1;
  __syncthreads();
  if (lane < kmax) {
    const int id = s_sel[lane];
    int r = 0;
    for (int m = 0; m < kmax; ++m) r += s_sel[m] < id;
    s_out[r] = id;
  }
  __syncthreads();
  if (lane < topk) crow[lane] = s_out[lane];
  int64_t t0 = cu_blk[b], t1 = cu_blk[b + 1];
  t0 = t0 < 0 ? 0 : (t0 > n_tokens ? n_tokens : t0);
  t1 = t1 < t0 ? t0 : (t1 > n_tokens ? n_tokens : t1);
  fill_token_rows(topk_idx + ((int64_t)h * n_tokens + t0) * topk, (t1 - t0) * topk, s_out, topk,
                  lane, 64);
}

// Rows of tokens outside every block ([0, cu_blk[0]) and [cu_blk[nb], n),
// clamped) are -1: the top-k kernels write only the tokens of blocks.
__global__ __launch_bounds__(256) void uncovered_rows_kernel(const int32_t* __restrict__ cu_blk,
                                                             int64_t nb, int64_t n_tokens,
                                                             int topk,
                                                             int32_t* __restrict__ topk_idx) {
  const int h = blockIdx.y;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tokens) return;
  int64_t lo = cu_blk[0], hi = cu_blk[nb];
  lo = lo < 0 ? 0 : (lo > n_tokens ? n_tokens : lo);
  hi = hi < lo ? lo : (hi > n_tokens ? n_tokens : hi);
  if (t >= lo && t < hi) return;
  int32_t* row = topk_idx + ((int64_t)h * n_tokens + t) * topk;
  for (int j = 0; j < topk; ++j) row[j] = -1;
}

struct SelectWs {
  float* pq;
  float* pk;
  float* partial;
  int32_t* first;
  double* scores;
  uint32_t* keys;  // class maxima of the scores (bounded_rows)
};

// Rows of this many blocks are selected behind a bound from class maxima (for
// topk <= 64): below, one wave holds the row in registers; above, the classes
// no longer fit a wave's registers.
inline bool bounded_rows(int64_t nb) { return nb > 64 * 32 && nb <= 4 * 64 * 32; }

void carve_select(Carver& ws, int64_t n, int64_t nb, int64_t hq, int64_t hkv,
                  int64_t d, SelectWs& s) {
  const int64_t nbc = nb > 0 ? nb : 1;
  s.pq = ws.take<float>((size_t)(nbc * hq * d));
  s.pk = ws.take<float>((size_t)(nbc * hkv * d));
  s.partial = ws.take<float>((size_t)(pool_partial_rows(n, nbc) *
                                      (hq > hkv ? hq : hkv) * d));
  s.first = ws.take<int32_t>((size_t)pool_first_count(n));
  s.scores = ws.take<double>((size_t)(hkv * nbc * nbc));
  s.keys = bounded_rows(nb) ? ws.take<uint32_t>((size_t)(hkv * nbc * SCORE_CLASSES *
                                                         ceil_div(nbc, SCORE_COLS)))
                            : nullptr;
}

}  // namespace lsrm

using namespace lsrm;

extern "C" size_t lsrm_select_blocks_workspace_size(int64_t n_tokens,
                                                    int64_t n_blocks,
                                                    int64_t hq, int64_t hkv,
                                                    int64_t head_dim) {
  if (n_tokens < 0 || n_blocks < 0 || hq <= 0 || hkv <= 0 || head_dim <= 0)
    return 0;
  Carver ws{nullptr, 0, 0};
  SelectWs s;
  carve_select(ws, n_tokens, n_blocks, hq, hkv, head_dim, s);
  return ws.used + 256;
}

// Shared body of lsrm_select_blocks (k given: pooled here) and
// lsrm_select_blocks_pooled (pooled_k given: the fp32 block means of k).
static int select_blocks_impl(const void* q, const void* k, const float* pooled_k, int dtype,
                              int64_t n_tokens, int64_t hq, int64_t hkv, int64_t head_dim,
                              const int32_t* cu_seqblocks, int64_t batch,
                              const int32_t* cu_block_tokens, int64_t n_blocks, int64_t topk,
                              const int32_t* forced_blocks, int64_t n_forced, int force_self,
                              int32_t* topk_idx, int32_t* topk_compact, void* workspace,
                              size_t workspace_bytes, void* stream) {
  if (n_tokens < 0 || hq <= 0 || hkv <= 0 || head_dim <= 0 || batch <= 0 ||
      n_blocks < 0 || topk <= 0 || n_forced < 0 || !cu_seqblocks ||
      !cu_block_tokens || (n_forced > 0 && !forced_blocks) ||
      (n_tokens > 0 && (!q || !(k || pooled_k) || !topk_idx)) ||
      (n_blocks > 0 && !topk_compact))
    return LSRM_ERR_INVALID_ARG;
  if (hq % hkv != 0) return LSRM_ERR_INVALID_ARG;
  if (dtype < LSRM_F32 || dtype > LSRM_BF16) return LSRM_ERR_UNSUPPORTED;
  if (head_dim > SEL_MAXD || topk > SEL_MAXK || n_blocks > SEL_MAX_CAND)
    return LSRM_ERR_UNSUPPORTED;
  const size_t need = lsrm_select_blocks_workspace_size(n_tokens, n_blocks, hq,
                                                        hkv, head_dim);
  if (workspace_bytes < need || !workspace) return LSRM_ERR_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  if (n_blocks == 0) {  // every token lies outside the (empty) block list
    if (n_tokens > 0) {
      hipLaunchKernelGGL(uncovered_rows_kernel, dim3(ceil_div(n_tokens, 256), (unsigned)hkv),
                         dim3(256), 0, st, cu_block_tokens, n_blocks, n_tokens, (int)topk,
                         topk_idx);
      LSRM_CHECK_LAUNCH();
    }
    return LSRM_OK;
  }
  Carver ws{reinterpret_cast<char*>(align_up((size_t)workspace, 256)), 0,
            workspace_bytes - 256};
  SelectWs s;
  carve_select(ws, n_tokens, n_blocks, hq, hkv, head_dim, s);
  if (!ws.ok()) return LSRM_ERR_WORKSPACE;

  int rc = launch_block_mean_pool(q, dtype, n_tokens, hq * head_dim,
                                  cu_block_tokens, n_blocks, s.pq, LSRM_F32,
                                  s.partial, s.first, st);
  if (rc) return rc;
  const float* pk = pooled_k;
  if (!pk) {
    rc = launch_block_mean_pool(k, dtype, n_tokens, hkv * head_dim, cu_block_tokens, n_blocks,
                                s.pk, LSRM_F32, s.partial, s.first, st);
    if (rc) return rc;
    pk = s.pk;
  }
  const unsigned nt = (unsigned)ceil_div(n_blocks, SCORE_COLS);
  hipLaunchKernelGGL(score_kernel,
                     dim3(nt, (unsigned)ceil_div(n_blocks, SCORE_ROWS), (unsigned)hkv),
                     dim3(256), 0, st, s.pq, pk, n_blocks, (int)hq, (int)hkv,
                     (int)head_dim, s.scores, topk <= 64 ? s.keys : nullptr);
  LSRM_CHECK_LAUNCH();
  const unsigned rows4 = (unsigned)ceil_div(n_blocks * hkv, 4);
#define LSRM_TOPK_WAVE(M)                                                     \
  hipLaunchKernelGGL(topk_wave_kernel<M>, dim3(rows4), dim3(256), 0, st,      \
                     s.scores, n_blocks, cu_seqblocks, batch, cu_block_tokens, \
                     n_tokens, (int)hkv, (int)topk, forced_blocks,            \
                     (int)n_forced, force_self, topk_idx, topk_compact)
  if (n_blocks <= 64 * 4)
    LSRM_TOPK_WAVE(4);
  else if (n_blocks <= 64 * 8)
    LSRM_TOPK_WAVE(8);
  else if (n_blocks <= 64 * 16)
    LSRM_TOPK_WAVE(16);
  else if (n_blocks <= 64 * 32)
    LSRM_TOPK_WAVE(32);
  else if (bounded_rows(n_blocks) && topk <= 64) {
#define LSRM_TOPK_BOUND(NM)                                                               \
  hipLaunchKernelGGL(topk_bound_kernel<NM>, dim3((unsigned)n_blocks, (unsigned)hkv),     \
                     dim3(64), 0, st, s.scores, s.keys, (int)nt, n_blocks, cu_seqblocks,   \
                     batch, cu_block_tokens, n_tokens, (int)topk, forced_blocks,           \
                     (int)n_forced, force_self, topk_idx, topk_compact)
    if (nt * SCORE_CLASSES <= 64 * 12)
      LSRM_TOPK_BOUND(12);
    else if (nt * SCORE_CLASSES <= 64 * 20)
      LSRM_TOPK_BOUND(20);
    else
      LSRM_TOPK_BOUND(32);
#undef LSRM_TOPK_BOUND
  } else
    hipLaunchKernelGGL(topk_kernel, dim3((unsigned)n_blocks, (unsigned)hkv),
                       dim3(256), 0, st, s.scores, n_blocks, cu_seqblocks,
                       batch, cu_block_tokens, n_tokens, (int)topk,
                       forced_blocks, (int)n_forced, force_self, topk_idx,
                       topk_compact);
#undef LSRM_TOPK_WAVE
  LSRM_CHECK_LAUNCH();
  hipLaunchKernelGGL(uncovered_rows_kernel, dim3(ceil_div(n_tokens, 256), (unsigned)hkv),
                     dim3(256), 0, st, cu_block_tokens, n_blocks, n_tokens, (int)topk, topk_idx);
  LSRM_CHECK_LAUNCH();
  return LSRM_OK;
}

extern "C" int lsrm_select_blocks(const void* q, const void* k, int dtype, int64_t n_tokens,
                                  int64_t hq, int64_t hkv, int64_t head_dim,
                                  const int32_t* cu_seqblocks, int64_t batch,
                                  const int32_t* cu_block_tokens, int64_t n_blocks, int64_t topk,
                                  const int32_t* forced_blocks, int64_t n_forced, int force_self,
                                  int32_t* topk_idx, int32_t* topk_compact, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  if (n_tokens > 0 && !k) return LSRM_ERR_INVALID_ARG;
  return select_blocks_impl(q, k, nullptr, dtype, n_tokens, hq, hkv, head_dim, cu_seqblocks,
                            batch, cu_block_tokens, n_blocks, topk, forced_blocks, n_forced,
                            force_self, topk_idx, topk_compact, workspace, workspace_bytes,
                            stream);
}

extern "C" int lsrm_select_blocks_pooled(const void* q, const float* pooled_k, int dtype,
                                         int64_t n_tokens, int64_t hq, int64_t hkv,
                                         int64_t head_dim, const int32_t* cu_seqblocks,
                                         int64_t batch, const int32_t* cu_block_tokens,
                                         int64_t n_blocks, int64_t topk,
                                         const int32_t* forced_blocks, int64_t n_forced,
                                         int force_self, int32_t* topk_idx,
                                         int32_t* topk_compact, void* workspace,
                                         size_t workspace_bytes, void* stream) {
  if (n_blocks > 0 && !pooled_k) return LSRM_ERR_INVALID_ARG;
  return select_blocks_impl(q, nullptr, pooled_k, dtype, n_tokens, hq, hkv, head_dim,
                            cu_seqblocks, batch, cu_block_tokens, n_blocks, topk, forced_blocks,
                            n_forced, force_self, topk_idx, topk_compact, workspace,
                            workspace_bytes, stream);
}
