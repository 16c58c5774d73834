// The filter network through a table over the pair distance.
//
// W(d) and W'(d) of a CFConv block are functions of one number.  A batch has
// 10^5..10^7 pairs, the functions are smooth on the scale of the radial
// basis' spacing, so the network is evaluated once per node of a uniform grid
// over [0, rc] (mlcg_filter_table, fp32 MFMA throughout), the pairs' rows are
// interpolated from four nodes (cubic Lagrange, values and derivatives each
// from their own table), and the reverse of that interpolation gives the
// adjoints of the nodes, on which the filter backward then runs.  The grid
// spacing has 11 significant bits and the grid at most 2^13 nodes, so the node
// distances are exact in fp32; a pair's place between them comes from its
// distance in double.
//
// The pairs are ordered by their interpolation stencil once per call (a
// stable counting sort: mlcg_pair_bins), so that a wave reads a stencil's
// table rows once for all its pairs, and the reverse accumulates a stencil's
// rows in registers.  Every sum has a fixed order.
#include "common.h"
#include "filter_gate.h"

#include <hip/hip_fp16.h>

namespace {

constexpr int kF = 128;
constexpr int kSortWaves = 4;
constexpr int kSortThreads = 1024;  // the first kSortWaves waves walk the pairs, all clear and scan
constexpr int kSortScanWaves = kSortThreads / MLCG_WAVE;
constexpr int kSortMaxGroups = 256;
constexpr int kMaxKeys = 8192;
constexpr int kRev = 64;      // records of a run (table_reverse_kernel)
constexpr int kRevWaves = 8;  // runs of a workgroup

// Position of a pair in the grid, in cells: 14 integer and 18 fraction bits,
// from the distance in double.  A float distance is off by up to 1e-6 A at 20
// A, the largest single error of the pairwise filters (5.4e-7 of the weight
// gradients); the fraction here resolves 3e-8 A.  kPastCut: at or past the
// cutoff of a cosine envelope, where the filter is zero.
constexpr int kFracBits = 18;
constexpr uint32_t kPastCut = 0xffffffffu;

__device__ __forceinline__ uint32_t grid_position(double d, double inv_h) {
  const double u = d * inv_h * (double)(1 << kFracBits);
  return u < 4294967294.0 ? (uint32_t)u : 0xfffffffeu;
}

// Stencil of a position: nodes key .. key + 3, clamped to the grid.
__device__ __forceinline__ int stencil_key(uint32_t u, int nkeys) {
  const int b = (int)(u >> kFracBits) - 1;
  return b < 0 ? 0 : (b > nkeys - 1 ? nkeys - 1 : b);
}

// Cubic Lagrange weights from the stencil's first node; zero past the cutoff.
__device__ __forceinline__ void stencil_weights(uint32_t u, int key, float w[4]) {
  const float t0 = (float)(u - ((uint32_t)key << kFracBits)) * (1.0f / (1 << kFracBits));
  const float t1 = t0 - 1.0f, t2 = t0 - 2.0f, t3 = t0 - 3.0f;
  const float m = u != kPastCut ? 1.0f : 0.0f;
  const float a = t0 * t1 * m, b = t2 * t3 * m;
  w[0] = t1 * b * (-1.0f / 6.0f);
  w[1] = t0 * b * 0.5f;
  w[2] = a * t3 * -0.5f;
  w[3] = a * t2 * (1.0f / 6.0f);
}

__device__ __forceinline__ int64_t live_pairs(const int32_t* n_dev, int64_t cap) {
  const int64_t np = *n_dev;
  return np < cap ? np : cap;
}

// Counting sort of the pairs by key in three launches, 28 us for 217 k pairs (six
// times the time of its bytes: three short latency-bound kernels).  Each wave
// counts and places a contiguous range, so that the order is stable without
// atomics between waves.

// Pairs of wave `w` of block `blk`: [lo, hi), contiguous, whole waves of 64.
__device__ __forceinline__ void wave_range(int64_t np, int blk, int groups, int w, int64_t& lo,
                                           int64_t& hi) {
  const int64_t waves = (int64_t)groups * kSortWaves;
  const int64_t per = ((np + waves - 1) / waves + 63) / 64 * 64;
  lo = ((int64_t)blk * kSortWaves + w) * per;
  hi = lo + per < np ? lo + per : np;
}

// Counts of every key among the block's pairs, and the pair distances.
__global__ __launch_bounds__(kSortThreads) void pair_key_count_kernel(
    const float* __restrict__ pos, const int32_t* __restrict__ pi,
    const int32_t* __restrict__ pj, const int32_t* __restrict__ n_dev, int64_t cap, double inv_h,
    int nkeys, float cut, float* __restrict__ dist, uint32_t* __restrict__ where,
    uint32_t* __restrict__ hist) {
  extern __shared__ uint32_t cnt[];  // [nkeys]
  for (int b = threadIdx.x; b < nkeys; b += kSortThreads) cnt[b] = 0u;
  __syncthreads();
  const int64_t np = live_pairs(n_dev, cap);
  int64_t lo, hi;
  wave_range(np, blockIdx.x, gridDim.x, threadIdx.x / MLCG_WAVE, lo, hi);
  if (threadIdx.x >= kSortWaves * MLCG_WAVE) hi = lo;
#pragma unroll 4
  for (int64_t p = lo + mlcg_lane(); p < hi; p += MLCG_WAVE) {
    const int64_t i = pi[p], j = pj[p];
    const float xi = pos[3 * i], yi = pos[3 * i + 1], zi = pos[3 * i + 2];
    const float xj = pos[3 * j], yj = pos[3 * j + 1], zj = pos[3 * j + 2];
    const float dx = xj - xi, dy = yj - yi, dz = zj - zi;
    // the filter forward's own fma order, so both routes have the same distances
    const float d = sqrtf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
    dist[p] = d;
    const double ex = (double)xj - xi, ey = (double)yj - yi, ez = (double)zj - zi;
    const uint32_t u =
        d < cut ? grid_position(sqrt(ex * ex + ey * ey + ez * ez), inv_h) : kPastCut;
    where[p] = u;
    atomicAdd(&cnt[stencil_key(u, nkeys)], 1u);
  }
  __syncthreads();
  uint32_t* h = hist + (int64_t)blockIdx.x * nkeys;
  for (int b = threadIdx.x; b < nkeys; b += kSortThreads) h[b] = cnt[b];
}

// Per key: the exclusive prefix of the blocks' counts (in place) and the total.
__global__ __launch_bounds__(256) void pair_key_offsets_kernel(uint32_t* __restrict__ hist,
                                                               int groups, int nkeys,
                                                               uint32_t* __restrict__ totals) {
  constexpr int kRows = kSortMaxGroups / 4;
  __shared__ uint32_t part[4][MLCG_WAVE];
  const int l = mlcg_lane(), s = threadIdx.x / MLCG_WAVE;
  const int b = blockIdx.x * MLCG_WAVE + l;
  const int first = s * kRows;
  uint32_t v[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r)
    v[r] = b < nkeys && first + r < groups ? hist[(int64_t)(first + r) * nkeys + b] : 0u;
  uint32_t sum = 0u;
#pragma unroll
  for (int r = 0; r < kRows; ++r) sum += v[r];
  part[s][l] = sum;
  __syncthreads();
  uint32_t run = 0u;
  for (int k = 0; k < s; ++k) run += part[k][l];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    if (b < nkeys && first + r < groups) hist[(int64_t)(first + r) * nkeys + b] = run;
    run += v[r];
  }
  if (s == 3 && b < nkeys) totals[b] = run;
}

// Writes the records {pair, i, j, grid position} in key order, stable in the
// pair index, and the keys' first positions.
__global__ __launch_bounds__(kSortThreads) void pair_key_scatter_kernel(
    const int32_t* __restrict__ pi, const int32_t* __restrict__ pj,
    const int32_t* __restrict__ n_dev, int64_t cap, int nkeys,
    const uint32_t* __restrict__ where, const uint32_t* __restrict__ hist,
    const uint32_t* __restrict__ totals, int32_t* __restrict__ start,
    int32_t* __restrict__ run_start, int4* __restrict__ recs) {
  extern __shared__ uint32_t off[];  // [kSortWaves][nkeys]
  __shared__ uint32_t wsum[2][kSortScanWaves];
  const int l = mlcg_lane(), w = threadIdx.x / MLCG_WAVE;
  for (int b = threadIdx.x; b < kSortWaves * nkeys; b += kSortThreads) off[b] = 0u;
  __syncthreads();
  const int64_t np = live_pairs(n_dev, cap);
  int64_t lo, hi;
  wave_range(np, blockIdx.x, gridDim.x, w, lo, hi);
  if (w >= kSortWaves) hi = lo;
  uint32_t* mine = off + (w < kSortWaves ? w : 0) * nkeys;
#pragma unroll 4
  for (int64_t p = lo + l; p < hi; p += MLCG_WAVE)
    atomicAdd(&mine[stencil_key(where[p], nkeys)], 1u);
  // first record and first run of every key: exclusive scans of the totals and
  // of the runs (of at most kRev records) they make, each thread over its own
  // stretch of consecutive keys
  const int per = (nkeys + kSortThreads - 1) / kSortThreads;
  const int k0 = threadIdx.x * per;
  uint32_t sum = 0u, runs = 0u;
  for (int b = k0; b < k0 + per && b < nkeys; ++b) {
    const uint32_t t = totals[b];
    sum += t;
    runs += (t + kRev - 1) / kRev;
  }
  uint32_t incl = sum, rincl = runs;
#pragma unroll
  for (int o = 1; o < MLCG_WAVE; o <<= 1) {
    const uint32_t up = __shfl_up(incl, o, MLCG_WAVE), rup = __shfl_up(rincl, o, MLCG_WAVE);
    if (l >= o) {
      incl += up;
      rincl += rup;
    }
  }
  if (l == MLCG_WAVE - 1) {
    wsum[0][w] = incl;
    wsum[1][w] = rincl;
  }
  __syncthreads();  // also: every wave's counts are complete
  uint32_t run = incl - sum, first_run = rincl - runs;
  for (int k = 0; k < w; ++k) {
    run += wsum[0][k];
    first_run += wsum[1][k];
  }
  for (int b = k0; b < k0 + per && b < nkeys; ++b) {
    const uint32_t t = totals[b];
    if (blockIdx.x == 0) {
      start[b] = (int32_t)run;
      run_start[b] = (int32_t)first_run;
    }
    uint32_t at = run + hist[(int64_t)blockIdx.x * nkeys + b];
#pragma unroll
    for (int k = 0; k < kSortWaves; ++k) {
      const uint32_t c = off[k * nkeys + b];
      off[k * nkeys + b] = at;
      at += c;
    }
    run += t;
    first_run += (t + kRev - 1) / kRev;
    if (blockIdx.x == 0 && b == nkeys - 1) {
      start[nkeys] = (int32_t)run;
      run_start[nkeys] = (int32_t)first_run;
    }
  }
  __syncthreads();
  for (int64_t p0 = lo; p0 < hi; p0 += MLCG_WAVE) {
    const int64_t p = p0 + l;
    const bool on = p < hi;
    const uint32_t u = on ? where[p] : 0u;
    const int key = stencil_key(u, nkeys);
    // lanes of this wave with the same key
    unsigned long long same = __ballot(on);
#pragma unroll
    for (int bit = 0; bit < 13; ++bit) {
      const bool one = (key >> bit) & 1;
      const unsigned long long m = __ballot(one);
      same &= one ? m : ~m;
    }
    if (on) {
      const int rank = __popcll(same & ((1ull << l) - 1ull));
      const uint32_t base = *(volatile uint32_t*)&mine[key];
      const int4 r = int4{(int)p, pi[p], pj[p], (int)u};
      recs[base + rank] = r;
      // the first lane of the group moves the counter past it, after every
      // lane of the group has read it (one wave: LDS operations in program
      // order; only this wave uses this counter)
      if (rank == 0) *(volatile uint32_t*)&mine[key] = base + (uint32_t)__popcll(same);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// ---------------------------------------------------------------------------
// Check of a table (see filter_gate.h).  Table of block k: [4][nodes + 1][128]
// = W, W', H, H' at d = 0, h, .., (nodes - 1) h and, last, at rc.
constexpr int kCheckRows = 32;  // odd nodes per workgroup

__device__ __forceinline__ unsigned wave_umax(unsigned v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned u = __shfl_xor(v, o, MLCG_WAVE);
    v = v > u ? v : u;
  }
  return v;
}

__device__ __forceinline__ unsigned abs_bits(float x) { return __float_as_uint(fabsf(x)); }

__global__ __launch_bounds__(256) void table_check_kernel(const float* __restrict__ tables,
                                                          int nodes, float t_rc,
                                                          unsigned* __restrict__ gates) {
  const int64_t plane = (int64_t)(nodes + 1) * kF;
  const int which = blockIdx.y & 3, blk = blockIdx.y >> 2;
  const float* T = tables + ((int64_t)blk * 4 + which) * plane;
  const int f = threadIdx.x & (kF - 1);
  const int half = threadIdx.x / kF;
  const int last_even = (nodes - 1) & ~1;
  unsigned err = 0u, big = 0u;
  const int o0 = blockIdx.x * kCheckRows;
#pragma unroll 4
  for (int r = half; r < kCheckRows; r += 2) {
    const int k = 2 * (o0 + r) + 1;  // odd node
    if (k >= last_even) break;
    int base = k - 3;
    base = base < 0 ? 0 : (base > last_even - 6 ? last_even - 6 : base);
    const float t = 0.5f * (float)(k - base);
    const float t1 = t - 1.0f, t2 = t - 2.0f, t3 = t - 3.0f;
    const float* c = T + (int64_t)base * kF + f;
    const float est = c[0] * (t1 * t2 * t3 * (-1.0f / 6.0f)) + c[2 * kF] * (t * t2 * t3 * 0.5f) +
                      c[4 * kF] * (t * t1 * t3 * -0.5f) + c[6 * kF] * (t * t1 * t2 * (1.0f / 6.0f));
    const float v = T[(int64_t)k * kF + f];
    const unsigned e = abs_bits(v - est), a = abs_bits(v);
    err = err > e ? err : e;
    big = big > a ? big : a;
  }
  if (blockIdx.x == 0 && half == 0) {
    // the cutoff distance itself, extrapolated over the last, partial cell
    const float t = t_rc, t1 = t - 1.0f, t2 = t - 2.0f, t3 = t - 3.0f;
    const float* c = T + (int64_t)(nodes - 4) * kF + f;
    const float est = c[0] * (t1 * t2 * t3 * (-1.0f / 6.0f)) + c[kF] * (t * t2 * t3 * 0.5f) +
                      c[2 * kF] * (t * t1 * t3 * -0.5f) + c[3 * kF] * (t * t1 * t2 * (1.0f / 6.0f));
    const unsigned e = abs_bits(c[4 * kF] - est);
    err = err > e ? err : e;
  }
  __shared__ unsigned red[2][4];
  err = wave_umax(err);
  big = wave_umax(big);
  if (mlcg_lane() == 0) {
    red[0][threadIdx.x / MLCG_WAVE] = err;
    red[1][threadIdx.x / MLCG_WAVE] = big;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const unsigned* r = red[threadIdx.x];
    const unsigned a = r[0] > r[1] ? r[0] : r[1], b = r[2] > r[3] ? r[2] : r[3];
    atomicMax(gates + blk * kGateWords + 4 * threadIdx.x + which, a > b ? a : b);
  }
}

// ---------------------------------------------------------------------------
// W, W' of the pairs from the table: a half-wave takes kSeg records in key
// order, keeps the stencil's rows in registers and writes whole rows.
constexpr int kSeg = 32;

template <typename T>
__device__ __forceinline__ void store_row4(T* row, int f, float4 v);
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef _Float16 halfx4_t __attribute__((ext_vector_type(4)));
template <>
__device__ __forceinline__ void store_row4<float>(float* row, int f, float4 v) {
  __builtin_nontemporal_store(floatx4_t{v.x, v.y, v.z, v.w},
                              reinterpret_cast<floatx4_t*>(row + f));
}
template <>
__device__ __forceinline__ void store_row4<__half>(__half* row, int f, float4 v) {
  __builtin_nontemporal_store(
      halfx4_t{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w},
      reinterpret_cast<halfx4_t*>(row + f));
}

__device__ __forceinline__ float4 lerp4(const float4* r, const float w[4]) {
  return float4{r[0].x * w[0] + r[1].x * w[1] + r[2].x * w[2] + r[3].x * w[3],
                r[0].y * w[0] + r[1].y * w[1] + r[2].y * w[2] + r[3].y * w[3],
                r[0].z * w[0] + r[1].z * w[1] + r[2].z * w[2] + r[3].z * w[3],
                r[0].w * w[0] + r[1].w * w[1] + r[2].w * w[2] + r[3].w * w[3]};
}

// Rows of the pairs: a wave reads a stencil's eight table rows once for all its
// pairs, so the launch is bound by the rows it writes: 217 k pairs, three blocks
// 133 us, 5.2 TB/s, where the network pair by pair takes 87-92 us a block; 3.0 M
// pairs in fp16 866 us, 5.6 TB/s, against 1447.
constexpr int kMaxBlocks = 8;  // blocks of a launch (blockIdx.y)
struct RowsBatch {
  void *W[kMaxBlocks], *Wd[kMaxBlocks];
};

template <typename T>
__global__ __launch_bounds__(256) void table_rows_kernel(
    const int4* __restrict__ recs, const int32_t* __restrict__ n_dev, int64_t cap, int nkeys,
    const float* __restrict__ tables, int64_t plane,
    const unsigned* __restrict__ gates, RowsBatch batch) {
  const int blk = blockIdx.y;
  if (!filter_table_serves(gates + blk * kGateWords)) return;
  const float* __restrict__ table = tables + (int64_t)blk * 4 * plane;
  T* __restrict__ W = static_cast<T*>(batch.W[blk]);
  T* __restrict__ Wd = static_cast<T*>(batch.Wd[blk]);
  const int64_t np = live_pairs(n_dev, cap);
  const int l = mlcg_lane(), hl = l & 31, hb = l & 32;
  const int64_t s0 = ((int64_t)blockIdx.x * 8 + (threadIdx.x >> 5)) * kSeg;
  if (s0 >= np) return;
  const int n = (int)(np - s0 < kSeg ? np - s0 : kSeg);
  const int4 r = recs[s0 + (hl < n ? hl : n - 1)];
  const int f = 4 * hl;
  float4 tw[4], td[4];
  int cur = -1;
  for (int k = 0; k < n; ++k) {
    const int p = __shfl(r.x, hb | k, MLCG_WAVE);
    const uint32_t u = (uint32_t)__shfl(r.w, hb | k, MLCG_WAVE);
    const int key = stencil_key(u, nkeys);
    if (key != cur) {
      const float* c = table + (int64_t)key * kF + f;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        tw[m] = *reinterpret_cast<const float4*>(c + m * kF);
        td[m] = *reinterpret_cast<const float4*>(c + plane + m * kF);
      }
      cur = key;
    }
    float w[4];
    stencil_weights(u, key, w);
    store_row4(W + (int64_t)p * kF, f, lerp4(tw, w));
    store_row4(Wd + (int64_t)p * kF, f, lerp4(td, w));
  }
}

// ---------------------------------------------------------------------------
// Reverse of the interpolation.  Pair adjoints formed from node vectors,
//   Wbar_p  = g2_i y_j + g2_j y_i + g1_i yd_j + g1_j yd_i
//   Wdbar_p = dd_p (g1_i y_j + g1_j y_i)
// are accumulated with the interpolation weights into the stencil's four
// nodes.  A wave takes one run: up to 64 records of one key, two features a
// lane, and writes one [8][128] block to the run's slot.
//
// Bound by the node rows (4 KiB a pair).  A key of R runs deals its records out
// in turn, so that every wave sweeps the batch from its first frame to its
// last: the waves of an XCD are in about the same frames at the same time and
// find some of their rows in its L2 (219 k pairs of 512 x 35 beads 22 %, 879 k of
// 512 x 100 beads 9 %).  The rest comes from the memory-side cache, 6.4 and 7.3
// TB/s: 105 and 450 us a block and 6 and 10 for table_combine_kernel, where the
// pair-by-pair backward takes 241-254 us at the smaller size.
//
// Bonded pairs share one distance, so a single key can hold a tenth of the
// pairs: a workgroup whose runs all have one key adds its waves' blocks first
// and writes one, to its first run's slot.
__device__ __forceinline__ float2 ld2(const float* __restrict__ a, int row, int f) {
  return *reinterpret_cast<const float2*>(a + (int64_t)row * kF + f);
}
__device__ __forceinline__ float2 cross2(float2 ai, float2 bj, float2 aj, float2 bi) {
  return float2{ai.x * bj.x + aj.x * bi.x, ai.y * bj.y + aj.y * bi.y};
}

// Key of run `run`: the last key whose first run is not past it (two rounds of
// 64 and up to 128 candidates; keys without records share their successor's
// first run and are passed over).
__device__ __forceinline__ int run_key(const int32_t* __restrict__ run_start, int nkeys,
                                       int run) {
  const int l = mlcg_lane();
  const int step = (nkeys + MLCG_WAVE - 1) / MLCG_WAVE;
  const int a = l * step;
  const unsigned long long m = __ballot(a < nkeys && run_start[a < nkeys ? a : 0] <= run);
  const int base = (__popcll(m) - 1) * step;
  int key = base;
  for (int x = 0; x < step; x += MLCG_WAVE) {
    const int b = base + x + l;
    const bool in = x + l < step && b < nkeys;
    const unsigned long long c = __ballot(in && run_start[in ? b : 0] <= run);
    key += __popcll(c);
  }
  return key - 1;
}

template <bool kTan, bool kYd>
__global__ __launch_bounds__(kRevWaves * MLCG_WAVE) void table_reverse_kernel(
    const int4* __restrict__ recs, const int32_t* __restrict__ start,
    const int32_t* __restrict__ run_start, int nkeys, const float* __restrict__ g2,
    const float* __restrict__ y, const float* __restrict__ g1, const float* __restrict__ yd,
    const float* __restrict__ dd, FilterGate gate, float* __restrict__ slots) {
  if (gate_closed(gate)) return;
  __shared__ __align__(16) float2 fold[kRevWaves][8][MLCG_WAVE];
  const int l = mlcg_lane();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int run0 = blockIdx.x * kRevWaves;
  const int run = run0 + wave;
  const int n_runs = run_start[nkeys];
  if (run >= n_runs) return;
  const int key = __builtin_amdgcn_readfirstlane(run_key(run_start, nkeys, run));
  const int first = run_start[key], parts = run_start[key + 1] - first;
  // the whole workgroup in one key (then none of its waves has returned above)
  const bool one_key = first <= run0 && first + parts >= run0 + kRevWaves;
  const int s0 = start[key] + (run - first);
  const int n = __builtin_amdgcn_readfirstlane((start[key + 1] - s0 + parts - 1) / parts);
  const int4 r = recs[s0 + (l < n ? l : n - 1) * parts];
  const float ddl = kTan ? dd[r.x] : 0.0f;
  float w_l[4];
  stencil_weights((uint32_t)r.w, key, w_l);
  const int f = 2 * l;
  float2 aw[4], ad[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) aw[m] = ad[m] = float2{0.f, 0.f};
  constexpr int kU = 4;  // records in flight
  for (int k = 0; k < n; k += kU) {
    float2 a[kU], b[kU], c[kU], e[kU], u[kU], v[kU], s[kU], t[kU];
#pragma unroll
    for (int x = 0; x < kU; ++x) {
      const int kk = k + x < n ? k + x : n - 1;
      const int i = __builtin_amdgcn_readlane(r.y, kk), j = __builtin_amdgcn_readlane(r.z, kk);
      a[x] = ld2(g2, i, f);
      b[x] = ld2(y, j, f);
      c[x] = ld2(g2, j, f);
      e[x] = ld2(y, i, f);
      if (kTan) {
        u[x] = ld2(g1, i, f);
        v[x] = ld2(g1, j, f);
      }
      if (kYd) {
        s[x] = ld2(yd, i, f);
        t[x] = ld2(yd, j, f);
      }
    }
#pragma unroll
    for (int x = 0; x < kU; ++x) {
      if (k + x < n) {  // uniform
        const int kk = k + x;
        float2 wb = cross2(a[x], b[x], c[x], e[x]);
        if (kYd) {
          const float2 q = cross2(u[x], t[x], v[x], s[x]);
          wb.x += q.x;
          wb.y += q.y;
        }
        float2 wdb = float2{0.f, 0.f};
        if (kTan) {
          const float dv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ddl), kk));
          const float2 q = cross2(u[x], b[x], v[x], e[x]);
          wdb = float2{dv * q.x, dv * q.y};
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const float wm =
              __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w_l[m]), kk));
          aw[m].x += wm * wb.x;
          aw[m].y += wm * wb.y;
          if (kTan) {
            ad[m].x += wm * wdb.x;
            ad[m].y += wm * wdb.y;
          }
        }
      }
    }
  }
  constexpr int kRows = kTan ? 8 : 4;
  if (!one_key) {
    float* o = slots + (int64_t)run * (8 * kF) + f;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      *reinterpret_cast<float2*>(o + m * kF) = aw[m];
      if (kTan) *reinterpret_cast<float2*>(o + (4 + m) * kF) = ad[m];
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    fold[wave][m][l] = aw[m];
    if (kTan) fold[wave][4 + m][l] = ad[m];
  }
  __syncthreads();
  for (int q = wave; q < kRows; q += kRevWaves) {
    float2 v = fold[0][q][l];
#pragma unroll
    for (int k = 1; k < kRevWaves; ++k) {
      const float2 u = fold[k][q][l];
      v.x += u.x;
      v.y += u.y;
    }
    *reinterpret_cast<float2*>(slots + (int64_t)run0 * (8 * kF) + q * kF + f) = v;
  }
}

// Node adjoints: node m takes row m - key of every slot of the keys m - 3 .. m.
// One workgroup per node, wave w the key m - 3 + w (its slots in order, four
// rows in flight), then the waves' sums in key order.
__device__ __forceinline__ void add_slots(const float* __restrict__ o, int first, int step,
                                          int count, bool tan, float2& w, float2& d) {
  for (int r = 0; r < count; r += 4) {
    float2 u[4], z[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int k = r + x < count ? r + x : count - 1;
      const float* p = o + (int64_t)(first + k * step) * (8 * kF);
      u[x] = *reinterpret_cast<const float2*>(p);
      z[x] = tan ? *reinterpret_cast<const float2*>(p + 4 * kF) : float2{0.f, 0.f};
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if (r + x < count) {
        w.x += u[x].x;
        w.y += u[x].y;
        d.x += z[x].x;
        d.y += z[x].y;
      }
    }
  }
}

// The nodes as pairs {0, m} of the positions (m h, 0, 0), for the kernels that
// then run on them.  Written here, by the first block whatever its gate: as
// buffers of the call they live as long as what reads them, a recorded graph
// included, without a launch of their own.
struct NodePairs {
  float h;
  float *pos, *dist;  // [nodes, 3], [nodes]
  int32_t *ij, *count;  // [2, nodes], [1]
};

template <bool kTan>
__global__ __launch_bounds__(256) void table_combine_kernel(
    const int32_t* __restrict__ run_start, int nkeys, const float* __restrict__ block_slots,
    int64_t slot_stride, int nodes, const unsigned* __restrict__ gates,
    float* __restrict__ block_wbar, float* __restrict__ block_wdbar, NodePairs np) {
  const int blk = blockIdx.y;
  if (blk == 0 && threadIdx.x == 0) {
    const int m = blockIdx.x;
    const float d = (float)m * np.h;  // exact
    np.pos[3 * m] = d;
    np.pos[3 * m + 1] = np.pos[3 * m + 2] = 0.0f;
    np.dist[m] = d;
    np.ij[m] = 0;
    np.ij[nodes + m] = m;
    if (m == 0) *np.count = nodes;
  }
  if (!filter_table_serves(gates + blk * kGateWords)) return;
  const float* __restrict__ slots = block_slots + blk * slot_stride;
  float* __restrict__ wbar = block_wbar + (int64_t)blk * nodes * kF;
  float* __restrict__ wdbar = block_wdbar + (int64_t)blk * nodes * kF;
  __shared__ float2 part[4][2][MLCG_WAVE];
  const int m = blockIdx.x, l = mlcg_lane();
  const int x = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int key = m - 3 + x;
  float2 w = float2{0.f, 0.f}, d = float2{0.f, 0.f};
  if (key >= 0 && key < nkeys) {
    const int a = run_start[key], e = run_start[key + 1];
    const float* o = slots + (3 - x) * kF + 2 * l;
    // workgroups of the reverse that lie inside the key wrote one slot
    const int g0 = (a + kRevWaves - 1) / kRevWaves, g1 = e / kRevWaves;
    if (g0 < g1) {
      add_slots(o, a, 1, g0 * kRevWaves - a, kTan, w, d);
      add_slots(o, g0 * kRevWaves, kRevWaves, g1 - g0, kTan, w, d);
      add_slots(o, g1 * kRevWaves, 1, e - g1 * kRevWaves, kTan, w, d);
    } else {
      add_slots(o, a, 1, e - a, kTan, w, d);
    }
  }
  part[x][0][l] = w;
  part[x][1][l] = d;
  __syncthreads();
  if (threadIdx.x < 2 * MLCG_WAVE) {
    const int h = threadIdx.x >> 6;
    float2 v = part[0][h][l];
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      v.x += part[k][h][l].x;
      v.y += part[k][h][l].y;
    }
    *reinterpret_cast<float2*>((h ? wdbar : wbar) + (int64_t)m * kF + 2 * l) = v;
  }
}

int sort_groups(int64_t cap) {
  const int64_t g = (cap + 1023) / 1024;
  return (int)(g < 1 ? 1 : (g < kSortMaxGroups ? g : kSortMaxGroups));
}

void allow_sort_lds_once() {
  static bool done[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64 || done[dev]) return;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(pair_key_scatter_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            kSortWaves * kMaxKeys * 4);
  done[dev] = true;
}

bool table_shape_ok(int nodes) { return nodes >= 16 && nodes <= kMaxKeys; }

}  // namespace

extern "C" int64_t mlcg_pair_bins_workspace_ints(int64_t max_pairs, int nodes) {
  if (max_pairs < 0 || !table_shape_ok(nodes)) return -1;
  return (int64_t)(sort_groups(max_pairs) + 1) * (nodes - 3) + max_pairs;
}

extern "C" int mlcg_pair_bins(const float* pos, const int32_t* pair_ij, int64_t pair_stride,
                              const int32_t* n_pairs_dev, int64_t max_pairs, float h,
                              int nodes, float cut, float* dist, int32_t* start, int32_t* run_start,
                              int32_t* records,
                              int32_t* workspace, int64_t workspace_ints, void* stream) {
  MLCG_REQUIRE(max_pairs >= 0 && max_pairs < (1LL << 31) && pair_stride >= max_pairs);
  MLCG_REQUIRE(table_shape_ok(nodes) && h > 0.0f);
  const double inv_h = 1.0 / (double)h;
  MLCG_REQUIRE(pos && pair_ij && n_pairs_dev && dist && start && run_start && records &&
               workspace);
  const int nkeys = nodes - 3;
  const int groups = sort_groups(max_pairs);
  MLCG_REQUIRE(workspace_ints >= (int64_t)(groups + 1) * nkeys + max_pairs);
  uint32_t* totals = reinterpret_cast<uint32_t*>(workspace);
  uint32_t* hist = totals + nkeys;
  uint32_t* where = hist + (int64_t)groups * nkeys;
  hipStream_t s = mlcg_stream(stream);
  allow_sort_lds_once();
  hipLaunchKernelGGL(pair_key_count_kernel, dim3(groups), dim3(kSortThreads),
                     sizeof(uint32_t) * nkeys, s, pos, pair_ij, pair_ij + pair_stride,
                     n_pairs_dev, max_pairs, inv_h, nkeys, cut, dist, where, hist);
  hipLaunchKernelGGL(pair_key_offsets_kernel, dim3(mlcg_div_up(nkeys, MLCG_WAVE)), dim3(256), 0,
                     s, hist, groups, nkeys, totals);
  hipLaunchKernelGGL(pair_key_scatter_kernel, dim3(groups), dim3(kSortThreads),
                     sizeof(uint32_t) * kSortWaves * nkeys, s, pair_ij, pair_ij + pair_stride,
                     n_pairs_dev, max_pairs, nkeys, where, hist, totals, start, run_start,
                     reinterpret_cast<int4*>(records));
  return mlcg_launch_status();
}

extern "C" int mlcg_filter_table_check(const float* tables, int num_blocks, int nodes,
                                       float h, float rc, uint32_t* gates, void* stream) {
  MLCG_REQUIRE(table_shape_ok(nodes) && num_blocks >= 1 && tables && gates);
  const float t_rc = (rc - (float)(nodes - 4) * h) / h;
  hipLaunchKernelGGL(table_check_kernel, dim3(mlcg_div_up(nodes / 2, kCheckRows), 4 * num_blocks),
                     dim3(256), 0, mlcg_stream(stream), tables, nodes, t_rc, gates);
  return mlcg_launch_status();
}

extern "C" int mlcg_filter_table_rows(const int32_t* records, const int32_t* n_pairs_dev,
                                      int64_t max_pairs, int nodes, const float* tables,
                                      const uint32_t* gates, int num_blocks, int f16,
                                      void* const* outputs, void* stream) {
  MLCG_REQUIRE(table_shape_ok(nodes) && max_pairs >= 0 && num_blocks >= 1);
  if (max_pairs == 0) return MLCG_OK;
  MLCG_REQUIRE(records && n_pairs_dev && tables && gates && outputs);
  const int64_t plane = (int64_t)(nodes + 1) * kF;
  const int4* recs = reinterpret_cast<const int4*>(records);
  for (int first = 0; first < num_blocks; first += kMaxBlocks) {
    const int n = num_blocks - first < kMaxBlocks ? num_blocks - first : kMaxBlocks;
    RowsBatch batch = {};
    for (int k = 0; k < n; ++k) {
      batch.W[k] = outputs[2 * (first + k)];
      batch.Wd[k] = outputs[2 * (first + k) + 1];
      MLCG_REQUIRE(batch.W[k] && batch.Wd[k]);
    }
    const dim3 grid(mlcg_div_up(max_pairs, 8 * kSeg), n);
    const float* t = tables + (int64_t)first * 4 * plane;
    const uint32_t* g = gates + first * kGateWords;
    if (f16)
      hipLaunchKernelGGL((table_rows_kernel<__half>), grid, dim3(256), 0, mlcg_stream(stream),
                         recs, n_pairs_dev, max_pairs, nodes - 3, t, plane, g,
                         batch);
    else
      hipLaunchKernelGGL((table_rows_kernel<float>), grid, dim3(256), 0, mlcg_stream(stream),
                         recs, n_pairs_dev, max_pairs, nodes - 3, t, plane, g,
                         batch);
  }
  return mlcg_launch_status();
}

extern "C" int64_t mlcg_filter_table_reverse_workspace_floats(int64_t max_pairs, int nodes) {
  if (max_pairs < 0 || !table_shape_ok(nodes)) return -1;
  return ((max_pairs + kRev - 1) / kRev + nodes) * (8 * kF);
}

extern "C" int mlcg_filter_table_reverse(const int32_t* records, const int32_t* start,
                                         const int32_t* run_start, int64_t max_pairs, int nodes,
                                         const float* gagg2,
                                         const float* y, const float* gagg1, const float* ydot,
                                         const float* ddot, const uint32_t* gate, float* slots,
                                         int64_t slot_floats, void* stream) {
  MLCG_REQUIRE(table_shape_ok(nodes) && max_pairs >= 0);
  MLCG_REQUIRE(records && start && run_start && gagg2 && y && gate && slots);
  MLCG_REQUIRE(!gagg1 || ddot);
  MLCG_REQUIRE(slot_floats >= mlcg_filter_table_reverse_workspace_floats(max_pairs, nodes));
  const FilterGate g{gate, 1};
  const int nkeys = nodes - 3;
  const int4* recs = reinterpret_cast<const int4*>(records);
  hipStream_t s = mlcg_stream(stream);
  // every key may leave one run partly filled
  const dim3 grid(mlcg_div_up((max_pairs + kRev - 1) / kRev + nkeys, kRevWaves));
#define MLCG_REV(T, Y)                                                                      \
  hipLaunchKernelGGL((table_reverse_kernel<T, Y>), grid, dim3(kRevWaves * MLCG_WAVE), 0, s, \
                     recs, start, run_start, nkeys, gagg2, y, gagg1, ydot, ddot, g, slots)
  if (gagg1 && ydot)
    MLCG_REV(true, true);
  else if (gagg1)
    MLCG_REV(true, false);
  else
    MLCG_REV(false, false);
#undef MLCG_REV
  return mlcg_launch_status();
}

extern "C" int mlcg_filter_table_combine(const int32_t* run_start, int64_t max_pairs, int nodes,
                                         int tangent, const float* slots, int num_blocks,
                                         const uint32_t* gates, float* wbar, float* wdbar,
                                         float h, float* node_pos, float* node_dist,
                                         int32_t* node_pair_ij, int32_t* node_count,
                                         void* stream) {
  MLCG_REQUIRE(table_shape_ok(nodes) && max_pairs >= 0 && num_blocks >= 1);
  MLCG_REQUIRE(run_start && slots && gates && wbar && wdbar);
  MLCG_REQUIRE(node_pos && node_dist && node_pair_ij && node_count);
  const NodePairs np{h, node_pos, node_dist, node_pair_ij, node_count};
  const int64_t stride = mlcg_filter_table_reverse_workspace_floats(max_pairs, nodes);
  const dim3 grid(nodes, num_blocks);
  if (tangent)
    hipLaunchKernelGGL((table_combine_kernel<true>), grid, dim3(256), 0, mlcg_stream(stream),
                       run_start, nodes - 3, slots, stride, nodes, gates, wbar, wdbar, np);
  else
    hipLaunchKernelGGL((table_combine_kernel<false>), grid, dim3(256), 0, mlcg_stream(stream),
                       run_start, nodes - 3, slots, stride, nodes, gates, wbar, wdbar, np);
  return mlcg_launch_status();
}
