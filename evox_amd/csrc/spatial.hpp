// Rows in spatial order: leaves of 64 neighbouring slots with their bounding boxes.
//
// A row's cell is its quantile in every objective, and the rows are put together cell by cell along the Z-order curve (the
// bits of the quantiles interleaved), so that the 64 rows of a leaf lie close together in every objective.  A leaf's low
// corner -- the smallest value per objective among its rows -- then rules whole leaves out at once: no row of a leaf whose
// low corner exceeds a row in some objective dominates that row.  A dominator has no larger quantile in any objective, so
// its cell comes no later on the curve (at the first interleaved bit that differs it has the 0): nothing behind the end of a
// row's own cell can dominate it, and the leaves nearest below are the likeliest.
#pragma once

#include "common.hpp"
#include "deal.hpp"
#include "order.hpp"

namespace evx {

constexpr int kLeafRows = 64;
constexpr int kGroupLeaves = 64;         // leaves under one box of the second level (4096 rows)
constexpr int kSpatialSamples = 256;     // rows whose values cut an objective into quantiles
constexpr int kSpatialObjectives = 16;   // the most objectives that take this way

// Boxes of a population of up to `rows` slots: leaves and groups, as rows of a structure of arrays.
__host__ __device__ inline int64_t spatial_leaves(int64_t rows) { return (rows + kLeafRows - 1) / kLeafRows; }
__host__ __device__ inline int64_t spatial_leaf_stride(int64_t rows) { return (spatial_leaves(rows) + kGroupLeaves - 1) / kGroupLeaves * kGroupLeaves; }
__host__ __device__ inline int64_t spatial_group_stride(int64_t rows) { return (spatial_leaf_stride(rows) / kGroupLeaves + 63) / 64 * 64; }

// The workgroup's table of ascending sample values of every objective (kSpatialSamples of them, as ordered keys): each
// workgroup ranks the same samples by counting, 1.2 us an objective per 256 threads, less than a launch of its own would cost.
// The low eight bits of a sample give way to its thread, which makes the samples distinct: one comparison each, and any
// ascending values will do for a table.
template <int M>
__device__ inline void spatial_quantiles(const float* __restrict__ xs, int npad, int n, uint32_t* table) {
  static_assert(kSpatialSamples == 256, "one sample per thread, eight bits to tell them apart");
  __shared__ __attribute__((aligned(16))) uint32_t sample[M][kSpatialSamples];
  // (each 256 threads of a larger workgroup take the next objective)
  const int t = threadIdx.x & (kSpatialSamples - 1), first = threadIdx.x / kSpatialSamples, step = blockDim.x / kSpatialSamples;
  const int i = (int)((int64_t)t * n / kSpatialSamples);
  for (int k = first; k < M; k += step) sample[k][t] = (ordered_key(xs[(int64_t)k * npad + i]) & ~255u) | t;
  __syncthreads();
  for (int k = first; k < M; k += step) {
    const uint32_t own = sample[k][t];
    int before = 0;
#pragma unroll 8
    for (int e = 0; e < kSpatialSamples; e += 4) {
      const uint4 s = *reinterpret_cast<const uint4*>(&sample[k][e]);
      before += (s.x < own) + (s.y < own) + (s.z < own) + (s.w < own);
    }
    table[k * kSpatialSamples + before] = own & ~255u;
  }
  __syncthreads();
}

// Quantile of a value, 0 .. 2^bits - 1: the samples that are no larger, never falling as the value grows.
__device__ inline uint32_t spatial_quantile(const uint32_t* table, uint32_t image, int bits) {
  int pos = 0;
#pragma unroll
  for (int step = kSpatialSamples / 2; step > 0; step >>= 1)
    if (table[pos + step - 1] <= image) pos += step;
  return (uint32_t)pos >> (8 - bits);
}

// Bucket of a row: the leading bits of its cell's number on the curve.  Objective k gives bit b of its quantile to the b-th
// round of bits; the last round may hold only the first objectives.
template <int M>
__device__ inline int spatial_bucket(const float (&x)[M], const uint32_t* table, int bucket_bits) {
  uint32_t q[M];
#pragma unroll
  for (int k = 0; k < M; ++k) q[k] = spatial_quantile(table + k * kSpatialSamples, ordered_key(x[k]), 8);
  uint32_t z = 0;
  int bits = 0;
  for (int b = 7; b >= 0 && bits < bucket_bits; --b)
#pragma unroll
    for (int k = 0; k < M; ++k)
      if (bits < bucket_bits) {
        z = (z << 1) | ((q[k] >> b) & 1u);
        ++bits;
      }
  return (int)(z << (bucket_bits - bits));
}

// One more row in bucket b (none where b < 0).  Lanes of a wave that share a bucket with its first lanes send one addition, as
// in bucket_hist_kernel.
__device__ inline void count_in_bucket(int b, int* __restrict__ hist) {
  const int lane = threadIdx.x & 63;
  uint64_t todo = __builtin_amdgcn_ballot_w64(b >= 0);
  for (int round = 0; round < 3 && todo != 0ull; ++round) {
    const int leader = __builtin_amdgcn_readlane(b, __ffsll((unsigned long long)todo) - 1);
    const uint64_t same = __builtin_amdgcn_ballot_w64(b == leader) & todo;
    if (lane == __ffsll((unsigned long long)same) - 1) atomicAdd(&hist[leader], __popcll(same));
    todo &= ~same;
  }
  if ((todo >> lane) & 1ull) atomicAdd(&hist[b], 1);
}

// How many of the rows in a structure of arrays fall into every bucket (hist must be zero), and every row's bucket.
// count: the rows, in device memory; nothing is done for at most `least` of them (so in the kernels below).
template <int M>
__global__ __launch_bounds__(256) void spatial_bucket_kernel(const float* __restrict__ xs, int npad, const int* __restrict__ count,
                                                             int least, int bucket_bits, int* __restrict__ bucket,
                                                             int* __restrict__ hist, int64_t ws_step) {
  to_population(ws_step, xs, count, bucket, hist);
  const int n = *count;
  if (n <= least) return;
  __shared__ uint32_t table[kSpatialSamples * M];
  spatial_quantiles<M>(xs, npad, n, table);
  for (int i0 = blockIdx.x * 256; i0 < n; i0 += gridDim.x * 256) {
    const int i = i0 + threadIdx.x;
    int b = -1;
    if (i < n) {
      float x[M];
#pragma unroll
      for (int k = 0; k < M; ++k) x[k] = xs[(int64_t)k * npad + i];
      b = spatial_bucket<M>(x, table, bucket_bits);
      bucket[i] = b;
    }
    count_in_bucket(b, hist);
  }
}

// The rows to their slots: any order inside a bucket.  cursor: first free slot of every bucket; start: the buckets' first
// slots.  slot_row[slot]: the row there; slot_end[slot]: the end of its bucket.  Slots up to the next multiple of 128 are
// filled with NaN.
template <int M>
__global__ __launch_bounds__(256) void spatial_scatter_kernel(const float* __restrict__ xs, int npad, const int* __restrict__ count,
                                                              int least, const int* __restrict__ bucket, const int* __restrict__ start,
                                                              int* __restrict__ cursor, float* __restrict__ xs_sorted,
                                                              int* __restrict__ slot_row, int* __restrict__ slot_end,
                                                              const Ctrl* __restrict__ ctrl, int64_t ws_step) {
  to_population(ws_step, xs, count, bucket, start, cursor, xs_sorted, slot_row, slot_end, ctrl);
  const int n = *count;
  if (n <= least || ctrl->err != 0) return;
  const int lane = threadIdx.x & 63;
  for (int i0 = blockIdx.x * 256; i0 < ((n + 127) & ~127); i0 += gridDim.x * 256) {
    const int i = i0 + threadIdx.x;
    const int b = i < n ? bucket[i] : -1;
    float x[M];
#pragma unroll
    for (int k = 0; k < M; ++k) x[k] = i < n ? xs[(int64_t)k * npad + i] : __uint_as_float(0x7FC00000u);
    uint64_t todo = __builtin_amdgcn_ballot_w64(b >= 0);
    uint64_t group[3] = {0ull, 0ull, 0ull};
    int first[3] = {0, 0, 0};
#pragma unroll
    for (int round = 0; round < 3; ++round) {
      if (todo == 0ull) break;
      const int leader = __builtin_amdgcn_readlane(b, __ffsll((unsigned long long)todo) - 1);
      group[round] = __builtin_amdgcn_ballot_w64(b == leader) & todo;
      first[round] = __ffsll((unsigned long long)group[round]) - 1;
      todo &= ~group[round];
    }
    const uint64_t me = 1ull << lane;
    int add = (todo & me) ? 1 : 0;
#pragma unroll
    for (int round = 0; round < 3; ++round)
      if (group[round] != 0ull && lane == first[round]) add = __popcll(group[round]);
    int at = 0;
    if (add != 0) at = atomicAdd(&cursor[b], add);
    int p = b >= 0 ? at : i;
#pragma unroll
    for (int round = 0; round < 3; ++round) {
      if (group[round] == 0ull) continue;
      const int base = __builtin_amdgcn_readlane(at, first[round]);
      if (group[round] & me) p = base + __popcll(group[round] & (me - 1ull));
    }
    if (i < ((n + 127) & ~127)) {
#pragma unroll
      for (int k = 0; k < M; ++k) xs_sorted[(int64_t)k * npad + p] = x[k];
      slot_row[p] = i < n ? i : -1;
      slot_end[p] = i < n ? start[b + 1] : p + 1;
    }
  }
}

// Low and high corners of the leaves and low corners of the groups of 64 leaves.  A row that holds a NaN neither
// dominates nor is dominated: it counts for no corner.  A workgroup takes one group, a wave every sixteenth leaf of it.
// m objectives; leaf_lo / leaf_hi: [m][leaf_stride], group_lo: [m][group_stride]; corners of empty leaves are +inf / -inf.
constexpr int kBoxThreads = 1024;
__global__ __launch_bounds__(kBoxThreads) void leaf_box_kernel(const float* __restrict__ xs, const int* __restrict__ count,
                                                               int least, int npad, int m,
                                                               int64_t leaf_stride, int64_t group_stride,
                                                               float* __restrict__ leaf_lo, float* __restrict__ leaf_hi,
                                                               float* __restrict__ group_lo, const Ctrl* __restrict__ ctrl,
                                                               int64_t ws_step) {
  to_population(ws_step, xs, leaf_lo, leaf_hi, group_lo, ctrl, count);
  const int n = *count;
  if (n <= least || (int64_t)blockIdx.x * kGroupLeaves * kLeafRows >= n || ctrl->err != 0) return;
  __shared__ float low[kSpatialObjectives][kGroupLeaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int l = wave; l < kGroupLeaves; l += kBoxThreads / 64) {
    const int64_t leaf = (int64_t)blockIdx.x * kGroupLeaves + l;
    const int64_t j = leaf * kLeafRows + lane;
    bool bad = j >= n;
    for (int k = 0; k < m; ++k) bad |= j < n && xs[(int64_t)k * npad + j] != xs[(int64_t)k * npad + j];
    for (int k = 0; k < m; ++k) {
      float lo = bad ? INFINITY : xs[(int64_t)k * npad + j];
      float hi = bad ? -INFINITY : lo;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, off));
        hi = fmaxf(hi, __shfl_xor(hi, off));
      }
      if (lane == 0) {
        leaf_lo[(int64_t)k * leaf_stride + leaf] = lo;
        leaf_hi[(int64_t)k * leaf_stride + leaf] = hi;
        low[k][l] = lo;
      }
    }
  }
  __syncthreads();
  for (int k = wave; k < m; k += kBoxThreads / 64) {
    float lo = low[k][lane];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) lo = fminf(lo, __shfl_xor(lo, off));
    if (lane == 0) group_lo[(int64_t)k * group_stride + blockIdx.x] = lo;
  }
}

// ---------------------------------------------------------------- first front only
//
// mask[i] = 1 when no row dominates row i: `non_dominate_rank(f) == 0`, the only thing that
// src/evox/workflows/eval_monitor.py:301-302 and :333-335 keep of the ranks.  Four steps: (1) rows that a champion, one of some
// sampled rows and rows of low sums, dominates are dropped and the rest is copied together; (2) with two or three
// objectives, where more than kFrontGridLeast are left, so are the rows that a row of a smaller cell of a grid dominates;
// (3) up to kFrontPairsRows rows left are compared pair by pair; (4) more are put in spatial order and compared by leaves.
// Which of the steps have work is decided on the device, by the number of rows left (a kernel with nothing to do takes
// 1.6 us).  Only the scan of the buckets in (4) waits for other workgroups, those before its own, and not forever: where the
// wait runs out no row is reported, and the status says so.
constexpr int kFrontPairsRows = 65536;
constexpr int kFrontSamples = 256;      // sampled rows; those that no other sample dominates serve as champions
// Of these at most this many.  32 / 64 / 128, us a call: 1 000 003 x 3 around a sphere 247 / 238 / 232, 30 000 x 4 111 / 104 / 96;
// uniform 30 000 x 5, where the few that matter are among any 32, 25.5 / 26.6 / 27.0.
constexpr int kFrontChampions = 64;
// With more objectives hardly any row is dominated by a sample (uniform 30 000 x 7 32 us, 73 with samples; x 8 55 and 105).
constexpr int kFrontFilterObjectives = 6;
// Champions besides: rows of low sums.  Where a few rows dominate the rest, these are among them.  A few where samples serve
// too (each champion costs every row a comparison), more where they stand alone.
constexpr int front_lowest(int m) { return m <= kFrontFilterObjectives ? 4 : 16; }
constexpr int kFrontRowsPerThread = 4;
constexpr int kFrontStretchRows = 256;  // rows of which the lowest is found, at least,
constexpr int kFrontStretches = 1024;   // and how many such stretches, at most
__host__ __device__ inline int front_stretch_rows(int n) {
  const int rows = (n + kFrontStretches - 1) / kFrontStretches;
  return rows < kFrontStretchRows ? kFrontStretchRows : rows;
}
constexpr int kFrontGridPopulation = 16384;  // step 2 is launched for populations of more rows,
constexpr int kFrontGridLeast = 20480;       // and has work when step 1 leaves more than these (compared pair by pair in 45 us)
constexpr int kFrontGrid = 256;       // cells of the grid of step 2 along an objective,
constexpr int kFrontGridSmall = 128;  // and in three objectives up to kFrontGridSmallRows rows, where both passes over its
constexpr int kFrontGridSmallRows = 131072;  // cells fit one workgroup (a launch costs 4 us of host time)

// Rows left after step 1, after step 2 and between its two passes over the rows, and whether any row of the population
// holds a NaN or an infinity.
struct FrontCount {
  int rows;
  int rows_grid;
  int nonfinite;
  int rows_between;
};

// Clears the control block and the counters, where front_lowest_kernel is not launched.
__global__ __launch_bounds__(256) void front_reset_kernel(Ctrl* __restrict__ ctrl, FrontCount* __restrict__ count, int64_t ws_step) {
  to_population(ws_step, ctrl, count);
  uint32_t* words = reinterpret_cast<uint32_t*>(ctrl);
  for (int i = threadIdx.x; i < (int)(sizeof(Ctrl) / 4); i += 256) words[i] = 0u;
  if (threadIdx.x == 0) *count = FrontCount{0, 0, 0};
}

// lowest[b]: the row of the lowest sum in stretch b of the rows, its sum before it (as an ordered key; all ones where every
// sum of the stretch is infinite or NaN).  A row of a low sum lies near the front, and in a population that a few rows dominate
// it is one of them, which a sample by position may well miss: 60 000 x 8, one row dominates all others, 850 us without these
// rows, 19 with.  Also clears the control block and the counters.
template <int M>
__global__ __launch_bounds__(256) void front_lowest_kernel(const float* __restrict__ f, int64_t stride_row, int64_t stride_col,
                                                           int64_t f_step, int n, unsigned long long* __restrict__ lowest,
                                                           Ctrl* __restrict__ ctrl, FrontCount* __restrict__ count, int64_t ws_step) {
  f += (int64_t)blockIdx.z * f_step;
  to_population(ws_step, lowest, ctrl, count);
  if (blockIdx.x == 0) {
    uint32_t* words = reinterpret_cast<uint32_t*>(ctrl);
    for (int i = threadIdx.x; i < (int)(sizeof(Ctrl) / 4); i += 256) words[i] = 0u;
    if (threadIdx.x == 0) *count = FrontCount{0, 0, 0};
  }
  __shared__ unsigned long long part[4];
  const int64_t rows = front_stretch_rows(n), first = (int64_t)blockIdx.x * rows;
  const int64_t end = first + rows < n ? first + rows : n;
  unsigned long long best = ~0ull;
#pragma unroll 4
  for (int64_t i = first + threadIdx.x; i < end; i += 256) {
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < M; ++k) sum += f[i * stride_row + k * stride_col];
    const unsigned long long own = ((unsigned long long)ordered_key(sum) << 32) | (unsigned long long)i;
    if (fabsf(sum) <= 3.4028234663852886e38f && own < best) best = own;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long other = __shfl_xor(best, off);
    best = other < best ? other : best;
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x != 0) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) best = part[w] < best ? part[w] : best;
  lowest[blockIdx.x] = best;
}

template <int M>
__device__ inline bool row_dominates(const float (&a)[M], const float (&b)[M]) {
  bool no_worse = true, better = false;
#pragma unroll
  for (int k = 0; k < M; ++k) {
    no_worse &= a[k] <= b[k];
    better |= a[k] < b[k];
  }
  return no_worse && better;
}

// The same in vector arithmetic, positive where a dominates b: the bitwise OR of the differences b - a, whose signs are
// exact (dominance.hpp).  Needs a to be finite, -0.0 stored as +0.0, and no NaN in b.
template <int M>
__device__ inline int dominance_sign(const float (&a)[M], const float (&b)[M]) {
  uint32_t o = 0u;
#pragma unroll
  for (int k = 0; k < M; ++k) o |= __float_as_uint(b[k] - a[k]);
  return (int)o;
}

// A whole small population in one launch.  A workgroup has 64 rows, one to a lane, in each of its waves; the waves take all
// rows in turn, 64 at a time, through LDS.  Every pair is compared, so it serves where the three launches of the steps below
// cost more than that.
constexpr int front_small_waves(int m) { return m <= 8 ? 16 : 8; }  // (of 64 * m values in LDS each)
template <int M>
__global__ __launch_bounds__(1024) void front_small_kernel(const float* __restrict__ f, int64_t stride_row, int64_t stride_col,
                                                           int64_t f_step, int n, uint8_t* __restrict__ mask, Ctrl* __restrict__ ctrl,
                                                           int64_t ws_step) {
  f += (int64_t)blockIdx.z * f_step;
  mask += (int64_t)blockIdx.z * n;
  to_population(ws_step, ctrl);
  __shared__ __attribute__((aligned(16))) float tiles[front_small_waves(M)][M][64];
  __shared__ unsigned long long dominated;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), waves = (int)(blockDim.x >> 6);
  if (blockIdx.x == 0)  // (no wait here, so no error either)
    for (int i = threadIdx.x; i < (int)(sizeof(Ctrl) / 4); i += (int)blockDim.x) reinterpret_cast<uint32_t*>(ctrl)[i] = 0u;
  if (threadIdx.x == 0) dominated = 0ull;
  const int j = (int)blockIdx.x * 64 + lane;
  auto row = [&](int i, float pad, float (&x)[M]) {
    bool finite = true;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      x[k] = i < n ? f[i * stride_row + k * stride_col] + 0.0f : pad;  // (-0.0 as +0.0)
      finite &= fabsf(x[k]) <= 3.4028234663852886e38f;
    }
    return __builtin_amdgcn_ballot_w64(!finite) == 0ull;
  };
  float x[M];
  const bool own_finite = row(j, 0.0f, x);
  int beaten = 0;
  for (int c0 = 0; c0 < n; c0 += 64 * waves) {
    const int first = c0 + 64 * wave;
    float(&tile)[M][64] = tiles[wave];
    float mine[M];
    // (a row of the largest numbers exceeds no finite row in the differences below)
    const bool all_finite = row(first + lane, 3.4028234663852886e38f, mine) && own_finite;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < M; ++k) tile[k][lane] = mine[k];
    __syncthreads();
    const int count = min(64, n - first);
    if (all_finite) {
      for (int e = 0; e < count; e += 4) {
        uint32_t o[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < M; ++k) {
          const float4 t = *reinterpret_cast<const float4*>(&tile[k][e]);
          o[0] |= __float_as_uint(x[k] - t.x);
          o[1] |= __float_as_uint(x[k] - t.y);
          o[2] |= __float_as_uint(x[k] - t.z);
          o[3] |= __float_as_uint(x[k] - t.w);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) beaten = max(beaten, (int)o[u]);  // (dominance_sign)
      }
    } else {
      for (int e = 0; e < count; ++e) {
        float t[M];
#pragma unroll
        for (int k = 0; k < M; ++k) t[k] = tile[k][e];
        if (row_dominates<M>(t, x)) beaten = 1;
      }
    }
  }
  const uint64_t found = __builtin_amdgcn_ballot_w64(beaten > 0);
  if (lane == 0 && found != 0ull) atomicOr(&dominated, found);
  __syncthreads();
  if (wave == 0 && j < n) mask[j] = ((dominated >> lane) & 1ull) != 0ull ? 0 : 1;
}

// Copies those of a workgroup's 256 * kFrontRowsPerThread rows that are kept to the next free places of `to` (any order): one
// addition to the counter for all of them.  bucket / to_bucket: null, or what else goes along with a row.
template <int M>
__device__ inline void front_keep(const float (&x)[kFrontRowsPerThread][M], const int (&number)[kFrontRowsPerThread],
                                  const bool (&keep)[kFrontRowsPerThread], int* counter, float* __restrict__ to,
                                  int* __restrict__ to_of, int npad, int* scratch, const int* bucket = nullptr,
                                  int* __restrict__ to_bucket = nullptr) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t kept[kFrontRowsPerThread];
  int mine = 0;
#pragma unroll
  for (int r = 0; r < kFrontRowsPerThread; ++r) {
    kept[r] = __builtin_amdgcn_ballot_w64(keep[r]);
    mine += __popcll(kept[r]);
  }
  if (lane == 0) scratch[wave] = mine;
  __syncthreads();
  if (threadIdx.x == 0) scratch[4] = atomicAdd(counter, scratch[0] + scratch[1] + scratch[2] + scratch[3]);
  __syncthreads();
  int at = scratch[4];
  for (int v = 0; v < wave; ++v) at += scratch[v];
#pragma unroll
  for (int r = 0; r < kFrontRowsPerThread; ++r) {
    if (keep[r]) {
      const int p = at + __popcll(kept[r] & ((1ull << lane) - 1ull));
#pragma unroll
      for (int k = 0; k < M; ++k) to[(int64_t)k * npad + p] = x[r][k];
      to_of[p] = number[r];
      if (bucket != nullptr) to_bucket[p] = bucket[r];
    }
    at += __popcll(kept[r]);
  }
  __syncthreads();  // scratch is used again
}

// Step 1.  Every workgroup finds the champions for itself (with `lowest` front_lowest of the stretches' lowest rows, each of its
// share of them, and up to kFrontFilterObjectives objectives those of 256 sampled rows that no other dominates) and takes per
// rows per thread at a time.  left[k][p] / left_of[p]: the rows kept, in any order, and their numbers; mask: 1 for them, 0 for the
// others.  grid: null or the grid_cells cells of step 2, set to "empty" here; zero: what step 4 needs cleared.
template <int M>
__global__ __launch_bounds__(256) void front_filter_kernel(const float* __restrict__ f, int64_t stride_row, int64_t stride_col,
                                                           int64_t f_step, int n, int npad, int per,
                                                           const unsigned long long* __restrict__ lowest, float* __restrict__ left,
                                                           int* __restrict__ left_of, uint8_t* __restrict__ mask,
                                                           FrontCount* __restrict__ count, uint32_t* __restrict__ grid,
                                                           int grid_cells, uint32_t* __restrict__ zero, int zero_words,
                                                           int64_t ws_step) {
  f += (int64_t)blockIdx.z * f_step;
  mask += (int64_t)blockIdx.z * n;
  to_population(ws_step, lowest, left, left_of, count, grid, zero);
  for (int c = blockIdx.x * 256 + threadIdx.x; c < grid_cells; c += gridDim.x * 256) grid[c] = ~0u;
  for (int c = blockIdx.x * 256 + threadIdx.x; c < zero_words; c += gridDim.x * 256) zero[c] = 0u;
  constexpr bool kSampled = M <= kFrontFilterObjectives;
  constexpr int kLowest = front_lowest(M), kMost = (kSampled ? kFrontChampions : 0) + kLowest;
  static_assert(kFrontSamples == 256 && kMost % 4 == 0 && 256 % kLowest == 0, "one sample per thread; champions in fours");
  __shared__ __attribute__((aligned(16))) float sample[kSampled ? M : 1][kFrontSamples];
  __shared__ __attribute__((aligned(16))) float champion[kMost][(M + 3) / 4 * 4];
  __shared__ int champions;
  __shared__ int scratch[5];
  {
    auto read = [&](int64_t i, float (&x)[M]) {
      bool finite = true;
#pragma unroll
      for (int k = 0; k < M; ++k) {
        x[k] = f[i * stride_row + k * stride_col] + 0.0f;
        finite &= fabsf(x[k]) <= 3.4028234663852886e38f;
      }
      return finite;
    };
    auto enter = [&](const float (&x)[M]) {
      const int c = atomicAdd(&champions, 1);
#pragma unroll
      for (int k = 0; k < M; ++k) champion[c][k] = x[k];
    };
    float mine[M];
    bool finite = false;
    if constexpr (kSampled) {
      finite = read((int64_t)threadIdx.x * n / kFrontSamples, mine);
#pragma unroll
      for (int k = 0; k < M; ++k) sample[k][threadIdx.x] = mine[k];
    }
    if (threadIdx.x == 0) champions = 0;
    __syncthreads();
    if (lowest != nullptr) {
      const int stretches = (n + front_stretch_rows(n) - 1) / front_stretch_rows(n);
      unsigned long long best = ~0ull;
      for (int e = threadIdx.x; e < stretches; e += 256) best = lowest[e] < best ? lowest[e] : best;
#pragma unroll
      for (int off = 128 / kLowest; off > 0; off >>= 1) {
        const unsigned long long other = __shfl_xor(best, off);
        best = other < best ? other : best;
      }
      float low[M];
      if (threadIdx.x % (256 / kLowest) == 0 && best != ~0ull && read((int64_t)(uint32_t)best, low)) enter(low);
    }
    // (a sample that is not finite is no champion, and may wrongly keep another from being one: neither does harm)
    if constexpr (kSampled) {
      int beaten = 0;
#pragma unroll 2
      for (int e = 0; e < kFrontSamples; e += 4) {
        float4 o[M];
#pragma unroll
        for (int k = 0; k < M; ++k) o[k] = *reinterpret_cast<const float4*>(&sample[k][e]);
        float a[4][M];
#pragma unroll
        for (int k = 0; k < M; ++k) {
          a[0][k] = o[k].x;
          a[1][k] = o[k].y;
          a[2][k] = o[k].z;
          a[3][k] = o[k].w;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) beaten = max(beaten, dominance_sign<M>(a[u], mine));
      }
      __syncthreads();  // (the rows of low sums are in)
      if (finite && beaten <= 0) {
        const int c = atomicAdd(&champions, 1);
        if (c < kMost)
#pragma unroll
          for (int k = 0; k < M; ++k) champion[c][k] = mine[k];
      }
    }
    __syncthreads();
  }
  const int nc = min(champions, kMost);
  if (threadIdx.x < 4 && nc + threadIdx.x < kMost) {  // (up to a whole four with rows that dominate nothing finite)
#pragma unroll
    for (int k = 0; k < M; ++k) champion[nc + threadIdx.x][k] = 3.4028234663852886e38f;
  }
  __syncthreads();
  bool bad = false;
  for (int64_t i0 = (int64_t)blockIdx.x * 256 * per; i0 < n; i0 += (int64_t)gridDim.x * 256 * per) {
    float x[kFrontRowsPerThread][M];
    int number[kFrontRowsPerThread], beaten[kFrontRowsPerThread];
    bool keep[kFrontRowsPerThread];
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      const int64_t i = r < per ? i0 + r * 256 + threadIdx.x : n;
      number[r] = i < n ? (int)i : n;
      beaten[r] = 0;
#pragma unroll
      for (int k = 0; k < M; ++k) x[r][k] = i < n ? f[i * stride_row + k * stride_col] + 0.0f : 0.0f;  // (-0.0 as +0.0)
    }
    constexpr int kTogether = M <= 8 ? 4 : 1;  // champions whose LDS reads are in flight together, as far as registers go
    for (int c = 0; c < nc; c += kTogether) {
      float champ[kTogether][M];
#pragma unroll
      for (int u = 0; u < kTogether; ++u)
#pragma unroll
        for (int k = 0; k < M; ++k) champ[u][k] = champion[c + u][k];
#pragma unroll
      for (int r = 0; r < kFrontRowsPerThread; ++r)
        if (r < per)
#pragma unroll
          for (int u = 0; u < kTogether; ++u) beaten[r] = max(beaten[r], dominance_sign<M>(champ[u], x[r]));
    }
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      bool nan = false;
#pragma unroll
      for (int k = 0; k < M; ++k) {
        nan |= x[r][k] != x[r][k];
        bad |= !(fabsf(x[r][k]) <= 3.4028234663852886e38f);
      }
      keep[r] = number[r] < n && (beaten[r] <= 0 || nan);  // (a row with a NaN is not dominated)
      if (number[r] < n) mask[number[r]] = keep[r] ? 1 : 0;
    }
    front_keep<M>(x, number, keep, &count->rows, left, left_of, npad, scratch);
  }
  if (__syncthreads_or(bad) && threadIdx.x == 0) count->nonfinite = 1;
}

// Step 2, for two and three objectives.  All objectives but the last are cut into 2^bits quantiles; a cell keeps the
// smallest value of the last objective among its rows (front_grid_kernel), then the smallest of all cells that are smaller
// in every cut objective (front_grid_prefix_kernel, one objective after the other): a row no better than that is dominated
// (front_grid_filter_kernel, which also counts the rows it leaves per bucket of the spatial order).  What it leaves are the
// rows within about a cell of the front: 1 000 003 rows around a sphere, 35 000 of them on the front, go down to 134 000.
template <int M>
__device__ inline int front_cell(const float (&x)[M], const uint32_t* table, int bits) {
  const int c0 = (int)spatial_quantile(table, ordered_key(x[0]), bits);
  if constexpr (M == 2) return c0;
  return (c0 << bits) + (int)spatial_quantile(table + kSpatialSamples, ordered_key(x[1]), bits);
}

// Minimum over the lanes up to this one (shifts inside the DPP rows, then from row to row).
__device__ __forceinline__ uint32_t lanes_prefix_min(uint32_t v) {
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x111, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x112, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x114, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x118, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x142, 0xa, 0xf, false));
  return min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x143, 0xc, 0xf, false));
}
__device__ __forceinline__ uint32_t lanes_before(uint32_t prefix) {  // ... up to the lane before it
  const uint32_t up = __shfl_up(prefix, 1);
  return (threadIdx.x & 63) == 0 ? ~0u : up;
}

// The workgroup goes through its own rows first, `per` to a thread, on a grid of 64 cells along an objective in LDS: a row
// that one of these rows dominates there is dropped -- what it would have told the grid, its dominator tells at least as
// well -- and comes neither to the grid in memory nor to the second pass over the rows.  Of 630 000 rows left by step 1
// (1 000 003 x 3 around a sphere) some 260 000 go on.  The grid's cells lie 2^spread words apart: minima in one line of memory
// follow one another, some 55 ns each, and up to 900 of them fell on the 32 cells of a line.  Both together, with 1024 threads
// to a workgroup and each 256 of them ranking the samples of one objective: 38 us for 60, and 17 for 31 in
// front_grid_filter_kernel (a call 206 us for 241; 1 000 000 x 2 146 for 175, 100 000 x 3 97 for 102).  The minima are bound
// by the lines they meet in; all but 21 us of this kernel.
// to / to_of: the rows that go on; tables: the quantiles, for the pass that follows.
constexpr int kFrontGridBlock = 1024, kFrontLocal = 64;
template <int M>
__global__ __launch_bounds__(kFrontGridBlock) void front_grid_kernel(const float* __restrict__ left, const int* __restrict__ left_of,
                                                                     int npad, int per, int bits, FrontCount* __restrict__ count,
                                                                     float* __restrict__ to, int* __restrict__ to_of,
                                                                     uint8_t* __restrict__ mask, int population,
                                                                     uint32_t* __restrict__ tables, uint32_t* __restrict__ grid,
                                                                     int spread, int64_t ws_step) {
  mask += (int64_t)blockIdx.z * population;
  to_population(ws_step, left, left_of, count, to, to_of, tables, grid);
  const int rows = count->rows;
  if (rows <= kFrontGridLeast) return;
  constexpr int kStride = kFrontLocal + 1, kLines = M == 2 ? 1 : kFrontLocal;  // (a column's cells fall into different banks)
  __shared__ uint32_t table[kSpatialSamples * M];
  __shared__ uint32_t local[kLines * kStride];
  __shared__ int scratch[kFrontGridBlock / 64 + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int kWaves = kFrontGridBlock / 64;
  spatial_quantiles<M>(left, npad, rows, table);
  if (blockIdx.x == 0)
    for (int e = threadIdx.x; e < kSpatialSamples * M; e += kFrontGridBlock) tables[e] = table[e];
  for (int i0 = blockIdx.x * kFrontGridBlock * per; i0 < rows; i0 += gridDim.x * kFrontGridBlock * per) {
    for (int c = threadIdx.x; c < kLines * kStride; c += kFrontGridBlock) local[c] = ~0u;
    float x[kFrontRowsPerThread][M];
    int number[kFrontRowsPerThread], cell[kFrontRowsPerThread], near[kFrontRowsPerThread];
    uint32_t value[kFrontRowsPerThread];
    bool keep[kFrontRowsPerThread];
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      const int i = i0 + r * kFrontGridBlock + threadIdx.x;
      keep[r] = r < per && i < rows;
      number[r] = keep[r] ? left_of[i] : 0;
#pragma unroll
      for (int k = 0; k < M; ++k) x[r][k] = keep[r] ? left[(int64_t)k * npad + i] : 0.0f;
    }
    __syncthreads();  // (the cells are clear)
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      bool nan = false;
#pragma unroll
      for (int k = 0; k < M; ++k) nan |= x[r][k] != x[r][k];
      cell[r] = front_cell<M>(x[r], table, bits);
      near[r] = M == 2 ? cell[r] >> (bits - 6) : (cell[r] >> (2 * bits - 6)) * kStride + ((cell[r] & ((1 << bits) - 1)) >> (bits - 6));
      value[r] = keep[r] && !nan ? ordered_key(x[r][M - 1]) : ~0u;  // (a row with a NaN beats none and is beaten by none)
      if (value[r] != ~0u) atomicMin(&local[near[r]], value[r]);
    }
    __syncthreads();
    // every cell: the smallest of the cells before it along the line, then of those in the lines before it
    for (int line = wave; line < kLines; line += kWaves)
      local[line * kStride + lane] = lanes_before(lanes_prefix_min(local[line * kStride + lane]));
    __syncthreads();
    if constexpr (M == 3) {
      for (int column = wave; column < kFrontLocal; column += kWaves)
        local[lane * kStride + column] = lanes_before(lanes_prefix_min(local[lane * kStride + column]));
      __syncthreads();
    }
    uint64_t kept[kFrontRowsPerThread];
    int mine = 0;
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      if (value[r] != ~0u && local[near[r]] <= value[r]) {
        keep[r] = false;
        mask[number[r]] = 0;
        value[r] = ~0u;
      }
      // (what a plain load sees may be old, which costs an addition too many and no more)
      if (value[r] < grid[cell[r] << spread]) atomicMin(&grid[cell[r] << spread], value[r]);
      kept[r] = __builtin_amdgcn_ballot_w64(keep[r]);
      mine += __popcll(kept[r]);
    }
    if (lane == 0) scratch[wave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
      int all = 0;
      for (int v = 0; v < kWaves; ++v) all += scratch[v];
      scratch[kWaves] = atomicAdd(&count->rows_between, all);
    }
    __syncthreads();
    int at = scratch[kWaves];
    for (int v = 0; v < wave; ++v) at += scratch[v];
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      if (keep[r]) {
        const int p = at + __popcll(kept[r] & ((1ull << lane) - 1ull));
#pragma unroll
        for (int k = 0; k < M; ++k) to[(int64_t)k * npad + p] = x[r][k];
        to_of[p] = number[r];
      }
      at += __popcll(kept[r]);
    }
    __syncthreads();  // (cells and counts are used again)
  }
}

// Row b of `in` (kFrontGrid cells, 2^spread words apart) to column b of `out`: out[c][b] = min of in[b][0 .. c - 1].
__global__ __launch_bounds__(kFrontGrid) void front_grid_prefix_kernel(const uint32_t* __restrict__ in, int spread,
                                                                       uint32_t* __restrict__ out, int out_stride, const FrontCount* __restrict__ count,
                                                                       int64_t ws_step) {
  to_population(ws_step, in, out, count);
  if (count->rows <= kFrontGridLeast) return;
  __shared__ uint32_t last[kFrontGrid / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t v = in[((int64_t)blockIdx.x * kFrontGrid + threadIdx.x) << spread];
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t o = __shfl_up(v, off);
    if (lane >= off) v = min(v, o);
  }
  if (lane == 63) last[wave] = v;
  __syncthreads();
  uint32_t before = __shfl_up(v, 1);
  if (lane == 0) before = ~0u;
  for (int w = 0; w < wave; ++w) before = min(before, last[w]);
  out[(int64_t)threadIdx.x * out_stride + blockIdx.x] = before;
}

// Both passes over a grid of kFrontGridSmall^2 cells, in one workgroup: out[c0][c1] = min of in over all smaller c0 and c1.
constexpr int kFrontGridThreads = 1024;
constexpr size_t kFrontGridLds = sizeof(uint32_t) * (kFrontGridSmall * kFrontGridSmall + kFrontGridThreads);
__global__ __launch_bounds__(kFrontGridThreads) void front_grid_small_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                                             const FrontCount* __restrict__ count, int64_t ws_step) {
  to_population(ws_step, in, out, count);
  if (count->rows <= kFrontGridLeast) return;
  extern __shared__ uint32_t cells[];
  uint32_t* part = cells + kFrontGridSmall * kFrontGridSmall;  // minimum of a thread's sixteen cells
  constexpr int kEach = kFrontGridSmall * kFrontGridSmall / kFrontGridThreads;
  constexpr int kParts = kFrontGridSmall / kEach;  // threads to a row or column
  const int line = threadIdx.x / kParts, piece = threadIdx.x % kParts;
  uint32_t v[kEach];
  uint32_t least = ~0u;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    v[e] = in[line * kFrontGridSmall + piece * kEach + e];
    least = min(least, v[e]);
  }
  part[threadIdx.x] = least;
  __syncthreads();
  uint32_t before = ~0u;
  for (int p = 0; p < piece; ++p) before = min(before, part[line * kParts + p]);
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    cells[line * kFrontGridSmall + piece * kEach + e] = before;
    before = min(before, v[e]);
  }
  __syncthreads();
  // (column = thread within a row of cells, so that neighbouring lanes read neighbouring words)
  const int column = threadIdx.x % kFrontGridSmall, rows_piece = threadIdx.x / kFrontGridSmall;
  least = ~0u;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    v[e] = cells[(rows_piece * kEach + e) * kFrontGridSmall + column];
    least = min(least, v[e]);
  }
  part[rows_piece * kFrontGridSmall + column] = least;
  __syncthreads();
  before = ~0u;
  for (int p = 0; p < rows_piece; ++p) before = min(before, part[p * kFrontGridSmall + column]);
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    out[(rows_piece * kEach + e) * kFrontGridSmall + column] = before;
    before = min(before, v[e]);
  }
}

template <int M>
__global__ __launch_bounds__(256) void front_grid_filter_kernel(const float* __restrict__ left, const int* __restrict__ left_of,
                                                                int npad, int bits, FrontCount* __restrict__ count,
                                                                const uint32_t* __restrict__ tables, const uint32_t* __restrict__ below, float* __restrict__ to,
                                                                int* __restrict__ to_of, uint8_t* __restrict__ mask, int population,
                                                                int bucket_bits, int* __restrict__ to_bucket,
                                                                int* __restrict__ hist, int64_t ws_step) {
  mask += (int64_t)blockIdx.z * population;
  to_population(ws_step, left, left_of, count, tables, below, to, to_of, to_bucket, hist);
  if (count->rows <= kFrontGridLeast) return;
  const int rows = count->rows_between;
  __shared__ uint32_t table[kSpatialSamples * M];
  __shared__ int scratch[5];
  for (int e = threadIdx.x; e < kSpatialSamples * M; e += 256) table[e] = tables[e];
  __syncthreads();
  for (int i0 = blockIdx.x * 256 * kFrontRowsPerThread; i0 < rows; i0 += gridDim.x * 256 * kFrontRowsPerThread) {
    float x[kFrontRowsPerThread][M];
    int number[kFrontRowsPerThread], bucket[kFrontRowsPerThread];
    bool keep[kFrontRowsPerThread];
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      const int i = i0 + r * 256 + threadIdx.x;
      keep[r] = i < rows;
      number[r] = keep[r] ? left_of[i] : 0;
#pragma unroll
      for (int k = 0; k < M; ++k) x[r][k] = keep[r] ? left[(int64_t)k * npad + i] : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < kFrontRowsPerThread; ++r) {
      bool nan = false;
#pragma unroll
      for (int k = 0; k < M; ++k) nan |= x[r][k] != x[r][k];
      if (keep[r] && !nan && below[front_cell<M>(x[r], table, bits)] <= ordered_key(x[r][M - 1])) {
        keep[r] = false;
        mask[number[r]] = 0;
      }
      bucket[r] = keep[r] && hist != nullptr ? spatial_bucket<M>(x[r], table, bucket_bits) : -1;
      if (hist != nullptr) count_in_bucket(bucket[r], hist);
    }
    front_keep<M>(x, number, keep, &count->rows_grid, to, to_of, npad, scratch, hist != nullptr ? bucket : nullptr, to_bucket);
  }
}

// Whether a row of xs[.][first .. first + 31] dominates the lane's row x; rows >= n are padding.  The rows are scalar
// operands, in vector arithmetic where the population is finite: the last 32 rows once more where fewer are left (one by one
// they were a third of the pair step at 4090 x 8).
template <int M>
__device__ inline bool half_leaf_dominates(const float* __restrict__ xs, int npad, int first, int n, const float (&x)[M], bool all_finite) {
  if (all_finite && n >= 32) {
    first = min(first, n - 32);
    int worst = 0;
    constexpr int G = M <= 3 ? 32 : (M <= 5 ? 8 : (M <= 8 ? 4 : 2));  // rows whose values sit in scalar registers at once
#pragma unroll 1
    for (int g = 0; g < 32; g += G) {
      float xi[M][G];
#pragma unroll
      for (int k = 0; k < M; ++k)
#pragma unroll
        for (int u = 0; u < G; ++u) xi[k][u] = xs[(int64_t)k * npad + first + g + u];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        uint32_t o = 0u;
#pragma unroll
        for (int k = 0; k < M; ++k) o |= __float_as_uint(x[k] - xi[k][u]);
        worst = max(worst, (int)o);  // positive: no difference is negative and some is not zero
      }
    }
    return worst > 0;
  }
  bool beaten = false;
  for (int i = first; i < min(first + 32, n); ++i) {
    float xi[M];
#pragma unroll
    for (int k = 0; k < M; ++k) xi[k] = xs[(int64_t)k * npad + i];
    beaten |= row_dominates<M>(xi, x);
  }
  return beaten;
}

// Step 3.  Grid (row blocks of 256, kFrontPairsParts): a wave takes 64 of the rows left against one part of them, which
// streams past as scalar operands 32 at a time.  Brute force, but at the rate of the vector unit: 10 000 rows of three
// objectives on one front take 13 us this way, 300 as long waves over all slots below.
// (grid_step: step 2 exists)
constexpr int kFrontPairsParts = 64;
template <int M>
__global__ __launch_bounds__(256) void front_pairs_kernel(const float* __restrict__ left, const int* __restrict__ left_of,
                                                          int npad, uint8_t* __restrict__ mask, int population,
                                                          const FrontCount* __restrict__ count, int grid_step, int64_t ws_step) {
  mask += (int64_t)blockIdx.z * population;
  to_population(ws_step, left, left_of, count);
  int rows = count->rows;
  if (rows > kFrontGridLeast && grid_step != 0) rows = count->rows_grid;
  if (rows > kFrontPairsRows) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int j0 = (blockIdx.x * 4 + wave) * 64;
  int part = ((rows + kFrontPairsParts - 1) / kFrontPairsParts + 31) & ~31;
  if (part < 64) part = 64;
  const int i0 = blockIdx.y * part;
  if (j0 >= rows || i0 >= rows) return;
  const int i1 = min(i0 + part, rows);
  const int j = j0 + lane;
  const bool all_finite = count->nonfinite == 0;
  float x[M];
#pragma unroll
  for (int k = 0; k < M; ++k) x[k] = left[(int64_t)k * npad + j];  // (npad is a multiple of 128: there is such a place)
  bool beaten = false;
  for (int ib = i0; ib < i1; ib += 32) {
    beaten |= half_leaf_dominates<M>(left, npad, ib, i1, x, all_finite);
    if (__builtin_amdgcn_ballot_w64(!beaten && j < rows) == 0ull) break;
  }
  if (beaten && j < rows) mask[left_of[j]] = 0;
}

// Step 4, on the rows left in spatial order (slot_row: the row left that a slot holds).  A workgroup of four waves takes the
// 64 rows of one leaf (lane = row, the same in every wave).  The leaves up to the end of its last row's bucket whose low
// corner is no worse than the leaf's high corner are dealt to the waves, nearest first, and the rows of such a leaf stream
// past as scalar operands; a wave skips a leaf when no row still undecided reaches its low corner, and stops when every row
// of the workgroup has met a dominator.  After a few leaves only the rows that nothing near dominates are undecided, most
// of them rows of the front: if they are few, the waves take them one by one (front_row_beaten), which asks a leaf 64 rows
// at a time and only the leaves whose low corner is no worse than the one row.
constexpr int kFrontWaves = 4;
// Leaves per wave before that: 1 / 3 / 6, us a call around a sphere, 1 000 003 x 3 234 / 238 / 251, 100 000 x 8, where the rows
// seldom get few, 2490 / 2496 / 2363.
constexpr int kFrontBulkLeaves = 3;
// And the most rows it is done for: 8 / 24 / 48, 1 000 003 x 3 241 / 238 / 248, 100 000 x 5 503 / 454 / 545.
constexpr int kFrontFewRows = 24;

// Whether some row of the leaves up to `last` dominates the row x (the same in every lane); wave-cooperative.
template <int M>
__device__ inline bool front_row_beaten(const float (&x)[M], int last, const float* __restrict__ xs, int npad, int64_t leaf_stride,
                                        int64_t group_stride, const float* __restrict__ leaf_lo, const float* __restrict__ group_lo) {
  const int lane = threadIdx.x & 63;
  const int last_group = last / kGroupLeaves;
  for (int c0 = last_group / 64 * 64; c0 >= 0; c0 -= 64) {
    bool reach = c0 + lane <= last_group;
#pragma unroll
    for (int k = 0; k < M; ++k) reach &= group_lo[(int64_t)k * group_stride + c0 + lane] <= x[k];
    uint64_t groups = __builtin_amdgcn_ballot_w64(reach);
    while (groups != 0ull) {
      const int g = c0 + 63 - __builtin_clzll(groups);
      groups &= ~(1ull << (g - c0));
      bool near = g * kGroupLeaves + lane <= last;
#pragma unroll
      for (int k = 0; k < M; ++k) near &= leaf_lo[(int64_t)k * leaf_stride + g * kGroupLeaves + lane] <= x[k];
      uint64_t leaves = __builtin_amdgcn_ballot_w64(near);
      while (leaves != 0ull) {
        // two leaves at a time, their loads in flight together
        const int a = 63 - __builtin_clzll(leaves);
        leaves &= ~(1ull << a);
        const int b = leaves != 0ull ? 63 - __builtin_clzll(leaves) : a;
        leaves &= ~(1ull << b);
        const int ja = (g * kGroupLeaves + a) * kLeafRows + lane, jb = (g * kGroupLeaves + b) * kLeafRows + lane;
        float ra[M], rb[M];
#pragma unroll
        for (int k = 0; k < M; ++k) {
          ra[k] = xs[(int64_t)k * npad + ja];
          rb[k] = xs[(int64_t)k * npad + jb];
        }
        if (__builtin_amdgcn_ballot_w64(row_dominates<M>(ra, x) || row_dominates<M>(rb, x)) != 0ull) return true;
      }
    }
  }
  return false;
}

template <int M>
__global__ __launch_bounds__(64 * kFrontWaves) void first_front_leaf_kernel(
    const float* __restrict__ xs, const int* __restrict__ slot_row, const int* __restrict__ slot_end, const int* __restrict__ left_of,
    const FrontCount* __restrict__ state, const int* __restrict__ count, int npad, int64_t leaf_stride, int64_t group_stride,
    const float* __restrict__ leaf_lo, const float* __restrict__ leaf_hi, const float* __restrict__ group_lo,
    uint8_t* __restrict__ mask, int population, const Ctrl* __restrict__ ctrl, int64_t ws_step) {
  to_population(ws_step, xs, slot_row, slot_end, left_of, state, count, leaf_lo, leaf_hi, group_lo, ctrl);
  mask += (int64_t)blockIdx.z * population;
  const int n = *count;
  if (n <= kFrontPairsRows) return;
  __shared__ unsigned long long decided;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int own = (int)blockIdx.x;  // this workgroup's leaf
  const int j = own * kLeafRows + lane;
  if (ctrl->err != 0) {  // the scan of the buckets failed, nothing is valid: no row is reported (the status carries the error)
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < population; i += (int64_t)gridDim.x * blockDim.x) mask[i] = 0;
    return;
  }
  if (own * kLeafRows >= n) return;
  float xj[M], hi[M];
#pragma unroll
  for (int k = 0; k < M; ++k) xj[k] = xs[(int64_t)k * npad + j];
#pragma unroll
  for (int k = 0; k < M; ++k) hi[k] = leaf_hi[(int64_t)k * leaf_stride + own];
  const int last = __builtin_amdgcn_readfirstlane((slot_end[min(own * kLeafRows + kLeafRows - 1, n - 1)] - 1) / kLeafRows);
  const bool all_finite = state->nonfinite == 0;  // wave-uniform
  if (threadIdx.x == 0) decided = 0ull;
  __syncthreads();
  // (rows beyond the population and rows with a NaN wait for nothing: their comparisons never hold)
  bool real = j < n;
#pragma unroll
  for (int k = 0; k < M; ++k) real &= xj[k] == xj[k];
  const uint64_t rows = __builtin_amdgcn_ballot_w64(real);
  uint64_t open = rows;  // rows that have met no dominator yet, as this wave knows
  int turn = wave;       // leaves until this wave's next one
  int taken = 0;         // leaves this wave has taken
  bool few = false;
  const int last_group = last / kGroupLeaves;
  for (int c0 = last_group / 64 * 64; c0 >= 0 && open != 0ull && !few; c0 -= 64) {
    bool reach = c0 + lane <= last_group;
#pragma unroll
    for (int k = 0; k < M; ++k) reach &= group_lo[(int64_t)k * group_stride + c0 + lane] <= hi[k];
    uint64_t groups = __builtin_amdgcn_ballot_w64(reach);
    while (groups != 0ull && open != 0ull && !few) {
      const int g = c0 + 63 - __builtin_clzll(groups);
      groups &= ~(1ull << (g - c0));
      bool near = g * kGroupLeaves + lane <= last;
#pragma unroll
      for (int k = 0; k < M; ++k) near &= leaf_lo[(int64_t)k * leaf_stride + g * kGroupLeaves + lane] <= hi[k];
      uint64_t leaves = __builtin_amdgcn_ballot_w64(near);
      while (leaves != 0ull) {
        const int l = 63 - __builtin_clzll(leaves);
        leaves &= ~(1ull << l);
        if (turn != 0) {
          --turn;
          continue;
        }
        turn = kFrontWaves - 1;
        const int d = __builtin_amdgcn_readfirstlane(g * kGroupLeaves + l);
        bool need = ((open >> lane) & 1ull) != 0ull;
#pragma unroll
        for (int k = 0; k < M; ++k) need &= leaf_lo[(int64_t)k * leaf_stride + d] <= xj[k];
        if (__builtin_amdgcn_ballot_w64(need) == 0ull) continue;
        bool met = half_leaf_dominates<M>(xs, npad, d * kLeafRows, n, xj, all_finite);
        met |= half_leaf_dominates<M>(xs, npad, d * kLeafRows + 32, n, xj, all_finite);
        const uint64_t found = __builtin_amdgcn_ballot_w64(met) & open;
        if (found != 0ull && lane == 0) atomicOr(&decided, found);
        open &= ~(found | *reinterpret_cast<volatile unsigned long long*>(&decided));
        if (open == 0ull) break;
        if (++taken >= kFrontBulkLeaves && __popcll(open) <= kFrontFewRows) {
          few = true;
          break;
        }
      }
    }
  }
  if (__syncthreads_or(few)) {
    // (a wave that left early has not asked its share of the leaves: what is open now is open to the whole workgroup)
    deal_open_rows(
        wave, kFrontWaves, [&] { return rows & ~decided; }, [] { __syncthreads(); },
        [&](int r) {
          float x[M];
#pragma unroll
          for (int k = 0; k < M; ++k) x[k] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(xj[k]), r));
          if (front_row_beaten<M>(x, last, xs, npad, leaf_stride, group_stride, leaf_lo, group_lo) && lane == 0) atomicOr(&decided, 1ull << r);
        });
    __syncthreads();
  }
  if (wave == 0 && j < n && ((decided >> lane) & 1ull) != 0ull) mask[left_of[slot_row[j]]] = 0;
}

}  // namespace evx
