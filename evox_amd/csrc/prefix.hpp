// The dominance bit matrix of a large finite population without testing pair by pair.
//
// Same matrix as dominance.hpp (src/evox/operators/selection/non_dominate.py:6-26 in slot space, lower
// triangle), from the order of the rows in each objective.  With pos_k(i) = position of row i in the
// ascending order of objective k and upper_k(j) = number of rows whose value in objective k is at most row j's,
//     x[i,k] <= x[j,k]  <=>  pos_k(i) < upper_k(j),
// so the rows that are no worse than j in objective k are a prefix of that order, and the dominators of j are
// the intersection over k of the M prefixes, less the rows identical to j (kid(i) == kid(j): equal in every
// objective; a row of a larger slot has a larger key sum and is never in the intersection).  Infinities and
// NaN are left to the pairwise kernel (a NaN has no place in the order).
//
//  1. The slots in the order of every objective, pos[k][slot] and upper[k][slot]: by workgroups that sort in LDS
//     (objective_order_lds_kernel, objective_order_stream_kernel), for the largest populations by one segmented radix sort
//     (objective_order_kernel).
//  2. dominance_prefix_kernel: a workgroup takes a tile of 512 dominator slots (8 matrix words, 64 bytes of
//     every row; 256 slots above ten objectives, where the tables of 512 no longer fit the LDS) and a stretch
//     of rows below it.  Restricted to one word of the tile, the prefix of objective k that belongs to row j is
//     one of only 65 bit sets: the word's own slots sorted by pos_k, the first c of them.  The workgroup builds
//     in LDS, per objective: the tile's positions in ascending order (mp), a coarse index from position to the
//     number t of them that lie before it, for every t the byte counts c (how many of the first t fall into each
//     word), and the 65 bit sets of every word, kept complemented.  A lane then needs, per row and objective, one
//     look-up of t (the coarse index, then a comparison or two along mp), one 8-byte read of the counts and one
//     8-byte read of a bit set per word, ORed over the objectives and complemented once: about 55 instructions
//     per objective and 512 pairs, where the pairwise test needs 640.  While it holds the words of a row it also
//     leaves their popcount and the highest non-empty word for the count stage (peel.hpp), which then reads no
//     row again.
#pragma once

#include "common.hpp"
#include "order.hpp"
#include "peel.hpp"
#include "radix.hpp"
#include "two.hpp"

namespace evx {

constexpr int kPrefixMaxObjectives = 16;
constexpr int kPrefixWideObjectives = 10;  // up to here tiles of 8 words (14.4 KB of LDS per objective), above it of 4 (9.3 KB)
constexpr int kPrefixBuckets = 1024;       // entries of the coarse index per objective, at most (plus two)
constexpr int kPrefixThreads = 1024;
constexpr int kPrefixRowChunk = 32768;     // rows per workgroup, at most (`chunk`, a multiple of 64)
constexpr int kPrefixNearbyGroups = 256;  // groups of 64 rows in a part of the work on rows in spatial order, at most
constexpr int kPrefixMaxRows = 1 << 22;    // a position and a slot of the tile share one int

// LDS of dominance_prefix_kernel<M, WW>, per objective: bit sets and counts (the scratch of the build lies over
// them), sorted positions, the sorted (position, slot) pairs of the build, and the coarse index.
__host__ __device__ inline size_t prefix_lds_bytes(int m, int tile_words, int buckets) {
  const int tile_slots = 64 * tile_words;
  const size_t sets = sizeof(uint64_t) * tile_words * 65;
  const size_t counts = sizeof(uint64_t) * (tile_slots + 1);
  const size_t scratch = (sizeof(int) * (size_t)(buckets + 2 + tile_slots) + 7) & ~(size_t)7;  // histogram, claimed
  const size_t over = sets + counts > scratch ? sets + counts : scratch;
  const size_t positions = sizeof(int) * (tile_slots + 8);
  const size_t sorted = sizeof(int) * tile_slots;
  const size_t index = (sizeof(uint16_t) * (size_t)(buckets + 2) + 7) & ~(size_t)7;
  return (size_t)m * (over + positions + sorted + index);
}

// Positions are cut into at most kPrefixBuckets buckets of 2^shift positions.
__host__ __device__ inline int prefix_bucket_shift(int n) {
  int shift = 0;
  while (((n - 1) >> shift) + 1 > kPrefixBuckets) ++shift;
  return shift;
}

// pos[k * kstride + slot] = position of the slot's row in the ascending order of objective k, equal values in the
// order of the original row index (the order of a stable sort of the population as the caller holds it, which the
// ordering of the last front takes over: front_order_kernels below);
// upper[k * kstride + slot] = number of rows whose value in objective k is at most this slot's.
// `xs` = the fitness by original index, `slot_of` = original index -> slot.  The sorted (key, original index) pairs
// stay in buf.pairs[0] and param->orders_valid says so.
// Grid: the radix grid (all blocks resident).  Dynamic LDS: kRadixLdsBytes.  Nothing is done for a
// population with a NaN or an infinity.
__global__ __launch_bounds__(kRadixThreads) void objective_order_kernel(const float* __restrict__ xs, int npad, int n, int m,
                                                                        const int* __restrict__ slot_of,
                                                                        SortParam* __restrict__ param,
                                                                        Ctrl* __restrict__ ctrl, int* __restrict__ pos,
                                                                        int* __restrict__ upper, int* __restrict__ total0,
                                                                        int* __restrict__ witness0, RadixBuffers buf,
                                                                        unsigned spin_limit) {
  extern __shared__ int order_lds[];
  __shared__ int base[256];
  __shared__ int scratch[kRadixThreads];
  if (param->nonfinite != 0) return;
  if (call_failed(ctrl, scratch)) return;
  const unsigned gen0 = radix_generation_base(ctrl);
  if (blockIdx.x == 0) {
    radix_master(ctrl, gen0, 12, spin_limit, scratch);
    if (threadIdx.x == 0) ctrl->radix_epoch += 1;  // nobody reads it again in this kernel
    return;
  }
  if (blockIdx.x < kFirstSweeper) return;
  const int workers = gridDim.x - kFirstSweeper;
  const int wb = (int)blockIdx.x - kFirstSweeper;
  // the row totals that dominance_prefix_kernel accumulates start from nothing
  for (int j = wb * blockDim.x + threadIdx.x; j < n; j += workers * blockDim.x) {
    total0[j] = 0;
    witness0[j] = -1;
  }
  auto initial = [&](int k, int e) { return ((unsigned long long)ordered_key(xs[(int64_t)k * npad + e]) << 32) | (unsigned)e; };
  if (!radix_sort_segments(buf, m, n, initial, ctrl, gen0, spin_limit, order_lds, base, scratch)) return;
  for (int k = 0; k < m; ++k) {
    const unsigned long long* __restrict__ sorted = buf.pairs[0] + (int64_t)k * buf.kstride;
    for (int p = wb * blockDim.x + threadIdx.x; p < n; p += workers * blockDim.x) {
      const unsigned long long pr = coherent_load(&sorted[p]);
      const uint32_t key = (uint32_t)(pr >> 32);
      const int slot = slot_of[(int)(unsigned)(pr & 0xFFFFFFFFull)];
      int e = p + 1;
      if (e < n && (uint32_t)(coherent_load(&sorted[e]) >> 32) == key) {
        // a run of equal values: its end by bisection (the first position whose key is larger, or n)
        int lo = p + 2, hi = n;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if ((uint32_t)(coherent_load(&sorted[mid]) >> 32) > key)
            hi = mid;
          else
            lo = mid + 1;
        }
        e = lo;
      }
      pos[(int64_t)k * buf.kstride + slot] = p;
      upper[(int64_t)k * buf.kstride + slot] = e;
    }
  }
  if (wb == 0 && threadIdx.x == 0) param->orders_valid = 1;
}

// The same orders for populations of at most kMidArgsortRows rows, in two launches without a wait between
// workgroups (the radix sort above spends 160 us on its twelve grid barriers whatever the size): the workgroups share
// the objectives out, and each produces a run of positions of its objective's order from all keys of that objective
// in its LDS (mid_argsort_slice); a second kernel derives pos and upper from the sorted pairs.
// Grid: any (one workgroup per compute unit).  Dynamic LDS: mid_sort_lds_bytes(n).
template <bool WIDE>
__global__ __launch_bounds__(kMidArgsortThreads) void objective_order_lds_kernel(const float* __restrict__ xs, int npad, int n, int m,
                                                                                 const SortParam* __restrict__ param,
                                                                                 const Ctrl* __restrict__ ctrl,
                                                                                 int* __restrict__ total0, int* __restrict__ witness0,
                                                                                 RadixBuffers buf) {
  extern __shared__ __attribute__((aligned(16))) uint64_t order_sort_lds[];
  if (param->nonfinite != 0 || ctrl->err != 0) return;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
    total0[j] = 0;
    witness0[j] = -1;
  }
  const int nb = (int)gridDim.x;
  const int per_objective = nb >= m ? nb / m : 1;  // workgroups that share an objective
  const int run = ((n + per_objective - 1) / per_objective + 15) & ~15;
  for (int item = blockIdx.x; item < per_objective * m; item += nb) {
    const int k = item % m, s0 = (item / m) * run;
    if (s0 >= n) continue;
    const float* __restrict__ col = xs + (int64_t)k * npad;
    unsigned long long* __restrict__ sorted = buf.pairs[0] + (int64_t)k * buf.kstride;
    mid_argsort_slice<WIDE>(
        order_sort_lds, n, s0, s0 + run, [&](int e) { return ordered_key(col[e]); },
        [&](int p, int e) { sorted[p] = ((unsigned long long)ordered_key(col[e]) << 32) | (unsigned)e; });
  }
}

// The same orders for larger populations, still without a wait between workgroups, in two launches: the rows are cut into `parts`
// shares of every objective's order, and a workgroup places the rows of one share.
// Rows are composites (key << 20 | original index: distinct, below 2^52).  Every workgroup of an objective sorts the
// same kOrderStreamSample composites (rows n i / sample); the composites between two of them are a share, which makes `parts` shares of
// about n / parts rows whatever the values are, equal ones included.
//  1. objective_shares_kernel: a workgroup takes `per` consecutive rows and groups them by their share, by bisection in the sample; where
//     the groups begin is left in offsets[objective][chunk][share].
//  2. objective_order_stream_kernel: a workgroup collects its share's groups in LDS, places them and writes its run of the order, and
//     positions and bounds by slot.  A share that does not fit `capacity` entries -- rows arranged so that the sample
//     misses where they crowd -- is taken in pieces instead, each collected in a pass over all keys: the largest stretch of composites from
//     the share's start that fits is found by bisection over the composites, a pass per step, as often as it takes.
// Placing is by buckets (of equal width in the value; where they crowd, of the index for the rows of the share's first and last
// value), every entry among those of its bucket; the network of radix.hpp only sorts what crowds in both.
// A workgroup that read all keys of its objective for its share, and sorted that by the network, took 78 us of vector issue for the
// reading alone at 200 000 rows (96 us, 20 more for positions and bounds in a launch of their own; 160 us and more by the radix sort
// above); now 15 + 42 us at 200 003 x 3 and 20 + 57 at 200 000 x 8: 7 the sample, 8 to 10 fetching the groups (chains of two reads), 9 to 13 the
// placing, 12 to 18 the scattered positions and bounds.
// Grid: m * parts workgroups of kOrderStreamThreads each.  Dynamic LDS: kOrderStreamLdsBytes.  n <= 2^20.
constexpr int kOrderStreamThreads = 1024;
constexpr int kOrderStreamCapacity = 16384;
constexpr int kOrderStreamPer = kOrderStreamCapacity / kOrderStreamThreads;
constexpr int kOrderStreamBuckets = 4 * kOrderStreamThreads;
constexpr uint32_t kOrderStreamCrowd = 48;  // entries of a bucket up to which every one looks at every other one
constexpr int kOrderStreamSample = 2048;
constexpr int kOrderStreamMaxRows = 1 << 20;
constexpr int kOrderStreamShare = 8192;  // rows of a share, at most, that the host aims at
constexpr int kOrderChunkPer = kOrderStreamShare / kOrderStreamThreads;  // rows of a thread in the first launch
constexpr int kOrderStreamMaxParts = 128;
// Words of the offsets and of the shares' bounds (two each), the first launch's other result.
__host__ __device__ inline size_t order_offsets_words(int m, int parts) { return (size_t)m * (size_t)parts * (size_t)(parts + 1); }
__host__ __device__ inline size_t order_bounds_words(int m, int parts) { return 2 * (size_t)m * (size_t)(parts + 1); }
constexpr size_t kOrderStreamLdsBytes = 8 * (size_t)kOrderStreamCapacity + 4 * (size_t)kOrderStreamBuckets;

// The rest of order_stream_place<PER, true> once some buckets crowd: cnt holds where the buckets begin, `held` the sizes of the thread's four and
// `run` where the first of them begins.  False, with comp as it was, if a crowded bucket holds several values.  word: one word.
template <int PER, typename BUCKET>
__device__ inline bool order_sample_place(unsigned long long* comp, const unsigned long long (&mine)[PER], int count, uint4 held, uint32_t run,
                                          uint32_t* cnt, uint32_t* word, BUCKET bucket_of_entry) {
  constexpr int kWaves = kOrderStreamThreads / 64;
  constexpr int kEntries = PER * kOrderStreamThreads;
  constexpr int kMostCrowded = kEntries / (int)(kOrderStreamCrowd + 1u);  // crowded buckets, at most
  static_assert(PER * kWaves * kMostCrowded <= 2 * kEntries, "the table takes the composites' place");
  static_assert(kEntries < (1 << 16) && kMostCrowded < (1 << 8), "number << 16 | first place");
  __shared__ uint32_t key_of[kMostCrowded];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // the crowded buckets are numbered from 1 on
  if (tid == 0) *word = 0u;
  __syncthreads();
  const uint32_t size[4] = {held.x, held.y, held.z, held.w};
  uint32_t first_of = run;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (size[i] > kOrderStreamCrowd) cnt[4 * tid + i] = (atomicAdd(word, 1u) + 1u) << 16 | first_of;
    first_of += size[i];
  }
  __syncthreads();
  uint32_t bucket[PER], number[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const bool live = tid + kOrderStreamThreads * r < count;
    bucket[r] = live ? bucket_of_entry(mine[r]) : 0u;
    number[r] = live ? cnt[bucket[r]] >> 16 : 0u;
    if (number[r] != 0u) key_of[number[r] - 1u] = (uint32_t)(mine[r] >> 20);  // (any member's)
  }
  __syncthreads();
  bool other = false;
#pragma unroll
  for (int r = 0; r < PER; ++r) other |= number[r] != 0u && key_of[number[r] - 1u] != (uint32_t)(mine[r] >> 20);
  if (__syncthreads_or(other)) return false;
  // members of a wave per crowded bucket, and how many lie in front of each
  uint32_t* const table = reinterpret_cast<uint32_t*>(comp);
  for (int i = tid; i < PER * kWaves * kMostCrowded; i += kOrderStreamThreads) table[i] = 0u;
  __syncthreads();
  uint32_t place[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    place[r] = 0u;
    uint64_t left = __builtin_amdgcn_ballot_w64(number[r] != 0u);
    while (left != 0ull) {  // (wave-uniform)
      const int at = __builtin_ctzll(left);
      const uint32_t of = (uint32_t)__builtin_amdgcn_readlane((int)number[r], at);
      const uint64_t same = __builtin_amdgcn_ballot_w64(number[r] == of);
      if (number[r] == of) place[r] = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
      if (lane == at) table[(r * kWaves + wave) * kMostCrowded + (int)of - 1] = (uint32_t)__popcll(same);
      left &= ~same;
    }
  }
  __syncthreads();
  if (tid < kMostCrowded) {
    uint32_t before = 0u;
    for (int w = 0; w < PER * kWaves; ++w) {
      const uint32_t here = table[w * kMostCrowded + tid];
      table[w * kMostCrowded + tid] = before;
      before += here;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER; ++r)
    if (number[r] != 0u) place[r] += (cnt[bucket[r]] & 0xFFFFu) + table[(r * kWaves + wave) * kMostCrowded + (int)number[r] - 1];
  __syncthreads();
  // (the others anywhere in their bucket, then by the members below them)
  uint32_t first[PER], end[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    first[r] = cnt[bucket[r]] & 0xFFFFu;
    end[r] = bucket[r] + 1u < (uint32_t)kOrderStreamBuckets ? cnt[bucket[r] + 1u] & 0xFFFFu : (uint32_t)count;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    if (tid + kOrderStreamThreads * r < count) {
      if (number[r] == 0u) place[r] = atomicAdd(&cnt[bucket[r]], 1u);
      comp[place[r]] = mine[r];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    if (tid + kOrderStreamThreads * r < count && number[r] == 0u) {
      place[r] = first[r];
      for (uint32_t q = first[r]; q < end[r]; ++q) place[r] += comp[q] < mine[r] ? 1u : 0u;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER; ++r)
    if (tid + kOrderStreamThreads * r < count) comp[place[r]] = mine[r];
  __syncthreads();
  return true;
}

// Places of `count` composites (entry tid + kOrderStreamThreads r of comp is `mine[r]`) in ascending order, by buckets; afterwards
// comp[place] holds them in that order.  False, with comp as it was, when they crowd.  cnt: kOrderStreamBuckets words; part, lo16, hi16: sixteen
// words each.  Every thread calls it, past a barrier behind the last write of comp; ends with one.
// BY_INDEX: the entries lie in the order of their indices, so that the members of a crowded bucket of one value need only be counted, a wave's
// by a ballot (half of 60 000 x 4 rows of four levels selected: 387 us where the middle levels of the sample went to the network, now 378; uniform values 302 as before).
template <int PER, bool BY_INDEX = false>
__device__ inline bool order_stream_place(unsigned long long* comp, int count, uint32_t* cnt, uint32_t* part, uint32_t* lo16, uint32_t* hi16) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int kWaves = kOrderStreamThreads / 64;
  constexpr unsigned long long kMask = (1ull << 52) - 1ull;
  unsigned long long mine[PER];
  uint32_t lo = 0xFFFFFFFFu, hi = 0u;
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int e = tid + kOrderStreamThreads * r;
    mine[r] = 0ull;
    if (e < count) {
      mine[r] = comp[bitonic_slot(e)] & kMask;
      const uint32_t key = (uint32_t)(mine[r] >> 20);
      lo = min(lo, key);
      hi = max(hi, key);
    }
  }
  const uint32_t wave_lo = wave_prefix_min(lo), wave_hi = ~wave_prefix_min(~hi);
  if (lane == 63) {
    lo16[wave] = wave_lo;
    hi16[wave] = wave_hi;
  }
  __syncthreads();
  for (int w = 0; w < kWaves; ++w) {
    lo = min(lo, lo16[w]);
    hi = max(hi, hi16[w]);
  }
  // (by value: finite values only; by ends: the rows of the smallest and of the largest value by their index, a quarter of the buckets each,
  // the others by value in between -- shares of one value or two)
  const float v0 = cost_of_key(lo), width = cost_of_key(hi) - v0;
  const bool by_value = lo < hi && width > 0.0f && width <= 3.4028234663852886e38f;
  const float scale = by_value ? (float)(kOrderStreamBuckets - 1) / width : 0.0f;
  uint32_t first_lo = 0u, first_hi = 0u;
  float scale_lo = 0.0f, scale_hi = 0.0f;
#pragma unroll 1
  for (int attempt = by_value ? 0 : 1; attempt < 2; ++attempt) {
    if (attempt == 1) {
      // the smallest and the largest index with either value
      uint32_t at[4] = {~0u, ~0u, ~0u, ~0u};
#pragma unroll
      for (int r = 0; r < PER; ++r) {
        if (tid + kOrderStreamThreads * r < count) {
          const uint32_t key = (uint32_t)(mine[r] >> 20), index = (uint32_t)(mine[r] & 0xFFFFFull);
          if (key == lo) at[0] = min(at[0], index), at[1] = min(at[1], ~index);
          if (key == hi) at[2] = min(at[2], index), at[3] = min(at[3], ~index);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t of_wave = wave_prefix_min(at[i]);
        if (lane == 63) cnt[16 * i + wave] = of_wave;
      }
      __syncthreads();
      for (int w = 0; w < kWaves; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) at[i] = min(at[i], cnt[16 * i + w]);
      __syncthreads();
      first_lo = at[0];
      first_hi = at[2];
      scale_lo = (float)(kOrderStreamBuckets / 4 - 1) / (float)(~at[1] - at[0] + 1u);
      scale_hi = (float)(kOrderStreamBuckets / 4 - 1) / (float)(~at[3] - at[2] + 1u);
    }
    auto bucket_of_entry = [&](unsigned long long c) -> uint32_t {
      const uint32_t key = (uint32_t)(c >> 20), index = (uint32_t)(c & 0xFFFFFull);
      const uint32_t t = by_value ? min((uint32_t)((cost_of_key(key) - v0) * scale), (uint32_t)kOrderStreamBuckets - 1u) : 0u;
      if (attempt == 0) return t;
      constexpr uint32_t kQuarter = (uint32_t)kOrderStreamBuckets / 4u;
      if (key == lo) return min((uint32_t)((float)(index - first_lo) * scale_lo), kQuarter - 1u);
      if (key == hi) return 3u * kQuarter + min((uint32_t)((float)(index - first_hi) * scale_hi), kQuarter - 1u);
      return kQuarter + t / 2u;
    };
    reinterpret_cast<uint4*>(cnt)[tid] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    uint32_t arrived[(PER + 1) / 2];  // (two to a word)
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const uint32_t at = tid + kOrderStreamThreads * r < count ? atomicAdd(&cnt[bucket_of_entry(mine[r])], 1u) : 0u;
      if (r & 1)
        arrived[r >> 1] |= at << 16;
      else
        arrived[r >> 1] = at;
    }
    __syncthreads();
    const uint4 held = reinterpret_cast<const uint4*>(cnt)[tid];
    const uint32_t sum = held.x + held.y + held.z + held.w;
    uint32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    if (lane == 63) part[wave] = incl;
    const bool crowded = __syncthreads_or(max(max(held.x, held.y), max(held.z, held.w)) > kOrderStreamCrowd) != 0;
    if (crowded && (!BY_INDEX || attempt == 1)) continue;
    uint32_t run = incl - sum;
    for (int w = 0; w < wave; ++w) run += part[w];
    reinterpret_cast<uint4*>(cnt)[tid] = make_uint4(run, run + held.x, run + held.x + held.y, run + held.x + held.y + held.z);
    __syncthreads();
    if constexpr (BY_INDEX) {
      if (__builtin_expect(crowded, 0)) {
        if (order_sample_place<PER>(comp, mine, count, held, run, cnt, lo16, bucket_of_entry)) return true;
        continue;
      }
    }
#pragma unroll
    for (int r = 0; r < PER; ++r)
      if (tid + kOrderStreamThreads * r < count) comp[cnt[bucket_of_entry(mine[r])] + ((arrived[r >> 1] >> (16 * (r & 1))) & 0xFFFFu)] = mine[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      if (tid + kOrderStreamThreads * r < count) {
        const uint32_t bucket = bucket_of_entry(mine[r]);
        const uint32_t first = cnt[bucket], end = bucket + 1u < (uint32_t)kOrderStreamBuckets ? cnt[bucket + 1u] : (uint32_t)count;
        uint32_t before = 0u;
        for (uint32_t q = first; q < end; q += 4) {  // (four members' reads in flight together)
#pragma unroll
          for (int u = 0; u < 4; ++u) before += comp[min(q + (uint32_t)u, end - 1u)] < mine[r] && q + (uint32_t)u < end ? 1u : 0u;
        }
        const uint32_t place = first + before;
        if (r & 1)
          arrived[r >> 1] = (arrived[r >> 1] & 0xFFFFu) | place << 16;
        else
          arrived[r >> 1] = (arrived[r >> 1] & 0xFFFF0000u) | place;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; ++r)
      if (tid + kOrderStreamThreads * r < count) comp[(arrived[r >> 1] >> (16 * (r & 1))) & 0xFFFFu] = mine[r];
    __syncthreads();
    return true;
  }
  return false;
}

constexpr unsigned long long kOrderBias = 0x4330000000000000ull;  // the bits of 2^52 as a double
constexpr unsigned long long kOrderEnd = 1ull << 52;               // above every composite

// per = ceil(n / parts) <= kOrderStreamShare.  grouped[k * kstride + row's place]: the composites of a chunk by share.
__global__ __launch_bounds__(kOrderStreamThreads) void objective_shares_kernel(const float* __restrict__ xs, int npad, int n, int m, int parts,
                                                                               int per, const SortParam* __restrict__ param,
                                                                               const Ctrl* __restrict__ ctrl, int* __restrict__ total0,
                                                                               int* __restrict__ witness0, int kstride,
                                                                               unsigned long long* __restrict__ grouped,
                                                                               uint32_t* __restrict__ offsets,
                                                                               unsigned long long* __restrict__ bounds) {
  extern __shared__ __attribute__((aligned(16))) double order_shares_lds[];
  __shared__ uint32_t part16[16];
  __shared__ uint32_t lo16[16];
  __shared__ uint32_t hi16[16];
  __shared__ unsigned long long bound_lds[kOrderStreamMaxParts + 1];
  __shared__ uint32_t group[kOrderStreamMaxParts];
  if (param->nonfinite != 0 || ctrl->err != 0) return;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
    total0[j] = 0;
    witness0[j] = -1;
  }
  double* const comp = order_shares_lds;
  unsigned long long* const composites = reinterpret_cast<unsigned long long*>(order_shares_lds);
  uint32_t* const cnt = reinterpret_cast<uint32_t*>(order_shares_lds + kOrderStreamSample);
  const int tid = threadIdx.x, lane = tid & 63;
  const int k = (int)blockIdx.x % m, chunk = (int)blockIdx.x / m;
  const float* __restrict__ col = xs + (int64_t)k * npad;
  const int e0 = min(chunk * per, n), e1 = min(e0 + per, n);
  uint32_t key[kOrderChunkPer];
#pragma unroll
  for (int r = 0; r < kOrderChunkPer; ++r) {  // (asked for ahead of the sample's sort)
    const int e = e0 + tid + kOrderStreamThreads * r;
    key[r] = e < e1 ? ordered_key(col[e]) : 0u;
  }
  for (int i = tid; i < kOrderStreamSample; i += kOrderStreamThreads) {
    const int e = (int)(((int64_t)i * n) / kOrderStreamSample);
    comp[bitonic_slot(i)] =
        __longlong_as_double((long long)(kOrderBias | (unsigned long long)ordered_key(col[e]) << 20 | (unsigned long long)(unsigned)e));
  }
  if (tid < kOrderStreamMaxParts) group[tid] = 0u;
  __syncthreads();
  const bool placed = order_stream_place<kOrderStreamSample / kOrderStreamThreads, true>(composites, kOrderStreamSample, cnt, part16, lo16, hi16);
  if (!placed) bitonic_sort_lds(comp, kOrderStreamSample);
  if (tid <= parts) {
    const int i = (int)(((int64_t)tid * kOrderStreamSample) / parts);
    const unsigned long long b = tid == 0 ? 0ull : tid == parts ? kOrderEnd : composites[placed ? i : bitonic_slot(i)] & (kOrderEnd - 1ull);
    bound_lds[tid] = b;
    if (chunk == 0) bounds[k * (parts + 1) + tid] = b;
  }
  __syncthreads();
  uint32_t where[kOrderChunkPer];  // share << 16 | place in its group
#pragma unroll
  for (int r = 0; r < kOrderChunkPer; ++r) {
    const int e = e0 + tid + kOrderStreamThreads * r;
    where[r] = 0u;
    if (e < e1) {
      const unsigned long long c = (unsigned long long)key[r] << 20 | (unsigned long long)(unsigned)e;
      int from = 0, until = parts;  // bound_lds[from] <= c < bound_lds[until]
      while (until - from > 1) {
        const int mid = (from + until) >> 1;
        if (bound_lds[mid] <= c)
          from = mid;
        else
          until = mid;
      }
      where[r] = (uint32_t)from << 16 | atomicAdd(&group[from], 1u);
    }
  }
  __syncthreads();
  if (tid < 64) {
    uint32_t before = 0u;
#pragma unroll
    for (int half = 0; half < kOrderStreamMaxParts / 64; ++half) {
      const uint32_t mine = group[64 * half + lane];
      uint32_t incl = mine;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t up = __shfl_up(incl, off);
        if (lane >= off) incl += up;
      }
      group[64 * half + lane] = before + incl - mine;
      before += __shfl(incl, 63);
    }
  }
  __syncthreads();
  unsigned long long* __restrict__ const out = grouped + (int64_t)k * kstride + e0;
#pragma unroll
  for (int r = 0; r < kOrderChunkPer; ++r) {
    const int e = e0 + tid + kOrderStreamThreads * r;
    if (e < e1) out[group[where[r] >> 16] + (where[r] & 0xFFFFu)] = (unsigned long long)key[r] << 20 | (unsigned long long)(unsigned)e;
  }
  uint32_t* __restrict__ const off = offsets + ((int64_t)k * parts + chunk) * (parts + 1);
  if (tid <= parts) off[tid] = tid < parts ? group[tid] : (uint32_t)(e1 - e0);
}

__global__ __launch_bounds__(kOrderStreamThreads) void objective_order_stream_kernel(const float* __restrict__ xs, int npad, int n, int m,
                                                                                     int parts, int per, int capacity,
                                                                                     const int* __restrict__ slot_of,
                                                                                     SortParam* __restrict__ param,
                                                                                     const Ctrl* __restrict__ ctrl,
                                                                                     const uint32_t* __restrict__ offsets,
                                                                                     const unsigned long long* __restrict__ bounds,
                                                                                     int* __restrict__ pos, int* __restrict__ upper,
                                                                                     RadixBuffers buf) {
  extern __shared__ __attribute__((aligned(16))) double order_stream_comp[];
  __shared__ int taken;           // composites of the present pass that lie in its range
  __shared__ int below_of[16];    // per wave: composites below the range
  __shared__ int upto_of[16];     // per wave: values up to that of the range's end
  __shared__ uint32_t part16[16];
  __shared__ uint32_t lo16[16];
  __shared__ uint32_t hi16[16];
  __shared__ int group_first[kOrderStreamMaxParts];  // of a chunk's rows of this share: the first one in the chunk, their number, their place here
  __shared__ int group_rows[kOrderStreamMaxParts];
  __shared__ int group_at[kOrderStreamMaxParts];
  __shared__ int share_rows;
  __shared__ int share_below;
  if (param->nonfinite != 0 || ctrl->err != 0) return;
  double* const comp = order_stream_comp;
  unsigned long long* const composites = reinterpret_cast<unsigned long long*>(order_stream_comp);
  uint32_t* const cnt = reinterpret_cast<uint32_t*>(order_stream_comp + kOrderStreamCapacity);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k = (int)blockIdx.x % m, part = (int)blockIdx.x / m;
  if (blockIdx.x == 0 && tid == 0) param->orders_valid = 1;
  const float* __restrict__ col = xs + (int64_t)k * npad;
  const unsigned long long* __restrict__ grouped = buf.pairs[1] + (int64_t)k * buf.kstride;
  unsigned long long* __restrict__ sorted = buf.pairs[0] + (int64_t)k * buf.kstride;
  int* __restrict__ const pos_k = pos + (int64_t)k * buf.kstride;
  int* __restrict__ const upper_k = upper + (int64_t)k * buf.kstride;
  constexpr unsigned long long kBias = kOrderBias, kEnd = kOrderEnd;
  auto as_entry = [&](unsigned long long c) { return __longlong_as_double((long long)(kBias | c)); };

  // ---- the share: between two members of the sorted sample, a group of every chunk
  unsigned long long lo = bounds[k * (parts + 1) + part];
  const unsigned long long end = bounds[k * (parts + 1) + part + 1];
  auto groups_of = [&](int share) {  // (called by every thread, past the last use of the lists; ends with a barrier)
    if (wave == 0) {
      int rows = 0, below = 0;
#pragma unroll
      for (int half = 0; half < kOrderStreamMaxParts / 64; ++half) {
        const int c = 64 * half + lane;
        const uint32_t* const off = offsets + ((int64_t)k * parts + min(c, parts - 1)) * (parts + 1) + share;
        const int first = c < parts ? (int)off[0] : 0, here = c < parts ? (int)off[1] - first : 0;
        int incl = here, firsts = first;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int up = __shfl_up(incl, o), up_first = __shfl_up(firsts, o);
          if (lane >= o) {
            incl += up;
            firsts += up_first;
          }
        }
        group_first[c] = first;
        group_rows[c] = here;
        group_at[c] = rows + incl - here;
        rows += __shfl(incl, 63);
        below += __shfl(firsts, 63);
      }
      if (lane == 0) {
        share_rows = rows;
        share_below = below;
      }
    }
    __syncthreads();
  };
  groups_of(part);

  // One pass over the objective's keys: the composites in [from, to) are counted (the return value) and, with `collect`,
  // the first `capacity` of them stored; *below = the composites smaller than `from`, *upto = the rows whose value is at most that
  // of `to`.  Most keys are told by two comparisons of floats (all are finite), the others by their composites.
  constexpr uint32_t kLowest = 0x00800000u, kHighest = 0xFF7FFFFFu;  // the keys of the finite values
  auto value_of = [&](uint32_t key) {  // (a bound of a bisection need not be the key of a value)
    return key < kLowest ? -INFINITY : key > kHighest ? INFINITY : cost_of_key(key);
  };
  auto pass = [&](unsigned long long from, unsigned long long to, bool collect, int* below, int* upto) {
    if (tid == 0) taken = 0;
    __syncthreads();
    const unsigned long long span = to - from;
    const float from_value = value_of((uint32_t)(from >> 20)), to_value = to == kEnd ? INFINITY : value_of((uint32_t)(to >> 20));
    int under = 0, most = 0;  // (wave-uniform)
    // (a wave takes 256 keys a step and fetches the keys of kAhead steps before it looks at the first of them)
    constexpr int kAhead = 8;
    for (int g0 = 256 * wave; g0 < n; g0 += kAhead * 4 * kOrderStreamThreads) {  // (wave-uniform)
      float4 q[kAhead];
#pragma unroll
      for (int a = 0; a < kAhead; ++a) {
        const int e0 = g0 + a * 4 * kOrderStreamThreads + 4 * lane;
        q[a] = make_float4(INFINITY, INFINITY, INFINITY, INFINITY);  // (beyond every value; in no range, whose last value is `to`'s or the largest one)
        if (e0 + 3 < n) {
          q[a] = *reinterpret_cast<const float4*>(col + e0);
        } else if (e0 < n) {
          q[a].x = col[e0];
          if (e0 + 1 < n) q[a].y = col[e0 + 1];
          if (e0 + 2 < n) q[a].z = col[e0 + 2];
        }
      }
#pragma unroll
      for (int a = 0; a < kAhead; ++a) {
        const int b0 = g0 + a * 4 * kOrderStreamThreads;
        if (b0 >= n) break;  // (wave-uniform)
        const int e0 = b0 + 4 * lane;
        const float v[4] = {q[a].x, q[a].y, q[a].z, q[a].w};
        uint64_t near[4];
        uint64_t any = 0ull;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint64_t less = __builtin_amdgcn_ballot_w64(v[u] < from_value);
          const uint64_t least = __builtin_amdgcn_ballot_w64(v[u] <= to_value);
          near[u] = least & ~less;
          under += __popcll(less);
          most += __popcll(least);
          any |= near[u];
        }
        if (any != 0ull) {  // (wave-uniform)
          unsigned long long c[4];
          uint64_t in[4];
          int here = 0;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            c[u] = ((unsigned long long)ordered_key(v[u]) << 20) | (unsigned long long)(unsigned)(e0 + u);
            const bool live = (near[u] >> lane & 1ull) != 0ull && e0 + u < n;
            in[u] = __builtin_amdgcn_ballot_w64(live && c[u] - from < span);
            under += __popcll(__builtin_amdgcn_ballot_w64(live && c[u] < from));
            here += __popcll(in[u]);
          }
          if (here != 0) {  // (wave-uniform)
            int at = 0;
            if (lane == 0) at = atomicAdd(&taken, here);
            at = __builtin_amdgcn_readfirstlane(at);
            if (collect) {
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const int mine = at + __popcll(in[u] & ((1ull << lane) - 1ull));
                if (((in[u] >> lane) & 1ull) != 0ull && mine < capacity) comp[bitonic_slot(mine)] = as_entry(c[u]);
                at += __popcll(in[u]);
              }
            }
          }
        }
      }
    }
    if (lane == 0) {
      below_of[wave] = under;
      upto_of[wave] = most;
    }
    __syncthreads();
    if (below != nullptr) {
      int sum = 0, sum_upto = 0;
#pragma unroll
      for (int w = 0; w < kOrderStreamThreads / 64; ++w) {
        sum += below_of[w];
        sum_upto += upto_of[w];
      }
      *below = sum;
      *upto = sum_upto;
    }
    const int count = taken;
    __syncthreads();  // (everybody has read the counters before the next pass clears them)
    return count;
  };

  const bool whole = share_rows <= capacity;  // (the same in every thread, as all that steers the loop)
  while (lo < end) {
    unsigned long long hi = end;
    int below = share_below, upto = 0, count = share_rows;
    if (whole) {
      // thirty-two lanes to a group
      for (int c = tid >> 5; c < parts; c += kOrderStreamThreads / 32) {
        const unsigned long long* __restrict__ const from = grouped + (int64_t)c * per + group_first[c];
        for (int i = tid & 31; i < group_rows[c]; i += 32) comp[bitonic_slot(group_at[c] + i)] = as_entry(from[i]);
      }
      __syncthreads();
    } else {
      count = pass(lo, hi, true, &below, &upto);
      // [lo, fits) holds at most one composite; [lo, over) too many
      unsigned long long fits = lo + 1ull, over = hi;
      if (count > capacity) {
        while (over - fits > 1ull) {
          const unsigned long long mid = fits + (over - fits) / 2ull;
          if (pass(lo, mid, false, nullptr, nullptr) <= capacity)
            fits = mid;
          else
            over = mid;
        }
        hi = fits;
        count = pass(lo, hi, true, &below, &upto);
      }
    }
    if (count > 0) {
      bool placed;
      if (count <= 4 * kOrderStreamThreads)
        placed = order_stream_place<4>(composites, count, cnt, part16, lo16, hi16);
      else if (count <= 8 * kOrderStreamThreads)
        placed = order_stream_place<8>(composites, count, cnt, part16, lo16, hi16);
      else
        placed = order_stream_place<kOrderStreamPer>(composites, count, cnt, part16, lo16, hi16);
      if (!placed) {
        int padded = kRowsBitonicMin;
        while (padded < count) padded <<= 1;
        for (int e = count + tid; e < padded; e += kOrderStreamThreads) comp[bitonic_slot(e)] = (double)INFINITY;
        __syncthreads();
        bitonic_sort_lds(comp, padded);
      }
      auto entry_at = [&](int e) { return composites[placed ? e : bitonic_slot(e)] & (kEnd - 1ull); };
      const uint32_t hi_key = (uint32_t)(hi >> 20);
      if (whole && hi < kEnd && (uint32_t)(entry_at(count - 1) >> 20) == hi_key) {
        // (rows of the last value lie in the next shares too, up to the last share that begins no later than that value ends)
        const unsigned long long* const bound = bounds + k * (parts + 1);
        int share = part + 1, behind = parts;  // bound[share] is of that value, bound[behind] of a larger one
        while (behind - share > 1) {
          const int mid = (share + behind) >> 1;
          if ((uint32_t)(bound[mid] >> 20) == hi_key)
            share = mid;
          else
            behind = mid;
        }
        __syncthreads();
        if (tid == 0) taken = 0;
        groups_of(share);
        int equal = 0;
        for (int c = tid >> 5; c < parts; c += kOrderStreamThreads / 32)
          for (int i = tid & 31; i < group_rows[c]; i += 32) equal += (uint32_t)(grouped[(int64_t)c * per + group_first[c] + i] >> 20) == hi_key ? 1 : 0;
        if (equal != 0) atomicAdd(&taken, equal);
        __syncthreads();
        upto = share_below + taken;
      }
      for (int e = tid; e < count; e += kOrderStreamThreads) {
        const unsigned long long c = entry_at(e);
        const uint32_t key = (uint32_t)(c >> 20);
        const int slot = slot_of[(int)(c & 0xFFFFFull)];
        sorted[below + e] = ((unsigned long long)key << 32) | (c & 0xFFFFFull);
        // the rows of its value or a smaller one: up to the first entry of a larger value, or beyond this range where `hi` cuts its value
        int last = e + 1;
        if (last < count && (uint32_t)(entry_at(last) >> 20) == key) {
          int from = e + 2, until = count;
          while (from < until) {
            const int mid = (from + until) >> 1;
            if ((uint32_t)(entry_at(mid) >> 20) > key)
              until = mid;
            else
              from = mid + 1;
          }
          last = from;
        }
        pos_k[slot] = below + e;
        upper_k[slot] = hi < kEnd && key == hi_key ? upto : below + last;
      }
      __syncthreads();
    }
    lo = hi;
  }
}

__global__ __launch_bounds__(256) void objective_positions_kernel(int n, int m, const int* __restrict__ slot_of,
                                                                  SortParam* __restrict__ param, const Ctrl* __restrict__ ctrl,
                                                                  int* __restrict__ pos, int* __restrict__ upper, RadixBuffers buf) {
  if (param->nonfinite != 0 || ctrl->err != 0) return;
  for (int64_t at = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; at < (int64_t)n * m; at += (int64_t)gridDim.x * blockDim.x) {
    const int k = (int)(at / n), p = (int)(at - (int64_t)k * n);
    const unsigned long long* __restrict__ sorted = buf.pairs[0] + (int64_t)k * buf.kstride;
    const unsigned long long pr = sorted[p];
    const uint32_t key = (uint32_t)(pr >> 32);
    const int slot = slot_of[(int)(unsigned)(pr & 0xFFFFFFFFull)];
    int e = p + 1;
    if (e < n && (uint32_t)(sorted[e] >> 32) == key) {
      // a run of equal values: its end by bisection (the first position whose key is larger, or n)
      int lo = p + 2, hi = n;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((uint32_t)(sorted[mid] >> 32) > key)
          hi = mid;
        else
          lo = mid + 1;
      }
      e = lo;
    }
    pos[(int64_t)k * buf.kstride + slot] = p;
    upper[(int64_t)k * buf.kstride + slot] = e;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) param->orders_valid = 1;
}

// The value that the neighbouring lane (lane ^ 1) passes in, by two DPP quad permutations.
__device__ inline uint64_t pair_exchange(uint64_t v) {
  const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)v, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
  const int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(v >> 32), 0xB1, 0xF, 0xF, true);
  return (uint64_t)(uint32_t)lo | ((uint64_t)(uint32_t)hi << 32);
}

// d[2p], d[2p+1] = the p-th 16-byte piece of this lane's row.  Afterwards they hold piece (lane & 3) of the row of
// lane (lane & ~3) + p: the 4 x 4 transpose of the pieces among four neighbouring lanes, in two exchanges (with the
// lane one away, then with the lane two away), every dword moved by one DPP quad permutation.
__device__ inline void quad_transpose_pieces(uint64_t (&d)[8], int lane) {
  int v[16];
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    v[2 * w] = (int)(uint32_t)d[w];
    v[2 * w + 1] = (int)(uint32_t)(d[w] >> 32);
  }
  const bool odd = (lane & 1) != 0, high = (lane & 2) != 0;
  // piece p occupies v[4p .. 4p+3]
#pragma unroll
  for (int h = 0; h < 2; ++h)  // pieces 2h and 2h+1 against the lane one away
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      int& even = v[4 * (2 * h) + x];
      int& oddp = v[4 * (2 * h + 1) + x];
      const int send = odd ? even : oddp;
      const int recv = __builtin_amdgcn_mov_dpp(send, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
      even = odd ? recv : even;
      oddp = odd ? oddp : recv;
    }
#pragma unroll
  for (int h = 0; h < 2; ++h)  // pieces h and h+2 against the lane two away
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      int& low = v[4 * h + x];
      int& hi = v[4 * (h + 2) + x];
      const int send = high ? low : hi;
      const int recv = __builtin_amdgcn_mov_dpp(send, 0x4E, 0xF, 0xF, true);  // quad_perm [2,3,0,1]
      low = high ? recv : low;
      hi = high ? hi : recv;
    }
#pragma unroll
  for (int w = 0; w < 8; ++w) d[w] = (uint64_t)(uint32_t)v[2 * w] | ((uint64_t)(uint32_t)v[2 * w + 1] << 32);
}

// ---- The row totals alone, without the matrix: nothing is written where a tile's words would lie, so the rows need not be
// in slot order.  In spatial order -- by the leading bits of their positions, an objective's after the other's -- a tile of
// 512 rows and a group of 64 rows lie in boxes of their own, and a tile whose box does not lie below the group's in
// every objective holds no dominator of its rows: of the pairs of tile and group 13 % are left at 200 000 x 8 (directions
// on a sphere), 17 % for uniform fitness, where the triangle of the slot order is 50 %.  The order of the slots is one
// more objective: a dominator's slot lies before the first slot with the row's key, which leaves out the row itself and
// its equals.
// 200 000 x 8, us: the order 68 (cells 16, gather 22, pairs 16), the totals 251 -- LDS look-ups as before, a quarter as many --
// against 760 in slot order; the selection 1176 -> 743.
constexpr int kNearbyCodeBits = 12;
constexpr int kNearbyCells = 1 << kNearbyCodeBits;

// cell[slot] = the row's cell, place[slot] = its place among the rows of that cell, hist = the number of rows in every cell.
// A workgroup counts its rows in LDS and takes its places of a cell with one addition (an addition per row, and another one
// for its place: 19 us each at 200 000 rows).
constexpr int kNearbyCellThreads = 1024, kNearbyCellRows = 4;  // rows per thread
__global__ __launch_bounds__(kNearbyCellThreads) void nearby_cells_kernel(const int* __restrict__ pos, int n, int kstride, int m,
                                                                          const SortParam* __restrict__ param, uint16_t* __restrict__ cell,
                                                                          int* __restrict__ place, int* __restrict__ hist) {
  __shared__ int count[kNearbyCells];
  if (param->nonfinite != 0) return;
  for (int c = threadIdx.x; c < kNearbyCells; c += kNearbyCellThreads) count[c] = 0;
  __syncthreads();
  const float scale = 4096.0f / (float)n;
  const int j0 = (int)blockIdx.x * kNearbyCellThreads * kNearbyCellRows + (int)threadIdx.x;
  uint32_t code[kNearbyCellRows] = {};
  int at[kNearbyCellRows];
  int bits = 0;
  for (int level = 11; bits < kNearbyCodeBits; --level)
    for (int k = 0; k < m && bits < kNearbyCodeBits; ++k, ++bits)
#pragma unroll
      for (int u = 0; u < kNearbyCellRows; ++u) {
        const int j = j0 + u * kNearbyCellThreads;
        const uint32_t q = j < n ? (uint32_t)((float)pos[(int64_t)k * kstride + j] * scale) : 0u;
        code[u] = (code[u] << 1) | ((q >> level) & 1u);
      }
#pragma unroll
  for (int u = 0; u < kNearbyCellRows; ++u) at[u] = j0 + u * kNearbyCellThreads < n ? atomicAdd(&count[code[u]], 1) : 0;
  __syncthreads();
  for (int c = threadIdx.x; c < kNearbyCells; c += kNearbyCellThreads) {
    const int mine = count[c];
    if (mine != 0) count[c] = atomicAdd(&hist[c], mine);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kNearbyCellRows; ++u) {
    const int j = j0 + u * kNearbyCellThreads;
    if (j < n) {
      cell[j] = (uint16_t)code[u];
      place[j] = count[code[u]] + at[u];
    }
  }
}

// slot_at[i] = the slot at place i of the spatial order (any order inside a cell: the totals do not depend on it).
__global__ __launch_bounds__(256) void nearby_scatter_kernel(const uint16_t* __restrict__ cell, const int* __restrict__ place, int n,
                                                             const SortParam* __restrict__ param, const Ctrl* __restrict__ ctrl,
                                                             const int* __restrict__ start, int* __restrict__ slot_at) {
  if (param->nonfinite != 0 || ctrl->err != 0) return;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) slot_at[start[cell[j]] + place[j]] = j;
}

// Order blockIdx.y (below m: that of an objective; m: that of the slots) of the rows at 256 places: positions and
// bounds by place (columns `stride` apart), and the box of every 64 places: smallest and
// largest position, largest bound.
__global__ __launch_bounds__(256) void nearby_gather_kernel(const int* __restrict__ pos, const int* __restrict__ upper,
                                                            const uint32_t* __restrict__ kid, int n, int kstride, int m,
                                                            const SortParam* __restrict__ param, const Ctrl* __restrict__ ctrl,
                                                            const int* __restrict__ slot_at, int stride, int* __restrict__ pos_at, int* __restrict__ upper_at, int group_stride,
                                                            int* __restrict__ group_lo, int* __restrict__ group_top,
                                                            int* __restrict__ group_hi) {
  if (param->nonfinite != 0 || ctrl->err != 0) return;
  const int k = blockIdx.y, i = blockIdx.x * 256 + (int)threadIdx.x;
  int p = 0x7FFFFFFF, top = 0, u = 0;
  if (i < n) {
    const int slot = slot_at[i];
    p = k < m ? pos[(int64_t)k * kstride + slot] : slot;
    u = k < m ? upper[(int64_t)k * kstride + slot] : (int)kid[slot];
    top = p;
    pos_at[(int64_t)k * stride + i] = p;
    upper_at[(int64_t)k * stride + i] = u;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    p = min(p, __shfl_xor(p, off));
    top = max(top, __shfl_xor(top, off));
    u = max(u, __shfl_xor(u, off));
  }
  const int group = i >> 6;
  if ((threadIdx.x & 63) == 0 && group < group_stride) {
    group_lo[(int64_t)k * group_stride + group] = p;
    group_top[(int64_t)k * group_stride + group] = top;
    group_hi[(int64_t)k * group_stride + group] = u;
  }
}

// The box of every tile, the groups that it can have dominators of (near[tile * groups ...]: the smallest position of the
// tile lies below the largest bound of the group in every objective), and the work: parts of `cap` groups of a tile's list in
// `full`, what is left of the lists in `rest`, counted in queue[0] and queue[1].  The tiles differ by a factor of fifty (a
// tile at the foot of the population is near to all groups): a workgroup per tile and quarter of the groups ended 200 us
// after the average one at 200 000 x 8.  A workgroup per tile.
template <int M>
__global__ __launch_bounds__(256) void nearby_pairs_kernel(const int* __restrict__ group_lo, const int* __restrict__ group_top,
                                                           const int* __restrict__ group_hi, int groups, int tile_groups, int cap,
                                                           const SortParam* __restrict__ param, const Ctrl* __restrict__ ctrl,
                                                           int* __restrict__ box, uint16_t* __restrict__ near_list, int* __restrict__ near_count,
                                                           int2* __restrict__ full, int2* __restrict__ rest, int* __restrict__ queue) {
  __shared__ int lo[M];
  __shared__ int found, first_item;
  if (param->nonfinite != 0 || ctrl->err != 0) return;
  const int tile = blockIdx.x, lane = threadIdx.x & 63;
  if (threadIdx.x == 0) found = 0;
  if ((int)threadIdx.x < M * 8) {  // (up to eight groups to a tile)
    const int k = (int)threadIdx.x >> 3, u = (int)threadIdx.x & 7, g = tile * tile_groups + u;
    const bool have = u < tile_groups && g < groups;
    int low = have ? group_lo[(int64_t)k * groups + g] : 0x7FFFFFFF;
    int top = have ? group_top[(int64_t)k * groups + g] : 0;
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
      low = min(low, __shfl_xor(low, off));
      top = max(top, __shfl_xor(top, off));
    }
    if (u == 0) {
      lo[k] = low;
      box[(tile * M + k) * 2] = low;
      box[(tile * M + k) * 2 + 1] = top;
    }
  }
  __syncthreads();
  uint16_t* const list = near_list + (int64_t)tile * groups;
  for (int g0 = 0; g0 < groups; g0 += blockDim.x) {
    const int g = g0 + (int)threadIdx.x;
    int hi[M];  // (all loads before any use)
#pragma unroll
    for (int k = 0; k < M; ++k) hi[k] = group_hi[(int64_t)k * groups + (g < groups ? g : 0)];
    bool near = g < groups;
#pragma unroll
    for (int k = 0; k < M; ++k) near &= lo[k] < hi[k];
    const uint64_t members = __builtin_amdgcn_ballot_w64(near);
    int at = 0;
    if (lane == 0 && members != 0ull) at = atomicAdd(&found, __popcll(members));
    at = __shfl(at, 0);
    if (near) list[at + __popcll(members & ((1ull << lane) - 1ull))] = (uint16_t)g;
  }
  __syncthreads();
  const int parts = found / cap;
  if (threadIdx.x == 0) {
    near_count[tile] = found;
    if (parts > 0) first_item = atomicAdd(&queue[0], parts);
    if (found > parts * cap) rest[atomicAdd(&queue[1], 1)] = make_int2(tile, parts);
  }
  __syncthreads();
  for (int p = threadIdx.x; p < parts; p += blockDim.x) full[first_item + p] = make_int2(tile, p);
}

// Inclusive scan over the 64 lanes of a wave: shifts inside the DPP rows of sixteen lanes, then a row's last lane to the
// rows behind it -- six vector instructions, where a permute through LDS is a round trip each.  op(0, v) == v.
template <class Op>
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, Op op) {
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));  // row_shr 1, 2, 4, 8
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));         // row_bcast 15: into rows 1 and 3
  return op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));      // row_bcast 31: into rows 2 and 3
}
template <class Op>
__device__ __forceinline__ uint64_t wave_scan_halves(uint64_t v, Op op) {  // (nothing passes from the lower half to the upper)
  return (uint64_t)wave_scan((uint32_t)v, op) | ((uint64_t)wave_scan((uint32_t)(v >> 32), op) << 32);
}

// A workgroup takes TT neighbouring tiles of WW words (TT = 2 with WW = 8: the whole 128-byte line of every row).
// grid.x = the ceil(nwords / (WW * TT)) tile groups of dominator slots, rounded up to a multiple of 128 / (WW * TT),
// grid.y = stretches of `chunk` rows, counted from the first row of the tile or (bands) from row 0 (rows above the
// tile have no word there).  Dynamic LDS: TT * prefix_lds_bytes(M, WW, buckets).  Writes the words of its tiles in
// every row of the stretch and adds their popcount to total0[row]; witness0[row] = the highest non-empty word so far
// (both start from objective_order_kernel's 0 and -1).  Sets param->totals_valid.  mode: bit 0 = the row totals,
// bit 1 = the matrix.  NEARBY: the totals alone, of rows in spatial order, by workgroups that take parts of
// the work until none is left.  unless_front0 (null: always run): the size of front 0, known from a launch with mode 1 and the
// count stage; when it holds `enough` rows nobody will read the matrix, and the launch (mode 2) does nothing.
struct NearbyWork {
  const int* box;         // [tile][objective]: smallest and largest position
  const uint16_t* near_list;  // [tile][groups]
  const int* near_count;
  const int2 *full, *rest;  // (tile, part of its list)
  int* queue;             // how many of either, and the next one to take
  int cap;                // groups per part, at most kPrefixNearbyGroups
};
template <int M, int WW, int TT, bool NEARBY = false>
__global__ __launch_bounds__(kPrefixThreads) void dominance_prefix_kernel(const int* __restrict__ pos, const int* __restrict__ upper,
                                                                          const uint32_t* __restrict__ kid,
                                                                          uint64_t* __restrict__ dom, int n, int kstride,
                                                                          int64_t wstride, int nwords, int shift, int buckets,
                                                                          int chunk, int bands, int mode, int* __restrict__ total0,
                                                                          int* __restrict__ witness0, SortParam* __restrict__ param,
                                                                          const Ctrl* __restrict__ ctrl, const int* __restrict__ unless_front0, int enough,
                                                                          NearbyWork work) {
  static_assert(!NEARBY || TT == 1, "a tile of rows in spatial order");
  constexpr int TS = 64 * WW, T = kPrefixThreads;
  constexpr int TPL = 16 / (WW * TT);  // workgroups that share a 128-byte line of the matrix
  constexpr int MPL = TS / 64;  // members of the tile per lane when a wave walks through them
  extern __shared__ uint64_t prefix_lds[];
  if (param->nonfinite != 0 || ctrl->err != 0) return;  // (after a failed wait nobody has written the positions, which index the tables)
  if (unless_front0 != nullptr && *unless_front0 >= enough) return;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) param->totals_valid = 1;  // for the count stage
  __shared__ uint16_t nearby[NEARBY ? kPrefixNearbyGroups : 1];
  __shared__ int nearby_item;
  __shared__ int tile_lo[M], tile_span[M], tile_shift[M];
  for (;;) {
  int tid = (int)threadIdx.x;
  // (what hangs on the thread alone is computed anew for every part: kept across them it took 128 registers and spilled)
  if constexpr (NEARBY) asm volatile("" : "+v"(tid));
  const int lane = tid & 63, wave = tid >> 6;
  int tile, r0 = 0, r1 = n, nearby_count = 0;
  if constexpr (NEARBY) {
    // the next part of the work; the grid ends when none is left
    __syncthreads();  // (the tables of the part before are no longer read)
    if (tid == 0) nearby_item = atomicAdd(&work.queue[2], 1);
    __syncthreads();
    const int item = nearby_item, fulls = work.queue[0];
    if (item >= fulls + work.queue[1]) return;
    const int2 part = item < fulls ? work.full[item] : work.rest[item - fulls];
    tile = part.x;
    nearby_count = min(work.cap, work.near_count[tile] - part.y * work.cap);
    for (int g = tid; g < nearby_count; g += T) nearby[g] = work.near_list[(int64_t)tile * nwords + part.y * work.cap + g];
    if (tid < M) {  // (positions of such a tile lie close together: its coarse index covers those only)
      const int low = work.box[(tile * M + tid) * 2], high = work.box[(tile * M + tid) * 2 + 1];
      int wide = 0;
      while (((high - low) >> wide) >= kPrefixBuckets) ++wide;
      tile_lo[tid] = low;
      tile_span[tid] = high - low + 1;  // (the bucket of every bound above the tile)
      tile_shift[tid] = wide;
    }
  } else {
    // Workgroups go to the eight dies in turn (linear index modulo 8), and a die has its own L2.  The tiles
    // that share the 128-byte lines of the matrix are given to consecutive workgroups of one die, which run
    // side by side over the same rows: their pieces of a line then meet in that L2 and leave as one line.
    const int64_t linear = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    const int die = (int)(linear & 7);
    const int seq = (int)blockIdx.x >> 3;  // this workgroup among those of its die in this row of the grid
    tile = TPL * ((seq / TPL) * 8 + die) + seq % TPL;
    if (tile * WW * TT >= nwords) return;
    const int first_slot = tile * WW * TT * 64;
    int64_t first_row = (int64_t)first_slot + (int64_t)blockIdx.y * chunk, end_row = first_row + chunk;
    if (bands) {  // the same rows for all tiles of a grid row: the tiles left of the diagonal in rows y * chunk ...
      first_row = (int64_t)blockIdx.y * chunk;
      end_row = first_row + chunk;
      if (first_row < first_slot) first_row = first_slot;
    }
    if (first_row >= n || first_row >= end_row) return;
    r0 = (int)first_row;
    r1 = (int)(end_row < n ? end_row : n);
  }
  const int w0 = tile * WW * TT;  // the first word of the workgroup's TT tiles (tile `sub` starts WW * sub words on)
  const int slot0 = w0 * 64;
  const int HB = buckets + 2;  // entries of the coarse index per objective
  // per objective k (all arrays [M][...]):
  constexpr int kSetWords = WW * 65;                 // sets[k][w][c]: the slots of the first c members of word w
  constexpr int kOver = kSetWords + TS + 1;          // ... then counts[k][t]: eight byte counts, members of each word among the first t
  const int scratch_words = (HB + TS + 1) / 2;       // histogram and claimed pairs of the build, in the same place
  const int over = kOver > scratch_words ? kOver : scratch_words;
  // the tables of tile `sub` of the workgroup (TT = 2: the two tiles of a 128-byte line, so that the workgroup writes
  // whole lines; their tables fit the LDS up to four objectives)
  const size_t tile_lds_words = prefix_lds_bytes(M, WW, buckets) / sizeof(uint64_t);
  uint64_t* tile_lds = prefix_lds;
  uint64_t* sets = nullptr;
  uint64_t* counts = nullptr;
  int* mp = nullptr;           // [M][TS + 8]: positions ascending, then INT_MAX
  int* sorted = nullptr;       // [M][TS]: position << 9 | slot in tile, ascending
  uint16_t* index = nullptr;   // [M][HB]: members in earlier buckets
  int live = 0;                // slots of the tile that hold a row
  int tile_slot0 = slot0;
  auto select_tile = [&](int sub) {
    tile_lds = prefix_lds + (size_t)sub * tile_lds_words;
    sets = tile_lds;
    counts = sets + kSetWords;
    mp = reinterpret_cast<int*>(tile_lds + (size_t)M * over);
    sorted = mp + M * (TS + 8);
    index = reinterpret_cast<uint16_t*>(sorted + M * TS);
    tile_slot0 = slot0 + sub * TS;
    live = n - tile_slot0 < TS ? n - tile_slot0 : TS;
  };
  auto hist_of = [&](int k) { return reinterpret_cast<int*>(tile_lds + (size_t)k * over); };  // [HB]
  auto claimed_of = [&](int k) { return hist_of(k) + HB; };                                      // [TS]
  const int index_stride = (HB + 3) & ~3;
  auto bucket_of_bound = [&](int k, int e) {  // the bucket of a bound; of a position p likewise
    if constexpr (!NEARBY) return e >> shift;
    const int past = e - tile_lo[k];
    return min(past > 0 ? past : 0, tile_span[k]) >> tile_shift[k];
  };

  for (int sub = 0; sub < TT; ++sub) {
  select_tile(sub);
  // ---- the tile's slots by position, objective by objective
  for (int t = tid; t < M * HB; t += T) hist_of(t / HB)[t % HB] = 0;
  for (int t = tid; t < M * (TS + 8); t += T) mp[t] = 0x7FFFFFFF;
  __syncthreads();
  constexpr int PER = (M * TS + T - 1) / T;
  int mine[PER];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int item = tid + u * T;
    const int k = item / TS, i = item - k * TS;
    mine[u] = -1;
    if (item < M * TS && i < live) {
      const int p = pos[(int64_t)k * kstride + tile_slot0 + i];
      mine[u] = (p << 9) | i;
      atomicAdd(&hist_of(k)[bucket_of_bound(k, p)], 1);
    }
  }
  __syncthreads();
  if (wave < M) {  // exclusive prefix of the bucket counts of objective `wave`: a lane adds up kPer consecutive buckets
    constexpr int kPer = (kPrefixBuckets + 2 + 63) / 64;  // (odd: the lanes' reads fall into different banks)
    int count[kPer], sum = 0;
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      const int b = lane * kPer + c;
      count[c] = b < HB ? hist_of(wave)[b] : 0;
      sum += count[c];
    }
    int before = (int)wave_scan((uint32_t)sum, [](uint32_t a, uint32_t b) { return a + b; }) - sum;
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      const int b = lane * kPer + c;
      if (b < HB) index[wave * index_stride + b] = (uint16_t)before;
      before += count[c];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    if (mine[u] >= 0) {
      const int k = (tid + u * T) / TS;
      const int b = bucket_of_bound(k, mine[u] >> 9);
      const int r = atomicSub(&hist_of(k)[b], 1) - 1;
      claimed_of(k)[(int)index[k * index_stride + b] + r] = mine[u];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    if (mine[u] >= 0) {
      const int k = (tid + u * T) / TS;
      const int b = bucket_of_bound(k, mine[u] >> 9);
      const int t0 = index[k * index_stride + b], t1 = index[k * index_stride + b + 1];
      int before = 0;
      for (int t = t0; t < t1; ++t) before += claimed_of(k)[t] < mine[u] ? 1 : 0;
      sorted[k * TS + t0 + before] = mine[u];
      mp[k * (TS + 8) + t0 + before] = mine[u] >> 9;
    }
  }
  __syncthreads();
  // ---- counts[k][t] and the single bits of sets[k][w][c + 1]; a wave per objective, a lane per MPL members
  for (int t = tid; t < M * kSetWords; t += T) sets[(size_t)(t / kSetWords) * over + t % kSetWords] = 0ull;
  __syncthreads();
  for (int k = wave; k < M; k += T / 64) {
    uint64_t one[MPL];
    uint64_t sum = 0ull;
#pragma unroll
    for (int c = 0; c < MPL; ++c) {
      const int t = MPL * lane + c;
      one[c] = t < live ? 1ull << (8 * ((sorted[k * TS + t] & (TS - 1)) >> 6)) : 0ull;
      sum += one[c];
    }
    // byte-wise counts: at most 64 per byte, no carry between bytes
    const uint64_t incl = wave_scan_halves(sum, [](uint32_t a, uint32_t b) { return a + b; });
    uint64_t run = incl - sum;  // members before this lane's eight
    uint64_t* const cnt = counts + (size_t)k * over;
    uint64_t* const set = sets + (size_t)k * over;
#pragma unroll
    for (int c = 0; c < MPL; ++c) {
      const int t = MPL * lane + c;
      cnt[t] = run;
      if (t < live) {
        const int i = sorted[k * TS + t] & (TS - 1);
        const int w = i >> 6;
        const int rank_in_word = (int)((run >> (8 * w)) & 255ull);
        set[w * 65 + rank_in_word + 1] = 1ull << (i & 63);
      }
      run += one[c];
    }
    if (lane == 63) cnt[TS] = run;
  }
  __syncthreads();
  // ---- sets[k][w][c] = OR of the single bits up to c; a wave per (objective, word)
  for (int item = wave; item < M * WW; item += T / 64) {
    const int k = item / WW, w = item - k * WW;
    uint64_t* const col = sets + (size_t)k * over + w * 65;
    const uint64_t incl = wave_scan_halves(col[lane + 1], [](uint32_t a, uint32_t b) { return a | b; });
    col[lane + 1] = ~incl;  // kept complemented: a row ORs the complements of its M sets (three-input ORs) and
    if (lane == 0) col[0] = ~0ull;  // complements once
  }
  __syncthreads();

  }  // tiles of the workgroup

  // ---- the rows of the stretch, 64 at a time per wave; the inputs of a wave's next rows are fetched while it
  // works on the present ones
  const int groups = NEARBY ? nearby_count : (r1 - r0 + 63) / 64;
  int e_next[M];
  int same_next = 0;
  auto row_of = [&](int g) { return r0 + (NEARBY ? (int)nearby[g] : g) * 64 + lane; };
  auto fetch = [&](int g) {
    const int j = row_of(g);
    const int jc = j < n ? j : n - 1;
#pragma unroll
    for (int k = 0; k < M; ++k) e_next[k] = upper[(int64_t)k * kstride + jc];
    same_next = NEARBY ? pos[(int64_t)(M - 1) * kstride + jc] : (int)kid[jc];  // (NEARBY: its place in the order of the slots)
  };
  if (wave < groups) fetch(wave);
  for (int g = wave; g < groups; g += T / 64) {
    const int j = row_of(g);
    int e[M];
#pragma unroll
    for (int k = 0; k < M; ++k) e[k] = e_next[k];
    const int same_from = same_next;  // slots from here on hold rows with the key of row j, or larger keys
    if (g + T / 64 < groups) fetch(g + T / 64);
    uint64_t dd[TT][WW];  // per tile: slots that are worse than row j in some objective, then its dominators
    int dominators = 0, highest = -1;
#pragma unroll
    for (int sub = 0; sub < TT; ++sub) {
      select_tile(sub);
      const int tw0 = w0 + sub * WW;
      uint64_t(&d)[WW] = dd[sub];
      // t[k] = members of objective k that lie before upper_k(j): those of the earlier buckets plus those of the
      // bucket itself that do (positions ascend, so the members from t on that lie before it are consecutive)
      int t[M];
      bool more = false;
#pragma unroll
      for (int k = 0; k < M; ++k) t[k] = index[k * index_stride + bucket_of_bound(k, e[k])];
#pragma unroll
      for (int k = 0; k < M; ++k) {
        const int m0 = mp[k * (TS + 8) + t[k]], m1 = mp[k * (TS + 8) + t[k] + 1];
        const int a0 = m0 < e[k] ? 1 : 0, a1 = m1 < e[k] ? 1 : 0;
        t[k] += a0 + a1;
        more |= a1 != 0;
      }
      if (__builtin_amdgcn_ballot_w64(more) != 0ull) {  // three or more members of the tile in one bucket: rare
#pragma unroll
        for (int k = 0; k < M; ++k)
          while (mp[k * (TS + 8) + t[k]] < e[k]) ++t[k];
      }
#pragma unroll
      for (int w = 0; w < WW; ++w) d[w] = 0ull;
#pragma unroll
      for (int k = 0; k < M; ++k) {
        const uint64_t c8 = counts[(size_t)k * over + t[k]];
        const uint64_t* const set = sets + (size_t)k * over;
#pragma unroll
        for (int w = 0; w < WW; ++w) d[w] |= set[w * 65 + (int)((c8 >> (8 * w)) & 255ull)];
      }
#pragma unroll
      for (int w = 0; w < WW; ++w) d[w] = ~d[w];
      // rows identical to j and everything after them: only near the diagonal (wave-uniform test; NEARBY: the last
      // of its orders, that of the slots, has left them out)
      if (!NEARBY && __builtin_amdgcn_ballot_w64(same_from < tile_slot0 + TS) != 0ull) {
#pragma unroll
        for (int w = 0; w < WW; ++w) {
          const int first = (tw0 + w) * 64;
          if (same_from <= first)
            d[w] = 0ull;
          else if (same_from < first + 64)
            d[w] &= (1ull << (same_from - first)) - 1ull;
        }
      }
      // what the count stage wants to know of the row, so that it does not have to read it again
#pragma unroll
      for (int w = 0; w < WW; ++w) {
        dominators += __popcll(d[w]);
        highest = d[w] != 0ull ? tw0 + w : highest;
      }
    }
    if constexpr (NEARBY) {
      if (j < n && dominators != 0) {
        atomicAdd(&total0[same_from], dominators);
        witness0[same_from] = same_from >> 6;  // (no word above this one: where a peel of the matrix would begin to look)
      }
      continue;
    }
    if (j < n && (mode & 1) && dominators != 0) {
      atomicAdd(&total0[j], dominators);
      atomicMax(&witness0[j], highest);
    }
    if (!(mode & 2)) continue;
    if constexpr (WW == 8 && TT == 2) {
      // Eight neighbouring lanes transpose the eight 16-byte pieces of their rows' lines (four of each tile): inside
      // the quads as below, then the lower quad hands its pieces of the second tile to the upper quad for the upper
      // quad's pieces of the first.  A store instruction then writes the whole 128-byte line of a row from eight
      // lanes side by side: one request of a line to memory instead of two of half a line.
      quad_transpose_pieces(dd[0], lane);
      quad_transpose_pieces(dd[1], lane);
      const bool upper_quad = (lane & 4) != 0;
      uint64_t other[8];  // piece (lane & 7) of the rows of the other quad
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const uint64_t send = upper_quad ? dd[0][x] : dd[1][x];
        const int lo = __shfl_xor((int)(uint32_t)send, 4);
        const int hi = __shfl_xor((int)(uint32_t)(send >> 32), 4);
        other[x] = (uint64_t)(uint32_t)lo | ((uint64_t)(uint32_t)hi << 32);
      }
      const int j8 = j - (lane & 7);  // the first row of this lane's eight
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        // rows 0..3 of the eight belong to the lower quad, rows 4..7 to the upper one
        const int q = p & 3;
        const bool own = (p >= 4) == upper_quad;
        const uint64_t a = own ? (upper_quad ? dd[1][2 * q] : dd[0][2 * q]) : other[2 * q];
        const uint64_t b = own ? (upper_quad ? dd[1][2 * q + 1] : dd[0][2 * q + 1]) : other[2 * q + 1];
        if (j8 + p < n)
          *reinterpret_cast<ulonglong2*>(dom + (int64_t)(j8 + p) * wstride + w0 + 2 * (lane & 7)) = make_ulonglong2(a, b);
      }
      continue;
    }
#pragma unroll
    for (int sub = 0; sub < TT; ++sub) {
      const int tw0 = w0 + sub * WW;
      uint64_t(&d)[WW] = dd[sub];
      if constexpr (WW == 8) {
        // Four neighbouring lanes exchange their 16-byte pieces (a 4 x 4 transpose through DPP moves), so that a
        // store instruction writes the whole 64 bytes of a row from four lanes side by side -- one request per row
        // to the memory system instead of four requests of 16 bytes from four instructions.  With two tiles per
        // workgroup the two halves of a row's line follow one another and leave the cache as one line.
        quad_transpose_pieces(d, lane);
        const int jq = j - (lane & 3);  // the first row of this lane's four
#pragma unroll
        for (int p = 0; p < 4; ++p)
          if (jq + p < n)
            *reinterpret_cast<ulonglong2*>(dom + (int64_t)(jq + p) * wstride + tw0 + 2 * (lane & 3)) =
                make_ulonglong2(d[2 * p], d[2 * p + 1]);
      } else {
        // tiles of four words: two neighbouring lanes exchange one piece each, a store writes the 32 bytes of a row
        static_assert(WW == 4, "tiles of four or eight words");
        const bool odd = (lane & 1) != 0;
        const uint64_t s0 = odd ? d[0] : d[2], s1 = odd ? d[1] : d[3];
        const uint64_t g0 = pair_exchange(s0), g1 = pair_exchange(s1);
        const uint64_t a0 = odd ? g0 : d[0], a1 = odd ? g1 : d[1];  // piece (lane & 1) of the even lane's row
        const uint64_t b0 = odd ? d[2] : g0, b1 = odd ? d[3] : g1;  // piece (lane & 1) of the odd lane's row
        const int jp = j - (lane & 1);
        if (jp < n) *reinterpret_cast<ulonglong2*>(dom + (int64_t)jp * wstride + tw0 + 2 * (lane & 1)) = make_ulonglong2(a0, a1);
        if (jp + 1 < n)
          *reinterpret_cast<ulonglong2*>(dom + (int64_t)(jp + 1) * wstride + tw0 + 2 * (lane & 1)) = make_ulonglong2(b0, b1);
      }
    }
  }
  if constexpr (!NEARBY) break;
  }  // parts of the work (NEARBY)
}

}  // namespace evx
