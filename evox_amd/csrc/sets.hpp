// Populations of up to 1024 rows and three to eight objectives, one workgroup each, without comparing pairs: the dominators of a row
// from the orders of the rows in every objective.
//
// Reference semantics: non_dominate_rank (src/evox/operators/selection/non_dominate.py:172-195, batched :107-125),
// crowding_distance (:198-231) and nd_environmental_selection (:234-254).
//
// The rows no worse than row j in objective k are a prefix of the rows in the order of that objective: up to the last row that
// shares j's value.  The prefixes, one bit per row, lie in a table in LDS, one entry per position; the AND of a row's entries
// over the objectives is its row of the dominance matrix, but for the row itself and its copies (rows equal in every objective),
// which are taken out.  NaN sorts last and no other row's prefix reaches it; a row that holds one has no dominators.  The words go
// straight into the registers that the peeling works on (few_peel).
//   * orders: by buckets as in two_small_place, up to four objectives side by side;
//   * table: a lane takes sixteen consecutive positions of one word of 32 rows, a scan over the lanes carries the prefixes on;
//   * crowding distances: the last front's rows in the order of an objective are read off that order by counting.
//
// Comparing all pairs (batched_kernel) is six vector instructions for three objectives and 64 pairs: 35 of the 60 us of 1024
// populations of 512 x 3, and more than that above three objectives.  Here an objective costs a row its bucket, the bits of sixteen
// positions and W / 2 reads of 16 bytes: a table entry of all words of a row, so that a lane reads them in pieces of 16 bytes, four
// words further on per segment, so that the lanes that write meet different banks.  512 rows of up to five objectives leave room for
// four workgroups on a compute unit (36 KB of LDS, 64 registers).  Bound by vector issue and LDS in equal parts: of the 41 us of 1024
// populations of 512 x 3 the orders take 12, the table 5, the fronts and their distances 10, the gather 10 (64 MB); the narrow
// instance still has 7 VGPRs in scratch at three objectives, 10 at four, 22 at five, 27 at eight.  us per selection of half the rows,
// pairs -> orders: 1024 x (512 x 3) 64 -> 41, 512 x (700 x 3) 67 -> 50, 390 x (1000 x 3) 129 -> 60, 1024 x (390 x 5)
// 146 -> 54, 1024 x (390 x 8) 210 -> 87.
#pragma once

#include "few.hpp"

namespace evx {

constexpr int kSetsRows = 1024;
constexpr int kSetsObjectives = 8;
constexpr int kSetsGroup = 4;        // objectives that are sorted side by side
constexpr int kSetsSegment = 16;     // positions per lane while the table is written
constexpr int kSetsNarrowRows = 32 * 16;  // up to here a wave writes two words of the table at once, and all words in one go

constexpr int kSetsEntry = 16;  // words (32 rows each) of a table entry: 512 rows; a larger population's table is written in two panels
// Four words between the segments: lanes that write the same position of their segments meet different banks.
__host__ __device__ inline size_t sets_table_bytes(int rows) {
  return 4 * ((size_t)rows * kSetsEntry + 4 * (size_t)(rows / kSetsSegment));
}
// What the sort of a group of objectives holds: per objective 2 rows counters, and keys by bucket.
__host__ __device__ inline size_t sets_sort_bytes(int rows, int m) {
  const int side = m < kSetsGroup ? m : kSetsGroup;
  return (size_t)side * rows * (8 + 4);
}
// What follows the peeling: fitness by objective, distances, ranks, order; costs and places of the last front in every objective or
// what few_position needs.
__host__ __device__ inline size_t sets_finish_bytes(int rows, int m) {
  const size_t front = (size_t)m * rows * (4 + 2);
  const size_t position = (size_t)rows * (16 + 8 + 2) + 32;
  return (size_t)rows * (4 * (size_t)m + 4 + 2 + 2) + (front > position ? front : position);
}
__host__ __device__ inline size_t sets_lds_bytes(int rows, int m) {
  size_t most = sets_table_bytes(rows);
  if (sets_sort_bytes(rows, m) > most) most = sets_sort_bytes(rows, m);
  if (sets_finish_bytes(rows, m) > most) most = sets_finish_bytes(rows, m);
  return (most + 15) / 16 * 16 + 2 * (size_t)m * rows;
}

// The OR over the lanes of the same word up to and with this one: rows of sixteen lanes, pairs of them, with WIDE all four.
template <bool WIDE>
__device__ inline uint32_t sets_prefix_or(uint32_t x) {
  uint32_t v = x;
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  if constexpr (WIDE) v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

// Grid: one workgroup of rows rounded up to 64 threads per population; thread j holds row j.  WORDS: 64-bit words of a matrix row at
// most, 8 (up to 512 rows) or 16.
template <int M, int WORDS>
__global__ __launch_bounds__(64 * WORDS) __attribute__((amdgpu_waves_per_eu(WORDS == 8 ? (M <= 5 ? 8 : 6) : 4, 8))) void sets_kernel(
    BatchedArgs a) {
  constexpr bool kWide = WORDS > 8;
  constexpr int kPanels = kWide ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) uint8_t sets_lds[];
  __shared__ __attribute__((aligned(16))) uint64_t front[2][kFewWords];
  __shared__ __attribute__((aligned(16))) uint32_t lows[M][16];
  __shared__ __attribute__((aligned(16))) uint32_t highs[M][16];
  __shared__ __attribute__((aligned(16))) uint32_t parts[M][16];
  const int j = threadIdx.x, lane = j & 63;
  const int wave = __builtin_amdgcn_readfirstlane(j >> 6);
  const int n = a.n, rows = blockDim.x, waves = rows >> 6;
  const bool valid = j < n;
  uint16_t* const orders = reinterpret_cast<uint16_t*>(sets_lds + sets_lds_bytes(rows, M) - 2 * (size_t)M * rows);  // rows by objective
  const float* __restrict__ f = a.f + (int64_t)blockIdx.x * a.f_stride_b;

  EVX_BATCH_TRACE(0);
  float x[M];
  bool nan = !valid;
#pragma unroll
  for (int k = 0; k < M; ++k) {
    x[k] = valid ? f[(int64_t)j * a.f_stride_row + (int64_t)k * a.f_stride_col + (j >= a.n_first ? a.f_second : 0)] : 0.0f;
    nan |= x[k] != x[k];
  }

  // ---- the words of row j: which rows are no worse anywhere
  uint32_t row[2 * WORDS];
#pragma unroll
  for (int w = 0; w < 2 * WORDS; ++w) row[w] = ~0u;
  bool alone = false;                  // some objective's value is this row's only
  uint64_t id_low = 0ull;              // the first position of its value in objectives 0 .. 5, ten bits each
  [[maybe_unused]] uint32_t id_high = 0u;  // ... in objectives 6 and 7
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const uint32_t key = ordered_key(x[k]);
    const bool finite = valid && fabsf(x[k]) <= 3.4028234663852886e38f;
    const uint32_t lo = wave_prefix_min(finite ? key : 0xFFFFFFFFu), hi = ~wave_prefix_min(finite ? ~key : 0xFFFFFFFFu);
    if (lane == 63) {
      lows[k][wave] = lo;
      highs[k][wave] = hi;
    }
  }
#pragma unroll
  for (int k0 = 0; k0 < M; k0 += kSetsGroup) {
    constexpr int kMost = M < kSetsGroup ? M : kSetsGroup;
    const int side = M - k0 < kSetsGroup ? M - k0 : kSetsGroup;  // (a constant once the loops are unrolled)
    uint32_t* const cnt = reinterpret_cast<uint32_t*>(sets_lds);                      // 2 rows counters per objective
    uint32_t* const keys = cnt + (size_t)kMost * 2 * rows;                            // by bucket
    uint32_t bucket[kMost], arrived[kMost], place[kMost];
    bool crowds = false;
#pragma unroll 1
    for (int attempt = 0;; ++attempt) {  // (buckets of equal width in the value; where one is crowded, in the key, whatever comes)
#pragma unroll
      for (int c = 0; c < side; ++c) reinterpret_cast<uint2*>(cnt)[(size_t)c * rows + j] = make_uint2(0u, 0u);
      __syncthreads();
#pragma unroll
      for (int c = 0; c < side; ++c) {
        const uint32_t lo = min_before_wave(lows[k0 + c], waves), hi = max_before_wave(highs[k0 + c], waves);
        const uint32_t key = ordered_key(x[k0 + c]);
        bucket[c] = attempt == 0 ? bucket_by_value(key, lo, hi, 2 * rows) : bucket_by_image(key, lo, hi, 2 * rows);
        arrived[c] = valid ? atomicAdd(&cnt[(size_t)c * 2 * rows + bucket[c]], 1u) : 0u;
      }
      __syncthreads();
      bool crowded = false;
#pragma unroll
      for (int c = 0; c < side; ++c) {
        const uint2 mine = reinterpret_cast<const uint2*>(cnt)[(size_t)c * rows + j];
        const uint32_t incl = wave_prefix_sum(mine.x + mine.y);
        if (lane == 63) parts[c][wave] = incl;
        place[c] = incl - mine.x - mine.y;  // (its part inside the wave, for now)
        crowded |= max(mine.x, mine.y) > kTwoSmallCrowd;
      }
      crowds = __syncthreads_or(crowded);
      if (!crowds || attempt == 1) break;
    }
#pragma unroll
    for (int c = 0; c < side; ++c) {
      uint2* const mine = reinterpret_cast<uint2*>(cnt) + (size_t)c * rows + j;
      const uint32_t run = place[c] + sum_before_wave(parts[c], wave);
      *mine = make_uint2(run, run + mine->x);
    }
    __syncthreads();
    uint32_t first[kMost], end[kMost];
#pragma unroll
    for (int c = 0; c < side; ++c) {
      first[c] = cnt[(size_t)c * 2 * rows + bucket[c]];
      end[c] = bucket[c] + 1u < 2u * (uint32_t)rows ? cnt[(size_t)c * 2 * rows + bucket[c] + 1u] : (uint32_t)n;
      if (valid) keys[(size_t)c * rows + first[c] + arrived[c]] = ordered_key(x[k0 + c]);
    }
    __syncthreads();
    if (crowds) {  // (values of a few levels: buckets of one value are told by a mark on the others' counter)
#pragma unroll
      for (int c = 0; c < side; ++c)
        if (valid && keys[(size_t)c * rows + first[c]] != ordered_key(x[k0 + c])) cnt[(size_t)c * 2 * rows + bucket[c]] = ~0u;
      __syncthreads();
    }
    uint32_t upto[kMost];  // rows no worse in the objective, and rows that share its value (16 bits each)
#pragma unroll
    for (int c = 0; c < side; ++c) {
      const uint32_t key = ordered_key(x[k0 + c]);
      const uint32_t slot = first[c] + arrived[c];
      uint32_t smaller = 0u, equal = 0u, equal_before = 0u;
      if (valid && crowds && cnt[(size_t)c * 2 * rows + bucket[c]] != ~0u) {
        equal = end[c] - first[c];
        equal_before = arrived[c];
      } else if (valid) {
        for (uint32_t q = first[c]; q < end[c]; q += 4) {  // (four members' reads in flight together)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t at = q + (uint32_t)u;
            const uint32_t other = keys[(size_t)c * rows + min(at, end[c] - 1u)];
            const bool in = at < end[c];
            smaller += in && other < key ? 1u : 0u;
            equal += in && other == key ? 1u : 0u;
            equal_before += at < slot && other == key ? 1u : 0u;
          }
        }
      }
      const uint32_t lower = valid ? first[c] + smaller : (uint32_t)j;
      upto[c] = (lower + equal) | equal << 16;
      alone |= equal < 2u;
      orders[(size_t)(k0 + c) * rows + lower + equal_before] = (uint16_t)j;  // (rows of one value in any order, for now)
      if (k0 + c < 6)
        id_low |= (uint64_t)lower << (10 * (k0 + c));
      else
        id_high |= lower << (10 * (k0 + c - 6));
    }
    __syncthreads();
    EVX_BATCH_TRACE(6);
    // ---- the table, and the row's words off it, in panels of 512 rows
    uint32_t* const table = reinterpret_cast<uint32_t*>(sets_lds);
#pragma unroll 1
    for (int c = 0; c < side; ++c) {  // (a loop: its sixteen words in flight for one objective after the other, or they do not fit the registers)
      uint32_t last = upto[0];
#pragma unroll
      for (int other = 1; other < kMost; ++other) last = c == other ? upto[other] : last;
      const uint32_t shares = last >> 16;
      last &= 0xFFFFu;
      uint16_t* const by_value = orders + (size_t)(k0 + c) * rows;
      uint32_t before_in_value = 0u;
#pragma unroll
      for (int panel = 0; panel < kPanels; ++panel) {
        const int segment = kWide ? lane : lane & 31;
        const bool writes = kSetsSegment * segment < rows;
        const int words = min(rows / 32 - panel * 16, 16);
        for (int word = kWide ? wave : j >> 5; word < words; word += kWide ? waves : 2 * waves) {  // (wave-uniform)
          const uint4* const from = reinterpret_cast<const uint4*>(by_value + kSetsSegment * segment);
          uint32_t pairs[8];
          if (writes) {
            const uint4 low = from[0], high = from[1];
            pairs[0] = low.x; pairs[1] = low.y; pairs[2] = low.z; pairs[3] = low.w;
            pairs[4] = high.x; pairs[5] = high.y; pairs[6] = high.z; pairs[7] = high.w;
          } else {
#pragma unroll
            for (int t = 0; t < 8; ++t) pairs[t] = ~0u;  // (row 65535: in no word)
          }
          const uint32_t base = 32u * (uint32_t)(panel * 16 + word);
          auto bit_of = [&](int t) {
            const uint32_t at = ((t & 1) ? pairs[t >> 1] >> 16 : pairs[t >> 1] & 0xFFFFu) - base;
            return at < 32u ? 1u << at : 0u;
          };
          // (once for the total, once more for the entries: sixteen words held in between would not fit the registers)
          uint32_t run = 0u;
#pragma unroll
          for (int t = 0; t < kSetsSegment; ++t) run |= bit_of(t);
          const uint32_t incl = sets_prefix_or<kWide>(run);
          run = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x138, 0xf, 0xf, false);  // wave_shr:1
          if (segment == 0) run = 0u;
          if (writes) {
            uint32_t* const to = table + (size_t)kSetsSegment * segment * kSetsEntry + 4 * segment + word;
#pragma unroll
            for (int t = 0; t < kSetsSegment; ++t) {
              run |= bit_of(t);
              to[t * kSetsEntry] = run;
            }
          }
        }
        __syncthreads();
        if (valid) {
          const uint32_t p = last - 1u;
          const uint4* const from = reinterpret_cast<const uint4*>(table + (size_t)p * kSetsEntry + 4 * (p / kSetsSegment));
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (4 * q < words) {  // (words behind the last one of 32 rows hold anything, and are cleared below)
              const uint4 v = from[q];
              row[16 * panel + 4 * q] &= v.x;
              row[16 * panel + 4 * q + 1] &= v.y;
              row[16 * panel + 4 * q + 2] &= v.z;
              row[16 * panel + 4 * q + 3] &= v.w;
            }
          }
          if (shares >= 2u) {  // the rows before it that share its value: their bits are in its entry, not in that of the value before
            const uint32_t less = last - shares;  // rows of smaller values
            const uint4* const from_less = reinterpret_cast<const uint4*>(table + (size_t)(less - 1u) * kSetsEntry + 4 * ((less - 1u) / kSetsSegment));
            const int mine_word = (j >> 5) - 16 * panel;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if (4 * q < words && 4 * q <= mine_word) {
                const uint4 v = from[q], l = less != 0u ? from_less[q] : make_uint4(0u, 0u, 0u, 0u);
                const uint32_t same[4] = {v.x & ~l.x, v.y & ~l.y, v.z & ~l.z, v.w & ~l.w};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                  const int w = 4 * q + u;
                  before_in_value += (uint32_t)__popc(w < mine_word ? same[u] : w == mine_word ? same[u] & ((1u << (j & 31)) - 1u) : 0u);
                }
              }
            }
          }
        }
        __syncthreads();
      }
      if (valid && shares >= 2u) by_value[last - shares + before_in_value] = (uint16_t)j;  // (read behind the peeling's barriers)
    }
  }
  EVX_BATCH_TRACE(7);
  // Copies of the row are no worse anywhere either: the rows of the same places in all objectives.  The first one of them stands for
  // all in everybody's words, and is taken out of its copies' own.  Rows that could have some meet in a hash table that keeps the first
  // row of a cell; rows whose cell went to another kind of row try again with another hash (the kind of a cell's first row is done, so
  // this ends; three or four times).
  int standing = j;
  const bool may_have_copies = valid && !nan && !alone;
  if (__syncthreads_or(may_have_copies)) {
    uint64_t* const all_low = reinterpret_cast<uint64_t*>(sets_lds);
    uint32_t* const all_high = reinterpret_cast<uint32_t*>(all_low + rows);
    uint4* const cells = reinterpret_cast<uint4*>(all_high + rows);  // 4 rows words
    all_low[j] = id_low;
    if (M > 6) all_high[j] = id_high;
    bool open = may_have_copies;
    for (uint32_t salt = 0u; __syncthreads_or(open); ++salt) {
      cells[j] = make_uint4(~0u, ~0u, ~0u, ~0u);
      __syncthreads();
      uint32_t hash = ((uint32_t)id_low ^ salt * 0x9E3779B9u) * 0x85EBCA6Bu;
      hash = (hash ^ hash >> 15 ^ (uint32_t)(id_low >> 32) ^ id_high * 0xC2B2AE35u) * 0x27D4EB2Fu;
      uint32_t* const cell = reinterpret_cast<uint32_t*>(cells) + (uint32_t)(((uint64_t)(hash ^ hash >> 13) * (4u * (uint32_t)rows)) >> 32);
      if (open) atomicMin(cell, (uint32_t)j);
      __syncthreads();
      if (open) {
        const int other = (int)*cell;
        bool same = all_low[other] == id_low;
        if (M > 6) same = same && all_high[other] == id_high;
        if (same) standing = other;
        open = !same;
      }
    }
    const uint64_t stands = __builtin_amdgcn_ballot_w64(standing == j);
    if (lane == 0) front[0][wave] = stands;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 2 * WORDS; ++w)
      if (32 * w < rows) row[w] &= reinterpret_cast<const uint32_t*>(front[0])[w];
    __syncthreads();
  }
#pragma unroll
  for (int w = 0; w < 2 * WORDS; ++w) {
    if (nan || 32 * w >= rows) row[w] = 0u;
    if (w == standing >> 5) row[w] &= ~(1u << (standing & 31));
  }
  EVX_BATCH_TRACE(1);

  // ---- fronts
  float* const fit = reinterpret_cast<float*>(sets_lds);  // by objective, `rows` apart
  float* const dist = fit + (size_t)M * rows;               // by row
  uint16_t* const rank_lds = reinterpret_cast<uint16_t*>(dist + rows);
  uint16_t* const order = rank_lds + rows;  // rows by (rank, index), then the selection order
  uint8_t* const rest = reinterpret_cast<uint8_t*>(order + rows);
#pragma unroll
  for (int k = 0; k < M; ++k) fit[(size_t)k * rows + j] = x[k];
  if (j < kFewWords) front[0][j] = front[1][j] = 0ull;
  uint64_t words[WORDS];
#pragma unroll
  for (int w = 0; w < WORDS; ++w) words[w] = (uint64_t)row[2 * w + 1] << 32 | row[2 * w];
  __syncthreads();
  const FewFronts got = few_peel<WORDS>(a, words, front, order, nullptr);
  const int rank = got.rank, worst = got.worst, worst_start = got.worst_start, nv = got.nv;
  if (a.rank_all && valid) a.rank_all[(int64_t)blockIdx.x * n + j] = rank;
  if (a.out_f == nullptr) return;  // rank-only mode
  rank_lds[j] = (uint16_t)rank;
  __syncthreads();
  EVX_BATCH_TRACE(2);

  // ---- crowding distances of the last front (:198-231 with mask = rank == worst).  Its rows in the order of an objective: thread j
  // stands for position j of that order, and counts the front's rows before it.
  float* const costs = reinterpret_cast<float*>(rest);                               // by objective and place in the front
  uint16_t* const places = reinterpret_cast<uint16_t*>(costs + (size_t)M * rows);  // by objective and row
  uint64_t in_front[M];
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const int at = valid ? orders[(size_t)k * rows + j] : 0;
    in_front[k] = __builtin_amdgcn_ballot_w64(valid && rank_lds[at] == (uint16_t)worst);
    if (lane == 0) parts[k][wave] = (uint32_t)__popcll(in_front[k]);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const uint32_t before = sum_before_wave(parts[k], wave);
    if (in_front[k] >> lane & 1ull) {
      const int at = orders[(size_t)k * rows + j];
      const uint32_t place = before + (uint32_t)__popcll(in_front[k] & ((1ull << lane) - 1ull));
      costs[(size_t)k * rows + place] = cost_of_key(ordered_key(fit[(size_t)k * rows + at]));
      places[(size_t)k * rows + at] = (uint16_t)place;
    }
  }
  __syncthreads();
  float d = -INFINITY;
  if (rank == worst) {
    bool boundary = false;
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const float* const cost = costs + (size_t)k * rows;
      const int p = places[(size_t)k * rows + j];
      if (p == 0 || p == nv - 1) {
        boundary = true;
      } else {
        const float term = (cost[p + 1] - cost[p - 1]) / (cost[nv - 1] - cost[0]);
        acc = k == 0 ? term : acc + term;
      }
    }
    d = boundary ? INFINITY : acc;
  }
  dist[j] = d;
  EVX_BATCH_TRACE(3);
  // ---- index-stable top-k on the last front by (-distance, row index) (:253); thread q has its row q, in index order
  {
    uint32_t* const cnt = reinterpret_cast<uint32_t*>(rest);
    uint64_t* const comps = reinterpret_cast<uint64_t*>(cnt + 4 * (size_t)rows);
    uint16_t* const ids = reinterpret_cast<uint16_t*>(comps + rows + 4);
    __syncthreads();
    const int mine = j < nv ? order[worst_start + j] : 0;
    const int p = few_position(j < nv ? ordered_key(-dist[mine]) : 0u, nv, rows, cnt, comps, ids, parts[0], lows[0], highs[0]);
    if (j < nv && p < a.stop_count - worst_start) order[worst_start + p] = (uint16_t)mine;  // (every row has been read from there)
  }
  __syncthreads();
  EVX_BATCH_TRACE(4);
  few_gather(a, order, rank_lds, dist, fit, rows);
  EVX_BATCH_TRACE(5);
}

}  // namespace evx
