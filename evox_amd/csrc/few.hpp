// A population of a few hundred to 1024 rows, three to eight objectives: the dominance matrix by the whole device, everything
// behind it -- fronts, crowding distances, selection order, gather -- by one workgroup.  Two launches.
//
// Reference semantics: non_dominate_rank (src/evox/operators/selection/non_dominate.py:172-195), crowding_distance (:198-231)
// and nd_environmental_selection (:234-254).
//
// One workgroup alone (batched.hpp) is bound by the vector issue of its one compute unit while it compares the pairs (700 rows:
// 21 of 46 us); the pipeline for larger populations pays an exchange between workgroups per front for no more than 1024 rows,
// and two more launches (1024 x 3: 45 us).  Here the pairs of 32 dominators and 64 rows are a wave's each, and the second launch holds
// a row's words in its thread's registers: a front is sixteen ANDs and one barrier.  It is bound by the two launches and
// by the chains of LDS round trips behind the fronts.
#pragma once

#include "two_small.hpp"

namespace evx {

constexpr int kFewRows = 1024;
constexpr int kFewObjectives = 8;
constexpr int kFewWords = kFewRows / 64;
constexpr int kFewCounting = 96;  // entries that a thread may compare one by one before buckets place the candidates faster

// Which of 32 rows, whose fitness lies in LDS (MS floats each; those from `left` on do not count), dominate this lane's row.
// finite: every value of the 32 rows and of the wave's rows is (dominance.hpp: the arithmetic form of the test).
template <int M>
__device__ __forceinline__ uint32_t few_half_word(const float* dominator, int left, float (&xj)[M], bool finite) {
  constexpr int MS = (M + 3) & ~3;
  uint32_t acc = 0u;
  if (finite) {
#pragma unroll
    for (int k = 0; k < M; ++k) xj[k] += 0.0f;  // (-0.0 becomes +0.0)
#pragma unroll 8
    for (int t = 31; t >= 0; --t) {
      float v[MS];
#pragma unroll
      for (int q = 0; q < MS / 4; ++q) {
        const float4 piece = *reinterpret_cast<const float4*>(dominator + t * MS + 4 * q);
        v[4 * q] = piece.x;
        v[4 * q + 1] = piece.y;
        v[4 * q + 2] = piece.z;
        v[4 * q + 3] = piece.w;
      }
      uint32_t o = 0u;
#pragma unroll
      for (int k = 0; k < M; ++k) o |= __float_as_uint(xj[k] - v[k]);
      acc = shift_in_positive(acc, t < left ? o : 0u);
    }
  } else {
#pragma unroll 2
    for (int t = 31; t >= 0; --t) {
      uint64_t le = t < left ? ~0ull : 0ull, lt = 0ull;
#pragma unroll
      for (int k = 0; k < M; ++k) {
        const float v = dominator[t * MS + k];
        le &= __builtin_amdgcn_ballot_w64(v <= xj[k]);
        lt |= __builtin_amdgcn_ballot_w64(v < xj[k]);
      }
      acc = shift_in(acc, le & lt);
    }
  }
  return acc;
}

// Word w of row j's matrix row at words[w * n + j]: which of the rows 64 w .. 64 w + 63 dominate row j.  Grid: (words, rows / 128,
// populations) workgroups of four waves: two groups of 64 rows times the two halves of a word.
template <int M>
__global__ __launch_bounds__(256) void few_dominance_kernel(BatchedArgs a, uint64_t* __restrict__ words, int64_t ws_step) {
  constexpr int MS = (M + 3) & ~3;
  __shared__ __attribute__((aligned(16))) float dominator[64 * MS];
  to_population(ws_step, words);
  const int tid = threadIdx.x, lane = tid & 63;
  const int half = __builtin_amdgcn_readfirstlane((tid >> 6) & 1);  // (known to be uniform)
  const float* __restrict__ f = a.f + (int64_t)blockIdx.z * a.f_stride_b;
  auto fitness_at = [&](int i, int k) {
    return f[(int64_t)i * a.f_stride_row + (int64_t)k * a.f_stride_col + (i >= a.n_first ? a.f_second : 0)];
  };
  const int i0 = (int)blockIdx.x * 64;
  if (tid < 64) {
#pragma unroll
    for (int k = 0; k < M; ++k) dominator[tid * MS + k] = i0 + tid < a.n ? fitness_at(i0 + tid, k) : 0.0f;
  }
  const int j = (int)blockIdx.y * 128 + (tid >> 7) * 64 + lane;
  const bool valid = j < a.n;
  float xj[M];
  bool finite = true;
#pragma unroll
  for (int k = 0; k < M; ++k) {
    xj[k] = valid ? fitness_at(j, k) : 0.0f;
    finite &= fabsf(xj[k]) <= 3.4028234663852886e38f;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < M; ++k) finite &= fabsf(dominator[lane * MS + k]) <= 3.4028234663852886e38f;
  const bool all_finite = __builtin_amdgcn_ballot_w64(!finite) == 0ull;
  const uint32_t acc = few_half_word<M>(dominator + half * 32 * MS, a.n - i0 - half * 32, xj, all_finite);
  if (valid) reinterpret_cast<uint32_t*>(words)[2 * ((int64_t)blockIdx.x * a.n + j) + half] = acc;
}

// Dynamic LDS of the workgroup that finishes a population of n rows with nt >= n threads: the placement's counters and entries,
// fitness by objective, costs by position, distances, three orders.
__host__ __device__ inline size_t few_finish_lds_bytes(int nt, int n, int m) {
  const size_t rows = (size_t)round_up(n, 64);
  return (size_t)nt * (4 * 4 + 8) + 32 + rows * (4 * (size_t)m + 4 + 4 + 2 + 2 + 2);
}

// Place of this thread's candidate (thread q < nv holds candidate q; entry: its key, then q) in the ascending order of the entries,
// by buckets: as two_small_place, for an item per thread.  bucket: a map of the key to 0 .. 4 nt - 1 that never decreases.  False when
// more than kTwoSmallCrowd candidates of different keys share one.  Every thread calls it.
// Candidates of one key that fill a bucket (values of a few levels, copies, distances of zero) are placed by their indices: the few buckets
// that can be as full are numbered, and a wave counts its candidates of each by a ballot.  1000 rows of one front, all equal, us per selection
// of half of them, three / eight objectives: by counting 112 / 245, like this 30 / 56; values of four levels, 700 x 8: 65 -> 45, of sixteen, 1000 x 8: 68 -> 53.
// cnt: 4 nt words; comps: nv entries; ids: nv; part: 16 words.
constexpr uint32_t kFewCrowd = 40;  // candidates of a bucket up to which each one looks at all
__device__ inline bool few_place(uint64_t entry, uint32_t bucket, int nv, int nt, uint32_t* cnt, uint64_t* comps, uint16_t* ids, uint32_t* part,
                                 int& place) {
  const int q = threadIdx.x, lane = q & 63, wave = q >> 6;
  const bool cand = q < nv;
  reinterpret_cast<uint4*>(cnt)[q] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  const uint32_t arrived = cand ? atomicAdd(&cnt[bucket], 1u) : 0u;
  __syncthreads();
  const uint4 mine = reinterpret_cast<const uint4*>(cnt)[q];
  const uint32_t sum = mine.x + mine.y + mine.z + mine.w;
  const uint32_t incl = wave_prefix_sum(sum);
  if (lane == 63) part[wave] = incl;
  const bool crowds = __syncthreads_or(max(max(mine.x, mine.y), max(mine.z, mine.w)) > kFewCrowd) != 0;
  const uint32_t run = incl - sum + sum_before_wave(part, wave);
  reinterpret_cast<uint4*>(cnt)[q] = make_uint4(run, run + mine.x, run + mine.x + mine.y, run + mine.x + mine.y + mine.z);
  __syncthreads();
  uint32_t first = 0u, end = 0u;
  if (cand) {
    first = cnt[bucket];
    end = bucket + 1u < 4u * (uint32_t)nt ? cnt[bucket + 1u] : (uint32_t)nv;
    comps[first + arrived] = entry;
  }
  if (q < 4) part[q] = 0u;  // crowds; whether one of them is too large; those of different keys
  __syncthreads();
  if (crowds) {
    const bool big = end - first > kFewCrowd;
    if (big && arrived == 0u) cnt[bucket] = atomicAdd(&part[0], 1u);  // (its start has been read by all)
    __syncthreads();
    const int crowd_count = (int)part[0];  // (at most 1024 / (kFewCrowd + 1))
    uint32_t number = big ? cnt[bucket] : ~0u;
    if (big && (uint32_t)(comps[first] >> 32) != (uint32_t)(entry >> 32)) {
      atomicOr(&part[2 + (number >> 5)], 1u << (number & 31u));
      if (end - first > kTwoSmallCrowd) part[1] = 1u;
    }
    __syncthreads();
    if (part[1] != 0u) return false;
    const uint64_t mixed = (uint64_t)part[3] << 32 | part[2];
    if (big && (mixed >> number & 1ull)) number = ~0u;  // (each one looks at all)
    const int waves = nt >> 6;
    uint32_t below = 0u;
#pragma unroll 1
    for (int c = 0; c < crowd_count; ++c) {
      const uint64_t of = __builtin_amdgcn_ballot_w64(number == (uint32_t)c);
      if (number == (uint32_t)c) below = (uint32_t)__popcll(of & ((1ull << lane) - 1ull));
      if (lane == 0) ids[c * waves + wave] = (uint16_t)__popcll(of);
    }
    __syncthreads();
    if (number != ~0u) {
#pragma unroll 4
      for (int w = 0; w < wave; ++w) below += ids[number * waves + w];
      place = (int)(first + below);
      return true;
    }
  }
  uint32_t before = 0u;
  for (uint32_t at = first; at < end; at += 4) {  // (four members' reads in flight together)
#pragma unroll
    for (int u = 0; u < 4; ++u) before += comps[min(at + (uint32_t)u, end - 1u)] < entry && at + (uint32_t)u < end ? 1u : 0u;
  }
  place = (int)(first + before);
  return true;
}

// Position of this thread's candidate (thread q < nv holds candidate q with `key`) in the ascending order of (key, q): by
// buckets -- of equal width in the key's value or in the key, whichever fits its range, then the other --, or by counting where the
// candidates are few or crowd.
// lo, hi: smallest and largest key of a finite value, -inf and +inf / NaN outside.  Every thread of the workgroup calls it.
__device__ inline int few_position(uint32_t key, int nv, int nt, uint32_t* cnt, uint64_t* comps, uint16_t* ids, uint32_t* part, uint32_t* lo16,
                                   uint32_t* hi16) {
  const int q = threadIdx.x;
  const bool cand = q < nv;
  const int parts = nt / ((nv + 63) & ~63);  // threads that share the comparisons of a candidate
  __syncthreads();  // (comps, cnt and the costs of the call before are free)
  const uint64_t entry = ((uint64_t)key << 32) | (uint32_t)q;
  if (nv > kFewCounting * parts) {
    const uint32_t key_inf = ordered_key(INFINITY), key_neg_inf = ordered_key(-INFINITY);
    uint32_t lo = 0xFFFFFFFFu, hi = 0u;
    if (cand && key > key_neg_inf && key < key_inf) lo = hi = key;
    two_small_range(lo, hi, lo16, hi16, nt);
    const bool wide = lo < hi && (lo ^ hi) >> 31 == 0u && lo != 0x80000000u && hi - lo > 24u << 23;  // (values of one sign, none zero, over more than 24 binades)
#pragma unroll 1
    for (int attempt = 0; attempt < 2; ++attempt) {
      int place;
      if (few_place(entry, (attempt == 0) != wide ? bucket_by_value(key, lo, hi, 4 * nt) : bucket_by_image(key, lo, hi, 4 * nt), nv, nt, cnt, comps,
                    ids, part, place))
        return place;
    }
    __syncthreads();
  }
  if (q < nv + 4) comps[q] = cand ? entry : ~0ull;
  if (q < 4 && nv + q >= nt) comps[nv + q] = ~0ull;
  return position_by_counting(comps, reinterpret_cast<int*>(cnt), nv, q, nt);
}

// The fronts of a population (non_dominate.py:29-59): a row joins when none of its dominators is unranked.  Thread j holds the words of
// row j (words from the population's own on are zero).  front: zeroed, behind a barrier.  order: the rows by (rank, index), up to the
// front that reaches a.stop_count; rows behind it keep kRankUnset.  A front is WORDS ANDs of 64 bits, one barrier, and a fold of the
// front's words.
struct FewFronts {
  int rank;                     // of this thread's row (-1: no row)
  int worst, worst_start, nv;  // the last front: its rank, the rows before it, its rows
};
template <int WORDS>
__device__ __forceinline__ FewFronts few_peel(const BatchedArgs& a, uint64_t (&row)[WORDS], uint64_t (*front)[kFewWords], uint16_t* order,
                                              Ctrl* __restrict__ ctrl) {
  const int j = threadIdx.x, lane = j & 63;
  const int wave = __builtin_amdgcn_readfirstlane(j >> 6);
  int rank = j < a.n ? kRankUnset : -1;
  int level = 0, ranked = 0, nv = 0;
  for (;; ++level) {
    uint64_t* const cur = front[level & 1];
    uint64_t left = 0ull;
#pragma unroll
    for (int w = 0; w < WORDS; ++w) left |= row[w];
    const bool now = rank == kRankUnset && left == 0ull;
    if (now) rank = level;
    const uint64_t mine = __builtin_amdgcn_ballot_w64(now);
    if (lane == 0) cur[wave] = mine;
    __syncthreads();
    // rows of the front, and those of the waves before this one: a word per lane, four steps inside a row of sixteen lanes
    int held = __popcll(cur[lane & (kFewWords - 1)]);
    held += __builtin_amdgcn_update_dpp(0, held, 0x111, 0xf, 0xf, true);  // row_shr:1
    held += __builtin_amdgcn_update_dpp(0, held, 0x112, 0xf, 0xf, true);  // row_shr:2
    held += __builtin_amdgcn_update_dpp(0, held, 0x114, 0xf, 0xf, true);  // row_shr:4
    held += __builtin_amdgcn_update_dpp(0, held, 0x118, 0xf, 0xf, true);  // row_shr:8
    const int size = __builtin_amdgcn_readlane(held, kFewWords - 1);
    const int before = wave == 0 ? 0 : __builtin_amdgcn_readlane(held, wave - 1);
    if (now) order[ranked + before + __popcll(mine & ((1ull << lane) - 1ull))] = (uint16_t)j;
    if (size == 0 || ranked + size >= a.stop_count) {
      nv = size;
      break;
    }
    ranked += size;
#pragma unroll
    for (int w = 0; w < WORDS; w += 2) {
      const ulonglong2 gone = *reinterpret_cast<const ulonglong2*>(cur + w);
      row[w] &= ~gone.x;
      row[w + 1] &= ~gone.y;
    }
  }
  if (j == 0 && ctrl != nullptr) {
    ctrl->err = 0;
    ctrl->nfronts = level + 1;
    ctrl->worst = level;
    ctrl->worst_start = ranked;
    ctrl->nv = nv;
    ctrl->need = a.stop_count - ranked;
    ctrl->passes = level;
    ctrl->tail_done = 1;
  }
  return {rank, level, ranked, nv};
}

// The selected rows, in the order of `order`: everything that LDS holds by row (fit by objective, `rows` apart), and x from memory.
__device__ __forceinline__ void few_gather(const BatchedArgs& a, const uint16_t* order, const uint16_t* rank_lds, const float* dist,
                                           const float* fit, int rows) {
  const int j = threadIdx.x, lane = j & 63, nt = blockDim.x, m = a.m;
  const int wave = __builtin_amdgcn_readfirstlane(j >> 6);
  const int topk = a.stop_count;
  const int64_t ob = (int64_t)blockIdx.x * topk;
  for (int p = j; p < topk; p += nt) {
    const int src = order[p];
    a.out_rank[ob + p] = rank_lds[src];
    a.out_dist[ob + p] = dist[src];
  }
  for (int e = j; e < topk * m; e += nt) {
    const int p = e / m, k = e - p * m;
    a.out_f[ob * m + e] = fit[(size_t)k * rows + order[p]];
  }
  if (a.x != nullptr) {
    const uint8_t* __restrict__ xb = a.x + (int64_t)blockIdx.x * a.x_stride_b;
    uint8_t* __restrict__ dst = a.out_x + ob * a.x_row_bytes;
    if (!gather_whole_units(a, xb, dst, order, topk, j, nt)) {
      for (int p = wave; p < topk; p += nt >> 6) {
        const int src = order[p];
        const uint8_t* __restrict__ sp = xb + (int64_t)src * a.x_row_stride + (src >= a.n_first ? a.x_second : 0);
        uint8_t* __restrict__ dp = dst + (int64_t)p * a.x_row_bytes;
        if (a.x_unit >= 4) {
          for (int64_t b = lane * 4; b < a.x_row_bytes; b += 64 * 4)
            *reinterpret_cast<uint32_t*>(dp + b) = *reinterpret_cast<const uint32_t*>(sp + b);
        } else {
          for (int64_t b = lane; b < a.x_row_bytes; b += 64) dp[b] = sp[b];
        }
      }
    }
  }
}

// Everything behind the matrix, by one workgroup of nt >= n threads: thread j < n holds row j, the others help where candidates
// are placed and rows gathered.  WORDS: words of a row at most.  mine: row j's fitness is at fit_of(k).  words: as above.
template <int WORDS, class FitOf>
__device__ __forceinline__ void few_finish(const BatchedArgs& a, const uint64_t* words, Ctrl* __restrict__ ctrl, uint8_t* few_lds, uint64_t (*front)[kFewWords],
                                           uint32_t* part, uint32_t* lo16, uint32_t* hi16, FitOf fit_of) {
  const int nt = blockDim.x;
  const int m = a.m, n = a.n, rows = (n + 63) & ~63, W = rows >> 6;
  uint32_t* cnt = reinterpret_cast<uint32_t*>(few_lds);  // 4 nt
  uint64_t* comps = reinterpret_cast<uint64_t*>(cnt + 4 * (size_t)nt);  // nt + 4
  float* fit = reinterpret_cast<float*>(comps + nt + 4);                // by objective, `rows` apart
  float* scost = fit + (size_t)m * rows;
  float* dist = scost + rows;                                // by row
  uint16_t* order = reinterpret_cast<uint16_t*>(dist + rows);  // rows by (rank, index), then the selection order
  uint16_t* rank_lds = order + rows;
  uint16_t* ids = rank_lds + rows;
  const int j = threadIdx.x, lane = j & 63;
  const int wave = __builtin_amdgcn_readfirstlane(j >> 6);
  const bool valid = j < n;

  uint64_t row[WORDS];
#pragma unroll
  for (int w = 0; w < WORDS; ++w) row[w] = w < W && valid ? words[(int64_t)w * n + j] : 0ull;
  if (a.out_f != nullptr && valid)
    for (int k = 0; k < m; ++k) fit[(size_t)k * rows + j] = fit_of(k);
  if (lane < kFewWords && wave == 0) front[0][lane] = front[1][lane] = 0ull;
  __syncthreads();
  EVX_BATCH_TRACE(1);

  const FewFronts got = few_peel<WORDS>(a, row, front, order, ctrl);
  const int rank = got.rank, worst_start = got.worst_start, nv = got.nv;
  if (a.rank_all && valid) a.rank_all[(int64_t)blockIdx.x * n + j] = rank;
  if (a.out_f == nullptr) return;  // rank-only mode
  if (valid) {
    rank_lds[j] = (uint16_t)rank;
    dist[j] = -INFINITY;
  }
  EVX_BATCH_TRACE(2);

  // ---- crowding distances of the last front (:198-231 with mask = rank == worst); thread q is its candidate q, in index order
  const int need = a.stop_count - worst_start;
  __syncthreads();
  const bool cand = j < nv;
  const int mine_row = cand ? order[worst_start + j] : 0;
  bool boundary = false;
  float acc = 0.0f;
  // ... and, behind the objectives, the index-stable top-k on the last front by (-distance, row index) (:253).  (One piece of code for
  // both: a second copy of the placement costs half a microsecond of fetching it.)
#pragma unroll 1
  for (int k = 0;; ++k) {
    const float d = k == m && boundary ? INFINITY : acc;
    if (k == m) {
      EVX_BATCH_TRACE(3);
    }
    const uint32_t key = cand ? ordered_key(k == m ? -d : fit[(size_t)k * rows + mine_row]) : 0u;
    const int p = few_position(key, nv, nt, cnt, comps, ids, part, lo16, hi16);
    if (k == m) {
      if (cand) dist[mine_row] = d;
      if (cand && p < need) order[worst_start + p] = (uint16_t)mine_row;  // (every candidate has been read from there)
      break;
    }
    if (cand) scost[p] = cost_of_key(key);
    __syncthreads();
    if (cand) {
      if (p == 0 || p == nv - 1) {
        boundary = true;
      } else {
        const float term = (scost[p + 1] - scost[p - 1]) / (scost[nv - 1] - scost[0]);
        acc = k == 0 ? term : acc + term;
      }
    }
  }
  __syncthreads();

  EVX_BATCH_TRACE(4);
  few_gather(a, order, rank_lds, dist, fit, rows);
  EVX_BATCH_TRACE(5);
}

// Grid: one workgroup of rows rounded up to 64 threads per population.  ctrl: the control block that callers read the outcome from.
__global__ __launch_bounds__(kFewRows) void few_finish_kernel(BatchedArgs a, const uint64_t* __restrict__ words, Ctrl* __restrict__ ctrl,
                                                              int64_t ws_step) {
  extern __shared__ __attribute__((aligned(16))) uint8_t few_lds[];
  __shared__ __attribute__((aligned(16))) uint64_t front[2][kFewWords];
  __shared__ __attribute__((aligned(16))) uint32_t part[16];
  __shared__ __attribute__((aligned(16))) uint32_t lo16[16];
  __shared__ __attribute__((aligned(16))) uint32_t hi16[16];
  if (ws_step != 0) {
    words = reinterpret_cast<const uint64_t*>(reinterpret_cast<const char*>(words) + (int64_t)blockIdx.x * ws_step);
    ctrl = reinterpret_cast<Ctrl*>(reinterpret_cast<char*>(ctrl) + (int64_t)blockIdx.x * ws_step);
  }
  const float* __restrict__ f = a.f + (int64_t)blockIdx.x * a.f_stride_b;
  const int j = threadIdx.x;
  EVX_BATCH_TRACE(0);
  few_finish<kFewWords>(a, words, ctrl, few_lds, front, part, lo16, hi16, [&](int k) {
    return f[(int64_t)j * a.f_stride_row + (int64_t)k * a.f_stride_col + (j >= a.n_first ? a.f_second : 0)];
  });
}

// Up to 256 rows: the matrix too, by sixteen waves.  A wave has 64 rows and some of the half words (32 dominators each) of their
// words; the words go to LDS behind the layout of few_finish_lds_bytes, after the rows' fitness (rows of M rounded up to four floats).
constexpr int kFewWholeRows = 256;
constexpr int kFewWholeWords = kFewWholeRows / 64;
__host__ __device__ inline size_t few_whole_lds_bytes(int nt, int n, int m) {
  const size_t rows = (size_t)round_up(n, 64);
  return (few_finish_lds_bytes(nt, n, m) + 15) / 16 * 16 + rows * (4 * (size_t)batched_stage_stride(m) + rows / 8);
}
template <int M>
__global__ __launch_bounds__(kFewRows) void few_whole_kernel(BatchedArgs a) {
  constexpr int MS = (M + 3) & ~3;
  extern __shared__ __attribute__((aligned(16))) uint8_t few_lds[];
  __shared__ __attribute__((aligned(16))) uint64_t front[2][kFewWords];
  __shared__ __attribute__((aligned(16))) uint32_t part[16];
  __shared__ __attribute__((aligned(16))) uint32_t lo16[16];
  __shared__ __attribute__((aligned(16))) uint32_t hi16[16];
  const int nt = blockDim.x, n = a.n, rows = (n + 63) & ~63;
  float* const dominator = reinterpret_cast<float*>(few_lds + (few_finish_lds_bytes(nt, n, M) + 15) / 16 * 16);
  uint64_t* const words = reinterpret_cast<uint64_t*>(dominator + rows * MS);
  const float* __restrict__ f = a.f + (int64_t)blockIdx.x * a.f_stride_b;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  EVX_BATCH_TRACE(0);
  bool finite = true;
  if (tid < rows) {
    float mine[M];
#pragma unroll
    for (int k = 0; k < M; ++k)
      mine[k] = tid < n ? f[(int64_t)tid * a.f_stride_row + (int64_t)k * a.f_stride_col + (tid >= a.n_first ? a.f_second : 0)] : 0.0f;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      dominator[tid * MS + k] = mine[k];
      finite &= fabsf(mine[k]) <= 3.4028234663852886e38f;
    }
  }
  const bool all_finite = __syncthreads_and(finite) != 0;
  const int groups = rows >> 6, halves = 2 * groups;
  for (int item = wave; item < groups * halves; item += nt >> 6) {  // (wave-uniform)
    const int group = item % groups, half = item / groups;
    const int row = group * 64 + lane;
    float xj[M];
#pragma unroll
    for (int k = 0; k < M; ++k) xj[k] = dominator[row * MS + k];
    const uint32_t acc = few_half_word<M>(dominator + half * 32 * MS, n - half * 32, xj, all_finite);
    if (row < n) reinterpret_cast<uint32_t*>(words)[2 * ((half >> 1) * n + row) + (half & 1)] = acc;
  }
  __syncthreads();
  EVX_BATCH_TRACE(6);
  few_finish<kFewWholeWords>(a, words, nullptr, few_lds, front, part, lo16, hi16, [&](int k) { return dominator[tid * MS + k]; });
}

}  // namespace evx
