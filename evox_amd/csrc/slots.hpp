// The slot order (order.hpp) of populations of mid size in two launches, by sorted runs (runs.hpp).
//
// The first launch does what prepare_kernel does -- structure of arrays, row keys, the state cleared -- and sorts the keys
// of every 512 rows while it has them; the second finds every key's place among all keys and writes the slot-ordered arrays.
// Exact for any distribution of the keys: nothing queues up where they crowd or are equal.  Bound by the launches, the
// second one by its searches and by every workgroup's read of all keys.  20 000 x 3, us: 7.6 + 10.8, the five launches of
// the bucket sort 25 for uniform fitness and 31 for a front on a plane.
#pragma once

#include "dominance.hpp"
#include "order.hpp"
#include "runs.hpp"

namespace evx {

// blockIdx.x below `runs` = ceil(npad / kRunRows): a run.  The workgroups behind them only clear.
// sorted[p]: the keys of run p / kRunRows in ascending order; whose[p]: the row that each belongs to (p < n); bad[run]: does
// the run hold a NaN or an infinity.
// LEX: two objectives ranked without a matrix (two.hpp), the rows in the order of the first objective, then the second; the
// keys are 64-bit integers there, otherwise integers below 2^53 held as doubles.
template <bool LEX>
using SlotKey = std::conditional_t<LEX, uint64_t, double>;

template <bool MANY, bool LEX>
__global__ __launch_bounds__(kRunRows) void slot_runs_kernel(const float* __restrict__ f, int64_t stride_row, int64_t stride_col,
                                                             int n_first, const float* __restrict__ f2, int64_t stride_row2,
                                                             int64_t stride_col2, int n, int m, int npad, float* __restrict__ xs,
                                                             SlotKey<LEX>* __restrict__ sorted, int* __restrict__ whose,
                                                             unsigned long long* __restrict__ bad, uint32_t* __restrict__ zero_words,
                                                             int64_t n_zero_words, int runs, int64_t f_step,
                                                             int64_t f2_step, int64_t ws_step) {
  __shared__ SlotKey<LEX> lds[2 * kRunRows];
  if constexpr (MANY) {
    f += (int64_t)blockIdx.z * f_step;
    f2 += (int64_t)blockIdx.z * f2_step;
    to_population(ws_step, xs, sorted, whose, bad, zero_words);
  }
  if ((int)blockIdx.x < runs) {
    const int i = (int)blockIdx.x * kRunRows + (int)threadIdx.x;
    uint64_t key = 0ull;
    bool odd = false;
    if (i < npad) {
      for (int k = 0; k < m; ++k) {
        const float v = i < n_first ? f[(int64_t)i * stride_row + k * stride_col]
                        : i < n     ? f2[(int64_t)(i - n_first) * stride_row2 + k * stride_col2]
                                    : __uint_as_float(0x7FC00000u);
        xs[(int64_t)k * npad + i] = v;
        key = LEX ? (key << 32) | ordered_key(v) : key + (uint64_t)key_weight(k) * ordered_key(v);
        odd |= i < n && !(fabsf(v) <= 3.4028234663852886e38f);  // NaN or infinite
      }
    }
    const int any_odd = __syncthreads_or(odd);
    const SlotKey<LEX> held = i < n ? (SlotKey<LEX>)key : run_last_key<SlotKey<LEX>>();
    const int at = (int)blockIdx.x * kRunRows + run_position(held, lds);
    if (i < n) {
      sorted[at] = held;
      whose[at] = i;
    }
    if (threadIdx.x == 0) bad[blockIdx.x] = (unsigned long long)any_odd;
  }
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t w = tid; w < n_zero_words; w += (int64_t)gridDim.x * blockDim.x) zero_words[w] = 0u;
}

// Grid: ceil(n / share) workgroups, share <= kRunRankThreads / kRunLanes keys each.  Dynamic LDS: run_rank8_lds_bytes(n).
template <bool MANY, bool LEX>
__global__ __launch_bounds__(kRunRankThreads) void slot_places_kernel(const SlotKey<LEX>* __restrict__ sorted, const int* __restrict__ whose,
                                                                      const unsigned long long* __restrict__ bad, int n, int m, int npad,
                                                                      int share, const float* __restrict__ xs,
                                                                      uint64_t* __restrict__ key_sorted, uint32_t* __restrict__ kid_sorted,
                                                                      float* __restrict__ xs_sorted, int* __restrict__ orig_of,
                                                                      int* __restrict__ slot_of, SortParam* __restrict__ param_out,
                                                                      int64_t ws_step) {
  extern __shared__ __attribute__((aligned(16))) unsigned char slot_lds_bytes[];
  SlotKey<LEX>* const slot_lds = reinterpret_cast<SlotKey<LEX>*>(slot_lds_bytes);
  if constexpr (MANY) to_population(ws_step, sorted, whose, bad, xs, key_sorted, kid_sorted, xs_sorted, orig_of, slot_of, param_out);
  const int runs = runs_of(n);
  const int e0 = (int)blockIdx.x * share, e1 = min(n, e0 + share);
  const int sub = threadIdx.x & (kRunLanes - 1);
  const int entry = e0 + (int)threadIdx.x / kRunLanes, e = min(entry, e1 - 1);
  const bool work = e0 + (int)(threadIdx.x & ~63u) / kRunLanes < e1;  // (of the wave)
  RunSearch<SlotKey<LEX>> s;
  s.own = e / kRunRows;
  s.at = e % kRunRows;
  s.key = sorted[e];
  const int i = whose[e];
  const float first_value = work && sub < m ? xs[(int64_t)sub * npad + i] : 0.0f;  // (asked for before the searches)
  for (int first = 0; first < runs; first += kRunTile8) {
    const int here = min(kRunTile8, runs - first);
    __syncthreads();
    runs_to_lds(sorted, n, first, here, slot_lds);
    __syncthreads();
    if (work) run_search_all<kRunEqual>(slot_lds, first, here, s);
  }
  run_search_end<kRunEqual>(s);
  if (entry < e1) {
    const int slot = (int)s.smaller;
    // -0.0 is stored as +0.0: every comparison reads the same, and differences of equal values are +0.0
    if (sub < m) xs_sorted[(int64_t)sub * npad + slot] = first_value + 0.0f;
    for (int k = sub + kRunLanes; k < m; k += kRunLanes) xs_sorted[(int64_t)k * npad + slot] = xs[(int64_t)k * npad + i] + 0.0f;
    if (sub == 0) {
      orig_of[slot] = i;
      slot_of[i] = slot;
      key_sorted[slot] = (uint64_t)s.key;
      kid_sorted[slot] = (uint32_t)slot - s.equal;  // first slot holding this key: equal ids <=> equal keys
    }
  }
  if (blockIdx.x != 0) return;
  for (int t = n + (int)threadIdx.x; t < npad; t += blockDim.x) {
    orig_of[t] = -1;
    key_sorted[t] = ~0ull;
    kid_sorted[t] = (uint32_t)t;
    for (int k = 0; k < m; ++k) xs_sorted[(int64_t)k * npad + t] = __uint_as_float(0x7FC00000u);
  }
  if (threadIdx.x < 64) {
    unsigned long long any = 0ull;
    for (int r = threadIdx.x; r < runs; r += 64) any |= bad[r];
    any = __builtin_amdgcn_ballot_w64(any != 0ull);
    if (threadIdx.x == 0) {
      SortParam sp;
      sp.kmin = 0ull;
      sp.shift = 0;
      sp.buckets = 0;
      sp.nonfinite = any != 0ull;
      sp.totals_valid = 0;
      sp.orders_valid = 0;
      *param_out = sp;
    }
  }
}

}  // namespace evx
