// Stable orders of up to a few ten thousand keys by comparison alone: sorted runs, and positions by searching them.
//
// The keys are cut into runs of kRunRows consecutive positions.  A first launch sorts every run (a workgroup each); a
// second one derives the position of a key among all keys as the sum, over the runs, of how many of the run's keys
// precede it: a binary search per run in a workgroup's LDS, which holds the runs of all keys.  No workgroup waits for
// another inside a launch, nothing depends on how the keys are distributed (a histogram by value queues up thousands of
// additions where keys crowd or are equal), and ties go by position without a wider key: a key of an earlier run precedes
// an equal one, a key of a later run does not.
//
// What bounds it: (keys / kRunRows) searches of ten LDS reads per key, throughput of the LDS and of vector issue alike, and
// the launches themselves (4 us each).  20 001 keys of three objectives, us per launch in a loop of launches: sorting the
// runs 5.9, places with neighbours 9.3, places of one order 6.0; 2000 keys: 5.8, 3.9, 4.3.  Runs of 256 would double the
// searches, runs of 1024 double what the sorts take on a quarter of the compute units; fetching the runs into LDS is 0.5
// us of it (80 KB per workgroup, the same for all).
#pragma once

#include "common.hpp"

namespace evx {

constexpr int kRunRows = 512;          // keys per run = threads that sort it
constexpr int kRunMaxRows = 32768;     // 4-byte keys that one workgroup's LDS holds
constexpr int kRunLdsStride = kRunRows + 4;  // keys from one run to the next in LDS: sixteen runs' same entries fall into different banks
constexpr int kRunRankThreads = 1024;  // threads of a workgroup that searches
__host__ __device__ inline size_t run_rank_lds_bytes(int n) {
  return sizeof(uint32_t) * (size_t)kRunLdsStride * (size_t)((n + kRunRows - 1) / kRunRows);
}

// Does a key `other` precede the key `mine`: smaller, or equal where `first` says that its position is the earlier one?
template <class K>
__device__ __forceinline__ bool run_precedes(K other, K mine, bool first) {
  return other < mine || (first && other == mine);
}

// How many of the N (a power of two) ascending keys of `run` precede `mine`.
template <int N, class K>
__device__ __forceinline__ int run_search(const K* run, K mine, bool first) {
  int c = 0;
#pragma unroll
  for (int s = N / 2; s >= 1; s >>= 1) c += run_precedes(run[c + s - 1], mine, first) ? s : 0;
  return c + (run_precedes(run[c], mine, first) ? 1 : 0);
}

__device__ __forceinline__ uint32_t lane_value(uint32_t v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// The position of every thread's key among the keys of its workgroup of kRunRows threads (ascending, equal keys by
// thread): 64 keys of a wave by counting (the other lanes' keys come through scalar registers), then the sorted 64s of
// four waves, then the two halves of the workgroup by searching one another in LDS.  lds: 2 * kRunRows keys.
template <class K>
__device__ __forceinline__ int run_position(K key, K* lds) {
  static_assert(kRunRows == 512, "eight waves");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  K* const by_wave = lds;
  K* const by_half = lds + kRunRows;
  int at = 0;
#pragma unroll 8
  for (int i = 0; i < 64; ++i) at += run_precedes(lane_value(key, i), key, i < lane) ? 1 : 0;
  by_wave[wave * 64 + at] = key;
  __syncthreads();
  const int half = wave >> 2;
  int more = 0;
#pragma unroll
  for (int u = 1; u < 4; ++u) {
    const int w = (half << 2) | ((wave + u) & 3);
    more += run_search<64>(by_wave + w * 64, key, w < wave);
  }
  at += more;
  by_half[half * 256 + at] = key;
  __syncthreads();
  at += run_search<256>(by_half + (half ^ 1) * 256, key, half == 1);
  return at;
}

// The sorted runs of nv keys (run r at sorted + r * kRunRows, 16-byte aligned) into LDS; the last run is filled up with the
// largest key.  Called by every thread; the caller puts a barrier behind it.
__device__ __forceinline__ void runs_to_lds(const uint32_t* __restrict__ sorted, int nv, uint32_t* lds) {
  const int whole = nv & ~3;
#pragma unroll 4
  for (int e = threadIdx.x * 4; e < whole; e += blockDim.x * 4)
    *reinterpret_cast<uint4*>(lds + (e / kRunRows) * kRunLdsStride + (e % kRunRows)) = *reinterpret_cast<const uint4*>(sorted + e);
  const int padded = (nv + kRunRows - 1) / kRunRows * kRunRows;
  for (int e = whole + threadIdx.x; e < padded; e += blockDim.x)
    lds[(e / kRunRows) * kRunLdsStride + (e % kRunRows)] = e < nv ? sorted[e] : 0xFFFFFFFFu;
}

// Neighbours of a key among all keys: the largest key before it and the smallest behind it.
struct RunNeighbours {
  uint32_t before, behind;
};

// The sum / maximum / minimum over the G (4 or 8) consecutive lanes of a group, the same in all of them.
template <int G, class Op>
__device__ __forceinline__ uint32_t run_group(uint32_t v, Op op) {
  static_assert(G == 4 || G == 8, "rotations inside a row of sixteen lanes");
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false));  // lanes 1 0 3 2
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false));  // lanes 2 3 0 1
  if constexpr (G == 8) v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, false));  // the other four
  return v;
}

// A key whose place is being looked for, and what its searches have found so far.
struct RunSearch {
  uint32_t key;
  int own, at;  // its run, and its place in that
  uint32_t smaller, before, behind;
};

// U searches side by side: runs r0, r0 + G, ... (those below `runs`).
template <int G, int U, bool NEIGHBOURS>
__device__ __forceinline__ void run_search_some(const uint32_t* lds, int runs, int r0, RunSearch& q) {
  const uint32_t* c[U];  // (an address in LDS: a step is one read, one comparison, one selection and one addition)
  uint32_t bound[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r = r0 + G * u;
    c[u] = lds + (r < runs ? r : 0) * kRunLdsStride;
    bound[u] = r < q.own ? q.key : q.key - 1u;
  }
#pragma unroll
  for (int s = kRunRows / 2; s >= 1; s >>= 1) {
    uint32_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = c[u][s - 1];
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] += v[u] <= bound[u] ? s : 0;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r = r0 + G * u;
    const uint32_t* const run = lds + (r < runs ? r : 0) * kRunLdsStride;
    int n = (int)(c[u] - run) + (*c[u] <= bound[u] ? 1 : 0);
    if (q.key == 0u && r > q.own) n = 0;
    if (r == q.own) n = q.at;
    q.smaller += r < runs ? (uint32_t)n : 0u;
    if constexpr (NEIGHBOURS) {  // (read whether or not there is one: branches would put the reads one after the other)
      const uint32_t lower = run[n > 0 ? n - 1 : 0], upper = run[min(r == q.own ? n + 1 : n, kRunRows - 1)];
      if (r < runs && n > 0) q.before = max(q.before, lower);
      if (r < runs && n + (r == q.own ? 1 : 0) < kRunRows) q.behind = min(q.behind, upper);
    }
  }
}

// The place of a key among all keys, whose runs lie in LDS: the key at entry e (run e / kRunRows, place e % kRunRows in it),
// the same in the kRunLanes lanes that call it together, each with its share of the runs, four of them at a time (a search
// is a chain of ten LDS round trips).  The keys of a wave should be neighbours in their run: their searches then read the
// same words mostly, and four lanes per key mean four different words of a wave's read in the LDS banks instead of
// sixteen (terms of 20 001 x 3, forty runs, us: sixteen lanes per key 11.6, eight 12.0, four 9.3).
// The comparison `v precedes key` is v <= bound, the bound being the key or one less: one instruction per step.  A key
// of zero that no equal key precedes has no such bound; nothing precedes it.
// NEIGHBOURS: also the keys next to it (before: 0 where there is none; behind: meaningless at the last place).
constexpr int kRunLanes = 4;
template <bool NEIGHBOURS>
__device__ __forceinline__ int run_place(const uint32_t* lds, int runs, int e, RunNeighbours* next_to) {
  RunSearch q;
  q.own = e / kRunRows;
  q.at = e % kRunRows;
  q.key = lds[q.own * kRunLdsStride + q.at];
  q.smaller = 0u;
  q.before = 0u;
  q.behind = 0xFFFFFFFFu;
  int r0 = threadIdx.x & (kRunLanes - 1), left = runs;
  for (; left > 2 * kRunLanes; left -= 4 * kRunLanes, r0 += 4 * kRunLanes) run_search_some<kRunLanes, 4, NEIGHBOURS>(lds, runs, r0, q);
  if (left > kRunLanes)
    run_search_some<kRunLanes, 2, NEIGHBOURS>(lds, runs, r0, q);
  else if (left > 0)
    run_search_some<kRunLanes, 1, NEIGHBOURS>(lds, runs, r0, q);
  if constexpr (NEIGHBOURS) {
    next_to->before = run_group<kRunLanes>(q.before, [](uint32_t a, uint32_t b) { return max(a, b); });
    next_to->behind = run_group<kRunLanes>(q.behind, [](uint32_t a, uint32_t b) { return min(a, b); });
  }
  return (int)run_group<kRunLanes>(q.smaller, [](uint32_t a, uint32_t b) { return a + b; });
}

}  // namespace evx
