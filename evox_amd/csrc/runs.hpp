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

#include <type_traits>

#include "common.hpp"

namespace evx {

constexpr int kRunRows = 512;          // keys per run = threads that sort it
constexpr int kRunMaxRows = 32768;     // 4-byte keys that one workgroup's LDS holds
constexpr int kRunTile8 = 32;          // runs of 8-byte keys that it holds
constexpr int kRunRankThreads = 1024;  // threads of a workgroup that searches
// Keys from one run to the next in LDS: sixteen bytes more than a run, so that the runs' same entries fall into different banks.
template <class K>
struct RunLds {
  static constexpr int kStride = kRunRows + 16 / (int)sizeof(K);
};
__host__ __device__ inline int runs_of(int n) { return (n + kRunRows - 1) / kRunRows; }
__host__ __device__ inline size_t run_rank_lds_bytes(int n) { return sizeof(uint32_t) * RunLds<uint32_t>::kStride * (size_t)runs_of(n); }
__host__ __device__ inline size_t run_rank8_lds_bytes(int n) {  // (more keys: a tile after the other)
  return sizeof(uint64_t) * RunLds<uint64_t>::kStride * (size_t)(runs_of(n) < kRunTile8 ? runs_of(n) : kRunTile8);
}

// The key behind all others (no key of a row is larger; equal ones go by position).
template <class K>
__device__ __forceinline__ constexpr K run_last_key() {
  if constexpr (std::is_same_v<K, double>)
    return (double)INFINITY;
  else
    return ~(K)0;
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
__device__ __forceinline__ uint64_t lane_value(uint64_t v, int lane) {
  return ((uint64_t)lane_value((uint32_t)(v >> 32), lane) << 32) | lane_value((uint32_t)v, lane);
}

// (integers below 2^53: the hardware compares doubles at the rate of 32-bit values, 64-bit integers several times slower)
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __longlong_as_double((long long)lane_value((uint64_t)__double_as_longlong(v), lane));
}

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

// The sorted runs first .. first + runs - 1 of nv keys (run r at sorted + r * kRunRows) into LDS, in pieces of sixteen bytes
// where they are aligned so; the last run of all is filled up with the largest key.  Called by every thread; the caller puts a barrier behind it.
template <class K>
__device__ __forceinline__ void runs_to_lds(const K* __restrict__ sorted, int nv, int first, int runs, K* lds) {
  constexpr int kVec = 16 / (int)sizeof(K);
  sorted += (int64_t)first * kRunRows;
  const int count = min(nv - first * kRunRows, runs * kRunRows);
  const int whole = (reinterpret_cast<uintptr_t>(sorted) & 15u) == 0 ? count & ~(kVec - 1) : 0;
#pragma unroll 4
  for (int e = threadIdx.x * kVec; e < whole; e += blockDim.x * kVec)
    *reinterpret_cast<uint4*>(lds + (e / kRunRows) * RunLds<K>::kStride + (e % kRunRows)) = *reinterpret_cast<const uint4*>(sorted + e);
#pragma unroll 4
  for (int e = whole + threadIdx.x; e < runs * kRunRows; e += blockDim.x)
    lds[(e / kRunRows) * RunLds<K>::kStride + (e % kRunRows)] = e < count ? sorted[e] : run_last_key<K>();
}

// The sum / maximum / minimum over the kRunLanes consecutive lanes of a group, the same in all of them.
constexpr int kRunLanes = 4;
template <class Op>
__device__ __forceinline__ uint32_t run_group(uint32_t v, Op op) {
  static_assert(kRunLanes == 4, "permutations of four lanes");
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, false));     // lanes 1 0 3 2
  return op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, false));  // lanes 2 3 0 1
}
template <class Op>
__device__ __forceinline__ uint64_t run_group(uint64_t v, Op op) {
  auto permuted = [&](auto control) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, control.value, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), control.value, 0xf, 0xf, false);
    return ((uint64_t)hi << 32) | lo;
  };
  v = op(v, permuted(std::integral_constant<int, 0xB1>{}));
  return op(v, permuted(std::integral_constant<int, 0x4E>{}));
}

// A key whose place is being looked for, and what its searches have found so far.
template <class K>
struct RunSearch {
  K key;
  int own, at;  // its run, and its place in that
  uint32_t smaller = 0;   // how many keys precede it
  uint32_t equal = 0;     // kRunEqual: how many of them are equal to it
  K before = 0, behind = run_last_key<K>();  // the largest key before it (0 where there is none) and the smallest behind it (meaningless at the last place)
};

// What a search looks for besides the number of keys that precede the key.
constexpr int kRunTies = 0;        // (equal keys of earlier positions precede it)
constexpr int kRunNeighbours = 1;  // ... and its neighbours
constexpr int kRunSmaller = 2;     // (only smaller keys precede it)
constexpr int kRunEqual = 3;       // as kRunTies, and how many of the keys that precede it are equal to it

// U searches side by side in the runs `first` + r0, r0 + kRunLanes, ... of which LDS holds `runs`.
template <int U, int MODE, class K>
__device__ __forceinline__ void run_search_some(const K* lds, int first, int runs, int r0, RunSearch<K>& q) {
  const K* c[U];  // (an address in LDS: a step is one read, one comparison, one selection and one addition)
  K bound[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r = r0 + kRunLanes * u;
    c[u] = lds + (r < runs ? r : 0) * RunLds<K>::kStride;
    bound[u] = MODE != kRunSmaller && first + r < q.own ? q.key : q.key - (K)1;
  }
#pragma unroll
  for (int s = kRunRows / 2; s >= 1; s >>= 1) {
    K v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = c[u][s - 1];
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] += v[u] <= bound[u] ? s : 0;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r = r0 + kRunLanes * u;
    const bool own = MODE != kRunSmaller && first + r == q.own;
    const K* const run = lds + (r < runs ? r : 0) * RunLds<K>::kStride;
    int n = (int)(c[u] - run) + (*c[u] <= bound[u] ? 1 : 0);
    if (q.key == (K)0 && (MODE == kRunSmaller || first + r > q.own)) n = 0;
    if (own) n = q.at;
    q.smaller += r < runs ? (uint32_t)n : 0u;
    if constexpr (MODE == kRunEqual) {  // (seldom any: a second search only where the last key that precedes it is equal)
      if (r < runs && n > 0 && run[n - 1] == q.key) q.equal += (uint32_t)(n - run_search<kRunRows>(run, q.key, false));
    }
    if constexpr (MODE == kRunNeighbours) {  // (read whether or not there is one: branches would put the reads one after the other)
      const K lower = run[n > 0 ? n - 1 : 0], upper = run[min(own ? n + 1 : n, kRunRows - 1)];
      if (r < runs && n > 0) q.before = lower > q.before ? lower : q.before;
      if (r < runs && n + (own ? 1 : 0) < kRunRows) q.behind = upper < q.behind ? upper : q.behind;
    }
  }
}

// The searches for one key in the runs first .. first + runs - 1, which lie in LDS: q is the same in the kRunLanes lanes that
// call it together, each with its share of the runs, four of them at a time (a search is a chain of ten LDS round trips).
// The keys of a wave should be neighbours in their run: their searches then read the same words mostly, and four lanes
// per key mean four different words of a wave's read in the LDS banks instead of sixteen (terms of 20 001 x 3, forty
// runs, us: sixteen lanes per key 11.6, eight 12.0, four 9.3).
// The comparison `v precedes key` is v <= bound, the bound being the key or one less: one instruction per step.  A key
// of zero that no equal key precedes has no such bound; nothing precedes it.
template <int MODE, class K>
__device__ __forceinline__ void run_search_all(const K* lds, int first, int runs, RunSearch<K>& q) {
  int r0 = threadIdx.x & (kRunLanes - 1), left = runs;
  for (; left > 2 * kRunLanes; left -= 4 * kRunLanes, r0 += 4 * kRunLanes) run_search_some<4, MODE>(lds, first, runs, r0, q);
  if (left > kRunLanes)
    run_search_some<2, MODE>(lds, first, runs, r0, q);
  else if (left > 0)
    run_search_some<1, MODE>(lds, first, runs, r0, q);
}
// Once all runs have been searched: the sums over the group.  The key's place is q.smaller then.
template <int MODE, class K>
__device__ __forceinline__ void run_search_end(RunSearch<K>& q) {
  q.smaller = run_group(q.smaller, [](uint32_t a, uint32_t b) { return a + b; });
  if constexpr (MODE == kRunEqual) q.equal = run_group(q.equal, [](uint32_t a, uint32_t b) { return a + b; });
  if constexpr (MODE == kRunNeighbours) {
    q.before = run_group(q.before, [](K a, K b) { return a > b ? a : b; });
    q.behind = run_group(q.behind, [](K a, K b) { return a < b ? a : b; });
  }
}

}  // namespace evx
