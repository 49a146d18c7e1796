// Two objectives, up to 4096 rows, one workgroup per population, no dominance matrix.
//
// Reference semantics: non_dominate_rank (src/evox/operators/selection/non_dominate.py:172-195, batched :107-125),
// crowding_distance (:198-231) and nd_environmental_selection (:234-254) for M = 2.
//
// With the rows in the order of (f1, f2, index), a row is dominated exactly by the earlier rows whose f2 is smaller
// or equal and that are not copies of it, so front r is the set of strict prefix minima of f2 among the rows that
// fronts 0 .. r-1 have left (two.hpp does the same across workgroups for large populations).  Two objectives mean
// many thin fronts (C2: 20 fronts of 100 rows), which cost the matrix kernels an exchange between workgroups each;
// here a front is one prefix minimum over the registers of four waves, which hand it on from wave to wave.
//
// The orders:
//   * (f1, f2, index): by buckets (two_small_place): a monotone map of f1 to 4096 buckets, LDS counters, and every row
//     compared with the rows of its own bucket in full -- one pass, whatever ties there are, as long as no bucket is
//     crowded (none is tried where all f1 are the same, only one where a sample says that few are); else a stable LSD radix sort of (32-bit key, 16-bit payload) pairs, eight bits a pass, on f2 and then f1;
//   * the listing of the fronts by (rank, index): one or two passes of that sort on the ranks;
//   * the last front by either objective: its rows already stand in the order of f1, which backwards is that of f2;
//   * its order by the distance, for the index-stable top-k: by counting while it is small, by buckets, else by the sort.
// A pass of the sort ranks the items of a wave among those of equal digit through a table of lane masks (stable), keeps
// a counter per (digit, wave) and scans the 4096 counters once.
//
// What bounds it: chains of dependent instructions and LDS round trips inside one workgroup; of 2000 uniform rows the
// rounds of the peeling 20 us of 34, the order of (f1, f2) 5.5, the listing 3, the gather 3.  us per selection of half the
// rows (30 values each), in a loop of calls, with a hash table for shared f1, four or eight passes of the sort for the
// first order, sixteen waves with a barrier per front and the last front by counting or three sorts -> like this:
//   rows                        200          1024         2000         4096
//   uniform                     24.4 -> 15   38 -> 26     63.5 -> 37   112 -> 62
//   twenty fronts, shared f1    26.4 -> 15.6 34.6 -> 22   45 -> 28.3   71 -> 48
//   one front                   22.8 -> 14.8 88 -> 19.4   59.5 -> 26   99 -> 43
//   equal rows                  16 -> 15     77 -> 27     58 -> 35     96 -> 55
//   four levels                 21 -> 18     29 -> 29     48 -> 41     108 -> 62
#pragma once

#include <type_traits>

#include "batched.hpp"
#include "peel.hpp"
#include "two.hpp"

// Hook for timing builds; nothing otherwise.
#ifndef EVX_PASS_TRACE
#define EVX_PASS_TRACE(slot)
#endif

namespace evx {

constexpr int kTwoSmallThreads = 1024;
constexpr int kTwoSmallRows = 4096;
constexpr int kTwoSmallPer = kTwoSmallRows / kTwoSmallThreads;  // items of a thread in every pass
constexpr int kTwoSmallBuckets = 4096;   // of two_small_place: four counters per thread
constexpr uint32_t kTwoSmallCrowd = 64;  // rows of a bucket up to which every row of it looks at every other one
constexpr int kTwoSmallCounting = 192;   // last fronts of at most this many rows are ordered by counting, larger ones by buckets
constexpr int kTwoSmallTied = 512;       // ... up to which they are where many distances are equal: 500 rows, all equal, 28 -> 21 us; 1000 33 -> 38
constexpr int kTwoSmallWaves = 4;        // waves that peel: one per SIMD of the compute unit
constexpr int kTwoSmallRing = 64;        // rounds that a wave may be ahead of the next one
constexpr uint16_t kTwoSmallUnset = 0xFFFFu;
// dynamic LDS: keys and payloads of the sort twice over, its counters, the keys of both objectives by row, ranks,
// the three orders, the distances
constexpr size_t kTwoSmallLdsBytes = (size_t)kTwoSmallRows * (4 + 4 + 2 + 2 + 4 + 4 + 4 + 2 + 2 + 2 + 2 + 4);

// Inclusive prefix sum over the lanes of a wave (DPP row shifts and row broadcasts, as wave_prefix_min).
__device__ inline uint32_t wave_prefix_sum(uint32_t x) {
  uint32_t v = x;
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x113, 0xf, 0xf, false);  // row_shr:3
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xe, false);  // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xc, false);  // row_shr:8
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

// The sum, minimum or maximum of words 0 .. wave-1 of sixteen words in LDS, the same in every lane: lane i < wave
// takes word i, four DPP steps fold the first row of sixteen lanes, and its last lane holds the result.  (Every vector
// instruction of a workgroup of sixteen waves costs the compute unit sixteen issue slots; a fold written as sixteen
// selects and additions per lane was a third of a round of the peeling.)
__device__ inline uint32_t sum_before_wave(const uint32_t* sixteen, int wave) {
  const int lane = threadIdx.x & 63;
  int v = lane < wave ? (int)sixteen[lane & 15] : 0;
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xe, true);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xc, true);  // row_shr:8
  return (uint32_t)__builtin_amdgcn_readlane(v, 15);
}
__device__ inline uint32_t min_before_wave(const uint32_t* sixteen, int wave) {
  const int lane = threadIdx.x & 63;
  uint32_t v = lane < wave ? sixteen[lane & 15] : kTwoNone;
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)kTwoNone, (int)v, 0x111, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)kTwoNone, (int)v, 0x112, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)kTwoNone, (int)v, 0x114, 0xf, 0xe, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)kTwoNone, (int)v, 0x118, 0xf, 0xc, false));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
}
__device__ inline uint32_t max_before_wave(const uint32_t* sixteen, int wave) {
  const int lane = threadIdx.x & 63;
  uint32_t v = lane < wave ? sixteen[lane & 15] : 0u;
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xe, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xc, false));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
}

// One stable pass of the sort: items 0 .. count-1 of (key_in, pay_in) go to (key_out, pay_out) in the order of the
// digit (key >> shift) & 255, items of equal digit in the order they had.  Called by all kTwoSmallThreads threads.
// cnt: 4096 counters (wave * 256 + digit); part: 16 words; lanes_a: 16 KB of LDS that is free during the pass (with
// key_out, which is written only at the end: a table of 256 lane masks per wave).  Ends with a barrier.
//   1. every wave counts its items per digit, row by row (64 items): every lane sets its bit in the wave's table entry
//      of its digit (an LDS atomic) and reads the entry back -- the lanes of equal digit --, an item's rank within its
//      wave is the count so far plus the lanes of equal digit below it; the last lane of a digit's group adds the
//      group to the count and clears the entry (the ballots that find such a group without LDS, eight per row, cost
//      four times the vector instructions);
//   2. the 4096 counters are scanned in the order (digit, wave), four per thread;
//   3. the items go to their places.
template <bool PARTIAL>  // leave out the items whose key is kTwoSmallUnset; the others end up side by side
__device__ inline void two_small_pass(const uint32_t* key_in, const uint16_t* pay_in, uint32_t* key_out, uint16_t* pay_out,
                                      int count, int shift, uint32_t* cnt, uint32_t* part, uint32_t* lanes_a) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  EVX_PASS_TRACE(0);
  const int first = wave * (64 * kTwoSmallPer) + lane;  // a wave's items are consecutive, row by row
  const bool wave_has_items = first - lane < count;      // (wave-uniform)
  unsigned long long* const table = reinterpret_cast<unsigned long long*>(wave < 8 ? lanes_a : key_out) + (wave & 7) * 256;
  // (outside step 2, which lies between barriers, a wave only touches its own counters)
#pragma unroll
  for (int i = 0; i < 4; ++i) cnt[wave * 256 + lane + 64 * i] = 0u;
  uint32_t key[kTwoSmallPer];
  uint16_t pay[kTwoSmallPer];
  int rin[kTwoSmallPer];
#pragma unroll
  for (int r = 0; r < kTwoSmallPer; ++r) {
    key[r] = 0u;
    pay[r] = 0;
    rin[r] = 0;
  }
  if (wave_has_items) {
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    reinterpret_cast<uint4*>(table)[2 * lane] = zero;
    reinterpret_cast<uint4*>(table)[2 * lane + 1] = zero;
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < kTwoSmallPer; ++r) {
      const int e = first + r * 64;
      if (e < count) {
        key[r] = key_in[e];
        pay[r] = pay_in[e];
      }
    }
    EVX_PASS_TRACE(1);
#pragma unroll
    for (int r = 0; r < kTwoSmallPer; ++r) {
      const int e = first + r * 64;
      if (e - lane >= count) continue;  // (wave-uniform: a row without items)
      if (e < count && !(PARTIAL && key[r] == kTwoSmallUnset)) {
        const uint32_t d = (key[r] >> shift) & 255u;
        atomicOr(&table[d], 1ull << lane);
        const uint64_t same = table[d];
        const uint32_t prior = cnt[wave * 256 + d];
        rin[r] = (int)prior + __popcll(same & below);
        if ((same >> lane) == 1ull) {  // the group's last lane
          cnt[wave * 256 + d] = prior + (uint32_t)__popcll(same);
          table[d] = 0ull;
        }
      }
    }
  }
  EVX_PASS_TRACE(2);
  __syncthreads();
  EVX_PASS_TRACE(3);
  // exclusive scan of the counters in the order (digit, wave): thread t has digit t / 4 and the four waves from
  // 4 (t % 4) on (a wave's counters lie together, so that the lanes of a wave meet different banks in steps 1 and 3)
  {
    uint32_t* const mine = cnt + (tid & 3) * 4 * 256 + (tid >> 2);
    const uint32_t c0 = mine[0], c1 = mine[256], c2 = mine[512], c3 = mine[768];
    const uint32_t sum = c0 + c1 + c2 + c3;
    const uint32_t incl = wave_prefix_sum(sum);
    if (lane == 63) part[wave] = incl;
    EVX_PASS_TRACE(4);
    __syncthreads();
    EVX_PASS_TRACE(5);
    uint32_t run = incl - sum + sum_before_wave(part, wave);
    mine[0] = run;
    run += c0;
    mine[256] = run;
    run += c1;
    mine[512] = run;
    run += c2;
    mine[768] = run;
  }
  EVX_PASS_TRACE(6);
  __syncthreads();
  EVX_PASS_TRACE(7);
  if (wave_has_items) {
#pragma unroll
    for (int r = 0; r < kTwoSmallPer; ++r) {
      if (first + r * 64 < count && !(PARTIAL && key[r] == kTwoSmallUnset)) {
        const uint32_t d = (key[r] >> shift) & 255u;
        const int to = (int)cnt[wave * 256 + d] + rin[r];
        key_out[to] = key[r];
        pay_out[to] = pay[r];
      }
    }
  }
  EVX_PASS_TRACE(8);
  __syncthreads();
  EVX_PASS_TRACE(9);
}

// `passes` passes from the lowest digit up (1 .. 4); returns through the references where the result lies.  vary: the
// bits in which any two keys differ (or more bits); a digit in which no two keys differ needs no pass -- objectives
// that take few values, such as counts or multiples of a step, leave the low bits of their float32 images alike.
__device__ inline void two_small_sort(uint32_t*& key_a, uint16_t*& pay_a, uint32_t*& key_b, uint16_t*& pay_b, int count, int passes,
                                      uint32_t* cnt, uint32_t* part, uint32_t* lanes_a, uint32_t vary = 0xFFFFFFFFu) {
#pragma unroll 1  // (code that runs once waits for memory at every line of it)
  for (int p = 0; p < passes; ++p) {
    if (((vary >> (8 * p)) & 255u) == 0u) continue;  // (the same in every thread)
    two_small_pass<false>(key_a, pay_a, key_b, pay_b, count, 8 * p, cnt, part, lanes_a);
    uint32_t* tk = key_a;
    key_a = key_b;
    key_b = tk;
    uint16_t* tp = pay_a;
    pay_a = pay_b;
    pay_b = tp;
  }
}

// The smallest and the largest of the workgroup's values (smallest > largest: no thread had any).  lo16, hi16: sixteen words each.
// Ends with every thread past a barrier; the caller puts another one before lo16 and hi16 are written again.
__device__ inline void two_small_range(uint32_t& lo, uint32_t& hi, uint32_t* lo16, uint32_t* hi16, int nt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t wave_lo = wave_prefix_min(lo), wave_hi = ~wave_prefix_min(~hi);
  if (lane == 63) {
    lo16[wave] = wave_lo;
    hi16[wave] = wave_hi;
  }
  __syncthreads();
  lo = min_before_wave(lo16, nt / 64);
  hi = max_before_wave(hi16, nt / 64);
}

// Buckets 0 .. buckets - 1 for keys (ordered_key) whose finite ones lie between lo and hi: none lower than that of a smaller key,
// however the differences and products round.  By value: of equal width, everything but NaN in the first one where the width is
// zero or overflows.  By image: of equal width in the key (values over many binades), infinities in buckets of their own.
__device__ inline uint32_t bucket_by_value(uint32_t key, uint32_t lo, uint32_t hi, int buckets) {
  const float v0 = cost_of_key(lo), width = cost_of_key(hi) - v0;
  const float scale = lo < hi && width > 0.0f ? (float)(buckets - 1) / width : 0.0f;
  const float t = (cost_of_key(key) - v0) * scale;
  return key == 0xFFFFFFFFu || t >= (float)(buckets - 1) ? (uint32_t)buckets - 1u : t > 0.0f ? (uint32_t)t : 0u;
}
__device__ inline uint32_t bucket_by_image(uint32_t key, uint32_t lo, uint32_t hi, int buckets) {
  const float scale = lo < hi ? (float)(buckets - 3) / (float)(hi - lo) : 0.0f;
  return key < lo ? 0u : key > hi ? (uint32_t)buckets - 1u : 1u + min((uint32_t)((float)(key - lo) * scale), (uint32_t)buckets - 3u);
}

// Places of `count` items (item tid + nt r of thread tid of the nt in the workgroup; id below 65536, all different) in the ascending order of
// (comp, id).  bucket: a map of comp to 0 .. 4 nt - 1 that never decreases as comp grows.  False, with
// nothing but cnt and part touched, when a bucket holds more than kTwoSmallCrowd items.  twins: some item of this thread shares its comp
// with another one.  cnt: 4 nt words; part: 16 words; comps, ids: count entries each.  Bound by LDS: an
// atomic, a scan of four counters per thread and as many reads per item as its bucket has members.
template <int PER>
__device__ inline bool two_small_place(const uint64_t (&comp)[PER], const uint32_t (&id)[PER], const uint32_t (&bucket)[PER], int count,
                                       int nt, uint32_t* cnt, uint32_t* part, uint64_t* comps, uint16_t* ids, int (&place)[PER], bool& twins) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  reinterpret_cast<uint4*>(cnt)[tid] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  uint32_t arrived[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r)
    arrived[r] = tid + nt * r < count ? atomicAdd(&cnt[bucket[r]], 1u) : 0u;
  __syncthreads();
  const uint4 mine = reinterpret_cast<const uint4*>(cnt)[tid];
  const uint32_t sum = mine.x + mine.y + mine.z + mine.w;
  const uint32_t incl = wave_prefix_sum(sum);
  if (lane == 63) part[wave] = incl;
  const bool crowded = max(max(mine.x, mine.y), max(mine.z, mine.w)) > kTwoSmallCrowd;
  if (__syncthreads_or(crowded)) return false;
  const uint32_t run = incl - sum + sum_before_wave(part, wave);
  reinterpret_cast<uint4*>(cnt)[tid] = make_uint4(run, run + mine.x, run + mine.x + mine.y, run + mine.x + mine.y + mine.z);
  __syncthreads();
  uint32_t first[PER], end[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    first[r] = end[r] = 0u;
    if (tid + nt * r < count) {
      first[r] = cnt[bucket[r]];
      end[r] = bucket[r] + 1u < 4u * (uint32_t)nt ? cnt[bucket[r] + 1u] : (uint32_t)count;
      comps[first[r] + arrived[r]] = comp[r];
      ids[first[r] + arrived[r]] = (uint16_t)id[r];
    }
  }
  __syncthreads();
  twins = false;
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    int before = 0;
    for (uint32_t q = first[r]; q < end[r]; q += 4) {  // (four members' reads in flight together)
      uint64_t other[4];
      uint32_t other_id[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t at = min(q + (uint32_t)u, end[r] - 1u);
        other[u] = comps[at];
        other_id[u] = q + (uint32_t)u < end[r] ? (uint32_t)ids[at] : id[r];  // (the item itself counts for nothing)
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool another = other_id[u] != id[r];
        before += another && (other[u] < comp[r] || (other[u] == comp[r] && other_id[u] < id[r])) ? 1 : 0;
        twins |= another && other[u] == comp[r];
      }
    }
    place[r] = (int)first[r] + before;
  }
  return true;
}

// ---- The peeling.  Wave w < waves holds positions 64 PER w .. 64 PER (w + 1) - 1 of the (f1, f2, index) order, PER
// consecutive ones per lane; val holds f2 (kTwoNone for what is out of the sweep).  In round r a wave needs the smallest
// f2 of front r among the positions before its own, and tells the next wave the smallest up to its end: the waves go
// through the rounds one after the other, none waits for a later one but to keep kTwoSmallRing rounds of messages.  A
// message also carries how many rows the rounds before it have ranked, so the last wave sees the end a round late and
// raises `ended`; rounds that earlier waves went through by then count for nothing (their ranks lie above the last front's).
// Four waves, one per SIMD, because a round is bound by instruction issue: sixteen waves of a quarter of the positions
// spend sixteen issue slots on each of the seven steps of the prefix minimum.  Sixteen positions per lane above 2048 rows, eight
// below (2000 uniform rows: 20 us with four waves of eight, 22 with two of sixteen), four up to 256 (one wave, no messages).
struct TwoSmallPeel {
  unsigned long long ring[kTwoSmallWaves - 1][kTwoSmallRing];  // round + 1 << 48 | rows ranked << 32 | smallest f2
  int progress[kTwoSmallWaves];                                 // rounds whose message wave w has taken
  int ended;                                                    // 1 + the round of the last front, 0: not known yet
  int total, nv;                                                // rows ranked up to the last front, rows in it
};

template <int PER, bool COPIES>  // COPIES: some row has copies, counted at the first one's position (the other instance reads no count)
__device__ __forceinline__ void two_small_rounds(const uint32_t* val, const uint32_t* copies, uint16_t* rank_at, int n, int waves,
                                                 int ranked_already, int stop, TwoSmallPeel* st) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // (known to be uniform: the branches below are scalar)
  const bool first_wave = wave == 0, last_wave = wave == waves - 1;
  auto word = [](const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  const int at = (wave * 64 + lane) * PER;
  uint32_t v[PER];
  int ranked[PER], group[PER];  // group: a row and its copies
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    v[e] = at + e < n ? val[at + e] : kTwoNone;
    group[e] = COPIES && at + e < n ? 1 + (int)copies[at + e] : 1;
    ranked[e] = kTwoSmallUnset;
  }
  auto message = [&](int round) {
    return first_wave ? 0ull : __hip_atomic_load(&st->ring[wave - 1][round % kTwoSmallRing], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  unsigned long long in = message(0);
  int own = 0, before_last = 0;  // rows ranked by this wave so far; (last wave) by all waves before the last round
  for (int round = 0;; ++round) {
    int over = last_wave ? 0 : word(&st->ended);  // (asked for early)
    uint32_t before[PER];  // smallest of the lane's own earlier positions (so that no step below waits for the one before it)
    before[0] = kTwoNone;
#pragma unroll
    for (int e = 1; e < PER; ++e) before[e] = min(before[e - 1], v[e - 1]);
    const uint32_t incl = wave_prefix_min(min(before[PER - 1], v[PER - 1]));
    uint32_t running = (uint32_t)__builtin_amdgcn_update_dpp((int)kTwoNone, (int)incl, 0x138, 0xf, 0xf, false);  // wave_shr:1
    uint32_t lowest = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    int total = own;
    over = __builtin_amdgcn_readfirstlane(over);
    if (!first_wave) {
      // (the wave before never waits for this one's round; it leaves without a message only once `ended` is set)
      uint32_t in_lo, in_hi;
      for (;;) {
        in_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)in);
        in_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(in >> 32));
        if ((in_hi >> 16) == (uint32_t)round + 1u || over != 0) break;
        in = message(round);
        const int now_over = last_wave ? 0 : word(&st->ended);
        over |= __builtin_amdgcn_readfirstlane(now_over);
      }
      in = message(round + 1);  // (the next one: it may be there when this round is over)
      running = min(running, in_lo);
      lowest = min(lowest, in_lo);
      total += (int)(in_hi & 0xFFFFu);
      if (lane == 0) __hip_atomic_store(&st->progress[wave], round + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (!last_wave) {
      if (round >= kTwoSmallRing && round % (kTwoSmallRing / 2) == 0) {
        // room for the next half ring: the next wave has taken what lies there
        int taken;
        do {
          const int p = word(&st->progress[wave + 1]), now_over = word(&st->ended);
          taken = __builtin_amdgcn_readfirstlane(p);
          over |= __builtin_amdgcn_readfirstlane(now_over);
        } while (taken < round - kTwoSmallRing / 2 && over == 0);
      }
      if (over != 0) break;
      if (lane == 0)
        __hip_atomic_store(&st->ring[wave][round % kTwoSmallRing],
                           ((unsigned long long)(((uint32_t)round + 1u) << 16 | (uint32_t)total) << 32) | lowest, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
    } else if (round > 0) {
      total += ranked_already;  // (rows with a NaN: front 0)
      if (total >= stop) {      // reached at the latest when every row is ranked
        if (lane == 0) {
          st->total = total;
          st->nv = total - before_last;
          __hip_atomic_store(&st->ended, round, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        break;
      }
      before_last = total;
    }
    int add = 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const uint32_t mine = v[e];
      const bool now = mine < min(running, before[e]);  // (a row out of the sweep holds kTwoNone, which is below nothing)
      ranked[e] = now ? round : ranked[e];
      v[e] = now ? kTwoNone : mine;
      if constexpr (COPIES)
        add += now ? group[e] : 0;
      else
        add += __popcll(__builtin_amdgcn_ballot_w64(now));
    }
    own += COPIES ? wave_sum(add) : add;
  }
#pragma unroll
  for (int e = 0; e < PER; ++e)
    if (at + e < n) rank_at[at + e] = (uint16_t)ranked[e];
}

// Grid: one workgroup of kTwoSmallThreads per population; dynamic LDS kTwoSmallLdsBytes.  a.m == 2, a.n <= kTwoSmallRows.
__global__ __launch_bounds__(kTwoSmallThreads) void two_small_kernel(BatchedArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t two_small_lds[];
  __shared__ TwoSmallPeel peel[1];
  __shared__ __attribute__((aligned(16))) uint32_t part[16];
  __shared__ __attribute__((aligned(16))) uint32_t lo16[16];
  __shared__ __attribute__((aligned(16))) uint32_t hi16[16];
  __shared__ uint32_t vary_bits[2];  // (radix path) bits in which the keys of f1 / of f2 differ from those of row 0
  __shared__ int nan_rows_lds[1];
  __shared__ int tied_lds[1];  // many rows of the last front share a distance
  uint32_t* key_a = reinterpret_cast<uint32_t*>(two_small_lds);  // the sort's buffers
  uint32_t* key_b = key_a + kTwoSmallRows;
  uint16_t* pay_a = reinterpret_cast<uint16_t*>(key_b + kTwoSmallRows);
  uint16_t* pay_b = pay_a + kTwoSmallRows;
  uint32_t* cnt = reinterpret_cast<uint32_t*>(pay_b + kTwoSmallRows);
  uint32_t* k1 = cnt + kTwoSmallRows;  // ordered keys of the objectives by position of the (f1, f2, index) order
  uint32_t* k2 = k1 + kTwoSmallRows;
  float* dist = reinterpret_cast<float*>(k2 + kTwoSmallRows);  // of the last front's rows, by row; before that:
  uint32_t* lanes_a = reinterpret_cast<uint32_t*>(dist);       // the lane masks of the sort's first eight waves
  uint16_t* rank16 = reinterpret_cast<uint16_t*>(dist + kTwoSmallRows);  // ranks by position
  uint16_t* lexi = rank16 + kTwoSmallRows;     // row at every position
  uint16_t* first_at = lexi + kTwoSmallRows;   // position of the first copy of the row at every position (where there are copies)
  uint16_t* other16 = first_at + kTwoSmallRows;

  const int n = a.n;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* __restrict__ f = a.f + (int64_t)blockIdx.x * a.f_stride_b;
  auto fitness_at = [&](int i, int k) {
    return f[(int64_t)i * a.f_stride_row + (int64_t)k * a.f_stride_col + (i >= a.n_first ? a.f_second : 0)];
  };
  constexpr uint32_t kNanKey = 0xFFFFFFFFu;  // (ordered_key)

  EVX_BATCH_TRACE(0);
  // ---- keys, and the order of (f1, f2, index)
  bool has_copies = false;
  {
    uint32_t a1[kTwoSmallPer], a2[kTwoSmallPer], id[kTwoSmallPer], bucket[kTwoSmallPer];
    uint64_t comp[kTwoSmallPer];
    int place[kTwoSmallPer];
    uint32_t lo = 0xFFFFFFFFu, hi = 0u;  // of the finite values of f1
    const uint32_t key_inf = ordered_key(INFINITY), key_neg_inf = ordered_key(-INFINITY);
#pragma unroll
    for (int r = 0; r < kTwoSmallPer; ++r) {
      const int i = tid + kTwoSmallThreads * r;
      a1[r] = a2[r] = 0u;
      if (i < n) {
        a1[r] = ordered_key(fitness_at(i, 0));
        a2[r] = ordered_key(fitness_at(i, 1));
      }
      id[r] = (uint32_t)i;
      comp[r] = ((uint64_t)a1[r] << 32) | a2[r];
      if (i < n && a1[r] > key_neg_inf && a1[r] < key_inf) {
        lo = min(lo, a1[r]);
        hi = max(hi, a1[r]);
      }
    }
    if (tid == 0) {
      nan_rows_lds[0] = 0;
      tied_lds[0] = 0;
      peel->ended = 0;
    }
    if (tid < kTwoSmallWaves) peel->progress[tid] = 0;
    if (tid < (kTwoSmallWaves - 1) * kTwoSmallRing) (&peel->ring[0][0])[tid] = 0ull;
    two_small_range(lo, hi, lo16, hi16, kTwoSmallThreads);
    // By buckets of equal width in the value of f1, else in its image.  Where one f1 is that of many rows neither will do, and an attempt
    // that fails takes 3 us (additions to one counter): none is made where all values are the same, and no second one where sixty-four
    // rows of a sample share their f1 with four of them more often than if some eighty rows of the population did.
    bool ordered = false;
    auto place_by = [&](auto bucket_of) {
#pragma unroll
      for (int r = 0; r < kTwoSmallPer; ++r) bucket[r] = bucket_of(a1[r], lo, hi, kTwoSmallBuckets);
      return two_small_place<kTwoSmallPer>(comp, id, bucket, n, kTwoSmallThreads, cnt, part, reinterpret_cast<uint64_t*>(key_a), pay_a, place, has_copies);
    };
    if (__builtin_expect(lo < hi, 1)) {
      ordered = place_by([](uint32_t key, uint32_t from, uint32_t to, int buckets) { return bucket_by_value(key, from, to, buckets); });
      if (__builtin_expect(!ordered, 0)) {
        const uint32_t key = ordered_key(fitness_at((int)((unsigned)(lane * n) >> 6), 0));  // (by every wave for itself)
        int same = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) same += __popcll(__builtin_amdgcn_ballot_w64(key == (uint32_t)__builtin_amdgcn_readlane((int)key, 8 + 16 * u)));
        if (same * n <= 7 * n + 4 * 63 * 80)
          ordered = place_by([](uint32_t key, uint32_t from, uint32_t to, int buckets) { return bucket_by_image(key, from, to, buckets); });
      }
    }
    EVX_BATCH_TRACE(1);
    if (__builtin_expect(!ordered, 0)) {  // (the same in every thread) many rows share an f1
      __syncthreads();
      if (tid < 2) vary_bits[tid] = 0u;
#pragma unroll
      for (int r = 0; r < kTwoSmallPer; ++r) {
        const int i = tid + kTwoSmallThreads * r;
        if (i < n) {
          k1[i] = a1[r];
          k2[i] = a2[r];
          key_a[i] = a2[r];
          pay_a[i] = (uint16_t)i;
        }
      }
      __syncthreads();
      uint32_t v1 = 0u, v2 = 0u;
#pragma unroll
      for (int r = 0; r < kTwoSmallPer; ++r) {
        if (tid + kTwoSmallThreads * r < n) {
          v1 |= a1[r] ^ k1[0];
          v2 |= a2[r] ^ k2[0];
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        v1 |= (uint32_t)__shfl_xor((int)v1, off);
        v2 |= (uint32_t)__shfl_xor((int)v2, off);
      }
      if (lane == 0) {
        if (v1) atomicOr(&vary_bits[0], v1);
        if (v2) atomicOr(&vary_bits[1], v2);
      }
      __syncthreads();
      two_small_sort(key_a, pay_a, key_b, pay_b, n, 4, cnt, part, lanes_a, vary_bits[1]);
      for (int s = tid; s < n; s += kTwoSmallThreads) key_a[s] = k1[pay_a[s]];
      __syncthreads();
      two_small_sort(key_a, pay_a, key_b, pay_b, n, 4, cnt, part, lanes_a, vary_bits[0]);
      // by position: every thread takes what it moves out of the arrays by row before any of it is written
#pragma unroll
      for (int r = 0; r < kTwoSmallPer; ++r) {
        const int s = tid + kTwoSmallThreads * r;
        if (s < n) {
          id[r] = pay_a[s];
          a1[r] = k1[id[r]];
          a2[r] = k2[id[r]];
          place[r] = s;
        }
      }
      key_a = reinterpret_cast<uint32_t*>(two_small_lds);
      key_b = key_a + kTwoSmallRows;
      pay_a = reinterpret_cast<uint16_t*>(key_b + kTwoSmallRows);
      pay_b = pay_a + kTwoSmallRows;
      has_copies = true;  // (asked below)
      __syncthreads();
    }
    int nan_rows = 0;
#pragma unroll
    for (int r = 0; r < kTwoSmallPer; ++r) {
      if (tid + kTwoSmallThreads * r < n) {
        k1[place[r]] = a1[r];
        k2[place[r]] = a2[r];
        lexi[place[r]] = (uint16_t)id[r];
        nan_rows += a1[r] == kNanKey || a2[r] == kNanKey ? 1 : 0;
      }
    }
    if (nan_rows != 0) atomicAdd(&nan_rows_lds[0], nan_rows);
    has_copies = __syncthreads_or(has_copies) != 0;
  }
  EVX_BATCH_TRACE(2);
  const int nan_rows = nan_rows_lds[0];

  // ---- out of the sweep: rows with a NaN (nothing compares with them: front 0) and the copies of a row (they take
  // the rank of the first copy, which counts for all of them)
  uint32_t* copies = cnt;           // per position of a first row
  uint32_t* val = k2;
  if (__builtin_expect(nan_rows != 0 || has_copies, 0)) {
    val = key_a;
    uint32_t last_first = 0u;  // 1 + the last position of this thread that is not a copy, 0 = none
    bool is_copy[kTwoSmallPer];
#pragma unroll
    for (int e = 0; e < kTwoSmallPer; ++e) {
      const int s = kTwoSmallPer * tid + e;
      is_copy[e] = false;
      if (s < n) {
        const uint32_t a1 = k1[s], a2 = k2[s];
        const bool is_nan = a1 == kNanKey || a2 == kNanKey;
        is_copy[e] = !is_nan && s > 0 && k1[s - 1] == a1 && k2[s - 1] == a2;
        val[s] = is_nan || is_copy[e] ? kTwoNone : a2;
        if (!is_copy[e]) last_first = (uint32_t)s + 1u;
        copies[s] = 0u;
      }
    }
    // the first copy of a copy: the last position before it that is not one (a prefix maximum)
    const uint32_t incl = ~wave_prefix_min(~last_first);
    const uint32_t excl = ~(uint32_t)__builtin_amdgcn_update_dpp((int)0xFFFFFFFFu, (int)~incl, 0x138, 0xf, 0xf, false);  // wave_shr:1
    if (lane == 63) hi16[wave] = incl;
    __syncthreads();
    uint32_t carry = max(excl, max_before_wave(hi16, wave));
#pragma unroll
    for (int e = 0; e < kTwoSmallPer; ++e) {
      const int s = kTwoSmallPer * tid + e;
      if (s < n) {
        if (!is_copy[e]) carry = (uint32_t)s + 1u;
        first_at[s] = (uint16_t)(carry - 1u);  // (a copy always has a first row before it)
        if (is_copy[e]) atomicAdd(&copies[carry - 1u], 1u);
      }
    }
    __syncthreads();
  }
  EVX_BATCH_TRACE(3);
  const int stop = a.stop_count;
  {
    const int per = n <= 64 * 4 ? 4 : n <= 64 * kTwoSmallWaves * 8 ? 8 : 16;
    const int waves = (n + 64 * per - 1) / (64 * per);
    auto rounds = [&](auto positions) {
      if (has_copies)
        two_small_rounds<decltype(positions)::value, true>(val, copies, rank16, n, waves, nan_rows, stop, peel);
      else
        two_small_rounds<decltype(positions)::value, false>(val, copies, rank16, n, waves, nan_rows, stop, peel);
    };
    if (wave < waves) {
      if (per == 4)
        rounds(std::integral_constant<int, 4>());
      else if (per == 8)
        rounds(std::integral_constant<int, 8>());
      else
        rounds(std::integral_constant<int, 16>());
    }
    __syncthreads();
  }
  const int worst = peel->ended - 1, total = peel->total, nv = peel->nv;
  const int worst_start = total - nv;
  EVX_BATCH_TRACE(4);

  // ---- ranks by row into the sort's first buffer, and the rows of the last front put together in the order of (f1, f2, index)
  const bool selecting = a.out_f != nullptr;
  const bool by_value = !(worst == 0 && nan_rows != 0);  // (a last front with NaN rows is ordered by sorting below)
  int members = 0;
  uint32_t rank_of[kTwoSmallPer], m1[kTwoSmallPer], m2[kTwoSmallPer], m_row[kTwoSmallPer], m_first[kTwoSmallPer];
#pragma unroll
  for (int e = 0; e < kTwoSmallPer; ++e) {
    const int s = kTwoSmallPer * tid + e;
    rank_of[e] = kTwoSmallUnset;
    if (s < n) {
      m1[e] = k1[s];
      m2[e] = k2[s];
      m_row[e] = lexi[s];
      m_first[e] = has_copies ? (uint32_t)first_at[s] : (uint32_t)s;
      rank_of[e] = nan_rows != 0 && (m1[e] == kNanKey || m2[e] == kNanKey) ? 0u : (uint32_t)rank16[m_first[e]];
      if (rank_of[e] > (uint32_t)worst) rank_of[e] = kTwoSmallUnset;  // (not ranked, or in a round after the last front's)
      members += rank_of[e] == (uint32_t)worst ? 1 : 0;
    }
  }
  const uint32_t members_incl = wave_prefix_sum((uint32_t)members);
  if (lane == 63) part[wave] = members_incl;
  if (a.rank_all) {
#pragma unroll
    for (int e = 0; e < kTwoSmallPer; ++e)
      if (kTwoSmallPer * tid + e < n)
        a.rank_all[(int64_t)blockIdx.x * n + m_row[e]] = rank_of[e] == kTwoSmallUnset ? kRankUnset : (int)rank_of[e];
  }
  if (!selecting) return;  // rank-only mode
  __syncthreads();         // (also: every read of key_a as `val` is over, and every read of k1, k2, lexi and first_at)
  {
    uint32_t to = members_incl - (uint32_t)members + sum_before_wave(part, wave);
#pragma unroll
    for (int e = 0; e < kTwoSmallPer; ++e) {
      const int s = kTwoSmallPer * tid + e;
      if (s < n) {
        key_a[m_row[e]] = rank_of[e];
        pay_a[m_row[e]] = (uint16_t)m_row[e];
        if (rank_of[e] == (uint32_t)worst) {
          k1[to] = m1[e];
          k2[to] = m2[e];
          lexi[to] = (uint16_t)m_row[e];
          if (has_copies) {  // how many copies stand before this one, and how many there are
            first_at[to] = (uint16_t)((uint32_t)s - m_first[e]);
            other16[to] = (uint16_t)(1u + copies[m_first[e]]);
          }
          ++to;
        }
      }
    }
    __syncthreads();
  }
  EVX_BATCH_TRACE(5);

  // ---- distances of the last front: crowding_distance with the mask rank == worst, non_dominate.py:209-231.  Its rows,
  // leaving copies aside, stand in the ascending order of f1 and in the descending one of f2 (of two rows that share
  // either, one dominates the other); copies stand by index, in both orders.
  const int need = stop - worst_start;
  uint32_t d_row[kTwoSmallPer];
  float d_of[kTwoSmallPer];
  if (by_value) {
    const float span1 = cost_of_key(k1[nv - 1]) - cost_of_key(k1[0]);
    const float span2 = cost_of_key(k2[0]) - cost_of_key(k2[nv - 1]);
#pragma unroll
    for (int r = 0; r < kTwoSmallPer; ++r) {
      const int p = tid + kTwoSmallThreads * r;
      d_row[r] = 0u;
      d_of[r] = 0.0f;
      if (p < nv) {
        const int before = has_copies ? first_at[p] : 0, group = has_copies ? other16[p] : 1;
        const int q = nv - (p - before) - group + before;  // position in the order of f2
        d_row[r] = lexi[p];
        if (p == 0 || p == nv - 1 || q == 0 || q == nv - 1) {
          d_of[r] = INFINITY;
        } else {
          d_of[r] = (cost_of_key(k1[p + 1]) - cost_of_key(k1[p - 1])) / span1;
          d_of[r] += (cost_of_key(k2[nv - 2 - q]) - cost_of_key(k2[nv - q])) / span2;
        }
      }
    }
    const uint32_t key = ordered_key(d_of[0]);
    const uint64_t same = __builtin_amdgcn_ballot_w64(tid < nv && key == (uint32_t)__builtin_amdgcn_readlane((int)key, 32));
    if (lane == 0 && __popcll(same) >= 40) tied_lds[0] = 1;
    __syncthreads();  // (cnt, as `copies`, and k1, k2 are free from here on)
  }

  // ---- the ranked rows by (rank, index): the rows are in index order, a pass of the sort is stable
  two_small_pass<true>(key_a, pay_a, key_b, pay_b, n, 0, cnt, part, lanes_a);
  uint32_t* listed_rank = key_b;  // rank and row at every position of the listing
  uint16_t* listed = pay_b;
  if (worst >= 255) {
    two_small_pass<false>(key_b, pay_b, key_a, pay_a, total, 8, cnt, part, lanes_a);
    listed_rank = key_a;
    listed = pay_a;
  }
  uint32_t* const free32 = worst >= 255 ? key_b : key_a;  // the buffers of the sort that hold nothing now
  uint16_t* const free16 = worst >= 255 ? pay_b : pay_a;
  uint64_t* const comps = reinterpret_cast<uint64_t*>(k1);  // (k1 and k2)
  EVX_BATCH_TRACE(6);

  // ---- the order of the last front by (distance descending, index), non_dominate.py:253, into the listing: nobody reads
  // its rows there any more except where they are taken from it first
  const bool tied = by_value && tied_lds[0] != 0;  // (buckets would be crowded)
  if (by_value && (nv <= kTwoSmallCounting || __builtin_expect(tied && nv <= kTwoSmallTied, 0))) {
    uint64_t* tile = comps;  // nv + 4 entries
    int* below = reinterpret_cast<int*>(cnt);
    const bool cand = tid < nv;
    if (tid < nv + 4) tile[tid] = cand ? ((uint64_t)ordered_key(-d_of[0]) << 32) | d_row[0] : ~0ull;
    const int p = position_by_counting(tile, below, nv, tid, kTwoSmallThreads);
    if (cand) dist[d_row[0]] = d_of[0];
    if (cand && p < need) listed[worst_start + p] = (uint16_t)d_row[0];
  } else {
    bool placed = false;
    if (by_value && __builtin_expect(!tied, 1)) {
      uint64_t comp[kTwoSmallPer];
      uint32_t bucket[kTwoSmallPer];
      int place[kTwoSmallPer];
      uint32_t lo = 0xFFFFFFFFu, hi = 0u;  // keys of the finite distances
      const uint32_t key_neg_inf = ordered_key(-INFINITY);
#pragma unroll
      for (int r = 0; r < kTwoSmallPer; ++r) {
        const uint32_t key = ordered_key(-d_of[r]);
        comp[r] = key;
        if (tid + kTwoSmallThreads * r < nv && key != key_neg_inf && key != kNanKey) {
          lo = min(lo, key);
          hi = max(hi, key);
        }
      }
      two_small_range(lo, hi, lo16, hi16, kTwoSmallThreads);
#pragma unroll
      for (int r = 0; r < kTwoSmallPer; ++r) bucket[r] = bucket_by_image((uint32_t)comp[r], lo, hi, kTwoSmallBuckets);
      bool twins;
      placed = two_small_place<kTwoSmallPer>(comp, d_row, bucket, nv, kTwoSmallThreads, cnt, part, comps, lexi, place, twins);
      if (placed) {
#pragma unroll
        for (int r = 0; r < kTwoSmallPer; ++r) {
          if (tid + kTwoSmallThreads * r < nv) {
            dist[d_row[r]] = d_of[r];
            if (place[r] < need) listed[worst_start + place[r]] = (uint16_t)d_row[r];
          }
        }
      }
    }
    if (__builtin_expect(!placed, 0)) {
      // by the radix sort, candidate q = listed[worst_start + q] (in index order): many equal distances, or rows with a NaN.
      // d_by_row shares nothing with the sort's lane masks, which lie in k1 here.
      uint32_t* sk_a = free32;
      uint32_t* sk_b = k2;
      uint16_t* sp_a = free16;
      uint16_t* sp_b = first_at;
      uint32_t* const masks = k1;
      __syncthreads();
      if (by_value) {
#pragma unroll
        for (int r = 0; r < kTwoSmallPer; ++r)
          if (tid + kTwoSmallThreads * r < nv) dist[d_row[r]] = d_of[r];
      } else {
        float acc[kTwoSmallPer];
        bool boundary[kTwoSmallPer];
#pragma unroll
        for (int r = 0; r < kTwoSmallPer; ++r) {
          acc[r] = 0.0f;
          boundary[r] = false;
        }
#pragma unroll 1
        for (int k = 0; k < 2; ++k) {
          sk_a = free32;
          sk_b = k2;
          sp_a = free16;
          sp_b = first_at;
          for (int q = tid; q < nv; q += kTwoSmallThreads) {
            sk_a[q] = ordered_key(fitness_at(listed[worst_start + q], k));
            sp_a[q] = (uint16_t)q;
          }
          __syncthreads();
          two_small_sort(sk_a, sp_a, sk_b, sp_b, nv, 4, cnt, part, masks);
          for (int p = tid; p < nv; p += kTwoSmallThreads) other16[sp_a[p]] = (uint16_t)p;  // position of every candidate
          __syncthreads();
          const float span = cost_of_key(sk_a[nv - 1]) - cost_of_key(sk_a[0]);
#pragma unroll
          for (int r = 0; r < kTwoSmallPer; ++r) {
            const int q = tid + kTwoSmallThreads * r;
            if (q < nv) {
              const int p = other16[q];
              if (p == 0 || p == nv - 1) {
                boundary[r] = true;
              } else {
                const float term = (cost_of_key(sk_a[p + 1]) - cost_of_key(sk_a[p - 1])) / span;
                acc[r] = k == 0 ? term : acc[r] + term;
              }
            }
          }
          __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < kTwoSmallPer; ++r) {
          const int q = tid + kTwoSmallThreads * r;
          if (q < nv) dist[listed[worst_start + q]] = boundary[r] ? INFINITY : acc[r];
        }
      }
      __syncthreads();
      sk_a = free32;
      sk_b = k2;
      sp_a = free16;
      sp_b = first_at;
      for (int q = tid; q < nv; q += kTwoSmallThreads) {
        const int row = listed[worst_start + q];
        sk_a[q] = ordered_key(-dist[row]);
        sp_a[q] = (uint16_t)row;
      }
      __syncthreads();
      two_small_sort(sk_a, sp_a, sk_b, sp_b, nv, 4, cnt, part, masks);
      for (int p = tid; p < need; p += kTwoSmallThreads) listed[worst_start + p] = sp_a[p];
    }
  }
  __syncthreads();
  EVX_BATCH_TRACE(7);

  // ---- the selected rows
  const int topk = stop;
  const int64_t ob = (int64_t)blockIdx.x * topk;
  for (int p = tid; p < topk; p += kTwoSmallThreads) {
    const int src = listed[p];
    const float f1 = fitness_at(src, 0), f2 = fitness_at(src, 1);
    a.out_rank[ob + p] = p < worst_start ? (int)listed_rank[p] : worst;
    a.out_dist[ob + p] = p < worst_start ? -INFINITY : dist[src];
    a.out_f[(ob + p) * 2] = f1;
    a.out_f[(ob + p) * 2 + 1] = f2;
  }
  EVX_BATCH_TRACE(8);
  if (a.x != nullptr) {
    const uint8_t* __restrict__ xb = a.x + (int64_t)blockIdx.x * a.x_stride_b;
    uint8_t* __restrict__ dst = a.out_x + ob * a.x_row_bytes;
    if (!gather_whole_units(a, xb, dst, listed, topk, tid, kTwoSmallThreads)) {
      for (int p = wave; p < topk; p += kTwoSmallThreads / 64) {
        const int src = listed[p];
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
  EVX_BATCH_TRACE(9);
}

}  // namespace evx
