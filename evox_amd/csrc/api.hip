// C ABI of libevox_hip.so (declared in include/evox_hip.h): argument checks, workspace layout
// and kernel launches.  Nothing here allocates device memory or waits for the device, except
// evox_hip_read_status(); the selection entry points keep 320 bytes of pinned host memory per device (outcome_slot).
#include <string.h>

#include <atomic>
#include <mutex>
#include <new>
#include <type_traits>

#include "../../include/evox_hip.h"
#include "batched.hpp"
#include "calibrate.hpp"
#include "common.hpp"
#include "crowd.hpp"
#include "dominance.hpp"
#include "finish.hpp"
#include "hv.hpp"
#include "launch_words.hpp"
#include "order.hpp"
#include "peel.hpp"
#include "peel_lds.hpp"
#include "prefix.hpp"
#include "radix.hpp"
#include "records.hpp"
#include "runs.hpp"
#include "slots.hpp"
#include "spatial.hpp"
#include "stepped.hpp"
#include "two.hpp"
#include "two_small.hpp"
#include "few.hpp"
#include "sets.hpp"
#include "wide.hpp"

namespace evx {

constexpr int kMaxGrid = 4096;  // slots of the grid barrier

struct Options {
  int peel_blocks_per_cu = 2;
  int peel_witness = 1;
  int peel_record_blocks = 0;  // sweeping blocks of the record protocol, 16 .. 255 (plus the lister); 0 = by size
  int peel_records = 1;  // record protocol (all-to-all, no master) for populations up to kRecordsMaxRowsWide
  int peel_lds = 1;      // populations whose lower triangle fits the LDS of the device are peeled from LDS (peel_lds.hpp)
  int peel_lds_blocks = 0;  // sweeping workgroups of that kernel, 0 = by size
  int peel_stepped = 0;     // 1: the fronts are peeled one launch each by kernels that never wait for each other (stepped.hpp),
                            // and the last front is ordered likewise; 0: only where the persistent grids cannot be resident
  int64_t two_small_min_rows = 128;  // populations of two objectives and at least this many rows (at most 4096) that go to a
                                   // one-workgroup kernel take the one without a matrix (two_small.hpp); 0 = never
  int64_t few_max_rows = kFewRows;  // populations of three to eight objectives and at most this many rows that reach the entry points
                                    // with a workspace: matrix by the whole device, the rest by one workgroup (few.hpp); 0 = never
  int64_t sets_min_rows = 257;  // populations of three to eight objectives and at least this many rows that go to a one-workgroup
                                // kernel take the one that compares no pairs (sets.hpp); more than kSetsRows = never
  int64_t two_min_rows = 4097;  // populations of two objectives and at least this many rows are ranked without a matrix (two.hpp); 0 = never
  int64_t two_min_rows_partial = 4097;  // ... when the ranking may stop at the front that holds a given row (measured, us per
                                        // selection of half the rows, without / with a matrix: 5000 rows 110 / 178, 20 000 rows
                                        // 218 / 362, 50 000 rows 324 / 1181; all ranks: 5000 rows 140 / 332)
  int peel_tail = 1;        // that kernel also orders a small last front (0: always the kernels of finish.hpp)
  int tail_merged = 1;      // after such a peel, ordering (where still needed) and gather share one launch
  int launch_memory = 1;    // ... unless the last selection of this shape had a last front that the peel left alone
  unsigned spin_limit = 4000000u;
  int dominance_tile_words = 0;  // 0 = by size (2 or 4)
  int dominance_folded = 1;      // tiles of two words: only the blocks at or below the diagonal are launched
  int mid_argsort = 1;  // an argsort step of 8193 .. kMidArgsortRows positions in one kernel without waits (0: the radix sort)
  int small_sort = 1;  // populations up to kSmallSortRows rows are put in slot order by one kernel (0: bucket sort)
  int64_t prefix_min_rows = 65536;  // finite populations of at least 20/32 of this many rows and 3 objectives (40/32
                                    // with 2, fewer with more: 32769 at 4, 28672 at 8, 10240 at 16 -- prefix_least_rows) get
                                    // their matrix from the per-objective orders (prefix.hpp); 0 = never
  int64_t prefix_double_tile = 131072;  // order-based matrix, up to four objectives: from this many rows on a workgroup
                                        // takes both tiles of a 128-byte line; 0 = never
  int prefix_mode = 3;  // measurements: 1 = popcounts only, 2 = matrix only
  int prefix_bands = 1;  // stretches of the order-based matrix: 1 = bands of rows counted from row 0, 0 = from each tile's diagonal
  int batched_stage = 1;  // the one-workgroup kernel reads its dominators from a copy of the fitness in LDS when the populations
                          // have at most 256 rows and are no more than the device has compute units (0: by scalar loads always)
  int order_stream = 1;  // the per-objective orders of more than 32768 rows come from workgroups that place shares of
                         // them in LDS (0: from the radix sort whose workgroups wait for each other)
  int order_stream_capacity = 16384;  // entries that such a workgroup sorts at once (tests make it small: shares in pieces)
  int prefix_count_first = 1;  // a selection whose last two of this shape found all they keep in front 0 has the order-based
                               // kernel count dominators first and build the matrix only if front 0 falls short; 0 = never, 2 = always
  int64_t prefix_nearby = 1;  // those counts in spatial order: 1 = by size (nearby_totals_apply), 0 = never, else from this many rows on
};
static Options g_opt;
// The tunables that calls made from this thread use: those handed to evox_hip_options_use, else the process-wide ones.
static thread_local const Options* t_opt = nullptr;
static inline const Options& opt() { return t_opt != nullptr ? *t_opt : g_opt; }


struct Layout {
  int n, m, npad, nwords, kstride, buckets, prep_blocks;
  int64_t wstride;
  // byte offsets
  size_t ctrl, fsize, fronts_slot, fronts_orig, hist, zero_end, fstart, xs, key, partials, sortparam, bstart, bcursor,
      scanflags, tailbuf, records, two_ring, members, member_key, slot_of, xs_sorted, key_sorted, kid_sorted, orig_of, count, witness, total0, witness0, leaf_lo, leaf_hi, group_lo, rank, dist, perm, order, rpairs0, rpairs1, rtable, rtotals, pos, scost, dkey, wide, wide_bytes, dom, total;
};

static size_t align_up(size_t v) { return (v + 255) / 256 * 256; }
static size_t wide_workspace_need(int64_t n, int64_t m);  // (workspace of the kernels of wide.hpp, defined with them)
constexpr int kErrNotResident = -100;  // internal: the grid of a persistent kernel would not be resident at once

static bool make_layout(int64_t n, int64_t m, Layout* L) {
  if (n < 1 || m < 1 || n > 0x7FFFFF00ll || m > 65535) return false;
  L->n = (int)n;
  L->m = (int)m;
  L->npad = (int)round_up(n, 128);
  // the objectives are columns npad floats apart: at a multiple of 16 KB the same row of six or more columns
  // competes for one set of the scalar cache (pairwise matrix of 65536 rows x 8: 1.19 ms, of 49152 rows: 0.42 ms)
  if (L->npad % 4096 == 0 && n >= 16384) L->npad += 128;
  L->nwords = L->npad / 64;
  L->wstride = round_up(L->nwords, 16);
  L->kstride = (int)round_up(n, 64);
  // buckets of the slot sort: a power of two near 4 n, between 1024 and 65536
  int buckets = 1024;
  while (buckets < 65536 && buckets < 4 * n) buckets <<= 1;
  L->buckets = buckets;
  L->prep_blocks = (int)((L->npad + 255) / 256 < 1024 ? (L->npad + 255) / 256 : 1024);
  size_t o = 0;
  // --- cleared on every call: control block, front sizes, front bitmaps, sort histogram
  L->ctrl = o;        o = align_up(o + sizeof(Ctrl) + sizeof(unsigned long long) * kMaxGrid);
  L->fsize = o;       o = align_up(o + sizeof(int) * (size_t)(n + 2));
  L->fronts_slot = o; o = align_up(o + sizeof(uint64_t) * kFrontBuffers * kFrontStride * (size_t)L->nwords);
  L->fronts_orig = o; o = align_up(o + sizeof(uint64_t) * kFrontBuffers * kFrontStride * (size_t)L->nwords);
  L->hist = o;        o = align_up(o + sizeof(int) * (size_t)buckets);
  L->scanflags = o;   o = align_up(o + sizeof(unsigned long long) * 64);
  L->tailbuf = o;     o = align_up(o + (n <= 32768 ? sizeof(unsigned long long) * kTailCopies * kTailRows : 0));
  L->records = o;     o = align_up(o + (n <= 32768 ? sizeof(unsigned long long) * kLdsPeelRecordUnits : (n <= kRecordsMaxRowsWide ? sizeof(unsigned long long) * kRecRing * (n > kRecordsMaxRows ? kRecUnitsWide : kRecUnits) : 0)));
  // the hand-over rings of the two-objective ranking (two.hpp)
  L->two_ring = o;    o = align_up(o + (m == 2 && n <= kTwoMaxRows ? sizeof(unsigned long long) * kTwoRingStride * (size_t)((n + kTwoChunk - 1) / kTwoChunk) : 0));
  L->zero_end = o;
  L->fstart = o;     o = align_up(o + sizeof(int) * (size_t)(n + 2));
  L->xs = o;         o = align_up(o + sizeof(float) * (size_t)m * L->npad);
  L->key = o;        o = align_up(o + sizeof(uint64_t) * (size_t)L->npad);
  L->partials = o;   o = align_up(o + sizeof(unsigned long long) * 3 * (size_t)L->prep_blocks);
  L->sortparam = o;  o = align_up(o + sizeof(SortParam));
  L->bstart = o;     o = align_up(o + sizeof(int) * (size_t)(buckets + 1));
  L->bcursor = o;    o = align_up(o + sizeof(int) * (size_t)buckets);
  L->members = o;    o = align_up(o + sizeof(int) * (size_t)n);
  L->member_key = o; o = align_up(o + sizeof(uint64_t) * (size_t)n);
  L->xs_sorted = o;  o = align_up(o + sizeof(float) * (size_t)m * L->npad);
  L->key_sorted = o; o = align_up(o + sizeof(uint64_t) * (size_t)L->npad);
  L->kid_sorted = o; o = align_up(o + sizeof(uint32_t) * (size_t)L->npad);
  L->orig_of = o;    o = align_up(o + sizeof(int) * (size_t)L->npad);
  L->slot_of = o;    o = align_up(o + sizeof(int) * (size_t)n);
  L->count = o;      o = align_up(o + sizeof(int) * (size_t)n);
  L->witness = o;    o = align_up(o + sizeof(int) * (size_t)n);
  // popcount and highest non-empty word of every row as the order-based dominance kernel leaves them (kept apart
  // from count / witness, which the peel consumes, so that the count stage can be repeated)
  L->total0 = o;     o = align_up(o + sizeof(int) * (size_t)n);
  L->witness0 = o;   o = align_up(o + sizeof(int) * (size_t)n);
  // boxes of the rows in spatial order (spatial.hpp)
  const size_t box = m <= kSpatialObjectives ? sizeof(float) * (size_t)m : 0;
  L->leaf_lo = o;    o = align_up(o + box * (size_t)spatial_leaf_stride(n));
  L->leaf_hi = o;    o = align_up(o + box * (size_t)spatial_leaf_stride(n));
  L->group_lo = o;   o = align_up(o + box * (size_t)spatial_group_stride(n));
  L->rank = o;       o = align_up(o + sizeof(int) * (size_t)n);
  L->dist = o;       o = align_up(o + sizeof(float) * (size_t)n);
  L->perm = o;       o = align_up(o + sizeof(int) * (size_t)n);
  L->order = o;      o = align_up(o + sizeof(int) * (size_t)n);
  // radix sort of large fronts: only populations that can have one get the buffers
  const size_t rseg = n > kRadixMinCandidates ? (size_t)m * L->kstride : 0;
  L->rpairs0 = o;    o = align_up(o + sizeof(unsigned long long) * rseg);
  L->rpairs1 = o;    o = align_up(o + sizeof(unsigned long long) * rseg);
  L->rtable = o;     o = align_up(o + (rseg ? sizeof(int) * (size_t)m * 256 * kRadixMaxWorkers : 0));
  L->rtotals = o;    o = align_up(o + (rseg ? sizeof(int) * (size_t)m * 256 : 0));
  L->pos = o;        o = align_up(o + sizeof(int) * (size_t)m * L->kstride);
  L->scost = o;      o = align_up(o + sizeof(float) * (size_t)m * L->kstride);
  L->dkey = o;       o = align_up(o + sizeof(uint32_t) * (size_t)L->kstride);
  L->dom = o;        o = align_up(o + sizeof(uint64_t) * (size_t)n * (size_t)L->wstride);
  // behind the matrix (the entry points that build none need only the bytes before it): the ordering of the last
  // front by kernels that never wait for each other (the tail of the stepped path)
  L->wide_bytes = wide_workspace_need(n, m);
  L->wide = o;       o = align_up(o + L->wide_bytes);
  L->total = o;
  return true;
}

struct Ws {
  Layout L;
  uint8_t* base;
  // several populations of one shape in the same launches (blockIdx.z): `step` bytes from the workspace of one to that
  // of the next, all laid out alike; 1 and 0 for a single population
  int batch = 1;
  int64_t step = 0;
  // above zero: the order-based dominance kernel has only counted so far; the count stage launches it again for the
  // matrix, and that launch does nothing when front 0 holds this many rows
  mutable int64_t matrix_unless = 0;
  template <class T>
  T* at(size_t off) const {
    return reinterpret_cast<T*>(base + off);
  }
  Ctrl* ctrl() const { return at<Ctrl>(L.ctrl); }
};

// The bit matrix and what lies behind it are the last regions: entry points that never build it need only the bytes before it.
static int open_ws(int64_t n, int64_t m, void* ws, size_t bytes, Ws* out, bool with_matrix = true) {
  if (!make_layout(n, m, &out->L)) return kErrBadArg;
  const size_t need = with_matrix ? out->L.total : out->L.dom;
  if (ws == nullptr || bytes < need || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  out->base = static_cast<uint8_t*>(ws);
  return 0;
}

// (The small host-side caches below are read and written by whichever threads call into the library: each slot is
// an atomic that holds a value derived from the device alone, so two threads that fill it at once store the same.)
static int device_cus() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = cached[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cached[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// What the last selections on this device found, for the choice of launches of the next one: some words of pinned host
// memory per device (launch_words.hpp), which the last kernel of a selection writes and the host reads at its next call of
// that shape without waiting for anything -- a stale or missing word costs a few microseconds, never a result.  Allocated
// at the first selection on a device that may allocate (not during a stream capture); null until then and for callers
// that may not.
static int* outcome_slot(LaunchWord meaning, int64_t n, int64_t m, bool may_allocate, hipStream_t s) {
  constexpr size_t bytes = sizeof(int) * kWordsPerMeaning * kLaunchWords;
  static std::atomic<int*> words[64];
  static std::atomic<bool> failed[64];
  static std::mutex mu;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  int* base = words[dev].load(std::memory_order_acquire);
  if (base == nullptr) {
    if (!may_allocate || failed[dev].load(std::memory_order_relaxed)) return nullptr;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
      (void)hipGetLastError();
      return nullptr;
    }
    std::lock_guard<std::mutex> lock(mu);
    base = words[dev].load(std::memory_order_acquire);
    if (base == nullptr) {
      void* p = nullptr;
      if (hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess || p == nullptr) {
        (void)hipGetLastError();
        failed[dev].store(true, std::memory_order_relaxed);
        return nullptr;
      }
      memset(p, 0, bytes);
      base = static_cast<int*>(p);
      words[dev].store(base, std::memory_order_release);
    }
  }
  return base + launch_word(meaning, n, m);
}

#define EVX_LAUNCH_CHECK()                          \
  do {                                              \
    hipError_t e_ = hipGetLastError();              \
    if (e_ != hipSuccess) return (int)e_;           \
  } while (0)

// ------------------------------------------------------------------ stages

template <int M, int IW>
static void launch_dominance_m(const Ws& w, int variant, hipStream_t s) {
  const Layout& L = w.L;
  dim3 grid((L.npad + 255) / 256, (L.nwords + IW - 1) / IW, w.batch);
  if (IW == 2) grid = dim3((L.npad + 127) / 128, (L.nwords + 3) / 4, w.batch);  // a block = two row groups x two tiles
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, w.at<float>(L.xs_sorted), w.at<uint64_t>(L.key_sorted),
                       w.at<uint32_t>(L.kid_sorted), w.at<uint64_t>(L.dom), L.n, L.npad, L.wstride, L.nwords,
                       w.at<SortParam>(L.sortparam), w.step);
  };
  if ((IW == 2 || IW == 4) && variant == kDomAuto && opt().dominance_folded) {
    const int row_blocks = IW == 2 ? (L.npad + 127) / 128 : (L.npad + 255) / 256;
    const int column = IW == 2 ? (row_blocks - 1) / 2 + 2 : row_blocks + 1;
    auto folded = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((row_blocks + 1) / 2, column, w.batch), dim3(256), 0, s, w.at<float>(L.xs_sorted),
                         w.at<uint64_t>(L.key_sorted), w.at<uint32_t>(L.kid_sorted), w.at<uint64_t>(L.dom), L.n, L.npad, L.wstride,
                         L.nwords, w.at<SortParam>(L.sortparam), row_blocks, w.step);
    };
    if (w.batch > 1)
      folded(dominance_folded_kernel<M, (IW == 2 ? 2 : 4), true>);
    else
      folded(dominance_folded_kernel<M, (IW == 2 ? 2 : 4), false>);
    return;
  }
  switch (variant) {
    case kDomTwoCompares: launch(dominance_kernel<M, IW, kDomTwoCompares>); break;
    case kDomKey64: launch(dominance_kernel<M, IW, kDomKey64>); break;
    case kDomKey32: launch(dominance_kernel<M, IW, kDomKey32>); break;
    default: launch(dominance_kernel<M, IW, kDomAuto>); break;
  }
}

template <int IW>
static void launch_dominance(const Ws& w, int variant, hipStream_t s) {
  const Layout& L = w.L;
  switch (L.m) {
    case 1: launch_dominance_m<1, IW>(w, variant, s); break;
    case 2: launch_dominance_m<2, IW>(w, variant, s); break;
    case 3: launch_dominance_m<3, IW>(w, variant, s); break;
    case 4: launch_dominance_m<4, IW>(w, variant, s); break;
    case 5: launch_dominance_m<5, IW>(w, variant, s); break;
    case 6: launch_dominance_m<6, IW>(w, variant, s); break;
    case 7: launch_dominance_m<7, IW>(w, variant, s); break;
    case 8: launch_dominance_m<8, IW>(w, variant, s); break;
    default: {
      // nine to sixteen objectives: the register kernel in its production form (tiles of four words, form chosen
      // on the device); the other tile sizes and the check variants, and more objectives, take the generic kernel
      if (IW == 4 && variant == kDomAuto && L.m <= 16) {
        auto wide = [&](auto kernel) {
          hipLaunchKernelGGL(kernel, dim3((L.npad + 255) / 256, (L.nwords + 3) / 4, w.batch), dim3(256), 0, s, w.at<float>(L.xs_sorted),
                             w.at<uint64_t>(L.key_sorted), w.at<uint32_t>(L.kid_sorted), w.at<uint64_t>(L.dom), L.n, L.npad,
                             L.wstride, L.nwords, w.at<SortParam>(L.sortparam), w.step);
        };
        switch (L.m) {
          case 9: wide(dominance_kernel<9, 4, kDomAuto>); return;
          case 10: wide(dominance_kernel<10, 4, kDomAuto>); return;
          case 11: wide(dominance_kernel<11, 4, kDomAuto>); return;
          case 12: wide(dominance_kernel<12, 4, kDomAuto>); return;
          case 13: wide(dominance_kernel<13, 4, kDomAuto>); return;
          case 14: wide(dominance_kernel<14, 4, kDomAuto>); return;
          case 15: wide(dominance_kernel<15, 4, kDomAuto>); return;
          default: wide(dominance_kernel<16, 4, kDomAuto>); return;
        }
      }
      dim3 grid((L.npad + 255) / 256, (L.nwords + IW - 1) / IW, w.batch);
      hipLaunchKernelGGL((dominance_any_m_kernel<IW>), grid, dim3(256), 0, s, w.at<float>(L.xs_sorted),
                         w.at<uint32_t>(L.kid_sorted), w.at<uint64_t>(L.dom), L.n, L.npad, L.wstride, L.nwords, L.m, w.step);
    }
  }
}

// Fitness -> structure of arrays + keys, state reset, then the slot sort (order.hpp).
// A population given in one part (n_first == n, second part unused) or in two.
struct Fitness {
  const float* f;
  int64_t sr, sc;
  int64_t n_first;
  const float* f2;
  int64_t sr2, sc2;
  int64_t step = 0, step2 = 0;  // several populations: elements from one population's fitness to the next one's
};

static Fitness one_part(const float* f, int64_t n, int64_t sr, int64_t sc, int64_t step = 0) {
  return Fitness{f, sr, sc, n, f, sr, sc, step, step};
}

static int grant_dynamic_lds(const void* kernel, size_t lds);

// Workgroups of one population that place its rows or candidates by searching the runs: one per compute unit, fewer where
// several populations share the launch (none waits for another: at least sixteen).
static int run_share_grid(const Ws& w) {
  const int share = device_cus() / w.batch;
  return share < 16 ? 16 : share;
}

// Up to this many rows the slot order comes from sorted runs: its searches grow with the square of the rows, the bucket sort's
// five launches hardly.  Whole calls, us, buckets / runs: rank 4097 x 3 109 / 99, 5000 x 9 85 / 74, 10 007 x 5 85.5 / 77.9, 20 000 x 3
// 213 / 209, 32 768 x 3 422 / 421, 40 000 x 3 540 / 542, 60 000 x 3 473 / 488; where keys crowd, 20 001 x 3 one front 112 / 104,
// 16 populations of 4000 x 8 in a launch 311 / 169.
constexpr int kSlotRunsRows = kRunMaxRows;

static int stage_prepare(const Ws& w, const Fitness& src, bool with_sort, hipStream_t s, bool lexicographic = false) {
  const Layout& L = w.L;
  if (src.f == nullptr || src.f2 == nullptr || src.n_first < 0 || src.n_first > L.n) return kErrBadArg;
  const int64_t zero_words = (int64_t)((L.zero_end - L.ctrl) / 4);
  // (every workgroup of small_sort_kernel reads its whole population to place sixteen rows: with several populations
  // in the launch, more workgroups than the device holds at once take turns -- 16 x 4096 rows: 102 us against 10 for
  // one population, the five launches of the bucket sort 30)
  const bool many = w.batch > 1;
  const bool small_sort_pays = w.batch == 1 || (int64_t)w.batch * (L.npad / kSmallSortGroup) <= 2 * device_cus();
  if (with_sort && !lexicographic && L.n <= kSmallSortRows && L.m <= kSmallSortObjectives && (int64_t)L.n * L.m <= kSmallSortValues &&
      opt().small_sort && small_sort_pays) {
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(L.npad / kSmallSortGroup, 1, w.batch), dim3(kSmallSortThreads), sizeof(double) * (size_t)L.npad, s, src.f,
                         src.sr, src.sc, (int)src.n_first, src.f2, src.sr2, src.sc2, L.n, L.m, L.npad, w.at<float>(L.xs),
                         w.at<SortParam>(L.sortparam), w.at<uint64_t>(L.key_sorted), w.at<uint32_t>(L.kid_sorted),
                         w.at<float>(L.xs_sorted), w.at<int>(L.orig_of), w.at<uint32_t>(L.ctrl), zero_words, src.step, src.step2, w.step);
    };
    if (many)
      launch(small_sort_kernel<true>);
    else
      launch(small_sort_kernel<false>);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  if (with_sort && L.n <= kSlotRunsRows) {
    const int runs = (L.npad + kRunRows - 1) / kRunRows;
    // (about as many workgroups as there are compute units share the clearing)
    const int grid = runs > device_cus() / w.batch ? runs : device_cus() / w.batch;
    const size_t lds = run_rank8_lds_bytes(L.n);
    int share = (int)round_up((L.n + run_share_grid(w) - 1) / run_share_grid(w), 16);  // (whole waves of sixteen keys)
    if (share > kRunRankThreads / kRunLanes) share = kRunRankThreads / kRunLanes;
    auto launch = [&](auto runs_kernel, auto places_kernel, auto* key_type) -> int {
      using Key = std::remove_pointer_t<decltype(key_type)>;
      hipLaunchKernelGGL(runs_kernel, dim3(grid, 1, w.batch), dim3(kRunRows), 0, s, src.f, src.sr, src.sc, (int)src.n_first, src.f2, src.sr2,
                         src.sc2, L.n, L.m, L.npad, w.at<float>(L.xs), w.at<Key>(L.key), w.at<int>(L.members),
                         w.at<unsigned long long>(L.partials), w.at<uint32_t>(L.ctrl), zero_words, runs, src.step, src.step2, w.step);
      EVX_LAUNCH_CHECK();
      if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(places_kernel), lds)) return e;
      hipLaunchKernelGGL(places_kernel, dim3((L.n + share - 1) / share, 1, w.batch), dim3(kRunRankThreads), lds, s, w.at<Key>(L.key),
                         w.at<int>(L.members), w.at<unsigned long long>(L.partials), L.n, L.m, L.npad, share, w.at<float>(L.xs),
                         w.at<uint64_t>(L.key_sorted), w.at<uint32_t>(L.kid_sorted), w.at<float>(L.xs_sorted), w.at<int>(L.orig_of),
                         w.at<int>(L.slot_of), w.at<SortParam>(L.sortparam), w.step);
      EVX_LAUNCH_CHECK();
      return 0;
    };
    if (lexicographic)
      return many ? launch(slot_runs_kernel<true, true>, slot_places_kernel<true, true>, (uint64_t*)nullptr)
                  : launch(slot_runs_kernel<false, true>, slot_places_kernel<false, true>, (uint64_t*)nullptr);
    return many ? launch(slot_runs_kernel<true, false>, slot_places_kernel<true, false>, (double*)nullptr)
                : launch(slot_runs_kernel<false, false>, slot_places_kernel<false, false>, (double*)nullptr);
  }
  auto launch_prepare = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(L.prep_blocks, 1, w.batch), dim3(256), 0, s, src.f, src.sr, src.sc, (int)src.n_first, src.f2,
                       src.sr2, src.sc2, L.n, L.m, L.npad, w.at<float>(L.xs), w.at<uint64_t>(L.key),
                       w.at<unsigned long long>(L.partials), w.at<uint32_t>(L.ctrl), zero_words, lexicographic ? 1 : 0, src.step,
                       src.step2, w.step);
  };
  if (many)
    launch_prepare(prepare_kernel<true>);
  else
    launch_prepare(prepare_kernel<false>);
  EVX_LAUNCH_CHECK();
  if (!with_sort) return 0;
  int blocks = (L.n + 255) / 256;
  if (blocks > 2048) blocks = 2048;
  auto launch_hist = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks, 1, w.batch), dim3(256), 0, s, w.at<uint64_t>(L.key), L.n,
                       w.at<unsigned long long>(L.partials), L.prep_blocks, L.buckets, w.at<int>(L.hist),
                       w.at<SortParam>(L.sortparam), w.step);
  };
  if (many)
    launch_hist(bucket_hist_kernel<true>);
  else
    launch_hist(bucket_hist_kernel<false>);
  EVX_LAUNCH_CHECK();
  auto launch_scan = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(L.buckets / 1024, 1, w.batch), dim3(256), 0, s, w.at<int>(L.hist), L.buckets,
                       w.at<int>(L.bstart), w.at<int>(L.bcursor), w.at<unsigned long long>(L.scanflags), w.ctrl(), w.step);
  };
  if (many)
    launch_scan(bucket_scan_kernel<true>);
  else
    launch_scan(bucket_scan_kernel<false>);
  EVX_LAUNCH_CHECK();
  auto launch_scatter = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks, 1, w.batch), dim3(256), 0, s, w.at<uint64_t>(L.key), L.n,
                       w.at<SortParam>(L.sortparam), w.at<int>(L.bcursor), w.at<int>(L.members), w.at<uint64_t>(L.member_key),
                       w.ctrl(), w.step);
  };
  if (many)
    launch_scatter(bucket_scatter_kernel<true>);
  else
    launch_scatter(bucket_scatter_kernel<false>);
  EVX_LAUNCH_CHECK();
  int pblocks = (L.npad + 255) / 256;
  if (pblocks > 2048) pblocks = 2048;
  auto launch_place = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(pblocks, 1, w.batch), dim3(256), 0, s, w.at<float>(L.xs), L.n, L.m,
                       L.npad, w.at<SortParam>(L.sortparam), w.at<int>(L.bstart), w.at<int>(L.members), w.at<uint64_t>(L.member_key),
                       w.at<uint64_t>(L.key_sorted), w.at<uint32_t>(L.kid_sorted), w.at<float>(L.xs_sorted), w.at<int>(L.orig_of), w.at<int>(L.slot_of),
                       w.ctrl(), w.step);
  };
  if (many)
    launch_place(bucket_place_kernel<true>);
  else
    launch_place(bucket_place_kernel<false>);
  EVX_LAUNCH_CHECK();
  return 0;
}

// From how many rows on the matrix comes from the per-objective orders: the pairwise kernel's work grows with the
// objectives (two compares each per pair), the other's hardly does, and it starts from some 160 us for the orders
// themselves.  Measured, a whole selection of uniform fitness in us, pairwise / from the orders:
//   x 3: 60 000 521 / 530;  x 4: 40 000 300 / 337, 50 000 406 / 376;  x 5: 40 000 295 / 335, 50 000 395 / 350;
//   x 6: 40 000 325 / 343, 50 000 439 / 352;  x 7: 33 000 302 / 315, 40 000 377 / 351;  x 8: 26 000 254 / 312,
//   33 000 335 / 325, 50 000 584 / 386;  x 9: 20 000 251 / 305, 26 000 342 / 323;  x 10: 20 000 269 / 315, 26 000 363 / 329;
//   x 12: 16 000 261 / 308, 20 000 312 / 307;  x 14: 16 000 301 / 327, 20 000 363 / 327;  x 16: 12 000 253 / 330,
//   16 000 342 / 344, 20 000 424 / 352;  x 2 (65 536 rows): 227 / 239, (100 000) 558 / 370.
// With the orders from shares that are placed by buckets (prefix.hpp, above kMidArgsortRows rows; they also order the last front):
//   x 3: 33 000 264 / 287 (one front: 284 / 214), 41 000 309 / 309 (shell 242 / 223), 52 000 385 / 344;  x 4: 33 000 215 / 212 (shell 205 / 177);
//   x 5: 33 000 218 / 205 (one front 324 / 223), 42 000 283 / 230;  x 6: 33 000 228 / 197;  x 7: 33 000 260 / 200 (one front 377 / 245).
// (Few levels share the loss and the gain: 41 000 x 3 of four 271 / 277, of eight 290 / 297;  33 000 x 4 of four 266 / 258.)
// As thirty-seconds of the tunable (20 of them are 40 960 rows; four to seven objectives begin where those orders do):
// Up to kMidArgsortRows rows the orders come from workgroups that sort in LDS and cost 60 to 90 us less:
//   x 8: 26 000 254 / 261, 32 768 322 / 295;  x 9: 16 000 212 / 224, 20 000 252 / 236;  x 10: 16 000 222 / 231,
//   20 000 268 / 245;  x 12: 12 000 198 / 210, 16 000 257 / 225;  x 16: 9000 220 / 215, 12 000 259 / 237.
static int64_t prefix_least_rows(int m) {
  int parts = m <= 2 ? 40 : m == 3 ? 20 : m <= 8 ? 16 : m <= 10 ? 12 : m <= 12 ? 10 : m <= 14 ? 9 : 8;
  if (opt().mid_argsort && m >= 8) parts = m == 8 ? 14 : m <= 10 ? 9 : m <= 12 ? 7 : m <= 14 ? 6 : 5;
  return opt().prefix_min_rows / 32 * parts + (opt().prefix_min_rows % 32 != 0 || (m >= 4 && m <= 7) ? 1 : 0);
}
static bool prefix_dominance_applies(const Layout& L) {
  if (opt().prefix_min_rows <= 0 || L.m < 2 || L.m > kPrefixMaxObjectives) return false;
  return L.n >= prefix_least_rows(L.m) && L.n > kRadixMinCandidates && L.n <= kPrefixMaxRows;
}
static int stage_dominance_prefix(const Ws& w, bool orders_only, hipStream_t s, int64_t count_first = 0);
static int dispatch_dominance_prefix(const Ws& w, hipStream_t s, int phase = 0);

static int dominance_tile_words(const Layout& L) {
  const int tile = opt().dominance_tile_words;
  if (tile != 0) return tile;
  return L.m >= 2 && L.m <= 8 && L.n <= (L.m >= 6 ? 32768 : 24576) ? 2 : 4;
}

// count_first: above zero, the caller keeps that many rows and expects front 0 to hold them (see Ws::matrix_unless).
static int stage_dominance(const Ws& w, int variant, hipStream_t s, int64_t count_first = 0) {
  // (kDomOrdersOnly: the first half of the path below alone, for measurements of the second)
  if (variant == kDomOrdersOnly) return prefix_dominance_applies(w.L) ? stage_dominance_prefix(w, true, s) : kErrBadArg;
  // (the orders of that path come from kernels whose workgroups wait for each other: not with the stepped path)
  // (nor for several populations in one launch: those orders come from a grid that fills the device)
  if (variant == kDomAuto && prefix_dominance_applies(w.L) && !opt().peel_stepped && w.batch == 1) return stage_dominance_prefix(w, false, s, count_first);
  // (the lower triangle in tiles of 4 words keeps every SIMD busy with several waves; up to about 24 000 rows of
  // two to eight objectives tiles of 2 words leave a shorter half-empty tail -- measured, us, tiles of 2 / 4:
  // 5000 x 3: 5.8 / 7.9, 16 000 x 3: 20.3 / 25.7, 20 000 x 2: 20.6 / 23.1, x 3: 27.6 / 31.3, x 8: 64.3 / 80.8,
  // 24 000 x 3: 38.8 / 39.8, 28 000 x 3: 49.1 / 48.1, x 8: 110.8 / 132.1, 50 000 x 3: 147.5 / 138.4 --; 8 and 16
  // are kept for measurements)
  const int tile = dominance_tile_words(w.L);
  if (tile >= 16)
    launch_dominance<16>(w, variant, s);
  else if (tile >= 8)
    launch_dominance<8>(w, variant, s);
  else if (tile >= 4)
    launch_dominance<4>(w, variant, s);
  else
    launch_dominance<2>(w, variant, s);
  EVX_LAUNCH_CHECK();
  return 0;
}

static int stage_count(const Ws& w, bool fill_dist, hipStream_t s, bool need_counts) {
  const Layout& L = w.L;
  int blocks = (L.n + 3) / 4;
  const int cap = device_cus() * 8;
  if (blocks > cap) blocks = cap;
  hipLaunchKernelGGL(count_kernel, dim3(blocks), dim3(256), 0, s, w.at<uint64_t>(L.dom), L.wstride, L.n,
                     w.at<int>(L.orig_of), w.at<int>(L.count), w.at<int>(L.rank), w.at<int>(L.witness),
                     w.at<uint64_t>(L.fronts_slot), w.at<uint64_t>(L.fronts_orig), w.at<int>(L.fsize),
                     fill_dist ? w.at<float>(L.dist) : (float*)nullptr, w.ctrl(), w.at<SortParam>(L.sortparam), need_counts ? 1 : 0);
  EVX_LAUNCH_CHECK();
  if (prefix_dominance_applies(L)) {
    // the order-based dominance kernel has left the popcounts: count_kernel above returned at once (the choice is
    // made on the device: a population with a NaN or an infinity went through the pairwise kernel and is counted there)
    hipLaunchKernelGGL(count_from_totals_kernel, dim3((L.n + 255) / 256 < 128 ? (L.n + 255) / 256 : 128), dim3(256), 0, s, w.at<int>(L.total0),
                       w.at<int>(L.witness0), L.n, w.at<int>(L.slot_of), w.at<int>(L.count), w.at<int>(L.rank),
                       w.at<int>(L.witness), w.at<uint64_t>(L.fronts_slot), w.at<uint64_t>(L.fronts_orig), w.at<int>(L.fsize),
                       fill_dist ? w.at<float>(L.dist) : (float*)nullptr, w.ctrl(), w.at<SortParam>(L.sortparam));
    EVX_LAUNCH_CHECK();
    if (w.matrix_unless > 0) {  // the size of front 0 is known now: the matrix, if anybody is going to read it
      if (int e = dispatch_dominance_prefix(w, s, 2)) return e;
      w.matrix_unless = 0;
    }
  }
  return 0;
}

static int grant_dynamic_lds(const void* kernel, size_t lds);

// Resident blocks per CU of the peel kernel for a dynamic-LDS size (cached: the query is not free).
// Returns a negative library code or positive hipError_t through *err and 0 on failure.
static int peel_blocks_per_cu(size_t lds, int* err) {
  struct Entry { size_t lds; int dev; int per_cu; };
  static Entry cache[16];
  static int used = 0;
  static std::mutex mu;
  int dev = 0;
  (void)hipGetDevice(&dev);
  {
    std::lock_guard<std::mutex> lock(mu);
    for (int i = 0; i < used; ++i)
      if (cache[i].lds == lds && cache[i].dev == dev) return cache[i].per_cu;
  }
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(peel_kernel), lds)) { *err = e; return 0; }
  int per_cu = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, peel_kernel, kPeelThreads, lds);
  if (e != hipSuccess) { *err = (int)e; return 0; }
  if (per_cu < 1) { *err = kErrBadArg; return 0; }
  {
    std::lock_guard<std::mutex> lock(mu);
    if (used < 16) cache[used++] = Entry{lds, dev, per_cu};
  }
  return per_cu;
}

// Grants only ever grow per (kernel, device), and are made one at a time: a thread that was given a large size never
// finds it taken back by another thread's smaller one between its grant and its launch.
static int grant_dynamic_lds(const void* kernel, size_t lds) {
  if (lds > 160 * 1024) return kErrBadArg;  // (what a workgroup of this device can have)
  if (lds <= 48 * 1024) return 0;
  struct Entry { const void* kernel; int dev; size_t lds; };
  static Entry table[128];
  static int used = 0;
  static std::mutex mu;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = -1;
  std::lock_guard<std::mutex> lock(mu);
  int at = -1;
  for (int i = 0; i < used; ++i)
    if (table[i].kernel == kernel && table[i].dev == dev) at = i;
  if (at >= 0 && table[at].lds >= lds) return 0;
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return (int)e;
  if (at >= 0)
    table[at].lds = lds;
  else if (used < 128)
    table[used++] = Entry{kernel, dev, lds};
  return 0;
}

// Sweeping workgroups of the LDS-resident peel for this population and the dynamic LDS each needs; 0 when the
// population does not fit (or the option is off).  Every workgroup takes a compute unit of its own.
constexpr size_t kLdsPeelBudget = 160 * 1024 - 512;

// Workgroups of peel_lds_kernel that a compute unit holds at once when each has `lds` bytes of dynamic LDS (asked of
// the runtime once per device and 8 KB step of the size, for the upper end of the step); 0 when the query fails.
static int lds_peel_per_cu(size_t lds) {
  static std::atomic<int> cache[64][24];  // 0 unknown, else the answer + 1
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64 || lds > kLdsPeelBudget) return 0;
  const int slot = (int)((lds + 8191) / 8192);
  int known = cache[dev][slot].load(std::memory_order_acquire);
  if (known == 0) {
    // (the attribute belongs to the (kernel, device) pair)
    // (both instances of the kernel: the one for several populations only moves its pointers first)
    int per_cu = 1 << 30;
    const size_t upper = (size_t)slot * 8192 < kLdsPeelBudget ? (size_t)slot * 8192 : kLdsPeelBudget;
    for (const void* kernel : {reinterpret_cast<const void*>(peel_lds_kernel<false>), reinterpret_cast<const void*>(peel_lds_kernel<true>)}) {
      if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsPeelBudget) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
      }
      int one = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&one, kernel, kLdsPeelThreads, upper) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
      }
      if (one < per_cu) per_cu = one;
    }
    known = per_cu + 1;
    cache[dev][slot].store(known, std::memory_order_release);
  }
  return known - 1;
}

// batch > 1: that many populations share the launch, each with this many sweeping workgroups (and its lister); up to
// four workgroups then share a compute unit where their LDS allows it, and the plan is the one with the most
// sweeping workgroups per population.
static int lds_peel_plan(const Layout& L, size_t* lds_out, int batch = 1) {
  if (!opt().peel_lds || L.n > 32768 || L.nwords > kLdsPeelThreads) return 0;  // (the lister keeps original indices in 16 bits and takes a bitmap word per thread)
  if (batch > 1) {
    size_t tail_need = opt().peel_tail ? peel_tail_lds_bytes(L.n, L.m) : 0;  // (a small last front is ordered in the kernel's LDS)
    if (tail_need > kLdsPeelBudget) tail_need = 0;
    int wanted = opt().peel_lds_blocks;
    if (wanted == 0) wanted = L.n / 64 < 32 ? 32 : L.n / 64;
    int best = 0;
    for (int per_cu = 1; per_cu <= 4; ++per_cu) {
      const int64_t share = (int64_t)per_cu * device_cus() / batch - 1;
      const int most = share < 255 ? (int)share : 255;
      if (most < 8) continue;
      const size_t limit = (size_t)160 * 1024 / per_cu - 1024;
      auto fits = [&](int sweepers) {
        const size_t b = lds_peel_bytes(L.n, L.nwords, sweepers);
        return b != 0 && b <= limit;
      };
      int sweepers = wanted < most ? wanted : most;
      while (sweepers < most && !fits(sweepers)) sweepers = sweepers + 8 < most ? sweepers + 8 : most;
      if (!fits(sweepers) || tail_need > limit || sweepers <= best) continue;
      const size_t lds = lds_peel_bytes(L.n, L.nwords, sweepers);
      if (lds_peel_per_cu(lds > tail_need ? lds : tail_need) < per_cu) continue;
      best = sweepers;
      *lds_out = lds;
    }
    return best;
  }
  const int most = device_cus() - 1 < 255 ? device_cus() - 1 : 255;  // + the lister; a record holds at least 4 units
  if (most < 8) return 0;
  auto fits = [&](int sweepers) {
    const size_t b = lds_peel_bytes(L.n, L.nwords, sweepers);
    return b != 0 && b <= kLdsPeelBudget;
  };
  if (!fits(most)) return 0;
  int sweepers = opt().peel_lds_blocks;
  if (sweepers == 0) {
    // by size: about 64 rows per workgroup, at least 32 workgroups
    sweepers = L.n / 64 < 32 ? 32 : L.n / 64;
  }
  if (sweepers > most) sweepers = most;
  while (sweepers < most && !fits(sweepers)) sweepers = sweepers + 8 < most ? sweepers + 8 : most;
  *lds_out = lds_peel_bytes(L.n, L.nwords, sweepers);
  return sweepers;
}

static int launch_lds_peel(const Ws& w, int64_t stop_count, bool want_perm, bool fill_dist, int sweepers, size_t lds, hipStream_t s,
                           bool order_last_front = false) {
  const Layout& L = w.L;
  if (stop_count < 1 || stop_count > L.n) return kErrBadArg;
  PeelTail tail;
  tail.mode = 0;
  tail.m = L.m;
  tail.npad = L.npad;
  tail.xs_sorted = w.at<float>(L.xs_sorted);
  tail.dist = w.at<float>(L.dist);
  tail.order = w.at<int>(L.order);
  tail.buffer = w.at<unsigned long long>(L.tailbuf);
  if (order_last_front && opt().peel_tail) {
    // a small last front is ordered by the peel kernel itself; its LDS must hold the candidates
    const size_t need = peel_tail_lds_bytes(L.n, L.m);
    if (need != 0 && need <= kLdsPeelBudget) {
      tail.mode = 2;
      if (lds < need) lds = need;
    }
  }
  // every workgroup waits for every other one, so the grid must be resident at once
  if ((int64_t)lds_peel_per_cu(lds) * device_cus() < (int64_t)(sweepers + 1) * w.batch) return kErrNotResident;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(sweepers + 1, 1, w.batch), dim3(kLdsPeelThreads), lds, s, w.at<uint64_t>(L.dom), L.wstride, L.nwords, L.n,
                       w.at<int>(L.orig_of), w.at<int>(L.rank), fill_dist ? w.at<float>(L.dist) : (float*)nullptr,
                       w.at<uint64_t>(L.fronts_slot), w.at<uint64_t>(L.fronts_orig), w.at<int>(L.fsize),
                       want_perm ? w.at<int>(L.perm) : (int*)nullptr, w.at<int>(L.fstart), w.ctrl(), (int)stop_count, opt().spin_limit,
                       w.at<unsigned long long>(L.records), sweepers, tail, w.step);
  };
  if (w.batch > 1)
    launch(peel_lds_kernel<true>);
  else
    launch(peel_lds_kernel<false>);
  EVX_LAUNCH_CHECK();
  return 0;
}

// Counts and peeling for the entry points: one kernel when the matrix fits the LDS of the device, else the count
// pass over the matrix followed by a peel kernel that rescans rows in memory.
static int stage_peel(const Ws& w, int64_t stop_count, bool want_perm, hipStream_t s);
static int stage_count(const Ws& w, bool fill_dist, hipStream_t s, bool need_counts = true);
static int peel_pass_plan(const Layout& L, int* blocks_out, int* use_witness_out);
static int stage_peel_stepped(const Ws& w, int64_t stop_count, bool want_perm, hipStream_t s);
static int count_and_peel_persistent(const Ws& w, int64_t stop_count, bool want_perm, bool fill_dist, hipStream_t s,
                                     bool order_last_front, bool* may_have_ordered, bool* always_orders);

// used_stepped: the fronts were peeled one launch each (stepped.hpp) -- asked for by the tunable, or because the grids
// of the persistent kernels would not be resident at once on this device; the last front is then left to the caller.
static int count_and_peel(const Ws& w, int64_t stop_count, bool want_perm, bool fill_dist, hipStream_t s,
                          bool order_last_front = false, bool* may_have_ordered = nullptr, bool* always_orders = nullptr,
                          bool* used_stepped = nullptr) {
  if (used_stepped) *used_stepped = false;
  int e = kErrNotResident;
  if (!opt().peel_stepped) e = count_and_peel_persistent(w, stop_count, want_perm, fill_dist, s, order_last_front, may_have_ordered, always_orders);
  if (e != kErrNotResident) return e;
  if (may_have_ordered) *may_have_ordered = false;
  if (always_orders) *always_orders = false;
  if (used_stepped) *used_stepped = true;
  if (int c = stage_count(w, fill_dist, s, true)) return c;
  return stage_peel_stepped(w, stop_count, want_perm, s);
}

static int count_and_peel_persistent(const Ws& w, int64_t stop_count, bool want_perm, bool fill_dist, hipStream_t s,
                                     bool order_last_front, bool* may_have_ordered, bool* always_orders) {
  size_t lds = 0;
  if (may_have_ordered) *may_have_ordered = false;
  if (always_orders) *always_orders = false;
  if (const int sweepers = lds_peel_plan(w.L, &lds, w.batch)) {
    const bool may = order_last_front && opt().peel_tail && peel_tail_lds_bytes(w.L.n, w.L.m) != 0 &&
                     peel_tail_lds_bytes(w.L.n, w.L.m) <= kLdsPeelBudget;
    if (may_have_ordered) *may_have_ordered = may;
    if (always_orders && may) {
      // Whatever the last front turns out to be, the peel kernel orders it: no front of this population is too
      // large for it, and no workgroup can have more rows in one front than its record holds (a level with such a
      // record goes through the bitmaps in memory and leaves the last front to the kernels after it).
      int units = 2;
      while (units * 2 * sweepers <= kRecUnits && units < 32) units *= 2;
      const int waves = kLdsPeelThreads / 64;
      const int rows_of_a_workgroup = (w.L.n + sweepers * waves - 1) / (sweepers * waves) * waves;
      *always_orders = peel_tail_applies(w.L.n, w.L.m) && rows_of_a_workgroup <= 2 + 3 * (units - 1);
    }
    return launch_lds_peel(w, stop_count, want_perm, fill_dist, sweepers, lds, s, order_last_front);
  }
  if (w.batch > 1) return kErrNotResident;  // (the kernels below take one population per launch)
  // (the witness passes read of a row only its highest dominator: the count stage then walks every row from the top
  // as far as that, instead of adding up all of it)
  int blocks = 0, use_witness = 0;
  if (int e = peel_pass_plan(w.L, &blocks, &use_witness)) return e;
  if (int e = stage_count(w, fill_dist, s, use_witness == 0)) return e;
  return stage_peel(w, stop_count, want_perm, s);
}

// Grid of the peel kernels that rescan rows in memory, and whether they use the witness pass (else the sweep pass,
// which needs the popcounts of the rows).
static int peel_pass_plan(const Layout& L, int* blocks_out, int* use_witness_out) {
  const size_t lds_limit = 160 * 1024 - 4096;
  const size_t bitmap = sizeof(uint64_t) * (size_t)L.nwords;
  const int cus = device_cus();
  // The grid never exceeds what the device holds at once (the blocks wait for one another).
  auto grid_for = [&](size_t lds, int* err) -> int {
    int per_cu = peel_blocks_per_cu(lds, err);
    if (per_cu > opt().peel_blocks_per_cu) per_cu = opt().peel_blocks_per_cu;
    int64_t blocks = (int64_t)cus * per_cu;
    if (blocks > kMaxGrid) blocks = kMaxGrid;
    const int64_t wpb = kPeelThreads / 64;
    const int64_t useful = kFirstSweeper + ((int64_t)L.n + wpb - 1) / wpb;  // master, lister + one wave per row
    return (int)(blocks < useful ? blocks : useful);
  };
  // The witness pass keeps two bitmaps in LDS and at most kWitnessChunks * 64 rows per sweeping
  // wave; populations too large for that use the sweep pass.
  int err = 0;
  int use_witness = opt().peel_witness && 2 * bitmap <= lds_limit;
  int blocks = 0;
  if (use_witness) {
    blocks = grid_for(2 * bitmap, &err);
    if (err) return err;
    const int64_t waves = (int64_t)(blocks - kFirstSweeper) * (kPeelThreads / 64);
    if (blocks <= kFirstSweeper || (L.n + waves - 1) / waves > kWitnessChunks * 64) use_witness = 0;
  }
  if (!use_witness) {
    if (bitmap > lds_limit) return kErrBadArg;
    blocks = grid_for(bitmap, &err);
    if (err) return err;
  }
  if (blocks <= kFirstSweeper) return kErrNotResident;
  *blocks_out = blocks;
  *use_witness_out = use_witness;
  return 0;
}

static int stage_peel(const Ws& w, int64_t stop_count, bool want_perm, hipStream_t s) {
  const Layout& L = w.L;
  if (stop_count < 1 || stop_count > L.n) return kErrBadArg;
  const size_t bitmap = sizeof(uint64_t) * (size_t)L.nwords;
  const int cus = device_cus();
  int blocks = 0, use_witness = 0;
  if (int e = peel_pass_plan(L, &blocks, &use_witness)) return e;
  if (use_witness && opt().peel_records && L.n <= kRecordsMaxRowsWide) {
    // all-to-all records: 1 lister + the sweeping blocks, all resident at once
    const int sweepers = cus >= 64 ? (opt().peel_record_blocks ? opt().peel_record_blocks : record_sweepers(L.n, L.m)) : 16;
    const int wpb = kRecThreads / 64;
    const int list_capacity = wpb * ((L.n + sweepers * wpb - 1) / (sweepers * wpb));
    const size_t rec_lds = bitmap + 24 * (size_t)list_capacity;  // queue (8 + 4 + 4) and ranked pairs (2 x 4) per row
    // every block waits for every other one: all of them must be resident at once
    int rec_per_cu = 0;
    const bool wide = L.n > kRecordsMaxRows;
    const void* kernel = wide ? reinterpret_cast<const void*>(peel_records_kernel<true>)
                              : reinterpret_cast<const void*>(peel_records_kernel<false>);
    const bool rows_fit = (int64_t)list_capacity <= (int64_t)wpb * kWitnessChunks * 64;  // what the waves' registers hold
    if (rows_fit && rec_lds <= 150 * 1024)
      if (int e = grant_dynamic_lds(kernel, rec_lds)) return e;
    const hipError_t oe = wide ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&rec_per_cu, peel_records_kernel<true>, kRecThreads, rec_lds)
                               : hipOccupancyMaxActiveBlocksPerMultiprocessor(&rec_per_cu, peel_records_kernel<false>, kRecThreads, rec_lds);
    if (oe != hipSuccess) return (int)oe;
    if (rows_fit && rec_lds <= 150 * 1024 && (int64_t)rec_per_cu * cus >= sweepers + 1) {
    hipLaunchKernelGGL(wide ? peel_records_kernel<true> : peel_records_kernel<false>, dim3(sweepers + 1), dim3(kRecThreads), rec_lds, s, w.at<uint64_t>(L.dom), L.wstride,
                       L.nwords, L.n, w.at<int>(L.orig_of), w.at<int>(L.rank), w.at<uint64_t>(L.fronts_slot),
                       w.at<uint64_t>(L.fronts_orig), w.at<int>(L.fsize), want_perm ? w.at<int>(L.perm) : (int*)nullptr,
                       w.at<int>(L.fstart), w.ctrl(), (int)stop_count, opt().spin_limit, w.at<int>(L.witness),
                       w.at<unsigned long long>(L.records), sweepers, list_capacity);
    EVX_LAUNCH_CHECK();
    return 0;
    }  // otherwise: the master protocol below, whose grid is sized to what fits
  }
  const size_t lds = bitmap * (use_witness ? 2 : 1);
  hipLaunchKernelGGL(peel_kernel, dim3(blocks), dim3(kPeelThreads), lds, s, w.at<uint64_t>(L.dom), L.wstride, L.nwords,
                     L.n, w.at<int>(L.orig_of), w.at<int>(L.count), w.at<int>(L.rank), w.at<uint64_t>(L.fronts_slot),
                     w.at<uint64_t>(L.fronts_orig), w.at<int>(L.fsize),
                     want_perm ? w.at<int>(L.perm) : (int*)nullptr, w.at<int>(L.fstart), w.ctrl(), (int)stop_count,
                     opt().spin_limit, w.at<int>(L.witness), use_witness);
  EVX_LAUNCH_CHECK();
  return 0;
}

// One launch per front, in groups; between groups the host waits for the stream and reads whether the pass that finds
// the ranking complete has run (the only place where this path waits).  stage_count must have left the full counts.
constexpr int kStepGroup = 16;
static int stage_peel_stepped(const Ws& w, int64_t stop_count, bool want_perm, hipStream_t s) {
  const Layout& L = w.L;
  if (stop_count < 1 || stop_count > L.n) return kErrBadArg;
  const size_t lds = sizeof(uint64_t) * (size_t)((L.nwords + 1) & ~1);
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(step_pass_kernel), lds)) return e;
  int sweepers = (L.n + kStepThreads / 64 - 1) / (kStepThreads / 64);
  const int cap = device_cus() * 8;
  if (sweepers > cap) sweepers = cap;
  const int listers = (L.nwords + kStepListWords - 1) / kStepListWords;
  // (front L.n - 1 is the last that can exist; the pass after a front is the one that sees it complete)
  for (int64_t level = 1; level <= (int64_t)L.n + 1;) {
    for (int k = 0; k < kStepGroup && level <= (int64_t)L.n + 1; ++k, ++level) {
      hipLaunchKernelGGL(step_pass_kernel, dim3(sweepers + listers), dim3(kStepThreads), lds, s, w.at<uint64_t>(L.dom), L.wstride,
                         L.nwords, L.n, w.at<int>(L.orig_of), w.at<int>(L.count), w.at<int>(L.rank), w.at<uint64_t>(L.fronts_slot),
                         w.at<uint64_t>(L.fronts_orig), w.at<int>(L.fsize), w.at<int>(L.fstart),
                         want_perm ? w.at<int>(L.perm) : (int*)nullptr, w.ctrl(), (int)stop_count, (int)level, sweepers);
      EVX_LAUNCH_CHECK();
    }
    int32_t head[16];
    hipError_t e = hipMemcpyAsync(head, w.ctrl(), sizeof(head), hipMemcpyDeviceToHost, s);
    if (e != hipSuccess) return (int)e;
    e = hipStreamSynchronize(s);
    if (e != hipSuccess) return (int)e;
    static_assert(offsetof(Ctrl, reserved) == 40 && sizeof(int32_t) * (10 + kStepDone + 1) <= sizeof(head), "Ctrl.reserved[kStepDone]");
    if (head[0] != 0 || head[10 + kStepDone] != 0) break;
  }
  return 0;
}

static RadixBuffers radix_buffers(const Ws& w) {
  RadixBuffers b;
  b.pairs[0] = w.at<unsigned long long>(w.L.rpairs0);
  b.pairs[1] = w.at<unsigned long long>(w.L.rpairs1);
  b.table = w.at<int>(w.L.rtable);
  b.totals = w.at<int>(w.L.rtotals);
  b.kstride = w.L.kstride;
  return b;
}

// Blocks of a radix kernel: master + idle slot + one worker per 1024 candidates, all resident.
static int radix_grid(const Layout& L) {
  int workers = (L.n + 1023) / 1024;
  const int cap = device_cus() * 2 - kFirstSweeper;
  if (workers > cap) workers = cap;
  if (workers > kRadixMaxWorkers) workers = kRadixMaxWorkers;
  if (workers < 1) workers = 1;
  return workers + kFirstSweeper;
}

// The last front of a population of at most kMidArgsortRows rows goes through the kernels with the sorted runs (finish.hpp),
// whose workgroups hold all its keys in LDS.
static bool crowd_mid_sort(const Layout& L) { return opt().mid_argsort != 0 && L.n > kMidSortMinCandidates && L.n <= kMidArgsortRows; }
// A larger population: a front of more than kMidSortMinCandidates and at most that many rows does; the other kernels return at
// once from it, and these from any other.
static bool crowd_mid_split(const Layout& L) { return opt().mid_argsort != 0 && L.n > kMidArgsortRows; }

// Grid of crowd_gather_kernel, crowd_sort_kernel and crowd_finish_kernel (finish.hpp): the radix grid when a front of this
// population can exceed kRadixMinCandidates rows (they then synchronise across blocks), else one block
// per 256 candidates and objective.
static int finish_grid(const Layout& L, int per_candidate_block) {
  if (crowd_mid_sort(L)) return device_cus();  // (crowd_gather_kernel with the LDS sorter: its LDS leaves room for one workgroup per compute unit: all resident)
  if (L.n > kRadixMinCandidates) {
    // The kernels choose on the device: a front of at most kRadixMinCandidates rows is still ordered by counting,
    // one work item per 256 candidates (and objective), and wants as many blocks as it has items -- a population
    // of 5000 rows has a radix grid of 7 blocks, on which the 110 items of a 2764-row front of ten objectives took
    // 0.59 ms.  More workers than the radix sort needs only idle at its barriers.
    int blocks = radix_grid(L);
    int wanted = (kRadixMinCandidates / 256) * per_candidate_block + kFirstSweeper;
    int cap = device_cus() * 2;
    if (cap > kRadixMaxWorkers + kFirstSweeper) cap = kRadixMaxWorkers + kFirstSweeper;
    if (wanted > cap) wanted = cap;
    return blocks > wanted ? blocks : wanted;
  }
  int blocks = ((L.n + 255) / 256) * per_candidate_block;
  return blocks < 1 ? 1 : blocks;
}

// The grid of one population when `batch` of them share a launch whose workgroups may wait for each other: the device
// holds `resident` such workgroups at once.
static int shared_grid(int grid, int resident, int batch) {
  if (batch <= 1) return grid;
  const int cap = resident / batch < 1 ? 1 : resident / batch;
  return grid < cap ? grid : cap;
}

constexpr int kNearbyMaxObjectives = 15;  // (the order of the slots is one more)
// From how many rows on the totals alone are counted in spatial order (their order costs 60 us, and what it saves hangs on
// the share of the pairs of tile and group that is left).  Whole selections whose front 0 holds what is kept, us, slot
// order / spatial order, all rows on a plane or (s) around a sphere with a part of front 0 kept:
//   x 3: 90 112 341 / 321, 100 000 (s) 277 / 291, 125 000 (s) 325 / 333, 131 072 481 / 383, (s) 390 / 334, 200 000 (s) 719 / 568;
//   x 4: 80 000 307 / 314, 90 112 339 / 327, 100 000 (s) 344 / 327, 200 000 899 / 614;
//   x 5: 57 344 288 / 294, 62 000 (s) 286 / 292, 65 536 303 / 301, (s) 304 / 300;
//   x 6: 57 344 (s) 302 / 307, 60 000 317 / 310;  x 8: 57 344 (s) 346 / 350, 60 000 380 / 360, 200 000 (s) 1176 / 743;
//   x 10: 57 344 (s) 371 / 381, 60 000 (s) 411 / 399;  x 11: 57 344 (s) 423 / 396;  x 15: 40 000 381 / 405, 57 344 (s) 543 / 501.
static int64_t nearby_least_rows(int m) { return m <= 3 ? 131072 : m == 4 ? 90112 : m == 5 ? 65536 : m <= 10 ? 60000 : 57344; }
static bool nearby_totals_apply(int n, int m) {
  const int64_t rule = opt().prefix_nearby;
  if (rule == 0 || m < 3 || m > kNearbyMaxObjectives) return false;  // (two objectives are ranked without totals)
  return n >= (rule == 1 ? nearby_least_rows(m) : rule);
}
template <int M>
static int launch_nearby_totals(const Ws& w, hipStream_t s);

// phase 0: totals and matrix in one launch (or what the tunable prefix_mode asks for); 1: the totals alone, and the
// pairwise kernel for a population that is not finite; 2: the matrix alone, unless front 0 holds w.matrix_unless rows.
template <int M>
static int launch_dominance_prefix(const Ws& w, hipStream_t s, int phase) {
  constexpr int WW = M <= kPrefixWideObjectives ? 8 : 4;  // words per tile: what the LDS holds tables for
  // up to four objectives the tables of two tiles fit: a workgroup then builds whole 128-byte lines of the matrix
  constexpr int TT = M <= 4 ? 2 : 1;
  const Layout& L = w.L;
  const int shift = prefix_bucket_shift(L.n);
  const int buckets = ((L.n - 1) >> shift) + 1;
  const int bands_wanted = opt().prefix_bands;
  // bands of rows shared by all tiles (their stores then fall into the same rows at about the same time) pay from
  // about 100 000 rows on: 200 000 x 8 1203 -> 1156 us, 100 000 x 8 441 -> 424, but 65536 x 3 181 -> 190
  const int bands = bands_wanted != 0 && L.n >= 98304 ? 1 : 0;
  // shorter stretches for smaller populations, so that the workgroups still outnumber the compute units
  const int chunk = L.n >= 131072 ? kPrefixRowChunk : (L.n >= 65536 ? kPrefixRowChunk / 2 : kPrefixRowChunk / 4);
  const int stretches = (L.n + chunk - 1) / chunk;
  auto launch = [&](auto kernel, int tt) -> int {
    const size_t lds = (size_t)tt * prefix_lds_bytes(M, WW, buckets);
    if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(kernel), lds)) return e;
    const int tiles = (int)round_up((L.nwords + WW * tt - 1) / (WW * tt), 128 / (WW * tt));
    hipLaunchKernelGGL(kernel, dim3(tiles, stretches), dim3(kPrefixThreads), lds, s, w.at<int>(L.pos), w.at<int>(L.scost),
                       w.at<uint32_t>(L.kid_sorted), w.at<uint64_t>(L.dom), L.n, L.kstride, L.wstride, L.nwords, shift, buckets,
                       chunk, bands, phase == 0 ? opt().prefix_mode : phase, w.at<int>(L.total0), w.at<int>(L.witness0),
                       w.at<SortParam>(L.sortparam), w.ctrl(), phase == 2 ? w.at<int>(L.fsize) : (const int*)nullptr, (int)w.matrix_unless,
                       NearbyWork{});
    EVX_LAUNCH_CHECK();
    return 0;
  };
  // (200 000 x 3: 957 -> 769 us, x 4: 972 -> 797; 100 000 x 3: 319 -> 317; 65536 x 3: 184 -> 220: half as many workgroups)
  if (phase == 1 && nearby_totals_apply(L.n, M)) {
    if constexpr (M >= 3 && M <= kNearbyMaxObjectives)
      if (int e = launch_nearby_totals<M>(w, s)) return e;
  } else if (TT == 2 && opt().prefix_double_tile > 0 && L.n >= opt().prefix_double_tile) {
    if (int e = launch(dominance_prefix_kernel<M, WW, TT>, TT)) return e;
  } else {
    if (int e = launch(dominance_prefix_kernel<M, WW, 1>, 1)) return e;
  }
  if (phase == 2) return 0;
  // a population with a NaN or an infinity: the pairwise kernel, on a grid that costs nothing when it has nothing to do
  hipLaunchKernelGGL(dominance_nonfinite_kernel<M>, dim3(device_cus() * 8), dim3(256), 0, s, w.at<float>(L.xs_sorted),
                     w.at<uint64_t>(L.key_sorted), w.at<uint32_t>(L.kid_sorted), w.at<uint64_t>(L.dom), L.n, L.npad, L.wstride,
                     L.nwords, w.at<SortParam>(L.sortparam));
  EVX_LAUNCH_CHECK();
  return 0;
}

// The row totals alone (phase 1) from the rows in spatial order.  What it needs besides the orders lies where the matrix
// would: nobody reads that before a second launch builds it.
template <int M>
static int launch_nearby_totals(const Ws& w, hipStream_t s) {
  const Layout& L = w.L;
  constexpr int MO = M + 1;
  constexpr int WW = MO <= kPrefixWideObjectives ? 8 : 4;
  const int stride = (int)round_up(L.n, 64), groups = stride / 64;
  size_t o = L.dom;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o = align_up(o + bytes);
    return at;
  };
  const int tiles = (groups + WW - 1) / WW;
  // (parts small enough that the last ones end together, large enough to be worth a tile's tables: 10 us against 0.3 per group)
  int cap = groups / 16;
  if (cap > kPrefixNearbyGroups) cap = kPrefixNearbyGroups;
  if (cap < 32) cap = 32;
  const size_t most_full = (size_t)tiles * (size_t)(groups / cap + 1);
  const size_t hist = take(sizeof(int) * kNearbyCells), flags = take(sizeof(unsigned long long) * 64), queue = take(sizeof(int) * 4);
  const size_t starts = take(sizeof(int) * (kNearbyCells + 1)), cursor = take(sizeof(int) * kNearbyCells);
  const size_t cell = take(sizeof(uint16_t) * (size_t)L.n), place = take(sizeof(int) * (size_t)L.n), slot_at = take(sizeof(int) * (size_t)L.n);
  const size_t pos_at = take(sizeof(int) * MO * (size_t)stride), upper_at = take(sizeof(int) * MO * (size_t)stride);
  const size_t lo = take(sizeof(int) * MO * (size_t)groups), top = take(sizeof(int) * MO * (size_t)groups),
               hi = take(sizeof(int) * MO * (size_t)groups);
  const size_t box = take(sizeof(int) * 2 * MO * (size_t)tiles), near_list = take(sizeof(uint16_t) * (size_t)tiles * (size_t)groups);
  const size_t near_count = take(sizeof(int) * (size_t)tiles), full = take(sizeof(int2) * most_full), rest = take(sizeof(int2) * (size_t)tiles);
  if (o > L.dom + sizeof(uint64_t) * (size_t)L.n * (size_t)L.wstride || groups > 65536) return kErrWorkspace;
  SortParam* const param = w.at<SortParam>(L.sortparam);
  hipLaunchKernelGGL(reset_state_kernel, dim3(16), dim3(256), 0, s, w.at<uint32_t>(hist), (int64_t)((queue - hist) / 4 + 4));
  EVX_LAUNCH_CHECK();
  const int cell_rows = kNearbyCellThreads * kNearbyCellRows;
  hipLaunchKernelGGL(nearby_cells_kernel, dim3((L.n + cell_rows - 1) / cell_rows), dim3(kNearbyCellThreads), 0, s, w.at<int>(L.pos), L.n,
                     L.kstride, M, param, w.at<uint16_t>(cell), w.at<int>(place), w.at<int>(hist));
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(bucket_scan_kernel<false>, dim3(kNearbyCells / 1024), dim3(256), 0, s, w.at<int>(hist), kNearbyCells, w.at<int>(starts),
                     w.at<int>(cursor), w.at<unsigned long long>(flags), w.ctrl(), (int64_t)0);
  EVX_LAUNCH_CHECK();
  int blocks = (L.n + 255) / 256;
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(nearby_scatter_kernel, dim3(blocks), dim3(256), 0, s, w.at<uint16_t>(cell), w.at<int>(place), L.n, param, w.ctrl(),
                     w.at<int>(starts), w.at<int>(slot_at));
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(nearby_gather_kernel, dim3((L.n + 255) / 256, MO), dim3(256), 0, s, w.at<int>(L.pos), w.at<int>(L.scost),
                     w.at<uint32_t>(L.kid_sorted), L.n, L.kstride, M, param, w.ctrl(), w.at<int>(slot_at), stride, w.at<int>(pos_at),
                     w.at<int>(upper_at), groups, w.at<int>(lo), w.at<int>(top), w.at<int>(hi));
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(nearby_pairs_kernel<MO>, dim3(tiles), dim3(256), 0, s, w.at<int>(lo), w.at<int>(top), w.at<int>(hi), groups, WW, cap, param,
                     w.ctrl(), w.at<int>(box), w.at<uint16_t>(near_list), w.at<int>(near_count), w.at<int2>(full), w.at<int2>(rest),
                     w.at<int>(queue));
  EVX_LAUNCH_CHECK();
  const auto kernel = dominance_prefix_kernel<MO, WW, 1, true>;
  const size_t lds = prefix_lds_bytes(MO, WW, kPrefixBuckets);
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(kernel), lds)) return e;
  const int grid = device_cus() * (lds <= 76 * 1024 ? 2 : 1);  // (what a compute unit holds at once)
  const NearbyWork work = {w.at<int>(box), w.at<uint16_t>(near_list), w.at<int>(near_count), w.at<int2>(full), w.at<int2>(rest), w.at<int>(queue), cap};
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kPrefixThreads), lds, s, w.at<int>(pos_at), w.at<int>(upper_at), (const uint32_t*)nullptr,
                     (uint64_t*)nullptr, L.n, stride, (int64_t)0, groups, 0, kPrefixBuckets, 0, 0, 1, w.at<int>(L.total0), w.at<int>(L.witness0),
                     param, w.ctrl(), (const int*)nullptr, 0, work);
  EVX_LAUNCH_CHECK();
  return 0;
}

// The matrix of a large finite population from the order of its rows in every objective (prefix.hpp).  The
// buffers of the crowding stage (radix pairs, pos, scost) are free until then and carry the orders.
template <int M>
static int launch_dominance_prefix(const Ws& w, hipStream_t s, int phase);

static int stage_dominance_prefix(const Ws& w, bool orders_only, hipStream_t s, int64_t count_first) {
  const Layout& L = w.L;
  // (the count stage launches the second phase: the peel that keeps the matrix in LDS has no count stage)
  size_t unused = 0;
  const int phase = count_first > 0 && !orders_only && opt().prefix_count_first && opt().prefix_mode == 3 &&
                            lds_peel_plan(L, &unused, 1) == 0 ? 1 : 0;
  if (phase == 1) w.matrix_unless = count_first;
  if (L.n <= kMidArgsortRows && opt().mid_argsort) {
    // the orders from workgroups that sort in LDS: two launches, no grid barrier (and no barrier words to reset)
    const size_t sort_lds = mid_sort_lds_bytes(L.n);
    const bool wide = L.n <= kMidArgsortWideRows;
    const void* const kernel = wide ? reinterpret_cast<const void*>(objective_order_lds_kernel<true>)
                                    : reinterpret_cast<const void*>(objective_order_lds_kernel<false>);
    if (int e = grant_dynamic_lds(kernel, sort_lds)) return e;
    if (wide)
      hipLaunchKernelGGL(objective_order_lds_kernel<true>, dim3(device_cus()), dim3(kMidArgsortThreads), sort_lds, s, w.at<float>(L.xs),
                         L.npad, L.n, L.m, w.at<SortParam>(L.sortparam), w.ctrl(), w.at<int>(L.total0), w.at<int>(L.witness0),
                         radix_buffers(w));
    else
      hipLaunchKernelGGL(objective_order_lds_kernel<false>, dim3(device_cus()), dim3(kMidArgsortThreads), sort_lds, s, w.at<float>(L.xs),
                         L.npad, L.n, L.m, w.at<SortParam>(L.sortparam), w.ctrl(), w.at<int>(L.total0), w.at<int>(L.witness0),
                         radix_buffers(w));
    EVX_LAUNCH_CHECK();
    int64_t blocks = ((int64_t)L.n * L.m + 255) / 256;
    if (blocks > device_cus() * 8) blocks = device_cus() * 8;
    hipLaunchKernelGGL(objective_positions_kernel, dim3((unsigned)blocks), dim3(256), 0, s, L.n, L.m, w.at<int>(L.slot_of),
                       w.at<SortParam>(L.sortparam), w.ctrl(), w.at<int>(L.pos), w.at<int>(L.scost), radix_buffers(w));
    EVX_LAUNCH_CHECK();
    return orders_only ? 0 : dispatch_dominance_prefix(w, s, phase);
  }
  // shares of one objective's order: as many as give every compute unit a workgroup, while they fit one (whole selections, us, shares /
  // radix sort below: 200 000 x 8 693 / 780, 250 000 x 8 826 / 910, 120 000 x 16 1100 / 1236)
  const int stream_parts = device_cus() / L.m < kOrderStreamMaxParts ? device_cus() / L.m : kOrderStreamMaxParts;
  if (opt().order_stream && L.n > kOrderStreamSample && L.n <= kOrderStreamMaxRows && (L.npad & 3) == 0 && stream_parts >= 1 &&
      stream_parts <= kOrderStreamSample && (int64_t)stream_parts * kOrderStreamShare >= L.n) {
    // larger populations likewise: the rows grouped by share of an objective's order, then the shares placed in LDS
    if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(objective_order_stream_kernel), kOrderStreamLdsBytes)) return e;
    const int parts = stream_parts;
    const int per = (L.n + parts - 1) / parts;
    // (the matrix is written behind these launches)
    unsigned long long* const bounds = w.at<unsigned long long>(L.dom);
    uint32_t* const offsets = w.at<uint32_t>(L.dom) + order_bounds_words(L.m, parts);
    const RadixBuffers buf = radix_buffers(w);
    hipLaunchKernelGGL(objective_shares_kernel, dim3(L.m * parts), dim3(kOrderStreamThreads),
                       8 * (size_t)kOrderStreamSample + 4 * (size_t)kOrderStreamBuckets, s, w.at<float>(L.xs), L.npad, L.n, L.m, parts, per,
                       w.at<SortParam>(L.sortparam), w.ctrl(), w.at<int>(L.total0), w.at<int>(L.witness0), buf.kstride, buf.pairs[1], offsets, bounds);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(objective_order_stream_kernel, dim3(L.m * parts), dim3(kOrderStreamThreads), kOrderStreamLdsBytes, s, w.at<float>(L.xs),
                       L.npad, L.n, L.m, parts, per, opt().order_stream_capacity, w.at<int>(L.slot_of), w.at<SortParam>(L.sortparam), w.ctrl(),
                       offsets, bounds, w.at<int>(L.pos), w.at<int>(L.scost), buf);
    EVX_LAUNCH_CHECK();
    return orders_only ? 0 : dispatch_dominance_prefix(w, s, phase);
  }
  const size_t lds = kRadixLdsBytes;
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(objective_order_kernel), lds)) return e;
  // more workers than one per 1024 rows: every one of them handles its share of all m segments
  int workers = (int)(((int64_t)L.n * L.m + 2047) / 2048);
  const int cap = (device_cus() * 2 < kRadixMaxWorkers + kFirstSweeper ? device_cus() * 2 : kRadixMaxWorkers + kFirstSweeper) - kFirstSweeper;
  if (workers > cap) workers = cap;
  if (workers + kFirstSweeper < radix_grid(L)) workers = radix_grid(L) - kFirstSweeper;
  hipLaunchKernelGGL(objective_order_kernel, dim3(workers + kFirstSweeper), dim3(kRadixThreads), lds, s, w.at<float>(L.xs), L.npad, L.n,
                     L.m, w.at<int>(L.slot_of), w.at<SortParam>(L.sortparam), w.ctrl(), w.at<int>(L.pos), w.at<int>(L.scost), w.at<int>(L.total0),
                     w.at<int>(L.witness0), radix_buffers(w), opt().spin_limit);
  EVX_LAUNCH_CHECK();
  // the barrier words of the control block restart from zero for the kernels that follow (the sort counted its
  // generations from a high base)
  const size_t first = offsetof(Ctrl, release);
  const int64_t words = (int64_t)((sizeof(Ctrl) + sizeof(unsigned long long) * kMaxGrid - first) / 4);
  hipLaunchKernelGGL(reset_state_kernel, dim3(16), dim3(256), 0, s, reinterpret_cast<uint32_t*>(w.base + L.ctrl + first), words);
  EVX_LAUNCH_CHECK();
  return orders_only ? 0 : dispatch_dominance_prefix(w, s, phase);
}

static int dispatch_dominance_prefix(const Ws& w, hipStream_t s, int phase) {
  switch (w.L.m) {
    case 2: return launch_dominance_prefix<2>(w, s, phase);
    case 3: return launch_dominance_prefix<3>(w, s, phase);
    case 4: return launch_dominance_prefix<4>(w, s, phase);
    case 5: return launch_dominance_prefix<5>(w, s, phase);
    case 6: return launch_dominance_prefix<6>(w, s, phase);
    case 7: return launch_dominance_prefix<7>(w, s, phase);
    case 8: return launch_dominance_prefix<8>(w, s, phase);
    case 9: return launch_dominance_prefix<9>(w, s, phase);
    case 10: return launch_dominance_prefix<10>(w, s, phase);
    case 11: return launch_dominance_prefix<11>(w, s, phase);
    case 12: return launch_dominance_prefix<12>(w, s, phase);
    case 13: return launch_dominance_prefix<13>(w, s, phase);
    case 14: return launch_dominance_prefix<14>(w, s, phase);
    case 15: return launch_dominance_prefix<15>(w, s, phase);
    case 16: return launch_dominance_prefix<16>(w, s, phase);
    default: return kErrBadArg;
  }
}

// Workgroups of kRunRows threads that order a small front of one population together (crowd_small_front): all of them are
// resident at once, a sixteenth of their threads candidates in a round.
static int crowd_small_blocks(const Ws& w) { return shared_grid(kFusedFrontRows * 16 / kRunRows, device_cus(), w.batch); }
// The largest front that goes that way where the sorted runs stand behind it.  Several populations share the device: a
// round of the workgroups that one of them gets, since every further round costs as much as the runs do -- 40 populations of
// 1400 x 4 around a sphere, last fronts of some 900 rows, us: 275 with up to 1024 rows there, 111 with up to 192.
static int crowd_small_rows(const Ws& w) {
  if (w.batch == 1) return kFusedFrontRows;
  const int round = crowd_small_blocks(w) * (kRunRows / 16);
  return round < kFusedSoloRows ? kFusedSoloRows : round;
}
// No front of the population is too large for crowd_small_front: the first of the ordering launches does it all.
static bool crowd_always_small(const Ws& w) {
  const Layout& L = w.L;
  return L.n <= (crowd_mid_sort(L) ? crowd_small_rows(w) : kFusedFrontRows) && (int64_t)L.n * L.m <= kFusedFrontValues && L.m <= kFusedFrontObjectives;
}

// Per-objective ordering of the candidates list[ctrl.worst_start ... + ctrl.nv).
// fused: 0 = the two kernels as stages of their own; 1 / 2 = a small front gets its distances (2: and the selection
// order) inside crowd_sort_kernel, and crowd_finish_kernel, given the same value, leaves it alone.
static CrowdArgs crowd_args(const Ws& w, const int* list, bool use_orders, int fused) {
  const Layout& L = w.L;
  CrowdArgs a;
  a.xs = w.at<float>(L.xs);
  a.npad = L.npad;
  a.list_base = list;
  a.ctrl = w.ctrl();
  a.m = L.m;
  a.kstride = L.kstride;
  a.pos = w.at<int>(L.pos);
  a.sorted_cost = w.at<float>(L.scost);
  a.buf = radix_buffers(w);
  a.spin_limit = opt().spin_limit;
  a.param = w.at<SortParam>(L.sortparam);
  a.use_orders = use_orders ? 1 : 0;
  a.fused = fused;
  a.mid_sort = crowd_mid_sort(L) ? 1 : (crowd_mid_split(L) ? 2 : 0);
  a.small_rows = crowd_small_rows(w);
  a.dist = w.at<float>(L.dist);
  a.dkey = w.at<uint32_t>(L.dkey);
  a.order = w.at<int>(L.order);
  a.runs = w.at<uint32_t>(L.xs_sorted);
  a.ws_step = w.step;
  return a;
}

// The three launches that read the orders of a large last front (of more than `above` rows) off the orders of the whole
// population.
static int stage_front_orders(const Ws& w, const int* list, int above, hipStream_t s) {
  const Layout& L = w.L;
  {
    const RadixBuffers b = radix_buffers(w);
    const int spans = (L.n + kFrontOrderSpan - 1) / kFrontOrderSpan;
    int* const number = reinterpret_cast<int*>(w.at<uint32_t>(L.dkey));  // free until the distances are known
    int* const per_span = b.table;
    hipLaunchKernelGGL(front_number_kernel, dim3((L.n + 1023) / 1024), dim3(256), 0, s, list, w.ctrl(),
                       w.at<SortParam>(L.sortparam), above, number);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(front_order_count_kernel, dim3(spans, L.m), dim3(256), 0, s, b.pairs[0], b.kstride, L.n, w.at<int>(L.rank),
                       w.ctrl(), w.at<SortParam>(L.sortparam), above, per_span);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(front_order_place_kernel, dim3(spans, L.m), dim3(256), 0, s, b.pairs[0], b.kstride, L.n,
                       w.at<int>(L.rank), w.ctrl(), w.at<SortParam>(L.sortparam), above, per_span, number, w.at<float>(L.xs), L.npad,
                       w.at<int>(L.pos), w.at<float>(L.scost));
    EVX_LAUNCH_CHECK();
  }
  return 0;
}

static size_t crowd_lds_bytes(const Layout& L, int fused) {
  size_t lds = sizeof(uint32_t) * kRadixMinCandidates + sizeof(uint64_t) * kRankTile;
  if (L.n > kRadixMinCandidates && kRadixLdsBytes > lds) lds = kRadixLdsBytes;
  if (fused != 0 && kFusedFrontLdsBytes > lds) lds = kFusedFrontLdsBytes;
  if (crowd_mid_sort(L) && mid_sort_lds_bytes(L.n) > lds) lds = mid_sort_lds_bytes(L.n);
  return lds;
}

// The first two of the launches that order a front from sorted runs (finish.hpp); the first alone where no front is too
// large for it.
static int launch_crowd_runs(const Ws& w, const CrowdArgs& a, int tail_flag, hipStream_t s) {
  const Layout& L = w.L;
  const int most = L.n < kRunMaxRows ? L.n : kRunMaxRows;
  const size_t runs_lds = a.mid_sort == 1 && a.fused != 0 ? kFusedFrontLdsBytes : sizeof(uint32_t) * 2 * kRunRows;
  const int small_blocks = crowd_small_blocks(w);
  int grid = (most + kRunRows - 1) / kRunRows * L.m;
  if (grid < small_blocks) grid = small_blocks;
  if (grid > 65536) grid = 65536;
  const void* const runs_kernel = w.batch > 1 ? reinterpret_cast<const void*>(crowd_runs_kernel<true>) : reinterpret_cast<const void*>(crowd_runs_kernel<false>);
  if (int e = grant_dynamic_lds(runs_kernel, runs_lds)) return e;
  if (w.batch > 1)
    hipLaunchKernelGGL(crowd_runs_kernel<true>, dim3(grid, 1, w.batch), dim3(kRunRows), runs_lds, s, a, tail_flag, small_blocks);
  else
    hipLaunchKernelGGL(crowd_runs_kernel<false>, dim3(grid), dim3(kRunRows), runs_lds, s, a, tail_flag, small_blocks);
  EVX_LAUNCH_CHECK();
  if (a.mid_sort == 1 && a.fused != 0 && crowd_always_small(w)) return 0;
  const size_t lds = run_rank_lds_bytes(most);
  const void* const terms_kernel = w.batch > 1 ? reinterpret_cast<const void*>(crowd_terms_kernel<true>) : reinterpret_cast<const void*>(crowd_terms_kernel<false>);
  if (int e = grant_dynamic_lds(terms_kernel, lds)) return e;
  if (w.batch > 1)
    hipLaunchKernelGGL(crowd_terms_kernel<true>, dim3(run_share_grid(w), 1, w.batch), dim3(kRunRankThreads), lds, s, a, tail_flag);
  else
    hipLaunchKernelGGL(crowd_terms_kernel<false>, dim3(run_share_grid(w)), dim3(kRunRankThreads), lds, s, a, tail_flag);
  EVX_LAUNCH_CHECK();
  return 0;
}

// The distances, and with `want_order` the selection order; `gather`: and the selected rows.
static int launch_crowd_pick(const Ws& w, const CrowdArgs& a, bool want_order, const GatherArgs* gather, int tail_flag, hipStream_t s) {
  const Layout& L = w.L;
  const int most = L.n < kRunMaxRows ? L.n : kRunMaxRows;
  const int runs = (most + kRunRows - 1) / kRunRows;
  if (w.batch > 1)
    hipLaunchKernelGGL(crowd_distances_kernel<true>, dim3(runs, 1, w.batch), dim3(kRunRows), 0, s, a, want_order ? 1 : 0, tail_flag);
  else
    hipLaunchKernelGGL(crowd_distances_kernel<false>, dim3(runs), dim3(kRunRows), 0, s, a, want_order ? 1 : 0, tail_flag);
  EVX_LAUNCH_CHECK();
  if (!want_order) return 0;
  const int grid = run_share_grid(w);
  const size_t picks_at = run_rank_lds_bytes(most);  // (a multiple of 16)
  const size_t lds = picks_at + (gather != nullptr ? sizeof(int2) * (size_t)((most + grid - 1) / grid) : 0);
  const GatherArgs g = gather != nullptr ? *gather : GatherArgs{};
  auto launch = [&](auto kernel) {
    if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(kernel), lds)) return e;
    hipLaunchKernelGGL(kernel, dim3(grid, 1, w.batch), dim3(kRunRankThreads), lds, s, a, g, tail_flag, (int)picks_at);
    return 0;
  };
  int e = 0;
  if (w.batch > 1)
    e = gather != nullptr ? launch(crowd_pick_kernel<true, true>) : launch(crowd_pick_kernel<true, false>);
  else
    e = gather != nullptr ? launch(crowd_pick_kernel<false, true>) : launch(crowd_pick_kernel<false, false>);
  if (e) return e;
  EVX_LAUNCH_CHECK();
  return 0;
}

// without_runs, here and below: the launches with the sorted runs are left out where a larger population has them beside the
// others, which then take a front of any size.
static int stage_crowd_sort(const Ws& w, const int* list, bool use_orders, int fused, hipStream_t s, bool after_peel_tail = false,
                            bool without_runs = false) {
  const Layout& L = w.L;
  const int tail_flag = after_peel_tail ? 1 : 0;
  if (crowd_mid_sort(L)) return launch_crowd_runs(w, crowd_args(w, list, false, fused), tail_flag, s);
  use_orders = use_orders && prefix_dominance_applies(L) && w.batch == 1;
  // a large front of a population whose matrix came from the per-objective orders: its own orders are read off
  // those (finish.hpp); the three kernels and those below choose on the device which of them has work
  CrowdArgs a = crowd_args(w, list, use_orders, fused);
  if (without_runs) a.mid_sort = 0;
  if (use_orders)
    if (int e = stage_front_orders(w, list, a.mid_sort == 2 ? kMidArgsortRows : kRadixMinCandidates, s)) return e;
  if (a.mid_sort == 2)
    if (int e = launch_crowd_runs(w, a, tail_flag, s)) return e;
  const size_t lds = crowd_lds_bytes(L, fused);
  const void* const kernel = w.batch > 1 ? reinterpret_cast<const void*>(crowd_sort_kernel<true>) : reinterpret_cast<const void*>(crowd_sort_kernel<false>);
  if (int e = grant_dynamic_lds(kernel, lds)) return e;
  // (the fused path ends with a barrier between all blocks: the grid must be resident at once, which a grid of at
  // most two blocks of 256 threads per compute unit is)
  int grid = finish_grid(L, L.m);
  if (fused != 0 && grid > device_cus() * 2) grid = device_cus() * 2;
  grid = shared_grid(grid, device_cus() * 2, w.batch);
  if (w.batch > 1)
    hipLaunchKernelGGL(crowd_sort_kernel<true>, dim3(grid, 1, w.batch), dim3(kRadixThreads), lds, s, a, tail_flag);
  else
    hipLaunchKernelGGL(crowd_sort_kernel<false>, dim3(grid), dim3(kRadixThreads), lds, s, a, tail_flag);
  EVX_LAUNCH_CHECK();
  return 0;
}

// Crowding distances of those candidates and, with want_order, the selection order; gather, where it is given: the
// selected rows too, behind the order (crowd_mid_sort populations only).
static int stage_crowd_finish(const Ws& w, const int* list, bool want_order, int fused, hipStream_t s, bool after_peel_tail = false,
                              const GatherArgs* gather = nullptr, bool without_runs = false) {
  const Layout& L = w.L;
  const int tail_flag = after_peel_tail ? 1 : 0;
  CrowdArgs a = crowd_args(w, list, false, fused);
  if (without_runs && a.mid_sort == 2) a.mid_sort = 0;
  if (gather == nullptr && fused != 0 && crowd_always_small(w)) return 0;  // (nothing is left to do)
  if (crowd_mid_sort(L)) return launch_crowd_pick(w, a, want_order, gather, tail_flag, s);
  if (gather != nullptr) return kErrBadArg;
  if (a.mid_sort == 2)
    if (int e = launch_crowd_pick(w, a, want_order, nullptr, tail_flag, s)) return e;
  const size_t lds = crowd_lds_bytes(L, 0);
  const void* const kernel = w.batch > 1 ? reinterpret_cast<const void*>(crowd_finish_kernel<true>) : reinterpret_cast<const void*>(crowd_finish_kernel<false>);
  if (int e = grant_dynamic_lds(kernel, lds)) return e;
  const int grid = shared_grid(finish_grid(L, 1), device_cus() * 2, w.batch);
  const int order_flag = want_order ? 1 : 0;
  if (w.batch > 1)
    hipLaunchKernelGGL(crowd_finish_kernel<true>, dim3(grid, 1, w.batch), dim3(kRadixThreads), lds, s, a, order_flag, tail_flag);
  else
    hipLaunchKernelGGL(crowd_finish_kernel<false>, dim3(grid), dim3(kRadixThreads), lds, s, a, order_flag, tail_flag);
  EVX_LAUNCH_CHECK();
  return 0;
}

// The copy of a result of 4-byte elements out of the workspace, as the last kernel of an entry point: the result, or
// `poison` in every element when a device-side wait of the call ran out.
static int copy_out(const Ctrl* ctrl, void* dst, const void* src, int64_t n, uint32_t poison, hipStream_t s, int batch = 1,
                    int64_t ws_step = 0, int* call_err = nullptr) {
  int64_t blocks = (n + 1023) / 1024;
  if (blocks > 1024) blocks = 1024;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(copy_or_poison_kernel, dim3((unsigned)blocks, 1, batch), dim3(256), 0, s, ctrl, static_cast<const uint32_t*>(src),
                     static_cast<uint32_t*>(dst), n, poison, ws_step, call_err);
  EVX_LAUNCH_CHECK();
  return 0;
}
constexpr uint32_t kPoisonIndex = 0xFFFFFFFFu;  // -1 as a rank or an order
constexpr uint32_t kPoisonFloat = 0x7FC00000u;  // NaN as a distance

template <int M>
static int launch_batched_m(const BatchedArgs& a, int64_t batch, hipStream_t s) {
  const int nt = (int)round_up(a.n, 64);
  // (few populations of at most 256 rows: every workgroup has a compute unit, and every wave a SIMD, to itself -- 200 x 3:
  // the matrix in 7.5 instead of 12 us; with two waves to a SIMD the scalar loads win: 512 x 3 14 against 16.5 us)
  const bool stage = batch <= device_cus() && nt <= 256 && M <= 8 && opt().batched_stage;
  const size_t lds = batched_lds_bytes(nt, M) + (stage ? batched_stage_bytes(nt, M) : 0);
  // the attribute belongs to the (kernel, device) pair: remembered per device
  static size_t granted[64] = {0};
  static std::mutex mu;  // (a smaller grant by another thread must not follow a larger one)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
  if (lds > 48 * 1024) {
    std::lock_guard<std::mutex> lock(mu);
    if (dev < 0 || lds > granted[dev]) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(batched_kernel<M>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return (int)e;
      if (dev >= 0) granted[dev] = lds;
    }
  }
  // grid.x carries the batch; very large batches go in slices
  for (int64_t b0 = 0; b0 < batch; b0 += 0x40000000ll) {
    BatchedArgs part = a;
    part.stage_fitness = stage ? 1 : 0;
    const int64_t nb = batch - b0 < 0x40000000ll ? batch - b0 : 0x40000000ll;
    part.f += b0 * a.f_stride_b;
    if (part.rank_all) part.rank_all += b0 * a.n;
    if (part.x) part.x += b0 * a.x_stride_b;
    if (part.out_x) part.out_x += b0 * a.stop_count * a.x_row_bytes;
    if (part.out_f) part.out_f += b0 * a.stop_count * a.m;
    if (part.out_rank) part.out_rank += b0 * a.stop_count;
    if (part.out_dist) part.out_dist += b0 * a.stop_count;
    hipLaunchKernelGGL(batched_kernel<M>, dim3((unsigned)nb), dim3(nt), lds, s, part);
    EVX_LAUNCH_CHECK();
  }
  return 0;
}

// Two objectives: one workgroup per population without a matrix (two_small.hpp), for up to kTwoSmallRows rows.
static int launch_two_small(const BatchedArgs& a, int64_t batch, hipStream_t s) {
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(two_small_kernel), kTwoSmallLdsBytes)) return e;
  for (int64_t b0 = 0; b0 < batch; b0 += 0x40000000ll) {
    BatchedArgs part = a;
    const int64_t nb = batch - b0 < 0x40000000ll ? batch - b0 : 0x40000000ll;
    part.f += b0 * a.f_stride_b;
    if (part.rank_all) part.rank_all += b0 * a.n;
    if (part.x) part.x += b0 * a.x_stride_b;
    if (part.out_x) part.out_x += b0 * a.stop_count * a.x_row_bytes;
    if (part.out_f) part.out_f += b0 * a.stop_count * a.m;
    if (part.out_rank) part.out_rank += b0 * a.stop_count;
    if (part.out_dist) part.out_dist += b0 * a.stop_count;
    hipLaunchKernelGGL(two_small_kernel, dim3((unsigned)nb), dim3(kTwoSmallThreads), kTwoSmallLdsBytes, s, part);
    EVX_LAUNCH_CHECK();
  }
  return 0;
}

// Rows that the one-workgroup kernels take: the matrix kernel up to kBatchedMaxRows, two objectives up to kTwoSmallRows.
static int64_t batched_rows_limit(int64_t m) {
  if (m < 1 || m > kBatchedMaxObjectives) return 0;
  return m == 2 && opt().two_small_min_rows > 0 ? kTwoSmallRows : kBatchedMaxRows;
}

// Few populations of at most 256 rows and three to eight objectives: sixteen waves each (few.hpp).
template <int M>
static int launch_few_whole_m(const BatchedArgs& a, int batch, hipStream_t s) {
  const int groups = (a.n + 63) / 64;
  const int nt = groups * 2 * groups * 64 < kFewRows ? groups * 2 * groups * 64 : kFewRows;  // (a wave per group and half word)
  const size_t lds = few_whole_lds_bytes(nt, a.n, M);
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(few_whole_kernel<M>), lds)) return e;
  hipLaunchKernelGGL(few_whole_kernel<M>, dim3(batch), dim3(nt), lds, s, a);
  EVX_LAUNCH_CHECK();
  return 0;
}
static int launch_few_whole(const BatchedArgs& a, int batch, hipStream_t s) {
  switch (a.m) {
    case 3: return launch_few_whole_m<3>(a, batch, s);
    case 4: return launch_few_whole_m<4>(a, batch, s);
    case 5: return launch_few_whole_m<5>(a, batch, s);
    case 6: return launch_few_whole_m<6>(a, batch, s);
    case 7: return launch_few_whole_m<7>(a, batch, s);
    default: return launch_few_whole_m<8>(a, batch, s);
  }
}

// Populations of three to eight objectives: one workgroup each, dominators from the orders of the objectives (sets.hpp).
template <int M>
static int launch_sets_m(const BatchedArgs& a, int64_t batch, hipStream_t s) {
  const int rows = (int)round_up(a.n, 64);
  const bool narrow = rows <= kSetsNarrowRows;
  const size_t lds = sets_lds_bytes(rows, M);
  const void* const kernel = narrow ? reinterpret_cast<const void*>(sets_kernel<M, 8>) : reinterpret_cast<const void*>(sets_kernel<M, 16>);
  if (int e = grant_dynamic_lds(kernel, lds)) return e;
  for (int64_t b0 = 0; b0 < batch; b0 += 0x40000000ll) {
    BatchedArgs part = a;
    const int64_t nb = batch - b0 < 0x40000000ll ? batch - b0 : 0x40000000ll;
    part.f += b0 * a.f_stride_b;
    if (part.rank_all) part.rank_all += b0 * a.n;
    if (part.x) part.x += b0 * a.x_stride_b;
    if (part.out_x) part.out_x += b0 * a.stop_count * a.x_row_bytes;
    if (part.out_f) part.out_f += b0 * a.stop_count * a.m;
    if (part.out_rank) part.out_rank += b0 * a.stop_count;
    if (part.out_dist) part.out_dist += b0 * a.stop_count;
    if (narrow)
      hipLaunchKernelGGL((sets_kernel<M, 8>), dim3((unsigned)nb), dim3(rows), lds, s, part);
    else
      hipLaunchKernelGGL((sets_kernel<M, 16>), dim3((unsigned)nb), dim3(rows), lds, s, part);
    EVX_LAUNCH_CHECK();
  }
  return 0;
}
static int launch_sets(const BatchedArgs& a, int64_t batch, hipStream_t s) {
  switch (a.m) {
    case 3: return launch_sets_m<3>(a, batch, s);
    case 4: return launch_sets_m<4>(a, batch, s);
    case 5: return launch_sets_m<5>(a, batch, s);
    case 6: return launch_sets_m<6>(a, batch, s);
    case 7: return launch_sets_m<7>(a, batch, s);
    default: return launch_sets_m<8>(a, batch, s);
  }
}

static int launch_batched(const BatchedArgs& a, int64_t batch, hipStream_t s) {
  // (1024 populations, us, all pairs against the orders of the objectives: 256 x 3 uniform 27 / 27, values of four levels 28 / 33, 192 x 3
  // 20 to 23 / 23 and 21 / 39; from 257 rows on no slower on any data: 257 x 3 46 / 31 and 48 / 37, 512 x 3 64 / 41, 390 x 5 146 / 54, 390 x 8 210 / 87,
  // with four levels 123 / 124)
  if (a.m >= 3 && a.m <= kSetsObjectives && a.n >= opt().sets_min_rows && a.n <= kSetsRows) return launch_sets(a, batch, s);
  if (a.m >= 3 && a.m <= kFewObjectives && a.n <= kFewWholeRows && batch <= device_cus() && opt().few_max_rows > 0)
    return launch_few_whole(a, (int)batch, s);
  if (a.m == 2 && opt().two_small_min_rows > 0 && (a.n >= opt().two_small_min_rows || a.n > kBatchedMaxRows))
    return launch_two_small(a, batch, s);
  switch (a.m) {
    case 1: return launch_batched_m<1>(a, batch, s);
    case 2: return launch_batched_m<2>(a, batch, s);
    case 3: return launch_batched_m<3>(a, batch, s);
    case 4: return launch_batched_m<4>(a, batch, s);
    case 5: return launch_batched_m<5>(a, batch, s);
    case 6: return launch_batched_m<6>(a, batch, s);
    case 7: return launch_batched_m<7>(a, batch, s);
    case 8: return launch_batched_m<8>(a, batch, s);
    case 9: return launch_batched_m<9>(a, batch, s);
    case 10: return launch_batched_m<10>(a, batch, s);
    case 11: return launch_batched_m<11>(a, batch, s);
    case 12: return launch_batched_m<12>(a, batch, s);
    case 13: return launch_batched_m<13>(a, batch, s);
    case 14: return launch_batched_m<14>(a, batch, s);
    case 15: return launch_batched_m<15>(a, batch, s);
    case 16: return launch_batched_m<16>(a, batch, s);
    default: return kErrBadArg;
  }
}

}  // namespace evx

using namespace evx;

// Populations that share those launches at most.  From 32 on the entry points without a workspace are the faster ones (64 x (300 x 3) 17 us
// against 33; the Python side goes by that), but a caller who is here would get the pipeline instead.
constexpr int kFewBatch = 64;
static bool few_applies(const Layout& L, const Fitness& fit, int batch);
static int stage_few(const Ws& w, const Fitness& fit, BatchedArgs a, hipStream_t s);
static bool two_applies(const Layout& L, int64_t stop_count);
static int many_two_share(const Layout& L, int64_t batch, int64_t stop_count);
static int stage_rank_two(const Ws& w, const Fitness& src, int64_t stop_count, bool fill_dist, int* rank_until, hipStream_t s);

extern "C" {

int evox_hip_abi_version(void) { return EVOX_HIP_ABI_VERSION; }

size_t evox_hip_workspace_bytes(int64_t n, int64_t m) {
  Layout L;
  return make_layout(n, m, &L) ? L.total : 0;
}

int evox_hip_workspace_layout(int64_t n, int64_t m, int64_t* out) {
  Layout L;
  if (out == nullptr || !make_layout(n, m, &L)) return kErrBadArg;
  out[0] = (int64_t)L.dom;
  out[1] = L.wstride;
  out[2] = L.nwords;
  out[3] = (int64_t)L.count;
  out[4] = (int64_t)L.rank;
  out[5] = (int64_t)L.dist;
  out[6] = (int64_t)L.perm;
  out[7] = (int64_t)L.fstart;
  out[8] = (int64_t)L.order;
  out[9] = (int64_t)L.ctrl;
  out[10] = (int64_t)L.orig_of;
  return 0;
}

int evox_hip_slot_sort_layout(int64_t n, int64_t m, int64_t* out) {
  Layout L;
  if (out == nullptr || !make_layout(n, m, &L)) return kErrBadArg;
  out[0] = (int64_t)L.key_sorted;
  out[1] = (int64_t)L.kid_sorted;
  out[2] = (int64_t)L.xs_sorted;
  out[3] = (int64_t)L.xs;
  out[4] = L.npad;
  out[5] = (int64_t)L.slot_of;
  return 0;
}

static int set_named(Options& o, const char* name, int64_t value) {
  if (name == nullptr) return kErrBadArg;
  if (!strcmp(name, "peel_blocks_per_cu") && value >= 1 && value <= 16) {
    o.peel_blocks_per_cu = (int)value;
  } else if (!strcmp(name, "peel_witness") && (value == 0 || value == 1)) {
    o.peel_witness = (int)value;
  } else if (!strcmp(name, "peel_record_blocks") && (value == 0 || (value >= 16 && value <= 255))) {
    o.peel_record_blocks = (int)value;
  } else if (!strcmp(name, "peel_records") && (value == 0 || value == 1)) {
    o.peel_records = (int)value;
  } else if (!strcmp(name, "peel_lds") && (value == 0 || value == 1)) {
    o.peel_lds = (int)value;
  } else if (!strcmp(name, "tail_merged") && (value == 0 || value == 1)) {
    o.tail_merged = (int)value;
  } else if (!strcmp(name, "launch_memory") && (value == 0 || value == 1)) {
    o.launch_memory = (int)value;
  } else if (!strcmp(name, "peel_stepped") && (value == 0 || value == 1)) {
    o.peel_stepped = (int)value;
  } else if (!strcmp(name, "few_max_rows") && value >= 0 && value <= kFewRows) {
    o.few_max_rows = value;
  } else if (!strcmp(name, "sets_min_rows") && value >= 1) {
    o.sets_min_rows = value;
  } else if (!strcmp(name, "two_small_min_rows") && value >= 0) {
    o.two_small_min_rows = value;
  } else if (!strcmp(name, "two_min_rows") && value >= 0) {
    o.two_min_rows = value;
    if (value < o.two_min_rows_partial) o.two_min_rows_partial = value;  // (a lower limit asked for counts for both)
  } else if (!strcmp(name, "two_min_rows_partial") && value >= 0) {
    o.two_min_rows_partial = value;
  } else if (!strcmp(name, "peel_tail") && (value == 0 || value == 1)) {
    o.peel_tail = (int)value;
  } else if (!strcmp(name, "peel_lds_blocks") && (value == 0 || (value >= 8 && value <= 255))) {
    o.peel_lds_blocks = (int)value;
  } else if (!strcmp(name, "spin_limit") && value >= 1 && value <= 0x7FFFFFFFll) {
    o.spin_limit = (unsigned)value;
  } else if (!strcmp(name, "dominance_tile_words") && (value == 0 || value == 2 || value == 4 || value == 8 || value == 16)) {
    o.dominance_tile_words = (int)value;
  } else if (!strcmp(name, "dominance_folded") && (value == 0 || value == 1)) {
    o.dominance_folded = (int)value;
  } else if (!strcmp(name, "small_sort") && (value == 0 || value == 1)) {
    o.small_sort = (int)value;
  } else if (!strcmp(name, "mid_argsort") && (value == 0 || value == 1)) {
    o.mid_argsort = (int)value;
  } else if (!strcmp(name, "prefix_min_rows") && value >= 0) {
    o.prefix_min_rows = value;
  } else if (!strcmp(name, "prefix_double_tile") && value >= 0) {
    o.prefix_double_tile = value;
  } else if (!strcmp(name, "prefix_mode") && value >= 1 && value <= 3) {
    o.prefix_mode = (int)value;
  } else if (!strcmp(name, "prefix_bands") && (value == 0 || value == 1)) {
    o.prefix_bands = (int)value;
  } else if (!strcmp(name, "batched_stage") && (value == 0 || value == 1)) {
    o.batched_stage = (int)value;
  } else if (!strcmp(name, "order_stream") && (value == 0 || value == 1)) {
    o.order_stream = (int)value;
  } else if (!strcmp(name, "order_stream_capacity") && value >= 1 && value <= kOrderStreamCapacity) {
    o.order_stream_capacity = (int)value;
  } else if (!strcmp(name, "prefix_count_first") && value >= 0 && value <= 2) {
    o.prefix_count_first = (int)value;
  } else if (!strcmp(name, "prefix_nearby") && value >= 0) {
    o.prefix_nearby = value;
  } else {
    return kErrBadArg;
  }
  return 0;
}

int evox_hip_set_option(const char* name, int64_t value) { return set_named(g_opt, name, value); }

struct evox_hip_options {
  evx::Options values;
};

evox_hip_options* evox_hip_options_create(void) {
  evox_hip_options* h = new (std::nothrow) evox_hip_options;
  if (h != nullptr) h->values = g_opt;
  return h;
}

void evox_hip_options_destroy(evox_hip_options* options) {
  if (options != nullptr && t_opt == &options->values) t_opt = nullptr;
  delete options;
}

int evox_hip_options_set(evox_hip_options* options, const char* name, int64_t value) {
  return options == nullptr ? kErrBadArg : set_named(options->values, name, value);
}

int evox_hip_options_use(const evox_hip_options* options) {
  t_opt = options == nullptr ? nullptr : &options->values;
  return 0;
}

int evox_hip_stage_prepare(const float* f, int64_t n, int64_t m, int64_t sr, int64_t sc, void* ws, size_t ws_bytes,
                           void* stream) {
  Ws w;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  return stage_prepare(w, one_part(f, n, sr, sc), true, (hipStream_t)stream);
}

int evox_hip_stage_dominance(int64_t n, int64_t m, int variant, void* ws, size_t ws_bytes, void* stream) {
  Ws w;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  return stage_dominance(w, variant, (hipStream_t)stream);
}

int evox_hip_stage_count(int64_t n, int64_t m, void* ws, size_t ws_bytes, void* stream) {
  Ws w;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  // as a stage of its own it may be repeated on one dominance matrix: start from a clean state
  const int64_t zero_words = (int64_t)((w.L.zero_end - w.L.ctrl) / 4);
  int blocks = (int)((zero_words + 255) / 256);
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(reset_state_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, w.at<uint32_t>(w.L.ctrl), zero_words);
  EVX_LAUNCH_CHECK();
  return stage_count(w, true, (hipStream_t)stream);
}

int evox_hip_stage_peel(int64_t n, int64_t m, int64_t stop_count, int32_t* rank_out, void* ws, size_t ws_bytes,
                        void* stream) {
  Ws w;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  // (the kernel that peels from LDS counts for itself; after stage_count it finds the same front 0 again.  As in the
  // selection it also orders a small last front: that part reads memory which stage_prepare clears, so a timing
  // of it repeats the stages from stage_prepare on)
  size_t lds = 0;
  if (const int sweepers = lds_peel_plan(w.L, &lds)) {
    if (int e = launch_lds_peel(w, stop_count, true, true, sweepers, lds, (hipStream_t)stream, true)) return e;
  } else if (int e = stage_peel(w, stop_count, true, (hipStream_t)stream)) {
    return e;
  }
  if (rank_out) return copy_out(w.ctrl(), rank_out, w.at<int>(w.L.rank), n, kPoisonIndex, (hipStream_t)stream);
  return 0;
}

int evox_hip_stage_crowding(int64_t n, int64_t m, void* ws, size_t ws_bytes, void* stream) {
  Ws w;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  if (int e = stage_crowd_sort(w, w.at<int>(w.L.perm), true, 0, (hipStream_t)stream)) return e;
  return stage_crowd_finish(w, w.at<int>(w.L.perm), false, 0, (hipStream_t)stream);
}

int evox_hip_stage_order(int64_t n, int64_t m, void* ws, size_t ws_bytes, void* stream) {
  Ws w;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  return stage_crowd_finish(w, w.at<int>(w.L.perm), true, 0, (hipStream_t)stream);
}

}  // extern "C"

// batch > 1: that many populations of one shape in the same launches (see select_rows); their ranks lie n elements apart.
static int rank_rows(const Fitness& fit, int64_t n, int64_t m, int64_t stop_count, int32_t* rank_out, void* ws, size_t ws_bytes,
                     hipStream_t s, int batch = 1, int64_t ws_step = 0) {
  Ws w;
  if (rank_out == nullptr || stop_count < 1 || stop_count > n) return kErrBadArg;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  if (batch > 1) {
    if (ws_step < (int64_t)w.L.total || (ws_step & 255) != 0 || ws_bytes < (size_t)ws_step * (size_t)batch) return kErrWorkspace;
    w.batch = batch;
    w.step = ws_step;
  }
  if (few_applies(w.L, fit, batch)) {
    BatchedArgs a = {};
    a.stop_count = (int)stop_count;
    a.rank_all = rank_out;
    return stage_few(w, fit, a, s);
  }
  if (batch == 1 ? two_applies(w.L, stop_count) : many_two_share(w.L, batch, stop_count) >= batch) {
    int* until = stop_count < n ? w.at<int>(w.L.order) : (int*)nullptr;
    const int e = stage_rank_two(w, fit, stop_count, false, until, s);
    if (e != kErrNotResident || batch > 1) {
      if (e) return e == kErrNotResident ? kErrBadArg : e;
      return copy_out(w.ctrl(), rank_out, until != nullptr ? until : w.at<int>(w.L.rank), n, kPoisonIndex, s, w.batch, w.step);
    }
  }
  if (int e = stage_prepare(w, fit, true, s)) return e;
  if (int e = stage_dominance(w, kDomAuto, s)) return e;
  if (batch > 1) {
    if (int e = count_and_peel_persistent(w, stop_count, false, false, s, false, nullptr, nullptr)) return e == kErrNotResident ? kErrBadArg : e;
  } else if (int e = count_and_peel(w, stop_count, false, false, s)) {
    return e;
  }
  return copy_out(w.ctrl(), rank_out, w.at<int>(w.L.rank), n, kPoisonIndex, s, w.batch, w.step);
}

extern "C" {

int evox_hip_non_dominate_rank_until(const float* f, int64_t n, int64_t m, int64_t sr, int64_t sc, int64_t stop_count,
                                     int32_t* rank_out, void* ws, size_t ws_bytes, void* stream) {
  return rank_rows(one_part(f, n, sr, sc), n, m, stop_count, rank_out, ws, ws_bytes, (hipStream_t)stream);
}

int evox_hip_non_dominate_rank(const float* f, int64_t n, int64_t m, int64_t sr, int64_t sc, int32_t* rank_out, void* ws,
                               size_t ws_bytes, void* stream) {
  return evox_hip_non_dominate_rank_until(f, n, m, sr, sc, n, rank_out, ws, ws_bytes, stream);
}

size_t evox_hip_first_front_workspace_bytes(int64_t n, int64_t m) {
  Layout L;
  return make_layout(n, m, &L) ? L.dom : 0;
}

}  // extern "C"

// The rows xs[k][.] of which *count are left, if more than `least`, into spatial order: xs_sorted, slot_row, slot_end and the
// boxes.  The histogram and the flags of its scan must be zero; counted: it holds the buckets' sizes already, and the rows'
// buckets are known.
static int spatial_bucket_bits(const Layout& L) {
  int bits = 10;
  while ((1 << bits) < L.buckets) ++bits;
  return bits;
}
template <int M>
static int stage_spatial_order(const Ws& w, const float* xs, float* xs_sorted, const int* count, int least, bool counted, hipStream_t s) {
  const Layout& L = w.L;
  int* const bucket = w.at<int>(L.members);
  int* const slot_row = w.at<int>(L.orig_of);
  int* const slot_end = w.at<int>(L.kid_sorted);
  int blocks = (L.npad + 255) / 256;
  if (blocks > 2048) blocks = 2048;
  if (!counted) {
    hipLaunchKernelGGL(spatial_bucket_kernel<M>, dim3(blocks < 1024 ? blocks : 1024, 1, w.batch), dim3(256), 0, s, xs, L.npad, count,
                       least, spatial_bucket_bits(L), bucket, w.at<int>(L.hist), w.step);
    EVX_LAUNCH_CHECK();
  }
  auto launch_scan = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(L.buckets / 1024, 1, w.batch), dim3(256), 0, s, w.at<int>(L.hist), L.buckets, w.at<int>(L.bstart),
                       w.at<int>(L.bcursor), w.at<unsigned long long>(L.scanflags), w.ctrl(), w.step);
  };
  w.batch > 1 ? launch_scan(bucket_scan_kernel<true>) : launch_scan(bucket_scan_kernel<false>);
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(spatial_scatter_kernel<M>, dim3(blocks, 1, w.batch), dim3(256), 0, s, xs, L.npad, count, least, bucket,
                     w.at<int>(L.bstart), w.at<int>(L.bcursor), xs_sorted, slot_row, slot_end, w.ctrl(), w.step);
  EVX_LAUNCH_CHECK();
  const int64_t leaf_stride = spatial_leaf_stride(L.n), group_stride = spatial_group_stride(L.n);
  hipLaunchKernelGGL(leaf_box_kernel, dim3((unsigned)(leaf_stride / kGroupLeaves), 1, w.batch), dim3(kBoxThreads), 0, s, xs_sorted,
                     count, least, L.npad, L.m, leaf_stride, group_stride, w.at<float>(L.leaf_lo), w.at<float>(L.leaf_hi),
                     w.at<float>(L.group_lo), w.ctrl(), w.step);
  EVX_LAUNCH_CHECK();
  return 0;
}

// Whether front_small_kernel takes a population, or `batch` of them.  One population around a sphere, it / the steps, us a call:
// 4096 x 3 13 / 21, 6000 x 3 17 / 21, 4096 x 5 18 / 27, 1000 x 8 15 / 19, 2000 x 8 24 / 19, 512 x 12 13 / 20, 1000 x 12 22 / 22,
// 512 x 16 20 / 25, 1000 x 16 34 / 29.  Where the workgroups no longer fit the device at once (two on a compute unit) the pairs
// are paid in full: 256 x 700 x 3 25 / 44, 1000 x 3 57 / 50; 256 x 700 x 8 96 / 140, 1000 x 8 147 / 116; 64 x 2000 x 2 36 / 26.
static bool front_small_fits(int n, int m, int batch) {
  if (n > 4096 || (int64_t)n * m > (m <= 8 ? 12288 : 8192)) return false;
  return n <= 768 || (int64_t)batch * ((n + 63) / 64) <= 2 * device_cus();
}

// The first front of up to kSpatialObjectives objectives (spatial.hpp).
template <int M>
static int first_front_steps(const Ws& w, const Fitness& fit, uint8_t* mask, hipStream_t s) {
  const Layout& L = w.L;
  if (front_small_fits(L.n, M, w.batch)) {
    const int tiles = (L.n + 63) / 64, waves = tiles < front_small_waves(M) ? tiles : front_small_waves(M);
    hipLaunchKernelGGL(front_small_kernel<M>, dim3((unsigned)tiles, 1, w.batch), dim3(64 * waves), 0, s, fit.f, fit.sr, fit.sc, fit.step,
                       L.n, mask, w.ctrl(), w.step);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  // The rows step 1 leaves stand in xs_sorted, those between the passes of step 2 in xs, those it leaves in xs_sorted again,
  // and the spatial order goes to xs.
  constexpr bool kGrid = M == 2 || M == 3;
  const bool grid_step = kGrid && L.n > kFrontGridPopulation;
  const bool order_step = L.n > kFrontPairsRows;
  FrontCount* const count = w.at<FrontCount>(L.fstart);
  const int* const counted = grid_step ? &count->rows_grid : &count->rows;
  float* const left = w.at<float>(L.xs_sorted);
  int* const left_of = w.at<int>(L.order);
  float* const to = grid_step ? w.at<float>(L.xs) : nullptr;
  int* const to_of = grid_step ? w.at<int>(L.perm) : nullptr;
  // (the cells before and after the prefix passes, where the radix sort's pairs go)
  uint32_t* const cells = grid_step ? w.at<uint32_t>(L.rpairs0) : nullptr;
  uint32_t* const turned = grid_step ? w.at<uint32_t>(L.rpairs1) : nullptr;
  const bool small_grid = M == 3 && L.n <= kFrontGridSmallRows;
  const int cell_bits = small_grid ? 7 : 8;
  const int grid_cells = !grid_step ? 0 : (M == 2 ? 1 << cell_bits : 1 << (2 * cell_bits));
  // (A cell to every 64 bytes, where they fit; side by side where one workgroup reads them all, which from 16 384 lines of
  // memory costs more than the minima save: 100 000 x 3 around a sphere took 112 us.)
  int spread = small_grid ? 0 : 4;
  while (spread > 0 && sizeof(uint32_t) * ((size_t)grid_cells << spread) > sizeof(unsigned long long) * (size_t)L.m * (size_t)L.kstride) --spread;
  // The rows of low sums cost a pass over the rows (and a launch that is needed anyway).  Without them, a population that a
  // few rows dominate which no sample holds goes on whole: pairs of up to 65 536 rows of four objectives take some 35 us then,
  // of 60 000 x 6 315, and 200 000 x 4 took 145 us where the rows of low sums leave 36.  (An entry per stretch of 256 rows or
  // more fits the 4 bytes that each of them has there.)
  const bool with_lowest = M > 4 || order_step;
  unsigned long long* const lowest = with_lowest ? w.at<unsigned long long>(L.witness) : nullptr;
  if (with_lowest) {
    const int stretches = (L.n + front_stretch_rows(L.n) - 1) / front_stretch_rows(L.n);
    hipLaunchKernelGGL(front_lowest_kernel<M>, dim3((unsigned)stretches, 1, w.batch), dim3(256), 0, s, fit.f, fit.sr, fit.sc, fit.step,
                       L.n, lowest, w.ctrl(), count, w.step);
  } else {
    hipLaunchKernelGGL(front_reset_kernel, dim3(1, 1, w.batch), dim3(256), 0, s, w.ctrl(), count, w.step);
  }
  EVX_LAUNCH_CHECK();
  // (fewer rows per thread as long as every workgroup, which finds the champions first, has a compute unit of its own)
  int blocks = (L.n + 256 * kFrontRowsPerThread - 1) / (256 * kFrontRowsPerThread);
  if (blocks > 1024) blocks = 1024;
  int per = kFrontRowsPerThread;
  while (per > 1 && (int64_t)w.batch * ((L.n + 128 * per - 1) / (128 * per)) <= device_cus()) per /= 2;
  const int filter_blocks = per < kFrontRowsPerThread ? (L.n + 256 * per - 1) / (256 * per) : blocks;
  hipLaunchKernelGGL(front_filter_kernel<M>, dim3(filter_blocks, 1, w.batch), dim3(256), 0, s, fit.f, fit.sr, fit.sc, fit.step, L.n, L.npad, per,
                     lowest, left, left_of, mask, count, cells, grid_cells << spread, w.at<uint32_t>(L.hist),
                     order_step ? (int)((L.tailbuf - L.hist) / 4) : 0, w.step);
  EVX_LAUNCH_CHECK();
  if constexpr (kGrid) {
    if (grid_step) {
      // (as many rows to a workgroup, up to four per thread, as leave every compute unit one: a workgroup drops what its own
      // rows dominate, 44 % of 1024 rows around a sphere and 58 % of 4096)
      uint32_t* const tables = w.at<uint32_t>(L.key);
      int grid_per = (int)(((int64_t)L.n * w.batch + (int64_t)kFrontGridBlock * device_cus() - 1) / ((int64_t)kFrontGridBlock * device_cus()));
      if (grid_per > kFrontRowsPerThread) grid_per = kFrontRowsPerThread;
      const int build_blocks = (L.n + kFrontGridBlock * grid_per - 1) / (kFrontGridBlock * grid_per);
      hipLaunchKernelGGL(front_grid_kernel<M>, dim3(build_blocks, 1, w.batch), dim3(kFrontGridBlock), 0, s, left, left_of, L.npad, grid_per,
                         cell_bits, count, to, to_of, mask, L.n, tables, cells, spread, w.step);
      EVX_LAUNCH_CHECK();
      const uint32_t* below = turned;
      if (small_grid) {
        if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(front_grid_small_kernel), kFrontGridLds)) return e;
        hipLaunchKernelGGL(front_grid_small_kernel, dim3(1, 1, w.batch), dim3(kFrontGridThreads), kFrontGridLds, s, cells, turned, count,
                           w.step);
        EVX_LAUNCH_CHECK();
      } else {
        hipLaunchKernelGGL(front_grid_prefix_kernel, dim3(M == 2 ? 1 : kFrontGrid, 1, w.batch), dim3(kFrontGrid), 0, s, cells, spread, turned,
                           M == 2 ? 1 : kFrontGrid, count, w.step);
        EVX_LAUNCH_CHECK();
        if (M == 3) {
          below = cells;
          hipLaunchKernelGGL(front_grid_prefix_kernel, dim3(kFrontGrid, 1, w.batch), dim3(kFrontGrid), 0, s, turned, 0, cells, kFrontGrid,
                             count, w.step);
          EVX_LAUNCH_CHECK();
        }
      }
      hipLaunchKernelGGL(front_grid_filter_kernel<M>, dim3(blocks, 1, w.batch), dim3(256), 0, s, to, to_of, L.npad, cell_bits, count,
                         tables, below, left, left_of, mask, L.n, spatial_bucket_bits(L), w.at<int>(L.members),
                         order_step ? w.at<int>(L.hist) : (int*)nullptr, w.step);
      EVX_LAUNCH_CHECK();
    }
  }
  const int pair_rows = L.n < kFrontPairsRows ? L.n : kFrontPairsRows;
  const int pair_parts = (pair_rows + 63) / 64 < kFrontPairsParts ? (pair_rows + 63) / 64 : kFrontPairsParts;  // (a part has 64 rows or more)
  hipLaunchKernelGGL(front_pairs_kernel<M>, dim3((pair_rows + 255) / 256, pair_parts, w.batch), dim3(256), 0, s, left, left_of,
                     L.npad, mask, L.n, count, grid_step ? 1 : 0, w.step);
  EVX_LAUNCH_CHECK();
  if (!order_step) return 0;
  float* const sorted = w.at<float>(L.xs);
  if (int e = stage_spatial_order<M>(w, left, sorted, counted, kFrontPairsRows, grid_step, s)) return e;
  hipLaunchKernelGGL((first_front_leaf_kernel<M>), dim3((unsigned)spatial_leaves(L.n), 1, w.batch), dim3(64 * kFrontWaves), 0, s,
                     sorted, w.at<int>(L.orig_of), w.at<int>(L.kid_sorted), left_of, count, counted, L.npad,
                     spatial_leaf_stride(L.n), spatial_group_stride(L.n), w.at<float>(L.leaf_lo), w.at<float>(L.leaf_hi),
                     w.at<float>(L.group_lo), mask, L.n, w.ctrl(), w.step);
  EVX_LAUNCH_CHECK();
  return 0;
}

// batch > 1: that many populations of one shape in the same launches, their workspaces (without the matrix) ws_step
// bytes apart, their masks n bytes.
static int first_front_rows(const Fitness& fit, int64_t n, int64_t m, uint8_t* mask_out, void* ws, size_t ws_bytes, hipStream_t s,
                            int batch = 1, int64_t ws_step = 0) {
  Ws w;
  if (mask_out == nullptr) return kErrBadArg;
  if (int e = open_ws(n, m, ws, ws_bytes, &w, false)) return e;
  const Layout& L = w.L;
  if (batch > 1) {
    if (ws_step < (int64_t)L.dom || (ws_step & 255) != 0 || ws_bytes < (size_t)ws_step * (size_t)batch) return kErrWorkspace;
    w.batch = batch;
    w.step = ws_step;
  }
  if (fit.f == nullptr) return kErrBadArg;
  switch (L.m) {
    case 1: return first_front_steps<1>(w, fit, mask_out, s);
    case 2: return first_front_steps<2>(w, fit, mask_out, s);
    case 3: return first_front_steps<3>(w, fit, mask_out, s);
    case 4: return first_front_steps<4>(w, fit, mask_out, s);
    case 5: return first_front_steps<5>(w, fit, mask_out, s);
    case 6: return first_front_steps<6>(w, fit, mask_out, s);
    case 7: return first_front_steps<7>(w, fit, mask_out, s);
    case 8: return first_front_steps<8>(w, fit, mask_out, s);
    case 9: return first_front_steps<9>(w, fit, mask_out, s);
    case 10: return first_front_steps<10>(w, fit, mask_out, s);
    case 11: return first_front_steps<11>(w, fit, mask_out, s);
    case 12: return first_front_steps<12>(w, fit, mask_out, s);
    case 13: return first_front_steps<13>(w, fit, mask_out, s);
    case 14: return first_front_steps<14>(w, fit, mask_out, s);
    case 15: return first_front_steps<15>(w, fit, mask_out, s);
    case 16: return first_front_steps<16>(w, fit, mask_out, s);
    default:
      if (int e = stage_prepare(w, fit, true, s)) return e;
      hipLaunchKernelGGL(first_front_any_m_kernel, dim3((L.n + 255) / 256, 1, w.batch), dim3(256), 0, s, w.at<float>(L.xs_sorted),
                         w.at<uint32_t>(L.kid_sorted), w.at<int>(L.orig_of), L.n, L.npad, L.m, mask_out, w.ctrl(), w.step);
  }
  EVX_LAUNCH_CHECK();
  return 0;
}

// batch > 1: as above; the masks lie mask_step bytes apart, the distances n elements.
static int crowding_rows(const Fitness& costs, int64_t n, int64_t m, const uint8_t* mask, int64_t mask_stride, int64_t mask_step,
                         float* dist_out, void* ws, size_t ws_bytes, hipStream_t s, int batch = 1, int64_t ws_step = 0) {
  Ws w;
  if (costs.f == nullptr || dist_out == nullptr) return kErrBadArg;
  if (int e = open_ws(n, m, ws, ws_bytes, &w, batch == 1)) return e;
  const Layout& L = w.L;
  if (batch > 1) {
    if (ws_step < (int64_t)L.dom || (ws_step & 255) != 0 || ws_bytes < (size_t)ws_step * (size_t)batch) return kErrWorkspace;
    w.batch = batch;
    w.step = ws_step;
  }
  if (int e = stage_prepare(w, costs, false, s)) return e;
  hipLaunchKernelGGL(compact_mask_kernel, dim3(1, 1, w.batch), dim3(1024), 0, s, mask, mask_stride, L.n, w.at<int>(L.perm),
                     w.at<float>(L.dist), w.ctrl(), mask_step, w.step);
  EVX_LAUNCH_CHECK();
  if (int e = stage_crowd_sort(w, w.at<int>(L.perm), false, 1, s)) return e;
  if (int e = stage_crowd_finish(w, w.at<int>(L.perm), false, 1, s)) return e;
  return copy_out(w.ctrl(), dist_out, w.at<float>(L.dist), n, kPoisonFloat, s, w.batch, w.step);
}

// Populations that share the launches of a first-front mask or of the crowding distances: their kernels need no
// matrix, so a copy of the workspace is small; as many as 1 GiB of workspace holds (for the crowding distances:
// and as the kernels that order a front, whose workgroups wait for each other, can be resident together).
static int many_small_share(const Layout& L, int64_t batch, bool crowding) {
  if (batch < 2) return 1;
  if (crowding && (L.n > kMidArgsortRows || (!opt().mid_argsort && L.n > kRadixMinCandidates))) return 1;
  int64_t share = (int64_t)(1ull << 30) / (int64_t)align_up(L.dom);
  if (crowding && share > device_cus() / 2) share = device_cus() / 2;
  if (share > 32768) share = 32768;
  if (share > batch) share = batch;
  if (share < 2) return 1;
  const int64_t passes = (batch + share - 1) / share;
  return (int)((batch + passes - 1) / passes);
}

extern "C" {

int evox_hip_first_front_mask(const float* f, int64_t n, int64_t m, int64_t sr, int64_t sc, uint8_t* mask_out, void* ws,
                              size_t ws_bytes, void* stream) {
  return first_front_rows(one_part(f, n, sr, sc), n, m, mask_out, ws, ws_bytes, (hipStream_t)stream);
}

size_t evox_hip_many_first_front_workspace_bytes(int64_t batch, int64_t n, int64_t m) {
  Layout L;
  if (batch < 1 || !make_layout(n, m, &L)) return 0;
  return align_up(L.dom) * (size_t)many_small_share(L, batch, false);
}

int evox_hip_many_first_front_mask(const float* f, int64_t batch, int64_t n, int64_t m, int64_t stride_batch, int64_t sr, int64_t sc,
                                   uint8_t* mask_out, void* ws, size_t ws_bytes, void* stream) {
  Layout L;
  if (f == nullptr || mask_out == nullptr || batch < 1 || !make_layout(n, m, &L)) return kErrBadArg;
  const int share = many_small_share(L, batch, false);
  for (int64_t b0 = 0; b0 < batch;) {
    const int64_t left = batch - b0;
    const int count = (int)(left < share ? left : share);
    if (int e = first_front_rows(one_part(f + b0 * stride_batch, n, sr, sc, stride_batch), n, m, mask_out + b0 * n, ws, ws_bytes,
                                 (hipStream_t)stream, count, count > 1 ? (int64_t)align_up(L.dom) : 0))
      return e;
    b0 += count;
  }
  return 0;
}

size_t evox_hip_many_crowding_workspace_bytes(int64_t batch, int64_t n, int64_t m) {
  Layout L;
  if (batch < 1 || !make_layout(n, m, &L)) return 0;
  const int share = many_small_share(L, batch, true);
  return share > 1 ? align_up(L.dom) * (size_t)share : L.total;
}

int evox_hip_many_crowding_distance(const float* costs, int64_t batch, int64_t n, int64_t m, int64_t stride_batch, int64_t sr,
                                    int64_t sc, const uint8_t* mask, int64_t mask_batch_stride, int64_t mask_stride, float* dist_out,
                                    void* ws, size_t ws_bytes, void* stream) {
  Layout L;
  if (costs == nullptr || dist_out == nullptr || batch < 1 || !make_layout(n, m, &L)) return kErrBadArg;
  const int share = many_small_share(L, batch, true);
  for (int64_t b0 = 0; b0 < batch;) {
    const int64_t left = batch - b0;
    const int count = (int)(left < share ? left : share);
    if (int e = crowding_rows(one_part(costs + b0 * stride_batch, n, sr, sc, stride_batch), n, m,
                              mask != nullptr ? mask + b0 * mask_batch_stride : nullptr, mask_stride, mask_batch_stride,
                              dist_out + b0 * n, ws, ws_bytes, (hipStream_t)stream, count, count > 1 ? (int64_t)align_up(L.dom) : 0))
      return e;
    b0 += count;
  }
  return 0;
}

int evox_hip_crowding_distance(const float* costs, int64_t n, int64_t m, int64_t sr, int64_t sc, const uint8_t* mask,
                               int64_t mask_stride, float* dist_out, void* ws, size_t ws_bytes, void* stream) {
  if (costs == nullptr) return kErrBadArg;
  return crowding_rows(one_part(costs, n, sr, sc), n, m, mask, mask_stride, 0, dist_out, ws, ws_bytes, (hipStream_t)stream);
}

}  // extern "C"

// Workspace of the standalone stable argsort: control block with barrier slots, two pair buffers, the
// per-block digit table and the digit totals.
struct SortLayout {
  int n, kstride, workers;
  size_t ctrl, pairs0, pairs1, table, totals, total;
};

static bool make_sort_layout(int64_t n, SortLayout* L) {
  if (n < 1 || n > 0x7FFFFF00ll) return false;
  L->n = (int)n;
  L->kstride = (int)round_up(n, 64);
  int workers = (int)((n + 1023) / 1024);
  if (workers > kRadixMaxWorkers) workers = kRadixMaxWorkers;
  L->workers = workers;
  size_t o = 0;
  L->ctrl = o;    o = align_up(o + sizeof(Ctrl) + sizeof(unsigned long long) * kMaxGrid);
  L->pairs0 = o;  o = align_up(o + sizeof(unsigned long long) * (size_t)L->kstride);
  L->pairs1 = o;  o = align_up(o + sizeof(unsigned long long) * (size_t)L->kstride);
  L->table = o;   o = align_up(o + sizeof(int) * 256 * (size_t)kRadixMaxWorkers);
  L->totals = o;  o = align_up(o + sizeof(int) * 256);
  L->total = o;
  return true;
}

// key_cap: see argsort_step_kernel (device memory or null; only the sort of more than kMidArgsortRows keys looks at it).
// call_err: the error word of the call that this step is a part of (or null).  The sort waits on a control block of its own:
// without that word, kernels that go by the call's would follow an order of -1.
static int argsort_step(const void* key, int kind, int64_t stride, int64_t n, const int32_t* prev_order, int32_t* order_out,
                        void* ws, size_t ws_bytes, void* stream, const int* key_cap = nullptr, int* call_err = nullptr) {
  SortLayout L;
  if (key == nullptr || order_out == nullptr || kind < 0 || kind > 2) return kErrBadArg;
  if (!make_sort_layout(n, &L)) return kErrBadArg;
  if (ws == nullptr || ws_bytes < L.total || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  hipStream_t s = (hipStream_t)stream;
  if (n <= kSmallArgsortRows) {
    const int npad = ((int)n + 127) & ~127;
    if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(small_argsort_kernel), sizeof(double) * (size_t)npad)) return e;
    hipLaunchKernelGGL(small_argsort_kernel, dim3(npad / kSmallArgsortGroup), dim3(kSmallArgsortThreads),
                       sizeof(double) * (size_t)npad, s, key, kind, stride, (int)n, prev_order, order_out);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  if (n <= kMidArgsortRows && opt().mid_argsort) {
    // (one workgroup per compute unit, each producing a run of slots; no workgroup waits for another)
    const size_t lds = mid_sort_lds_bytes((int)n);
    const bool wide = n <= kMidArgsortWideRows;
    if (int e = grant_dynamic_lds(wide ? reinterpret_cast<const void*>(mid_argsort_kernel<true>)
                                       : reinterpret_cast<const void*>(mid_argsort_kernel<false>), lds))
      return e;
    const int per = (int)round_up((n + device_cus() - 1) / device_cus(), 16);
    if (wide)
      hipLaunchKernelGGL(mid_argsort_kernel<true>, dim3((unsigned)((n + per - 1) / per)), dim3(kMidArgsortThreads), lds, s, key, kind,
                         stride, (int)n, prev_order, per, order_out);
    else
      hipLaunchKernelGGL(mid_argsort_kernel<false>, dim3((unsigned)((n + per - 1) / per)), dim3(kMidArgsortThreads), lds, s, key, kind,
                         stride, (int)n, prev_order, per, order_out);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  uint8_t* base = static_cast<uint8_t*>(ws);
  // every call starts from a cleared control block: barrier generations restart
  const int64_t zero_words = (int64_t)((L.pairs0 - L.ctrl) / 4);
  hipLaunchKernelGGL(reset_state_kernel, dim3(16), dim3(256), 0, s, reinterpret_cast<uint32_t*>(base + L.ctrl), zero_words);
  EVX_LAUNCH_CHECK();
  RadixBuffers b;
  b.pairs[0] = reinterpret_cast<unsigned long long*>(base + L.pairs0);
  b.pairs[1] = reinterpret_cast<unsigned long long*>(base + L.pairs1);
  b.table = reinterpret_cast<int*>(base + L.table);
  b.totals = reinterpret_cast<int*>(base + L.totals);
  b.kstride = L.kstride;
  int workers = L.workers;
  const int cap = device_cus() * 2 - kFirstSweeper;  // all blocks resident at once
  if (workers > cap) workers = cap;
  if (workers < 1) workers = 1;
  hipLaunchKernelGGL(argsort_step_kernel, dim3(workers + kFirstSweeper), dim3(kRadixThreads), kRadixLdsBytes, s, key, kind,
                     stride, L.n, prev_order, reinterpret_cast<Ctrl*>(base + L.ctrl), b, order_out, opt().spin_limit, key_cap);
  EVX_LAUNCH_CHECK();
  // (an order of -1 everywhere when one of the sort's grid barriers ran out)
  return copy_out(reinterpret_cast<const Ctrl*>(base + L.ctrl), order_out, nullptr, n, kPoisonIndex, s, 1, 0, call_err);
}

// One stable argsort step of int32 keys for each of `batch` populations in one launch (n <= kMidArgsortRows, the
// kernels that never wait): keys key_step bytes apart, orders order_step bytes apart.
static int argsort_step_many(const void* key, int64_t n, int batch, int64_t key_step, int32_t* order_out, int64_t order_step,
                             hipStream_t s) {
  if (n <= kSmallArgsortRows) {
    const int npad = ((int)n + 127) & ~127;
    if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(small_argsort_kernel), sizeof(double) * (size_t)npad)) return e;
    hipLaunchKernelGGL(small_argsort_kernel, dim3(npad / kSmallArgsortGroup, batch), dim3(kSmallArgsortThreads),
                       sizeof(double) * (size_t)npad, s, key, (int)kKeyInt32, (int64_t)1, (int)n, (const int*)nullptr, order_out, key_step,
                       order_step);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  if (n > kMidArgsortRows) return kErrBadArg;
  const size_t lds = mid_sort_lds_bytes((int)n);
  const bool wide = n <= kMidArgsortWideRows;
  if (int e = grant_dynamic_lds(wide ? reinterpret_cast<const void*>(mid_argsort_kernel<true>)
                                     : reinterpret_cast<const void*>(mid_argsort_kernel<false>), lds))
    return e;
  // (a population's share of the compute units, at least sixteen workgroups)
  int blocks = device_cus() / batch;
  if (blocks < 16) blocks = 16;
  const int per = (int)round_up((n + blocks - 1) / blocks, 16);
  const dim3 grid((unsigned)((n + per - 1) / per), (unsigned)batch);
  if (wide)
    hipLaunchKernelGGL(mid_argsort_kernel<true>, grid, dim3(kMidArgsortThreads), lds, s, key, (int)kKeyInt32, (int64_t)1, (int)n,
                       (const int*)nullptr, per, order_out, key_step, order_step);
  else
    hipLaunchKernelGGL(mid_argsort_kernel<false>, grid, dim3(kMidArgsortThreads), lds, s, key, (int)kKeyInt32, (int64_t)1, (int)n,
                       (const int*)nullptr, per, order_out, key_step, order_step);
  EVX_LAUNCH_CHECK();
  return 0;
}

// `batch` sorts of n <= kSmallArgsortRows positions in one launch: a workgroup per sort, or several sorts per
// workgroup when they are short.
template <int T, int R>
static int launch_rows_argsort(const void* key, int kind, int64_t batch_stride, int64_t stride, int64_t batch, int n,
                               const int32_t* prev_order, int32_t* order_out, hipStream_t s) {
  int group = 1;
  while (group * R < n) group <<= 1;  // threads per sort, a power of two
  if (group > T) return kErrBadArg;
  const int rows_per_block = T / group;
  const int row_stride = rows_per_block > 1 ? (n | 1) : n;
  const size_t lds = sizeof(double) * (size_t)rows_per_block * (size_t)row_stride;
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(rows_argsort_kernel<T, R>), lds)) return e;
  int64_t blocks = (batch + rows_per_block - 1) / rows_per_block;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL((rows_argsort_kernel<T, R>), dim3((unsigned)blocks), dim3(T), lds, s, key, kind, batch_stride, stride, batch, n,
                     rows_per_block, row_stride, prev_order, order_out);
  EVX_LAUNCH_CHECK();
  return 0;
}

static int launch_rows_bitonic(const void* key, int kind, int64_t batch_stride, int64_t stride, int64_t batch, int n,
                               const int32_t* prev_order, int32_t* order_out, hipStream_t s) {
  int npad = kRowsBitonicMin;
  while (npad < n) npad <<= 1;
  if (npad > kRowsArgsortMax) return kErrBadArg;
  const int threads = npad / 8 < 1024 ? npad / 8 : 1024;  // eight entries per thread and pass
  const size_t lds = sizeof(double) * (size_t)npad;
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(rows_bitonic_argsort_kernel), lds)) return e;
  const int64_t blocks = batch < 65536 ? batch : 65536;
  hipLaunchKernelGGL(rows_bitonic_argsort_kernel, dim3((unsigned)blocks), dim3(threads), lds, s, key, kind, batch_stride, stride,
                     batch, n, npad, prev_order, order_out);
  EVX_LAUNCH_CHECK();
  return 0;
}

extern "C" {

size_t evox_hip_argsort_workspace_bytes(int64_t n) {
  SortLayout L;
  return make_sort_layout(n, &L) ? L.total : 0;
}

int evox_hip_stable_argsort_step(const void* key, int kind, int64_t stride, int64_t n, const int32_t* prev_order,
                                 int32_t* order_out, void* ws, size_t ws_bytes, void* stream) {
  return argsort_step(key, kind, stride, n, prev_order, order_out, ws, ws_bytes, stream);
}

int evox_hip_stable_argsort_step_batched(const void* key, int kind, int64_t batch_stride, int64_t stride, int64_t batch,
                                         int64_t n, const int32_t* prev_order, int32_t* order_out, void* ws, size_t ws_bytes,
                                         void* stream) {
  SortLayout L;
  if (key == nullptr || order_out == nullptr || kind < 0 || kind > 2 || batch < 1) return kErrBadArg;
  if (!make_sort_layout(n, &L)) return kErrBadArg;
  if (ws == nullptr || ws_bytes < L.total || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  hipStream_t s = (hipStream_t)stream;
  // all sorts in one launch when a sort fits the LDS of a workgroup: by counting up to 256 positions (several
  // sorts per workgroup), through a bitonic network above that
  if (batch >= 2 && n <= kRowsArgsortMax) {
    if (n <= 256) return launch_rows_argsort<256, 1>(key, kind, batch_stride, stride, batch, (int)n, prev_order, order_out, s);
    return launch_rows_bitonic(key, kind, batch_stride, stride, batch, (int)n, prev_order, order_out, s);
  }
  const size_t key_bytes = 4;
  for (int64_t b = 0; b < batch; ++b) {
    const void* kb = static_cast<const uint8_t*>(key) + (size_t)(b * batch_stride) * key_bytes;
    if (int e = argsort_step(kb, kind, stride, n, prev_order ? prev_order + b * n : nullptr, order_out + b * n, ws, ws_bytes, stream))
      return e;
  }
  return 0;
}

}  // extern "C"

// ---- fitness of 8-byte elements (wide.hpp)
struct WideLayout {
  int n, m;
  size_t ctrl, key_lo, key_hi, key_mask, selected, boundary, ord_a, ord_b, terms, dist, neg_lo, neg_hi, order_a, order_b, front_dkey,
      front_ends, sort_ws, sort_bytes, total;
};

static bool make_wide_layout(int64_t n, int64_t m, WideLayout* L) {
  if (n < 1 || m < 1 || n > 0x7FFFFF00ll || m > 65535 || n * m > 0x7FFFFFFFll * 16) return false;
  L->n = (int)n;
  L->m = (int)m;
  const size_t nm = (size_t)n * (size_t)m;
  size_t o = 0;
  L->ctrl = o;      o = align_up(o + sizeof(WideCtrl));
  L->key_lo = o;    o = align_up(o + 4 * nm);
  L->key_hi = o;    o = align_up(o + 4 * nm);
  L->key_mask = o;  o = align_up(o + 4 * (size_t)n);
  L->selected = o;  o = align_up(o + (size_t)n);
  L->boundary = o;  o = align_up(o + 4 * (size_t)n);
  L->ord_a = o;     o = align_up(o + 4 * nm);
  L->ord_b = o;     o = align_up(o + 4 * nm);
  L->terms = o;     o = align_up(o + 8 * nm);
  L->dist = o;      o = align_up(o + 8 * (size_t)n);
  L->neg_lo = o;    o = align_up(o + 4 * (size_t)n);
  L->neg_hi = o;    o = align_up(o + 4 * (size_t)n);
  L->order_a = o;   o = align_up(o + 4 * (size_t)n);
  L->order_b = o;   o = align_up(o + 4 * (size_t)n);
  L->front_dkey = o; o = align_up(o + 8 * (size_t)n);
  L->front_ends = o; o = align_up(o + 8 * (size_t)m);
  SortLayout sort_layout;
  if (!make_sort_layout(n, &sort_layout)) return false;
  L->sort_bytes = sort_layout.total;
  L->sort_ws = o;   o = align_up(o + L->sort_bytes);
  L->total = o;
  return true;
}

static int wide_grid(int64_t items) {
  int64_t blocks = (items + 255) / 256;
  const int64_t cap = (int64_t)device_cus() * 8;
  if (blocks > cap) blocks = cap;
  return (int)(blocks < 1 ? 1 : blocks);
}

// The crowding distances of the rows selected by the mask, by the rank vector (rank == its largest set value) or all
// rows, into `dist` (double for out_kind 0, float for 1), and with neg_keys the sort keys of their negatives.
static int wide_distances(const WideLayout& L, uint8_t* base, const void* costs, int kind, int64_t sr, int64_t sc,
                          const uint8_t* mask, int64_t mask_stride, const int32_t* rank, void* dist, int out_kind, bool neg_keys,
                          hipStream_t s, int* outcome = nullptr) {
  const int n = L.n, m = L.m;
  WideCtrl* ctrl = reinterpret_cast<WideCtrl*>(base + L.ctrl);
  uint32_t* key_lo = reinterpret_cast<uint32_t*>(base + L.key_lo);
  uint32_t* key_hi = reinterpret_cast<uint32_t*>(base + L.key_hi);
  int* key_mask = reinterpret_cast<int*>(base + L.key_mask);
  uint8_t* selected = base + L.selected;
  int* boundary = reinterpret_cast<int*>(base + L.boundary);
  int* ord_a = reinterpret_cast<int*>(base + L.ord_a);
  int* ord_b = reinterpret_cast<int*>(base + L.ord_b);
  hipLaunchKernelGGL(wide_head_kernel, dim3(1), dim3(1024), 0, s, mask, mask_stride, rank, n, ctrl);
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(wide_keys_kernel, dim3(wide_grid((int64_t)n * m)), dim3(256), 0, s, costs, kind, sr, sc, n, m, mask, mask_stride,
                     rank, ctrl, key_lo, key_hi, key_mask, selected, boundary);
  EVX_LAUNCH_CHECK();
  // per objective: by cost (low half, then high half of its ordered image), then selected rows first; ties by row
  void* sort_ws = base + L.sort_ws;
  if (int e = evox_hip_stable_argsort_step_batched(key_lo, kKeyUint32, n, 1, m, n, nullptr, ord_a, sort_ws, L.sort_bytes, s)) return e;
  if (int e = evox_hip_stable_argsort_step_batched(key_hi, kKeyUint32, n, 1, m, n, ord_a, ord_b, sort_ws, L.sort_bytes, s)) return e;
  const int* order = ord_b;
  if (mask != nullptr || rank != nullptr) {
    if (int e = evox_hip_stable_argsort_step_batched(key_mask, kKeyInt32, 0, 1, m, n, ord_b, ord_a, sort_ws, L.sort_bytes, s)) return e;
    order = ord_a;
  }
  uint32_t* neg_lo = neg_keys ? reinterpret_cast<uint32_t*>(base + L.neg_lo) : nullptr;
  uint32_t* neg_hi = neg_keys ? reinterpret_cast<uint32_t*>(base + L.neg_hi) : nullptr;
  if (out_kind == 0) {
    double* terms = reinterpret_cast<double*>(base + L.terms);
    hipLaunchKernelGGL(wide_terms_kernel<double>, dim3(wide_grid((int64_t)n * m)), dim3(256), 0, s, costs, kind, sr, sc, n, m, order, ctrl,
                       terms, boundary);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(wide_sum_kernel<double>, dim3(wide_grid(n)), dim3(256), 0, s, terms, selected, boundary, ctrl, n, m,
                       static_cast<double*>(dist), neg_lo, neg_hi, outcome);
  } else {
    float* terms = reinterpret_cast<float*>(base + L.terms);
    hipLaunchKernelGGL(wide_terms_kernel<float>, dim3(wide_grid((int64_t)n * m)), dim3(256), 0, s, costs, kind, sr, sc, n, m, order, ctrl,
                       terms, boundary);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(wide_sum_kernel<float>, dim3(wide_grid(n)), dim3(256), 0, s, terms, selected, boundary, ctrl, n, m,
                       static_cast<float*>(dist), neg_lo, neg_hi, outcome);
  }
  EVX_LAUNCH_CHECK();
  return 0;
}

// Whether the selection of a population of n rows orders its last front without sorting the costs
// (wide_select_direct): up to kWideDirectRows rows, unless the last selection of this shape found a front of more
// than kWideDirectFront rows -- that path's work grows with the square of the front.
static bool wide_direct_applies(int64_t n, const int* outcome) {
  return n <= kWideDirectRows && (outcome == nullptr || __atomic_load_n(outcome, __ATOMIC_RELAXED) != 2);
}

// The distances of the rows of the last front (rank == the largest rank set) and the selection order of all rows by
// (rank, distance descending, row index), for populations of up to kWideDirectRows rows: one stable argsort step of
// the ranks lists the rows, the kernels of wide.hpp do the rest without sorting the costs.
static int wide_select_direct(const WideLayout& L, uint8_t* base, const void* costs, int kind, int64_t sr, int64_t sc,
                              const int32_t* rank, void* dist, int out_kind, int* order_out, hipStream_t s, int* outcome,
                              int batch = 1, int64_t ws_step = 0, int64_t cost_step = 0) {
  // batch > 1: that many populations in the same launches, their workspaces ws_step bytes, their costs cost_step bytes and
  // their rank vectors n entries apart (dist and order_out lie in the workspaces)
  const int n = L.n, m = L.m;
  WideCtrl* ctrl = reinterpret_cast<WideCtrl*>(base + L.ctrl);
  int* listing = reinterpret_cast<int*>(base + L.order_b);
  uint64_t* key = reinterpret_cast<uint64_t*>(base + L.terms);
  uint64_t* dkey = reinterpret_cast<uint64_t*>(base + L.front_dkey);
  int* ends = reinterpret_cast<int*>(base + L.front_ends);
  hipLaunchKernelGGL(wide_head_kernel, dim3(1, 1, batch), dim3(1024), 0, s, (const uint8_t*)nullptr, (int64_t)0, rank, n, ctrl, ws_step);
  EVX_LAUNCH_CHECK();
  if (batch > 1) {
    if (int e = argsort_step_many(rank, n, batch, (int64_t)n * 4, listing, ws_step, s)) return e;
  } else if (int e = evox_hip_stable_argsort_step(rank, kKeyInt32, 1, n, nullptr, listing, base + L.sort_ws, L.sort_bytes, s)) {
    return e;
  }
  // (sixteen lanes per candidate; the grids are sized for a front of all rows, which the kernels find out on the device)
  const int pair_grid = shared_grid(wide_grid((int64_t)n * 16), device_cus() * 8, batch);
  const int keys_grid = shared_grid(wide_grid((int64_t)n * m), device_cus() * 8, batch);
  const int dist_grid = (n + 15) / 16;  // (a group of lanes per row, n <= kWideDirectRows)
  auto launch = [&](auto* typed_dist) {
    using Out = std::remove_pointer_t<decltype(typed_dist)>;
    hipLaunchKernelGGL(wide_front_keys_kernel<Out>, dim3(keys_grid < m ? m : keys_grid, 1, batch), dim3(256), 0, s, costs, kind, sr, sc, n,
                       m, listing, ctrl, key, ends, typed_dist, ws_step, cost_step);
    hipLaunchKernelGGL(wide_front_dist_kernel<Out>, dim3(dist_grid, 1, batch), dim3(256), 0, s, costs, kind, sr, sc, n, m, listing, ctrl,
                       key, ends, typed_dist, dkey, ws_step, cost_step);
  };
  if (out_kind == 0)
    launch(static_cast<double*>(dist));
  else
    launch(static_cast<float*>(dist));
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(wide_front_order_kernel, dim3(pair_grid, 1, batch), dim3(256), 0, s, listing, ctrl, dkey, n, order_out, outcome, ws_step);
  EVX_LAUNCH_CHECK();
  return 0;
}

// The gathers of a selection by `order` in one launch: x (if any), the fitness rows, the ranks and the distances.
struct WideGather {
  const void* x;
  int64_t x_row_bytes, x_row_stride_bytes, x_step;
  const void* f_rows;
  int64_t f_row_bytes, f_row_stride_bytes, f_step;
  const int32_t* rank;
  const void* dist;
  int64_t dist_bytes, dist_step;
  void *out_x, *out_f, *out_rank, *out_dist;
};
static int wide_gather(const WideGather& a, const int* order, int64_t order_step, int64_t n, int64_t topk, int batch, hipStream_t s) {
  GatherParts parts;
  parts.parts = 0;
  parts.first[0] = 0;
  auto add_part = [&](const void* src, int64_t row_bytes, int64_t row_stride_bytes, int64_t src_step, void* dst) {
    if (row_bytes <= 0) return;
    uintptr_t bits = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) | (uintptr_t)row_bytes | (uintptr_t)row_stride_bytes;
    if (batch > 1) bits |= (uintptr_t)src_step | (uintptr_t)(topk * row_bytes);
    const int unit = bits % 16 == 0 ? 16 : bits % 8 == 0 ? 8 : bits % 4 == 0 ? 4 : 1;
    const int p = parts.parts++;
    parts.src[p] = static_cast<const uint8_t*>(src);
    parts.dst[p] = static_cast<uint8_t*>(dst);
    parts.row_bytes[p] = row_bytes;
    parts.row_stride_bytes[p] = row_stride_bytes;
    parts.src_step[p] = src_step;
    parts.dst_step[p] = topk * row_bytes;
    parts.unit[p] = unit;
    parts.first[p + 1] = parts.first[p] + topk * (row_bytes / unit);
  };
  if (a.x != nullptr) add_part(a.x, a.x_row_bytes, a.x_row_stride_bytes, a.x_step, a.out_x);
  add_part(a.f_rows, a.f_row_bytes, a.f_row_stride_bytes, a.f_step, a.out_f);
  add_part(a.rank, 4, 4, n * 4, a.out_rank);
  add_part(a.dist, a.dist_bytes, a.dist_bytes, a.dist_step, a.out_dist);
  const int grid = shared_grid(wide_grid(parts.first[parts.parts]), device_cus() * 8, batch);
  hipLaunchKernelGGL(gather_parts_kernel, dim3(grid, 1, batch), dim3(256), 0, s, parts, order, topk, order_step);
  EVX_LAUNCH_CHECK();
  return 0;
}

namespace evx {
static size_t wide_workspace_need(int64_t n, int64_t m) {
  WideLayout L;
  return make_wide_layout(n, m, &L) ? L.total : 0;
}
}  // namespace evx

// Two objectives without a matrix (two.hpp): the rows sorted by (f1, f2, index), the fronts as rounds of prefix
// minima handed from workgroup to workgroup, the listing by (rank, index) from one stable argsort of the ranks.
static bool two_applies(const Layout& L, int64_t stop_count) {
  const int64_t least = stop_count >= L.n ? opt().two_min_rows : (opt().two_min_rows_partial > opt().two_min_rows ? opt().two_min_rows_partial : opt().two_min_rows);
  return L.m == 2 && opt().two_min_rows > 0 && L.n >= least && L.n <= kTwoMaxRows && !opt().peel_stepped;
}

// Several populations at once take that path when their argsort of the ranks is one of the kernels that never wait
// and all their chains are resident together: how many of `batch` share a launch (0: none).
static int many_two_share(const Layout& L, int64_t batch, int64_t stop_count) {
  if (batch < 2 || !two_applies(L, stop_count) || L.n > kMidArgsortRows || !opt().mid_argsort) return 0;
  const int blocks = (L.n + kTwoChunk - 1) / kTwoChunk;
  int share = device_cus() * 2 / blocks;
  if (share > batch) share = (int)batch;
  if (share < 2) return 0;
  const int64_t passes = (batch + share - 1) / share;
  return (int)((batch + passes - 1) / passes);
}

// Leaves what count_and_peel leaves: ranks by original index (of every row), the listing, the front starts and sizes
// and the control block's description of the front that holds the stop_count-th row.  rank_until: optionally the
// ranks with the rows behind that front unset (n ints).
static int stage_rank_two(const Ws& w, const Fitness& src, int64_t stop_count, bool fill_dist, int* rank_until, hipStream_t s) {
  const Layout& L = w.L;
  if (stop_count < 1 || stop_count > L.n) return kErrBadArg;
  WideLayout WL;
  if (!make_wide_layout(L.n, L.m, &WL) || WL.total > L.wide_bytes) return kErrWorkspace;
  if (int e = stage_prepare(w, src, true, s, true)) return e;
  const int blocks = (L.n + kTwoChunk - 1) / kTwoChunk;
  // (every workgroup waits for the one before it: resident at once on any device with as many compute units)
  if ((int64_t)blocks * w.batch > device_cus() * 2) return kErrNotResident;
  const float* xs_sorted = w.at<float>(L.xs_sorted);
  hipLaunchKernelGGL(two_peel_kernel, dim3(blocks, 1, w.batch), dim3(kTwoThreads), 0, s, xs_sorted, xs_sorted + L.npad,
                     w.at<uint32_t>(L.kid_sorted), w.at<int>(L.orig_of), L.n, w.at<int>(L.rank),
                     fill_dist ? w.at<float>(L.dist) : (float*)nullptr, w.ctrl(), w.at<unsigned long long>(L.two_ring), opt().spin_limit,
                     (int)stop_count, w.step);
  EVX_LAUNCH_CHECK();
  int grid = (L.n + 255) / 256;
  if (grid > device_cus() * 8) grid = device_cus() * 8;
  grid = shared_grid(grid, device_cus() * 8, w.batch);
  hipLaunchKernelGGL(two_finish_kernel, dim3(grid, 1, w.batch), dim3(256), 0, s, w.at<uint32_t>(L.kid_sorted), w.at<int>(L.orig_of),
                     xs_sorted, xs_sorted + L.npad, L.n, w.at<int>(L.rank), w.ctrl(), w.step);
  EVX_LAUNCH_CHECK();
  if (w.batch > 1) {
    if (int e = argsort_step_many(w.at<int>(L.rank), L.n, w.batch, w.step, w.at<int>(L.perm), w.step, s)) return e;
  } else {
    uint8_t* wb = w.base + L.wide;
    if (int e = argsort_step(w.at<int>(L.rank), kKeyInt32, 1, L.n, nullptr, w.at<int>(L.perm), wb + WL.sort_ws, WL.sort_bytes, s,
                             &w.ctrl()->reserved[kTwoRounds], &w.ctrl()->err))
      return e;
  }
  hipLaunchKernelGGL(two_bounds_kernel, dim3(grid, 1, w.batch), dim3(256), 0, s, w.at<int>(L.perm), w.at<int>(L.rank), L.n,
                     w.at<int>(L.fstart), w.ctrl(), (int)stop_count, w.step);
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(two_sizes_kernel, dim3(grid, 1, w.batch), dim3(256), 0, s, w.at<int>(L.perm), w.at<int>(L.rank), L.n,
                     w.at<int>(L.fstart), w.at<int>(L.fsize), w.ctrl(), rank_until, w.step);
  EVX_LAUNCH_CHECK();
  return 0;
}

// Populations that two launches take (few.hpp): all whose rows fit the threads of one workgroup (against the pipeline, us
// per selection of half the rows in a loop of calls; the device alone is done with 300 x 3 in 12.5: 300 x 3 37 -> 17, 1000 x 3 45 -> 21, 1000 x 5 47 -> 31, 1000 x 8 82 -> 47; all ranks of 1000 x 3
// 64 -> 23), unless a tunable asks for a kernel of the pipeline.  The two parts of a population must have equal strides.
static bool few_applies(const Layout& L, const Fitness& fit, int batch) {
  if (L.n > opt().few_max_rows || L.m < 3 || L.m > kFewObjectives || batch > kFewBatch) return false;
  const Options usual;
  if (opt().peel_stepped || !opt().peel_lds || !opt().peel_records || !opt().peel_witness || !opt().peel_tail || !opt().tail_merged ||
      !opt().small_sort || !opt().dominance_folded || opt().dominance_tile_words || opt().peel_lds_blocks || opt().peel_record_blocks ||
      opt().spin_limit != usual.spin_limit)
    return false;
  return fit.n_first >= L.n || (fit.sr == fit.sr2 && fit.sc == fit.sc2 && ((fit.f2 - fit.f) * (int64_t)sizeof(float) == (const char*)fit.f2 - (const char*)fit.f));
}
static int stage_few(const Ws& w, const Fitness& fit, BatchedArgs a, hipStream_t s) {
  const Layout& L = w.L;
  a.f = fit.f;
  a.f_stride_b = fit.step;
  a.f_stride_row = fit.sr;
  a.f_stride_col = fit.sc;
  a.n = L.n;
  a.m = L.m;
  a.n_first = (int)(fit.n_first < L.n ? fit.n_first : L.n);
  a.f_second = fit.n_first < L.n ? (fit.f2 - fit.f) - fit.n_first * fit.sr : 0;
  const int nt = (int)round_up(L.n, 64);
  const dim3 grid(nt / 64, (nt + 127) / 128, w.batch);
  uint64_t* const words = w.at<uint64_t>(L.dom);
  switch (L.m) {
    case 3: hipLaunchKernelGGL(few_dominance_kernel<3>, grid, dim3(256), 0, s, a, words, w.step); break;
    case 4: hipLaunchKernelGGL(few_dominance_kernel<4>, grid, dim3(256), 0, s, a, words, w.step); break;
    case 5: hipLaunchKernelGGL(few_dominance_kernel<5>, grid, dim3(256), 0, s, a, words, w.step); break;
    case 6: hipLaunchKernelGGL(few_dominance_kernel<6>, grid, dim3(256), 0, s, a, words, w.step); break;
    case 7: hipLaunchKernelGGL(few_dominance_kernel<7>, grid, dim3(256), 0, s, a, words, w.step); break;
    default: hipLaunchKernelGGL(few_dominance_kernel<8>, grid, dim3(256), 0, s, a, words, w.step); break;
  }
  EVX_LAUNCH_CHECK();
  const size_t lds = few_finish_lds_bytes(nt, L.n, L.m);
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(few_finish_kernel), lds)) return e;
  hipLaunchKernelGGL(few_finish_kernel, dim3(w.batch), dim3(nt), lds, s, a, words, w.ctrl(), w.step);
  EVX_LAUNCH_CHECK();
  return 0;
}

// Shared body of the two selection entry points: the population is one part or two.
static int select_rows(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes, const void* x2,
                       int64_t x2_row_stride_bytes, const Fitness& fit, int64_t n, int64_t m, int64_t topk, void* out_x,
                       float* out_f, int32_t* out_rank, float* out_dist, int32_t* out_order, void* ws, size_t ws_bytes,
                       hipStream_t s, bool may_allocate, int batch = 1, int64_t ws_step = 0, int64_t x_step_bytes = 0,
                       int64_t x2_step_bytes = 0) {
  // batch > 1: that many populations of one shape in the same launches (the caller has checked that their grids are
  // resident together: many_populations_plan); their workspaces lie ws_step bytes apart, their decision vectors
  // x_step_bytes, their fitness fit.step elements, their results topk rows
  Ws w;
  if (out_f == nullptr || out_rank == nullptr || out_dist == nullptr) return kErrBadArg;
  if ((x == nullptr) != (out_x == nullptr) || (x == nullptr) != (x2 == nullptr)) return kErrBadArg;
  if (x != nullptr && (x_row_bytes < 0 || x_row_stride_bytes < 0 || x2_row_stride_bytes < 0)) return kErrBadArg;
  if (topk < 1 || topk > n) return kErrBadArg;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  const Layout& L = w.L;
  if (batch > 1) {
    if (ws_step < (int64_t)L.total || (ws_step & 255) != 0 || ws_bytes < (size_t)ws_step * (size_t)batch) return kErrWorkspace;
    w.batch = batch;
    w.step = ws_step;
  }
  int unit = 1;
  if (x != nullptr) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(x2) | reinterpret_cast<uintptr_t>(out_x) |
                           (uintptr_t)x_row_bytes | (uintptr_t)x_row_stride_bytes | (uintptr_t)x2_row_stride_bytes |
                           (uintptr_t)x_step_bytes | (uintptr_t)x2_step_bytes;
    unit = (bits % 16 == 0) ? 16 : (bits % 4 == 0) ? 4 : 1;
  }
  if (out_order == nullptr && few_applies(L, fit, batch) && (x == x2 || x_row_stride_bytes == x2_row_stride_bytes) && x_step_bytes == x2_step_bytes) {
    BatchedArgs a = {};
    a.stop_count = (int)topk;
    a.x = static_cast<const uint8_t*>(x);
    a.x_stride_b = x_step_bytes;
    a.x_row_stride = x_row_stride_bytes;
    a.x_row_bytes = x_row_bytes;
    a.x_unit = unit;
    if (fit.n_first < n) a.x_second = (static_cast<const uint8_t*>(x2) - static_cast<const uint8_t*>(x)) - fit.n_first * x_row_stride_bytes;
    a.out_x = static_cast<uint8_t*>(out_x);
    a.out_f = out_f;
    a.out_rank = out_rank;
    a.out_dist = out_dist;
    return stage_few(w, fit, a, s);
  }
  GatherArgs g = {};
  g.order = w.at<int>(L.order);
  g.listed = w.at<int>(L.perm);
  g.topk = (int)topk;
  g.x = static_cast<const uint8_t*>(x);
  g.x_row_stride = x_row_stride_bytes;
  g.x_row_bytes = x_row_bytes;
  g.out_x = static_cast<uint8_t*>(out_x);
  g.unit = unit;
  g.f = fit.f;
  g.f_stride_row = fit.sr;
  g.f_stride_col = fit.sc;
  g.n_first = (int)fit.n_first;
  g.x2 = static_cast<const uint8_t*>(x2);
  g.x2_row_stride = x2_row_stride_bytes;
  g.f2 = fit.f2;
  g.f2_stride_row = fit.sr2;
  g.f2_stride_col = fit.sc2;
  g.m = L.m;
  g.out_f = out_f;
  g.rank = w.at<int>(L.rank);
  g.out_rank = out_rank;
  g.dist = w.at<float>(L.dist);
  g.out_dist = out_dist;
  g.out_order = out_order;
  g.ctrl = w.ctrl();
  g.ws_step = w.step;
  g.x_step = x_step_bytes;
  g.x2_step = x2_step_bytes;
  g.f_step = fit.step;
  g.f2_step = fit.step2;
  int gather_blocks = (int)((topk + 3) / 4);
  if (gather_blocks > device_cus() * 8) gather_blocks = device_cus() * 8;
  const dim3 gather_grid(gather_blocks, 1, w.batch);
  auto launch_gather = [&](bool after_peel) {
    if (after_peel && w.batch > 1)
      hipLaunchKernelGGL(gather_after_peel_kernel<true>, gather_grid, dim3(256), 0, s, g);
    else if (after_peel)
      hipLaunchKernelGGL(gather_after_peel_kernel<false>, gather_grid, dim3(256), 0, s, g);
    else if (w.batch > 1)
      hipLaunchKernelGGL(gather_kernel<true>, gather_grid, dim3(256), 0, s, g);
    else
      hipLaunchKernelGGL(gather_kernel<false>, gather_grid, dim3(256), 0, s, g);
  };
  // Above kMidArgsortRows rows the launches with the sorted runs stand beside those for other fronts.  What the last
  // selection of the shape found says whether they are worth their four launches (a converged population's front is larger:
  // 70 000 x 3 on a plane 304 -> 288 us).
  bool without_runs = false;
  if (batch == 1 && crowd_mid_split(L) && opt().launch_memory) {
    g.outcome = outcome_slot(kWordRuns, n, m, may_allocate, s);
    const int small = L.m <= kFusedFrontObjectives ? (kFusedFrontValues / L.m < kFusedFrontRows ? kFusedFrontValues / L.m : kFusedFrontRows) : 0;
    g.outcome_from = small > kMidSortMinCandidates ? small : kMidSortMinCandidates;
    g.outcome_to = kMidArgsortRows;
    without_runs = g.outcome != nullptr && __atomic_load_n(g.outcome, __ATOMIC_RELAXED) == 2;
  }
  if (batch == 1 ? two_applies(L, topk) : many_two_share(L, batch, topk) >= batch) {
    const int e = stage_rank_two(w, fit, topk, true, nullptr, s);
    if (e != kErrNotResident || batch > 1) {
      if (e) return e == kErrNotResident ? kErrBadArg : e;
      // the last front by the ordering kernels, then the gather, as after a peel that leaves the last front alone
      if (int c = stage_crowd_sort(w, w.at<int>(L.perm), false, 2, s, false, without_runs)) return c;
      if (crowd_mid_sort(L)) return stage_crowd_finish(w, w.at<int>(L.perm), true, 2, s, false, &g);
      if (int c = stage_crowd_finish(w, w.at<int>(L.perm), true, 2, s, false, nullptr, without_runs)) return c;
      launch_gather(false);
      EVX_LAUNCH_CHECK();
      return 0;
    }
  }
  if (int e = stage_prepare(w, fit, true, s)) return e;
  // A population that keeps filling what is kept from front 0 alone (many objectives, or converged) has no use for
  // the matrix: where the order-based kernel would build it, the word of the launch memory says what the last two
  // selections of the shape found, and the kernel counts first when both had enough in front 0 (200 000 x 8, half
  // kept: the stage 0.98 -> 0.80 ms; a wrong guess costs a second launch, 0.92 ms, once).
  int64_t count_first = 0;
  if (batch == 1 && opt().launch_memory && opt().prefix_count_first && prefix_dominance_applies(L) && !opt().peel_stepped) {
    g.front0_note = outcome_slot(kWordFront0, n, m, may_allocate, s);
    g.front0_size = w.at<int>(L.fsize);
    g.front0_enough = (int)topk;
    if (opt().prefix_count_first == 2 || (g.front0_note != nullptr && __atomic_load_n(g.front0_note, __ATOMIC_RELAXED) == 3)) count_first = topk;
  }
  if (int e = stage_dominance(w, kDomAuto, s, count_first)) return e;
  bool peel_orders = false;  // the peel kernel orders a small last front itself (it says so in Ctrl.tail_done)
  bool peel_always_orders = false;  // ... and here every front is small enough: nothing is left to launch but the gather
  bool stepped = false;  // the fronts were peeled one launch each: the last front is ordered likewise, by the kernels of wide.hpp
  if (batch > 1) {
    if (int e = count_and_peel_persistent(w, topk, true, true, s, true, &peel_orders, &peel_always_orders)) return e == kErrNotResident ? kErrBadArg : e;
  } else if (int e = count_and_peel(w, topk, true, true, s, true, &peel_orders, &peel_always_orders, &stepped)) {
    return e;
  }
  g.order_from_peel = peel_always_orders ? 1 : 0;
  if (!crowd_mid_split(L))
    g.outcome = peel_orders && !peel_always_orders && opt().launch_memory
                    ? outcome_slot(batch > 1 ? kWordBatch : kWordLastFront, n, m, may_allocate, s) : nullptr;
  const int last_outcome = g.outcome != nullptr && g.outcome_to == 0 ? __atomic_load_n(g.outcome, __ATOMIC_RELAXED) : 0;
  // Where the peel kernel may have ordered the last front, the kernels that would order it look at Ctrl.tail_done and
  // return at once.  A launch that does nothing still costs 2 to 4.7 us, so with up to three objectives -- last
  // fronts of a few hundred rows, which the peel kernel orders -- all ordering stages and the gather share one
  // launch (crowd_gather_kernel); with more objectives the last front is usually too large for the peel kernel, and
  // the stages as kernels of their own order it faster than the shared launch does (20 000 x 5, a front of 2532 rows:
  // 138 us per selection).
  // What the last selection of this shape found decides where it is known: a population that has converged keeps
  // last fronts of thousands of rows, which the kernels of their own order 40 us faster (20 001 x 3, one front: 114
  // against 155 us), and a last front that the peel ordered will mostly be followed by another (2000 x 5: 55 -> 52.7 us
  // in the one launch, 57 in the four).
  const bool one_ordering_launch = peel_orders && opt().tail_merged && (L.m <= 3 ? last_outcome != 2 : last_outcome == 1);
  if (stepped) {
    // distances of the rows of the last front (the mask rank == worst), the order by (rank, distance descending, index)
    // from three stable argsort steps, the gather: the fitness is read from its structure-of-arrays copy
    WideLayout WL;
    if (!make_wide_layout(n, m, &WL) || WL.total > L.wide_bytes) return kErrWorkspace;
    uint8_t* wb = w.base + L.wide;
    int* const wide_outcome = opt().launch_memory ? outcome_slot(kWordWide, n, m, may_allocate, s) : nullptr;
    if (wide_direct_applies(n, wide_outcome)) {
      if (int e = wide_select_direct(WL, wb, w.at<float>(L.xs), kWideFloat32, 1, L.npad, w.at<int>(L.rank), w.at<float>(L.dist), 1,
                                     w.at<int>(L.order), s, wide_outcome))
        return e;
      g.outcome = nullptr;
      launch_gather(false);
      EVX_LAUNCH_CHECK();
      return 0;
    }
    if (int e = wide_distances(WL, wb, w.at<float>(L.xs), kWideFloat32, 1, L.npad, nullptr, 0, w.at<int>(L.rank), w.at<float>(L.dist), 1,
                               true, s, wide_outcome))
      return e;
    int* order_a = reinterpret_cast<int*>(wb + WL.order_a);
    int* order_b = reinterpret_cast<int*>(wb + WL.order_b);
    void* sort_ws = wb + WL.sort_ws;
    if (int e = evox_hip_stable_argsort_step(wb + WL.neg_lo, kKeyUint32, 1, n, nullptr, order_a, sort_ws, WL.sort_bytes, s)) return e;
    if (int e = evox_hip_stable_argsort_step(wb + WL.neg_hi, kKeyUint32, 1, n, order_a, order_b, sort_ws, WL.sort_bytes, s)) return e;
    if (int e = evox_hip_stable_argsort_step(w.at<int>(L.rank), kKeyInt32, 1, n, order_b, w.at<int>(L.order), sort_ws, WL.sort_bytes, s))
      return e;
    g.outcome = nullptr;
    launch_gather(false);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  if (peel_always_orders) {
    launch_gather(true);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  if (!one_ordering_launch) {
    if (int e = stage_crowd_sort(w, w.at<int>(L.perm), true, 2, s, peel_orders, without_runs)) return e;
    if (crowd_mid_sort(L) && !crowd_always_small(w)) return stage_crowd_finish(w, w.at<int>(L.perm), true, 2, s, peel_orders, &g);
    if (int e = stage_crowd_finish(w, w.at<int>(L.perm), true, 2, s, peel_orders, nullptr, without_runs)) return e;
    if (peel_orders)
      launch_gather(true);
    else
      launch_gather(false);
    EVX_LAUNCH_CHECK();
    return 0;
  }
  // the peel kernel may have ordered the last front: one launch for what is left of the ordering (nothing, then) and
  // the gather
  const size_t lds = crowd_lds_bytes(L, 2);
  const bool mid = crowd_mid_sort(L);
  const bool wide = L.n <= kMidArgsortWideRows;
  const bool many = w.batch > 1;
  auto instance = [&](auto one, auto several) { return many ? reinterpret_cast<const void*>(several) : reinterpret_cast<const void*>(one); };
  const void* const kernel = !mid   ? instance(crowd_gather_kernel<kRadixThreads, 0, false>, crowd_gather_kernel<kRadixThreads, 0, true>)
                             : wide ? instance(crowd_gather_kernel<kMidArgsortThreads, 1, false>, crowd_gather_kernel<kMidArgsortThreads, 1, true>)
                                    : instance(crowd_gather_kernel<kMidArgsortThreads, 2, false>, crowd_gather_kernel<kMidArgsortThreads, 2, true>);
  if (int e = grant_dynamic_lds(kernel, lds)) return e;
  int grid = finish_grid(L, L.m);  // resident at once: at most two blocks of 256 threads per compute unit
  if (grid > device_cus() * 2) grid = device_cus() * 2;
  grid = shared_grid(grid, mid ? device_cus() : device_cus() * 2, w.batch);
  const CrowdArgs ca = crowd_args(w, w.at<int>(L.perm), false, 2);
  if (mid && wide && many)
    hipLaunchKernelGGL((crowd_gather_kernel<kMidArgsortThreads, 1, true>), dim3(grid, 1, w.batch), dim3(kMidArgsortThreads), lds, s, ca, g);
  else if (mid && wide)
    hipLaunchKernelGGL((crowd_gather_kernel<kMidArgsortThreads, 1, false>), dim3(grid), dim3(kMidArgsortThreads), lds, s, ca, g);
  else if (mid && many)
    hipLaunchKernelGGL((crowd_gather_kernel<kMidArgsortThreads, 2, true>), dim3(grid, 1, w.batch), dim3(kMidArgsortThreads), lds, s, ca, g);
  else if (mid)
    hipLaunchKernelGGL((crowd_gather_kernel<kMidArgsortThreads, 2, false>), dim3(grid), dim3(kMidArgsortThreads), lds, s, ca, g);
  else if (many)
    hipLaunchKernelGGL((crowd_gather_kernel<kRadixThreads, 0, true>), dim3(grid, 1, w.batch), dim3(kRadixThreads), lds, s, ca, g);
  else
    hipLaunchKernelGGL((crowd_gather_kernel<kRadixThreads, 0, false>), dim3(grid), dim3(kRadixThreads), lds, s, ca, g);
  EVX_LAUNCH_CHECK();
  return 0;
}

extern "C" {

int evox_hip_nd_environmental_selection(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes, const float* f,
                                        int64_t n, int64_t m, int64_t sr, int64_t sc, int64_t topk, void* out_x,
                                        float* out_f, int32_t* out_rank, float* out_dist, int32_t* out_order, void* ws,
                                        size_t ws_bytes, void* stream) {
  if (f == nullptr) return kErrBadArg;
  return select_rows(x, x_row_bytes, x_row_stride_bytes, x, x_row_stride_bytes, one_part(f, n, sr, sc), n, m, topk, out_x,
                     out_f, out_rank, out_dist, out_order, ws, ws_bytes, (hipStream_t)stream, true);
}

int evox_hip_nd_environmental_selection_two_part(const void* x_a, int64_t x_a_row_stride_bytes, const void* x_b,
                                                 int64_t x_b_row_stride_bytes, int64_t x_row_bytes, const float* f_a,
                                                 int64_t n_a, int64_t f_a_stride_row, int64_t f_a_stride_col,
                                                 const float* f_b, int64_t n_b, int64_t f_b_stride_row,
                                                 int64_t f_b_stride_col, int64_t m, int64_t topk, void* out_x, float* out_f,
                                                 int32_t* out_rank, float* out_dist, int32_t* out_order, void* ws,
                                                 size_t ws_bytes, void* stream) {
  if (n_a < 0 || n_b < 0 || n_a > 0x7FFFFF00ll || n_b > 0x7FFFFF00ll) return kErrBadArg;
  // a part without rows may come with null pointers: it is never read, the other part stands in for it
  if (n_a == 0) {
    f_a = f_b;
    x_a = x_b;
  }
  if (n_b == 0) {
    f_b = f_a;
    x_b = x_a;
  }
  if (f_a == nullptr || f_b == nullptr) return kErrBadArg;
  const Fitness fit{f_a, f_a_stride_row, f_a_stride_col, n_a, f_b, f_b_stride_row, f_b_stride_col};
  return select_rows(x_a, x_row_bytes, x_a_row_stride_bytes, x_b, x_b_row_stride_bytes, fit, n_a + n_b, m, topk, out_x, out_f,
                     out_rank, out_dist, out_order, ws, ws_bytes, (hipStream_t)stream, true);
}

}  // extern "C"

// ---- Many populations of one shape (more rows than the one-workgroup kernel of batched.hpp takes): the stages of the
// pipeline run once for `share` populations at a time, population b in the workgroups with blockIdx.z == b on its own
// copy of the workspace.  The kernels whose workgroups wait for each other get 1 / share of the device each, so that
// all of them are resident together; that is possible where the peel keeps the matrix in LDS (up to 32 768 rows) and
// a population's matrix fits the LDS of its share of the compute units.  Reference: the batched loop of
// src/evox/operators/selection/non_dominate.py:107-125 (torch.vmap of the ranking, utils/op_register.py:26-51).
static int many_populations_share(const Layout& L, int64_t batch, int64_t stop_count) {
  if (const int two = many_two_share(L, batch, stop_count)) return two;  // every population a chain of workgroups (two.hpp)
  if (batch < 2 || opt().peel_stepped || !opt().peel_lds || L.n > 32768) return 0;
  if (!opt().mid_argsort && L.n > kRadixMinCandidates) return 0;  // (large last fronts would take the radix grid)
  int share = 4 * device_cus() / 9;  // at least eight sweeping workgroups and the lister per population, up to four on a compute unit
  if (share > batch) share = (int)batch;
  size_t lds = 0;
  while (share >= 2 && lds_peel_plan(L, &lds, share) == 0) --share;
  if (share < 2) return 0;
  // (two objectives where many_two_share does not apply -- the LDS sorter switched off: several populations are still
  // faster through the matrix kernels that they share than one after the other, unless few of them fit a launch)
  if (two_applies(L, stop_count) && share < 4 && L.n > 12288) return 0;
  const int64_t passes = (batch + share - 1) / share;
  return (int)((batch + passes - 1) / passes);  // even passes: 30 populations, 28 at a time at most -> 15 + 15
}

static size_t many_workspace_step(const Layout& L) { return align_up(L.total); }

extern "C" {

/* Workspace for evox_hip_many_*: one copy of the single-population workspace per population that shares a launch. */
size_t evox_hip_many_workspace_bytes(int64_t batch, int64_t n, int64_t m, int64_t stop_count) {
  Layout L;
  if (batch < 1 || !make_layout(n, m, &L)) return 0;
  const int share = many_populations_share(L, batch, stop_count);
  return many_workspace_step(L) * (size_t)(share > 1 ? share : 1);
}

int64_t evox_hip_many_populations_per_launch(int64_t batch, int64_t n, int64_t m, int64_t stop_count) {
  Layout L;
  if (batch < 1 || !make_layout(n, m, &L)) return 0;
  const int share = many_populations_share(L, batch, stop_count);
  return share > 1 ? share : 1;
}

int evox_hip_many_non_dominate_rank_until(const float* f, int64_t batch, int64_t n, int64_t m, int64_t stride_batch, int64_t sr,
                                          int64_t sc, int64_t stop_count, int32_t* rank_out, void* ws, size_t ws_bytes,
                                          void* stream) {
  Layout L;
  if (f == nullptr || rank_out == nullptr || batch < 1 || !make_layout(n, m, &L)) return kErrBadArg;
  const int share = many_populations_share(L, batch, stop_count);
  const size_t step = many_workspace_step(L);
  for (int64_t b0 = 0; b0 < batch;) {
    const int64_t left = batch - b0;
    const int count = share > 1 ? (int)(left < share ? left : share) : 1;
    const Fitness fit = one_part(f + b0 * stride_batch, n, sr, sc, stride_batch);
    if (int e = rank_rows(fit, n, m, stop_count, rank_out + b0 * n, ws, ws_bytes, (hipStream_t)stream, count, count > 1 ? (int64_t)step : 0))
      return e;
    b0 += count;
  }
  return 0;
}

int evox_hip_many_nd_environmental_selection(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes,
                                             int64_t x_batch_stride_bytes, const float* f, int64_t batch, int64_t n, int64_t m,
                                             int64_t stride_batch, int64_t sr, int64_t sc, int64_t topk, void* out_x, float* out_f,
                                             int32_t* out_rank, float* out_dist, void* ws, size_t ws_bytes, void* stream) {
  Layout L;
  if (f == nullptr || batch < 1 || !make_layout(n, m, &L) || topk < 1 || topk > n) return kErrBadArg;
  if ((x == nullptr) != (out_x == nullptr) || (x != nullptr && (x_row_bytes < 0 || x_batch_stride_bytes < 0))) return kErrBadArg;
  const int share = many_populations_share(L, batch, topk);
  const size_t step = many_workspace_step(L);
  for (int64_t b0 = 0; b0 < batch;) {
    const int64_t left = batch - b0;
    const int count = share > 1 ? (int)(left < share ? left : share) : 1;
    const Fitness fit = one_part(f + b0 * stride_batch, n, sr, sc, stride_batch);
    const uint8_t* xb = x != nullptr ? static_cast<const uint8_t*>(x) + b0 * x_batch_stride_bytes : nullptr;
    uint8_t* oxb = out_x != nullptr ? static_cast<uint8_t*>(out_x) + b0 * topk * x_row_bytes : nullptr;
    if (int e = select_rows(xb, x_row_bytes, x_row_stride_bytes, xb, x_row_stride_bytes, fit, n, m, topk, oxb, out_f + b0 * topk * m,
                            out_rank + b0 * topk, out_dist + b0 * topk, nullptr, ws, ws_bytes, (hipStream_t)stream, true, count,
                            count > 1 ? (int64_t)step : 0, x_batch_stride_bytes, x_batch_stride_bytes))
      return e;
    b0 += count;
  }
  return 0;
}

}  // extern "C"

// Parts of a sorted row of n values in dense_rank_kernel, `rows` rows in the launch: as many as there are compute units
// for each row, none smaller than one value per thread.  Every part reads all values before it, so more parts than
// compute units would only add reads.  The reads of the last part, a whole row by one workgroup, bound the kernel for long rows,
// and stay below what one workgroup takes for the row alone up to the most values there are: a row of 2^20 129 us against
// 1904, of 2^24 - 1 2404 against 32 915, 64 rows of 300 000 485 against 767.
static int dense_rank_parts(int64_t rows, int64_t n) {
  const int64_t most = (n + kDenseRankThreads - 1) / kDenseRankThreads, share = device_cus() / rows;
  return (int)(share < 1 ? 1 : share < most ? share : most);
}

extern "C" {

int evox_hip_dense_rank_rows(const void* sorted, int kind, const int64_t* index, int64_t batch, int64_t n, int64_t m, float* out,
                             void* stream) {
  if (sorted == nullptr || index == nullptr || out == nullptr || (kind != kWideFloat64 && kind != kWideInt64)) return kErrBadArg;
  if (batch < 1 || n < 1 || m < 1 || n >= (1ll << 24) || batch * m > 0x7FFFFFFFll) return kErrBadArg;
  hipStream_t s = (hipStream_t)stream;
  const int parts = dense_rank_parts(batch * m, n);
  const int per = (int)round_up((n + parts - 1) / parts, kDenseRankThreads);
  const dim3 grid((unsigned)(batch * m), (unsigned)((n + per - 1) / per));
  if (kind == kWideFloat64)
    hipLaunchKernelGGL(dense_rank_kernel<double>, grid, dim3(kDenseRankThreads), 0, s, static_cast<const double*>(sorted), index,
                       (int)n, (int)m, per, out);
  else
    hipLaunchKernelGGL(dense_rank_kernel<long long>, grid, dim3(kDenseRankThreads), 0, s, static_cast<const long long*>(sorted), index,
                       (int)n, (int)m, per, out);
  EVX_LAUNCH_CHECK();
  return 0;
}

size_t evox_hip_wide_workspace_bytes(int64_t n, int64_t m) {
  WideLayout L;
  return make_wide_layout(n, m, &L) ? L.total : 0;
}

int evox_hip_crowding_distance_wide(const void* costs, int kind, int64_t n, int64_t m, int64_t sr, int64_t sc, const uint8_t* mask,
                                    int64_t mask_stride, void* dist_out, int out_kind, void* ws, size_t ws_bytes, void* stream) {
  WideLayout L;
  if (costs == nullptr || dist_out == nullptr || (kind != kWideFloat64 && kind != kWideInt64) || (out_kind != 0 && out_kind != 1))
    return kErrBadArg;
  if (!make_wide_layout(n, m, &L)) return kErrBadArg;
  if (ws == nullptr || ws_bytes < L.total || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  return wide_distances(L, static_cast<uint8_t*>(ws), costs, kind, sr, sc, mask, mask_stride, nullptr, dist_out, out_kind, false,
                        (hipStream_t)stream);
}

int evox_hip_nd_environmental_selection_wide(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes, const void* f_rows,
                                             int64_t f_row_bytes, int64_t f_row_stride_bytes, const void* costs, int kind, int64_t n,
                                             int64_t m, int64_t sr, int64_t sc, const int32_t* rank, int64_t topk, void* out_x,
                                             void* out_f, int32_t* out_rank, void* out_dist, int out_kind, void* ws, size_t ws_bytes,
                                             void* stream) {
  WideLayout L;
  if (costs == nullptr || rank == nullptr || f_rows == nullptr || out_f == nullptr || out_rank == nullptr || out_dist == nullptr)
    return kErrBadArg;
  if ((kind != kWideFloat64 && kind != kWideInt64) || (out_kind != 0 && out_kind != 1)) return kErrBadArg;
  if ((x == nullptr) != (out_x == nullptr) || x_row_bytes < 0 || x_row_stride_bytes < 0 || f_row_bytes < 1 || f_row_stride_bytes < 0)
    return kErrBadArg;
  if (!make_wide_layout(n, m, &L) || topk < 1 || topk > n) return kErrBadArg;
  if (ws == nullptr || ws_bytes < L.total || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  hipStream_t s = (hipStream_t)stream;
  uint8_t* base = static_cast<uint8_t*>(ws);
  void* dist = base + L.dist;
  int* order_a = reinterpret_cast<int*>(base + L.order_a);
  int* order_b = reinterpret_cast<int*>(base + L.order_b);
  int* const outcome = opt().launch_memory ? outcome_slot(kWordWide, n, m, true, s) : nullptr;
  if (wide_direct_applies(n, outcome)) {
    if (int e = wide_select_direct(L, base, costs, kind, sr, sc, rank, dist, out_kind, order_a, s, outcome)) return e;
  } else {
    if (int e = wide_distances(L, base, costs, kind, sr, sc, nullptr, 0, rank, dist, out_kind, true, s, outcome)) return e;
    // rows by rank, then by distance descending (NaN last), then by index: one stable step per key part, least
    // significant first (src/evox/operators/selection/non_dominate.py:253, src/evox/utils/jit_fix_operator.py:246-250)
    void* sort_ws = base + L.sort_ws;
    if (int e = evox_hip_stable_argsort_step(base + L.neg_lo, kKeyUint32, 1, n, nullptr, order_a, sort_ws, L.sort_bytes, s)) return e;
    if (int e = evox_hip_stable_argsort_step(base + L.neg_hi, kKeyUint32, 1, n, order_a, order_b, sort_ws, L.sort_bytes, s)) return e;
    if (int e = evox_hip_stable_argsort_step(rank, kKeyInt32, 1, n, order_b, order_a, sort_ws, L.sort_bytes, s)) return e;
  }
  const int64_t dist_bytes = out_kind == 0 ? 8 : 4;
  const WideGather gather = {x, x_row_bytes, x_row_stride_bytes, 0, f_rows, f_row_bytes, f_row_stride_bytes, 0, rank, dist, dist_bytes, 0,
                             out_x, out_f, out_rank, out_dist};
  return wide_gather(gather, order_a, 0, n, topk, 1, s);
}

int evox_hip_many_nd_environmental_selection_wide(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes, int64_t x_batch_stride_bytes,
                                                  const void* f_rows, int64_t f_row_bytes, int64_t f_row_stride_bytes,
                                                  int64_t f_batch_stride_bytes, const void* costs, int kind, int64_t batch, int64_t n,
                                                  int64_t m, int64_t stride_batch, int64_t sr, int64_t sc, const int32_t* rank,
                                                  int64_t topk, void* out_x, void* out_f, int32_t* out_rank, void* out_dist,
                                                  int out_kind, void* ws, size_t ws_bytes, void* stream) {
  WideLayout L;
  if (batch < 1 || !make_wide_layout(n, m, &L) || topk < 1 || topk > n) return kErrBadArg;
  if ((kind != kWideFloat64 && kind != kWideInt64) || (out_kind != 0 && out_kind != 1)) return kErrBadArg;
  const int64_t step = (int64_t)align_up(L.total);
  const int64_t dist_bytes = out_kind == 0 ? 8 : 4;
  hipStream_t s = (hipStream_t)stream;
  int* const outcome = opt().launch_memory ? outcome_slot(kWordWide, n, m, true, s) : nullptr;
  const int64_t x_out_step = topk * x_row_bytes, f_out_step = topk * f_row_bytes;
  const bool together = batch > 1 && wide_direct_applies(n, outcome) && (n <= kSmallArgsortRows || opt().mid_argsort) &&
                        ws_bytes >= (size_t)step * (size_t)batch && batch <= 65535;
  if (!together) {  // one population after the other, each through the single-population entry point
    for (int64_t b = 0; b < batch; ++b) {
      const int e = evox_hip_nd_environmental_selection_wide(
          x ? static_cast<const char*>(x) + b * x_batch_stride_bytes : nullptr, x_row_bytes, x_row_stride_bytes,
          static_cast<const char*>(f_rows) + b * f_batch_stride_bytes, f_row_bytes, f_row_stride_bytes,
          static_cast<const char*>(costs) + b * stride_batch * 8, kind, n, m, sr, sc, rank + b * n, topk,
          out_x ? static_cast<char*>(out_x) + b * x_out_step : nullptr, static_cast<char*>(out_f) + b * f_out_step, out_rank + b * topk,
          static_cast<char*>(out_dist) + b * topk * dist_bytes, out_kind, ws, ws_bytes, stream);
      if (e) return e;
    }
    return 0;
  }
  if (costs == nullptr || rank == nullptr || f_rows == nullptr || out_f == nullptr || out_rank == nullptr || out_dist == nullptr)
    return kErrBadArg;
  if ((x == nullptr) != (out_x == nullptr) || x_row_bytes < 0 || x_row_stride_bytes < 0 || f_row_bytes < 1 || f_row_stride_bytes < 0)
    return kErrBadArg;
  if (ws == nullptr || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  uint8_t* base = static_cast<uint8_t*>(ws);
  void* dist = base + L.dist;
  int* order = reinterpret_cast<int*>(base + L.order_a);
  if (int e = wide_select_direct(L, base, costs, kind, sr, sc, rank, dist, out_kind, order, s, outcome, (int)batch, step, stride_batch * 8))
    return e;
  const WideGather gather = {x, x_row_bytes, x_row_stride_bytes, x_batch_stride_bytes, f_rows, f_row_bytes, f_row_stride_bytes,
                             f_batch_stride_bytes, rank, dist, dist_bytes, step, out_x, out_f, out_rank, out_dist};
  return wide_gather(gather, order, step, n, topk, (int)batch, s);
}

}  // extern "C"

extern "C" {

int evox_hip_nd_environmental_selection_wide_whole(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes, const void* f_rows,
                                                   int64_t f_row_bytes, int64_t f_row_stride_bytes, const void* costs, int kind,
                                                   int64_t n, int64_t m, int64_t sr, int64_t sc, int64_t topk, void* out_x, void* out_f,
                                                   int32_t* out_rank, void* out_dist, int out_kind, void* ws, size_t ws_bytes,
                                                   void* stream) {
  Ws w;
  if (costs == nullptr || f_rows == nullptr || out_f == nullptr || out_rank == nullptr || out_dist == nullptr) return kErrBadArg;
  if ((kind != kWideFloat64 && kind != kWideInt64) || (out_kind != 0 && out_kind != 1)) return kErrBadArg;
  if ((x == nullptr) != (out_x == nullptr) || x_row_bytes < 0 || x_row_stride_bytes < 0 || f_row_bytes < 1 || f_row_stride_bytes < 0)
    return kErrBadArg;
  if (n > kRunMaxRows || topk < 1 || topk > n) return kErrBadArg;
  if (int e = open_ws(n, m, ws, ws_bytes, &w)) return e;
  const Layout& L = w.L;
  WideLayout WL;
  if (!make_wide_layout(n, m, &WL) || WL.total > L.wide_bytes) return kErrWorkspace;
  uint8_t* const wb = w.base + L.wide;
  hipStream_t s = (hipStream_t)stream;
  // (regions of the 8-byte kernels' part of the workspace: the two halves of the keys lie side by side and hold whole
  // images, the image that is ranked lies where the terms go later)
  uint64_t* const runs = reinterpret_cast<uint64_t*>(wb + WL.key_lo);
  int* const whose = reinterpret_cast<int*>(wb + WL.ord_a);
  float* const images = reinterpret_cast<float*>(wb + WL.terms);
  const int all_runs = runs_of((int)n), most_shares = (int)((n + kWideShare - 1) / kWideShare);
  const size_t lds = run_rank8_lds_bytes((int)n);
  if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(value_images_kernel), lds)) return e;
  hipLaunchKernelGGL(value_runs_kernel, dim3(all_runs, (unsigned)m), dim3(kRunRows), 0, s, costs, kind, sr, sc, (int)n, runs, whose);
  EVX_LAUNCH_CHECK();
  hipLaunchKernelGGL(value_images_kernel, dim3(most_shares, (unsigned)m), dim3(kRunRankThreads), lds, s, runs, whose, kind, (int)n, (int)m,
                     images);
  EVX_LAUNCH_CHECK();
  const Fitness fit = one_part(images, n, m, 1);
  bool stepped = false;
  int ranked = kErrNotResident;
  if (two_applies(L, topk)) ranked = stage_rank_two(w, fit, topk, false, nullptr, s);
  if (ranked == kErrNotResident) {
    if (int e = stage_prepare(w, fit, true, s)) return e;
    if (int e = stage_dominance(w, kDomAuto, s)) return e;
    ranked = count_and_peel(w, topk, true, false, s, false, nullptr, nullptr, &stepped);
  }
  if (ranked) return ranked;
  if (stepped) {  // (its fronts have no listing: the order from the ranks alone)
    if (int e = copy_out(w.ctrl(), w.at<int>(L.order), w.at<int>(L.rank), n, kPoisonIndex, s)) return e;
    return evox_hip_nd_environmental_selection_wide(x, x_row_bytes, x_row_stride_bytes, f_rows, f_row_bytes, f_row_stride_bytes, costs,
                                                    kind, n, m, sr, sc, w.at<int>(L.order), topk, out_x, out_f, out_rank, out_dist,
                                                    out_kind, wb, L.wide_bytes, stream);
  }
  WideFront a = {};
  a.costs = costs;
  a.kind = kind;
  a.stride_row = sr;
  a.stride_col = sc;
  a.n = (int)n;
  a.m = (int)m;
  a.list_base = w.at<int>(L.perm);
  a.ctrl = w.ctrl();
  a.runs = runs;
  a.whose = whose;
  a.terms = wb + WL.terms;
  a.dist = wb + WL.dist;
  a.dist_runs = reinterpret_cast<uint64_t*>(wb + WL.front_dkey);
  a.dist_whose = reinterpret_cast<int*>(wb + WL.order_a);
  a.topk = (int)topk;
  auto unit_of = [](const void* src, const void* dst, int64_t row_bytes, int64_t stride) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) | (uintptr_t)row_bytes | (uintptr_t)stride;
    return bits % 16 == 0 ? 16 : bits % 8 == 0 ? 8 : bits % 4 == 0 ? 4 : 1;
  };
  a.x = static_cast<const uint8_t*>(x);
  a.x_row_bytes = x_row_bytes;
  a.x_row_stride = x_row_stride_bytes;
  a.x_unit = unit_of(x, out_x, x_row_bytes, x_row_stride_bytes);
  a.out_x = static_cast<uint8_t*>(out_x);
  a.f = static_cast<const uint8_t*>(f_rows);
  a.f_row_bytes = f_row_bytes;
  a.f_row_stride = f_row_stride_bytes;
  a.f_unit = unit_of(f_rows, out_f, f_row_bytes, f_row_stride_bytes);
  a.out_f = static_cast<uint8_t*>(out_f);
  a.rank = w.at<int>(L.rank);
  a.out_rank = out_rank;
  a.out_dist = out_dist;
  int runs_grid = all_runs * (int)m;
  if (runs_grid > 65536) runs_grid = 65536;
  const int shares = device_cus() / (int)m > most_shares ? device_cus() / (int)m : most_shares;  // workgroups of one objective
  const int picks = device_cus() > most_shares ? device_cus() : most_shares;
  auto launch = [&](auto terms_kernel, auto distances_kernel, auto pick_kernel) -> int {
    if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(terms_kernel), lds)) return e;
    if (int e = grant_dynamic_lds(reinterpret_cast<const void*>(pick_kernel), lds)) return e;
    hipLaunchKernelGGL(wide_front_runs_kernel, dim3(runs_grid), dim3(kRunRows), 0, s, a);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(terms_kernel, dim3(shares * (int)m), dim3(kRunRankThreads), lds, s, a);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(distances_kernel, dim3(all_runs), dim3(kRunRows), 0, s, a);
    EVX_LAUNCH_CHECK();
    hipLaunchKernelGGL(pick_kernel, dim3(picks), dim3(kRunRankThreads), lds, s, a);
    EVX_LAUNCH_CHECK();
    return 0;
  };
  if (out_kind == 0) return launch(wide_front_terms_kernel<double>, wide_front_distances_kernel<double>, wide_front_pick_kernel<double>);
  return launch(wide_front_terms_kernel<float>, wide_front_distances_kernel<float>, wide_front_pick_kernel<float>);
}

}  // extern "C"

// Scratch memory of the entry point that allocates nothing: part of the device image, one copy per GPU.  In host
// code the array's name stands for the symbol, not for device memory: its address on the current GPU comes from
// hipGetSymbolAddress, looked up once per device and kept.
static __device__ __align__(256) unsigned char scratch[EVOX_HIP_STATIC_SCRATCH_BYTES];
static std::atomic<void*> g_scratch_ptr[64];

static int static_scratch(void** out) {
  int dev = 0;
  const hipError_t de = hipGetDevice(&dev);
  if (de != hipSuccess) return (int)de;
  if (dev < 0 || dev >= 64) return kErrBadArg;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (p == nullptr || (reinterpret_cast<uintptr_t>(p) & 255u) != 0) return kErrWorkspace;
    g_scratch_ptr[dev].store(p, std::memory_order_release);  // (two first calls at once look up the same address)
  }
  *out = p;
  return 0;
}

extern "C" {

int evox_hip_nd_environmental_selection_static(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes,
                                               const float* f, int64_t n, int64_t m, int64_t sr, int64_t sc, int64_t topk,
                                               void* out_x, float* out_f, int32_t* out_rank, float* out_dist,
                                               int32_t* out_order, void* stream) {
  if (f == nullptr) return kErrBadArg;
  const size_t need = evox_hip_workspace_bytes(n, m);
  if (need == 0) return kErrBadArg;
  if (need > (size_t)EVOX_HIP_STATIC_SCRATCH_BYTES) return kErrStaticLimit;
  void* ws = nullptr;
  if (int e = static_scratch(&ws)) return e;
  // every call clears the part of the buffer that must start from zero (stage_prepare), whatever the call before
  // left there
  return select_rows(x, x_row_bytes, x_row_stride_bytes, x, x_row_stride_bytes, one_part(f, n, sr, sc), n, m, topk, out_x,
                     out_f, out_rank, out_dist, out_order, ws, (size_t)EVOX_HIP_STATIC_SCRATCH_BYTES, (hipStream_t)stream, false);
}

int64_t evox_hip_batched_max_rows(int64_t m) { return batched_rows_limit(m); }

int evox_hip_batched_non_dominate_rank(const float* f, int64_t batch, int64_t n, int64_t m, int64_t stride_batch,
                                       int64_t stride_row, int64_t stride_col, int32_t* rank_out, void* stream) {
  if (f == nullptr || rank_out == nullptr || batch < 1 || n < 1 || n > batched_rows_limit(m)) return kErrBadArg;
  BatchedArgs a = {};
  a.f = f;
  a.f_stride_b = stride_batch;
  a.f_stride_row = stride_row;
  a.f_stride_col = stride_col;
  a.n = (int)n;
  a.m = (int)m;
  a.stop_count = (int)n;
  a.rank_all = rank_out;
  return launch_batched(a, batch, (hipStream_t)stream);
}

int evox_hip_batched_nd_environmental_selection(const void* x, int64_t x_row_bytes, int64_t x_row_stride_bytes,
                                                int64_t x_batch_stride_bytes, const float* f, int64_t batch, int64_t n,
                                                int64_t m, int64_t stride_batch, int64_t stride_row, int64_t stride_col,
                                                int64_t topk, void* out_x, float* out_f, int32_t* out_rank, float* out_dist,
                                                void* stream) {
  if (f == nullptr || out_f == nullptr || out_rank == nullptr || out_dist == nullptr) return kErrBadArg;
  if (batch < 1 || n < 1 || n > batched_rows_limit(m) || topk < 1 || topk > n) return kErrBadArg;
  if ((x == nullptr) != (out_x == nullptr) || (x != nullptr && (x_row_bytes < 0 || x_row_stride_bytes < 0))) return kErrBadArg;
  BatchedArgs a = {};
  a.f = f;
  a.f_stride_b = stride_batch;
  a.f_stride_row = stride_row;
  a.f_stride_col = stride_col;
  a.n = (int)n;
  a.m = (int)m;
  a.stop_count = (int)topk;
  a.x = static_cast<const uint8_t*>(x);
  a.x_stride_b = x_batch_stride_bytes;
  a.x_row_stride = x_row_stride_bytes;
  a.x_row_bytes = x_row_bytes;
  a.out_x = static_cast<uint8_t*>(out_x);
  a.out_f = out_f;
  a.out_rank = out_rank;
  a.out_dist = out_dist;
  a.x_unit = 1;
  if (x != nullptr) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out_x) | (uintptr_t)x_row_bytes |
                           (uintptr_t)x_row_stride_bytes | (uintptr_t)x_batch_stride_bytes;
    a.x_unit = (bits % 16 == 0) ? 16 : (bits % 4 == 0) ? 4 : 1;
  }
  return launch_batched(a, batch, (hipStream_t)stream);
}

int evox_hip_small_nd_environmental_selection_two_part(const void* x_a, const void* x_b, int64_t x_row_bytes,
                                                       int64_t x_row_stride_bytes, const float* f_a, int64_t n_a,
                                                       const float* f_b, int64_t n_b, int64_t m, int64_t stride_row,
                                                       int64_t stride_col, int64_t topk, void* out_x, float* out_f,
                                                       int32_t* out_rank, float* out_dist, void* stream) {
  if (f_a == nullptr || f_b == nullptr || out_f == nullptr || out_rank == nullptr || out_dist == nullptr) return kErrBadArg;
  if (n_a < 1 || n_b < 1 || n_a + n_b > batched_rows_limit(m)) return kErrBadArg;
  const int64_t n = n_a + n_b;
  if (topk < 1 || topk > n) return kErrBadArg;
  if ((x_a == nullptr) != (out_x == nullptr) || (x_a == nullptr) != (x_b == nullptr)) return kErrBadArg;
  if (x_a != nullptr && (x_row_bytes < 0 || x_row_stride_bytes < 0)) return kErrBadArg;
  BatchedArgs a = {};
  a.f = f_a;
  a.f_stride_row = stride_row;
  a.f_stride_col = stride_col;
  a.n = (int)n;
  a.m = (int)m;
  a.stop_count = (int)topk;
  a.n_first = (int)n_a;
  // row i >= n_a of the population is row i - n_a of part b: f_a + i * stride_row + f_second
  a.f_second = (f_b - f_a) - n_a * stride_row;
  a.x = static_cast<const uint8_t*>(x_a);
  a.x_row_stride = x_row_stride_bytes;
  a.x_row_bytes = x_row_bytes;
  a.out_x = static_cast<uint8_t*>(out_x);
  a.out_f = out_f;
  a.out_rank = out_rank;
  a.out_dist = out_dist;
  a.x_unit = 1;
  if (x_a != nullptr) {
    a.x_second = (static_cast<const uint8_t*>(x_b) - static_cast<const uint8_t*>(x_a)) - n_a * x_row_stride_bytes;
    const uintptr_t bits = reinterpret_cast<uintptr_t>(x_a) | reinterpret_cast<uintptr_t>(x_b) | reinterpret_cast<uintptr_t>(out_x) |
                           (uintptr_t)x_row_bytes | (uintptr_t)x_row_stride_bytes;
    a.x_unit = (bits % 16 == 0) ? 16 : (bits % 4 == 0) ? 4 : 1;
  }
  return launch_batched(a, 1, (hipStream_t)stream);
}

int evox_hip_tournament_pick(const int64_t* parents, int64_t n_round, int64_t tournament_size, const float* fit,
                             int64_t n_candidates, int64_t n_keys, int64_t stride_row, int64_t stride_col, int64_t* out,
                             void* stream) {
  if (parents == nullptr || fit == nullptr || out == nullptr) return kErrBadArg;
  if (n_round < 0 || tournament_size < 1 || tournament_size > 0x7FFFFFFF || n_candidates < 1 || n_keys < 1 || n_keys > 0x7FFFFFFF)
    return kErrBadArg;
  if (n_round == 0) return 0;
  int64_t blocks = (n_round + 255) / 256;
  if (blocks > 65535) blocks = 65535;
  hipLaunchKernelGGL(tournament_pick_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, parents, n_round,
                     (int)tournament_size, fit, stride_row, stride_col, (int)n_keys, out);
  EVX_LAUNCH_CHECK();
  return 0;
}

int evox_hip_tournament_pick_keys(const int64_t* parents, int64_t n_round, int64_t tournament_size, int64_t n_candidates,
                                  int64_t n_keys, const void* const* keys, const int32_t* kinds, const int64_t* strides,
                                  int64_t* out, void* stream) {
  if (parents == nullptr || keys == nullptr || kinds == nullptr || strides == nullptr || out == nullptr) return kErrBadArg;
  if (n_round < 0 || tournament_size < 1 || tournament_size > 0x7FFFFFFF || n_candidates < 1 || n_keys < 1 || n_keys > 4)
    return kErrBadArg;
  TournamentKeys t = {};
  for (int k = 0; k < (int)n_keys; ++k) {
    if (keys[k] == nullptr || (kinds[k] != 0 && kinds[k] != 1)) return kErrBadArg;
    t.key[k] = keys[k];
    t.kind[k] = kinds[k];
    t.stride[k] = strides[k];
  }
  t.nkeys = (int)n_keys;
  if (n_round == 0) return 0;
  int64_t blocks = (n_round + 255) / 256;
  if (blocks > 65535) blocks = 65535;
  hipLaunchKernelGGL(tournament_pick_keys_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, parents, n_round,
                     (int)tournament_size, t, out);
  EVX_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"

// What the two uses of the points against the samples keep in their workspace.
struct HvBytes {
  size_t packed, partial, alpha, points, extreme, covered, cover;
};
static HvBytes hv_bytes(int64_t n, int64_t m, int64_t n_sample) {
  HvBytes b;
  const int64_t share = hv_share(n_sample);
  b.packed = align_up(sizeof(float) * (size_t)hv_packed((int)m) * (size_t)n_sample);
  b.partial = align_up(sizeof(float) * (size_t)((n_sample + share - 1) / share) * (size_t)n);
  b.alpha = align_up(sizeof(float) * (size_t)n);
  b.points = align_up(sizeof(float) * (size_t)n * (size_t)m);
  b.extreme = align_up(sizeof(float) * (size_t)kHvParts * (size_t)m);
  b.covered = align_up(sizeof(uint64_t) * (size_t)((n_sample + 63) / 64));
  b.cover = align_up(sizeof(int) * (size_t)n_sample);
  return b;
}
static bool hv_sizes_fit(int64_t n, int64_t n_sample) { return n >= 1 && n_sample >= 1 && n <= 0x7FFFFF00ll && n_sample <= 0x7FFFFF00ll; }

// The kernels are built for 1 to 8 objectives, for up to kHvRegs (their number read at run time) and for any number.
template <typename F>
static int hv_for_objectives(int64_t m, F&& launch) {
  switch (m) {
    case 1: return launch(std::integral_constant<int, 1>());
    case 2: return launch(std::integral_constant<int, 2>());
    case 3: return launch(std::integral_constant<int, 3>());
    case 4: return launch(std::integral_constant<int, 4>());
    case 5: return launch(std::integral_constant<int, 5>());
    case 6: return launch(std::integral_constant<int, 6>());
    case 7: return launch(std::integral_constant<int, 7>());
    case 8: return launch(std::integral_constant<int, 8>());
    default: break;
  }
  if (m <= kHvRegs) return launch(std::integral_constant<int, kHvRegs>());
  return launch(std::integral_constant<int, 0>());
}

static HvSplit hv_split_for(int64_t n, int64_t m, int64_t n_sample) { return hv_split(n, n_sample, hv_step((int)m), device_cus()); }

// cover: zero where the split has several parts.
template <int kMode>
static int hv_contribution_launches(const float* points_t, const HvSamples& samples, const float* alpha, int64_t n, int64_t m,
                                    int64_t n_sample, float scale, const HvSplit& split, float* packed, int* cover, float* partial,
                                    float* out, hipStream_t s) {
  const int64_t share = hv_share(n_sample);
  const int shares = (int)((n_sample + share - 1) / share);
  const unsigned blocks = (unsigned)((n_sample + 63) / 64);
  if (int e = hv_for_objectives(m, [&](auto objectives) {
        constexpr int M = decltype(objectives)::value;
        hipLaunchKernelGGL((hv_sample_weight_kernel<M, kMode>), dim3(blocks, split.parts), dim3(split.threads), 0, s, points_t, samples,
                           (int)n, (int)m, (int)n_sample, alpha, packed, cover);
        EVX_LAUNCH_CHECK();
        if (split.parts > 1) {
          hipLaunchKernelGGL((hv_weight_kernel<M, kMode>), dim3(blocks), dim3(64), 0, s, samples, (int)m, (int)n_sample, cover, alpha, packed);
          EVX_LAUNCH_CHECK();
        }
        hipLaunchKernelGGL(hv_point_partial_kernel<M>, dim3((unsigned)((n + 255) / 256), (unsigned)shares), dim3(256), 0, s, points_t,
                           packed, samples, (int)n, (int)m, (int)n_sample, (int)share, partial);
        EVX_LAUNCH_CHECK();
        return 0;
      }))
    return e;
  hipLaunchKernelGGL(hv_point_total_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, partial, samples, (int)n, (int)m, shares,
                     (int)n_sample, scale, out);
  EVX_LAUNCH_CHECK();
  return 0;
}

// covered: zero where the split has several parts.
template <int kMode>
static int hv_covered_launch(const float* points_t, const HvSamples& samples, int64_t n, int64_t m, int64_t n_sample,
                             const HvSplit& split, unsigned long long* covered, hipStream_t s) {
  return hv_for_objectives(m, [&](auto objectives) {
    constexpr int M = decltype(objectives)::value;
    hipLaunchKernelGGL((hv_covered_kernel<M, kMode>), dim3((unsigned)((n_sample + 63) / 64), split.parts), dim3(split.threads), 0, s,
                       points_t, samples, (int)n, (int)m, (int)n_sample, covered);
    EVX_LAUNCH_CHECK();
    return 0;
  });
}

static int hv_clear(void* words, int64_t n_words, hipStream_t s) {
  const int64_t blocks = (n_words + 255) / 256;
  hipLaunchKernelGGL(reset_state_kernel, dim3((unsigned)(blocks < 64 ? blocks : 64)), dim3(256), 0, s, static_cast<uint32_t*>(words), n_words);
  EVX_LAUNCH_CHECK();
  return 0;
}

extern "C" {

size_t evox_hip_hv_workspace_bytes(int64_t n, int64_t n_sample) {
  if (!hv_sizes_fit(n, n_sample)) return 0;
  const HvBytes b = hv_bytes(n, kHvRegs, n_sample);  // (the call's objectives are not known here)
  return b.packed + b.partial + b.cover;
}

int evox_hip_hv_contributions(const float* fit_t, const float* samples_t, const float* alpha, int64_t n, int64_t m,
                              int64_t n_sample, float scale, float* out, void* ws, size_t ws_bytes, void* stream) {
  if (fit_t == nullptr || samples_t == nullptr || alpha == nullptr || out == nullptr || m < 1 || m > 65535) return kErrBadArg;
  const size_t need = evox_hip_hv_workspace_bytes(n, n_sample);
  if (need == 0) return kErrBadArg;
  if (ws == nullptr || ws_bytes < need || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  const HvBytes b = hv_bytes(n, kHvRegs, n_sample);
  uint8_t* base = static_cast<uint8_t*>(ws);
  int* cover = reinterpret_cast<int*>(base + b.packed + b.partial);
  const HvSplit split = hv_split_for(n, m, n_sample);
  if (split.parts > 1) {
    if (int e = hv_clear(cover, n_sample, (hipStream_t)stream)) return e;
  }
  const HvSamples samples = {samples_t, 1, n_sample, nullptr, nullptr, 0, 0};
  return hv_contribution_launches<kHvPlain>(fit_t, samples, alpha, n, m, n_sample, scale, split, reinterpret_cast<float*>(base), cover,
                                            reinterpret_cast<float*>(base + b.packed), out, (hipStream_t)stream);
}

size_t evox_hip_hype_workspace_bytes(int64_t n, int64_t m, int64_t n_sample) {
  if (!hv_sizes_fit(n, n_sample) || m < 1 || m > kHvRegs) return 0;
  const HvBytes b = hv_bytes(n, m, n_sample);
  return b.packed + b.partial + b.alpha + b.points + b.extreme + b.cover;
}

int evox_hip_hype_contributions(const float* f, int64_t stride_row, int64_t stride_col, int64_t n, int64_t m, const float* ref,
                                int64_t ref_stride, int64_t pop_size, const float* u, int64_t n_sample, float* out, void* ws,
                                size_t ws_bytes, void* stream) {
  const size_t need = evox_hip_hype_workspace_bytes(n, m, n_sample);
  if (need == 0 || f == nullptr || ref == nullptr || u == nullptr || out == nullptr || pop_size < 1) return kErrBadArg;
  if (ws == nullptr || ws_bytes < need || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  hipStream_t s = (hipStream_t)stream;
  const HvBytes b = hv_bytes(n, m, n_sample);
  uint8_t* at = static_cast<uint8_t*>(ws);
  float* packed = reinterpret_cast<float*>(at);
  float* partial = reinterpret_cast<float*>(at += b.packed);
  float* alpha = reinterpret_cast<float*>(at += b.partial);
  float* points = reinterpret_cast<float*>(at += b.alpha);
  float* extreme = reinterpret_cast<float*>(at += b.points);
  int* cover = reinterpret_cast<int*>(at += b.extreme);
  const int parts = hv_parts(n);
  const HvSplit split = hv_split_for(n, m, n_sample);
  hipLaunchKernelGGL(hv_points_kernel<false>, dim3((unsigned)parts + 1), dim3(256), 0, s, f, stride_row, stride_col, ref, ref_stride,
                     (int)n, (int)m, parts, points, extreme, alpha, pop_size, reinterpret_cast<uint32_t*>(cover),
                     split.parts > 1 ? n_sample : 0);
  EVX_LAUNCH_CHECK();
  const HvSamples samples = {u, m, 1, extreme, ref, ref_stride, parts};
  return hv_contribution_launches<kHvHype>(points, samples, alpha, n, m, n_sample, 1.0f, split, packed, cover, partial, out, s);
}

size_t evox_hip_hv_covered_workspace_bytes(int64_t n_sample) {
  if (n_sample < 1 || n_sample > 0x7FFFFF00ll) return 0;
  return hv_bytes(1, 1, n_sample).covered;
}

int evox_hip_hv_covered_count(const float* points_t, const float* samples_t, int64_t n, int64_t m, int64_t n_sample,
                              int64_t* out_count, void* ws, size_t ws_bytes, void* stream) {
  if (points_t == nullptr || samples_t == nullptr || out_count == nullptr || n < 1 || n > 65535ll * 1024 || m < 1 || m > 65535)
    return kErrBadArg;
  const size_t need = evox_hip_hv_covered_workspace_bytes(n_sample);
  if (need == 0) return kErrBadArg;
  if (ws == nullptr || ws_bytes < need || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  hipStream_t s = (hipStream_t)stream;
  unsigned long long* covered = static_cast<unsigned long long*>(ws);
  const HvSplit split = hv_split_for(n, m, n_sample);
  if (split.parts > 1) {
    if (int e = hv_clear(covered, 2 * ((n_sample + 63) / 64), s)) return e;
  }
  const HvSamples samples = {samples_t, 1, n_sample, nullptr, nullptr, 0, 0};
  if (int e = hv_covered_launch<kHvPlain>(points_t, samples, n, m, n_sample, split, covered, s)) return e;
  hipLaunchKernelGGL(hv_covered_total_kernel<false>, dim3(1), dim3(1024), 0, s, covered, (int)((n_sample + 63) / 64), samples, (int)m,
                     (int)n_sample, out_count, (float*)nullptr);
  EVX_LAUNCH_CHECK();
  return 0;
}

size_t evox_hip_hv_estimate_workspace_bytes(int64_t n, int64_t m, int64_t n_sample) {
  if (!hv_sizes_fit(n, n_sample) || m < 1 || m > kHvRegs) return 0;
  const HvBytes b = hv_bytes(n, m, n_sample);
  return b.points + b.extreme + b.covered;
}

int evox_hip_hv_estimate(const float* objs, int64_t stride_row, int64_t stride_col, int64_t n, int64_t m, const float* ref,
                         int64_t ref_stride, const float* u, int64_t n_sample, float* out, void* ws, size_t ws_bytes, void* stream) {
  const size_t need = evox_hip_hv_estimate_workspace_bytes(n, m, n_sample);
  if (need == 0 || objs == nullptr || ref == nullptr || u == nullptr || out == nullptr) return kErrBadArg;
  if (ws == nullptr || ws_bytes < need || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0) return kErrWorkspace;
  hipStream_t s = (hipStream_t)stream;
  const HvBytes b = hv_bytes(n, m, n_sample);
  uint8_t* at = static_cast<uint8_t*>(ws);
  float* points = reinterpret_cast<float*>(at);
  float* extreme = reinterpret_cast<float*>(at += b.points);
  unsigned long long* covered = reinterpret_cast<unsigned long long*>(at += b.extreme);
  const int parts = hv_parts(n);
  const HvSplit split = hv_split_for(n, m, n_sample);
  hipLaunchKernelGGL(hv_points_kernel<true>, dim3((unsigned)parts), dim3(256), 0, s, objs, stride_row, stride_col, ref, ref_stride,
                     (int)n, (int)m, parts, points, extreme, (float*)nullptr, (int64_t)0, reinterpret_cast<uint32_t*>(covered),
                     split.parts > 1 ? 2 * ((n_sample + 63) / 64) : 0);
  EVX_LAUNCH_CHECK();
  const HvSamples samples = {u, m, 1, extreme, ref, ref_stride, parts};
  if (int e = hv_covered_launch<kHvMetric>(points, samples, n, m, n_sample, split, covered, s)) return e;
  hipLaunchKernelGGL(hv_covered_total_kernel<true>, dim3(1), dim3(1024), 0, s, covered, (int)((n_sample + 63) / 64), samples, (int)m,
                     (int)n_sample, (int64_t*)nullptr, out);
  EVX_LAUNCH_CHECK();
  return 0;
}

int evox_hip_calibration_launch(int kind, int64_t blocks, int64_t iterations, float* scratch_out, void* stream) {
  if (scratch_out == nullptr || kind < 0 || kind > 3 || blocks < 1 || blocks > 65535 || iterations < 1 || iterations > 10000000)
    return kErrBadArg;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)blocks), block(256);
  if (kind == 0)
    hipLaunchKernelGGL(calibrate_kernel<0>, grid, block, 0, s, scratch_out, (int)iterations, 1.0f, 2.0f);
  else if (kind == 1)
    hipLaunchKernelGGL(calibrate_kernel<1>, grid, block, 0, s, scratch_out, (int)iterations, 1.0f, 2.0f);
  else if (kind == 2)
    hipLaunchKernelGGL(calibrate_kernel<2>, grid, block, 0, s, scratch_out, (int)iterations, 1.0f, 2.0f);
  else
    hipLaunchKernelGGL(calibrate_kernel<3>, grid, block, 0, s, scratch_out, (int)iterations, 1.0f, 2.0f);
  EVX_LAUNCH_CHECK();
  return 0;
}

int evox_hip_dominance_plan(int64_t n, int64_t m, int64_t* out2) {
  Layout L;
  if (out2 == nullptr || !make_layout(n, m, &L)) return kErrBadArg;
  out2[0] = prefix_dominance_applies(L) ? 0 : dominance_tile_words(L);
  out2[1] = prefix_dominance_applies(L);
  return 0;
}

int evox_hip_peel_plan(int64_t n, int64_t m, int64_t* out3) {
  Layout L;
  if (out3 == nullptr || !make_layout(n, m, &L)) return kErrBadArg;
  size_t lds = 0;
  const int sweepers = lds_peel_plan(L, &lds);
  out3[0] = sweepers != 0;
  out3[1] = sweepers;
  out3[2] = (int64_t)lds;
  return 0;
}

int evox_hip_read_status(const void* ws, void* stream, int32_t* host_out8) {
  if (host_out8 == nullptr) return kErrBadArg;
  if (ws == nullptr) {  // the library's own scratch memory on the current device (the entry point that takes no workspace)
    void* own = nullptr;
    if (int e = static_scratch(&own)) return e;
    ws = own;
  }
  // the control block is the first region of the workspace
  hipError_t e = hipMemcpyAsync(host_out8, ws, 8 * sizeof(int32_t), hipMemcpyDeviceToHost, (hipStream_t)stream);
  if (e != hipSuccess) return (int)e;
  e = hipStreamSynchronize((hipStream_t)stream);
  if (e != hipSuccess) return (int)e;
  return host_out8[0];
}

}  // extern "C"
