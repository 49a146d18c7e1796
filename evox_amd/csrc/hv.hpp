// Monte-Carlo hypervolume: the other users of a pairwise "no worse in every objective" test, points
// against samples instead of rows against rows.
//
// HypE's contributions (src/evox/algorithms/mo/hype.py:12-39):
//   pds[s, i] = all_k fit[i, k] - sample[s, k] <= 0                               (hype.py:30)
//   ds[s]     = number of points with pds[s, .], minus one when it is not zero    (hype.py:31-32)
//   f[i]      = sum_s pds[s, i] ? alpha[ds[s]] : 0                                (hype.py:34-36)
// The metric (src/evox/metrics/hv.py:13-19):
//   covered[s] = any_i all_k sample[s, k] < point[i, k]                           (hv.py:18)
//
// Bound by vector issue: a test costs M compares, and a few thousand points against a hundred thousand samples are
// 10^8 tests, some 5 us of the device.  What the kernels have to see to is that enough waves are there to hide the
// loads of the other side.  Whether a sample is covered, and by how many points, is decided by a workgroup that holds 64
// samples, one to a lane, in each of its waves; the waves take the points in turn, hv_step at a time, as scalar operands.
// Where the samples are too few to fill the device, several workgroups have the same samples and share the points.
// (A wave that took all the points of its samples was alone with the latency of every scalar load: 129 us for 1001 x 3
// against 100 000 samples, 27 us this way; counts and weights of 2000 x 3 against 10 000, 25 us before, 15 now.)  The sums
// over the samples have the points in the lanes and read the samples, packed with their weights, from LDS, eight reads in
// flight (47 us with scalar loads, 11 now); their order of summation is part of the results and has stayed.
#pragma once

#include "common.hpp"
#include "hv_split.hpp"

namespace evx {

constexpr int kHvTile = 128;         // samples that a workgroup of the sums holds in LDS at a time
constexpr int kHvMaxShares = 64;     // shares of the samples in the sums, at most (bounds the workspace)
constexpr int kHvParts = 64;         // workgroups that look for the box of the points, at most
constexpr int kHvRegs = 16;          // objectives held in registers; more are re-read from memory
constexpr int kHvPacked = 20;        // floats per packed sample, at most (16 objectives, the weight, whole 16-byte pieces)
// Weights that one thread computes in ascending order, at least: those of a sample that up to 14 points cover, which decide
// between the points, are the plain products.  (A HypE call on 2000 x 3 against 10 000 samples takes 47 us with 4, 14 or 32, on
// 5000 x 3 against 20 000 80, 80 or 83.)
constexpr int kHvAlphaShare = 14;
// Steps after which the waves of a workgroup tell each other what is covered.  8 / 32 / 128, us a call: uniform 100 000 x 3
// against 10 000 samples 137 / 155 / 180, 20 000 x 3 against 100 000 279 / 282 / 315, up to 5000 points 3 % apart at most.
constexpr int kHvMeet = 32;

__host__ __device__ constexpr int hv_packed(int m) { return (m + 1 + 3) & ~3; }

// Samples per share of the sums: whole eights, at least 256, at most kHvMaxShares shares.  (A share is added up in ascending
// order and the shares in theirs: points that cover equally weighted samples in another order differ by a rounding, and the
// order of a selection among them with it, so the length of a share belongs to the results.)
__host__ inline int64_t hv_share(int64_t n_sample) {
  int64_t len = (n_sample + kHvMaxShares - 1) / kHvMaxShares;
  if (len < 256) len = 256;
  return (len + 7) & ~7ll;
}
__host__ inline int hv_parts(int64_t n) {
  const int64_t parts = (n + 255) / 256;
  return (int)(parts < kHvParts ? parts : kHvParts);
}

// The samples of a kernel: sample[s, k] = u[s * row + k * col], as it is (parts == 0) or moved into the box of the points,
// whose far corner (metric: u * bound) or near corner (HypE: u * (ref - low) + low) is the extreme of `parts` rows of m.
enum { kHvPlain = 0, kHvMetric = 1, kHvHype = 2 };
struct HvSamples {
  const float* u;
  int64_t row, col;
  const float* extreme;
  const float* ref;
  int64_t ref_stride;
  int parts;
};

// max / min as torch reduces them: a NaN wins.
template <bool kMax>
__device__ inline float hv_extreme(float a, float b) {
  if (a != a) return a;
  if (b != b) return b;
  return kMax ? fmaxf(a, b) : fminf(a, b);
}
template <bool kMax>
__device__ inline float hv_wave_extreme(float v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v = hv_extreme<kMax>(v, __shfl_xor(v, d));
  return v;
}
// Objective k's extreme over all parts, in every lane of the calling wave (all of its lanes call; parts <= 64).
template <bool kMax>
__device__ inline float hv_corner(const HvSamples& in, int m, int k) {
  const int lane = threadIdx.x & 63;
  return hv_wave_extreme<kMax>(in.extreme[(lane < in.parts ? lane : 0) * m + k]);
}
// Multiplied and added in two roundings, as the reference's two statements are.
template <int kMode>
__device__ inline float hv_sample(const HvSamples& in, int m, int64_t s, int k) {
#pragma clang fp contract(off)
  const float u = in.u[s * in.row + k * in.col];
  if constexpr (kMode == kHvMetric) return u * hv_corner<true>(in, m, k);
  if constexpr (kMode == kHvHype) {
    const float low = hv_corner<false>(in, m, k);
    const float scaled = u * (in.ref[k * in.ref_stride] - low);
    return scaled + low;
  }
  return u;
}

// The reference's test is on the difference (hype.py:30): inf - inf is NaN and fails it.  With one side finite it is the
// plain comparison (differences do not underflow).
template <bool kFinite>
__device__ inline bool hv_no_worse(float fit, float sample) {
  return kFinite ? fit <= sample : fit - sample <= 0.0f;
}
__device__ inline bool hv_finite(float v) { return fabsf(v) <= 3.4028234663852886e38f; }

// points_t[k][i] = value of row i in objective k: |f - ref| for the metric, f for HypE; extreme[part][k] = the largest
// (smallest for HypE) of the part's rows.  With alpha, one more workgroup writes the weights of a sample covered by
// j + 1 points, alpha[j] = prod_{1 <= i <= j} (pop - i) / (n - i) / (j + 1), infinities as the largest numbers and NaN as
// zero (hype.py:14-24), in the precision of the reference's statements, whose cumprod is a scan too: a thread has
// kHvAlphaShare of them or more in ascending order, the threads' products are scanned.  Largest relative error against 64
// bits over n = 50 to 5000 with half of them kept: 5.0e-7, that of the cumprod on the same device 5.4e-7.
// zero: what the workgroups that share samples add up in, cleared here.
template <bool kMetric>
__global__ __launch_bounds__(256) void hv_points_kernel(const float* __restrict__ f, int64_t row, int64_t col,
                                                        const float* __restrict__ ref, int64_t ref_stride, int n, int m, int parts,
                                                        float* __restrict__ points_t, float* __restrict__ extreme,
                                                        float* __restrict__ alpha, int64_t pop, uint32_t* __restrict__ zero,
                                                        int64_t zero_words) {
  for (int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x; w < zero_words; w += (int64_t)gridDim.x * 256) zero[w] = 0u;
  __shared__ float wave_extreme[4];
  __shared__ float product[256];
  const int t = threadIdx.x;
  if ((int)blockIdx.x == parts) {
    const int share = max(kHvAlphaShare, (n + 255) / 256);
    const int j0 = min(n, t * share), j1 = min(n, j0 + share);
    auto quotient = [&](int j) { return j == 0 ? 1.0f : (float)(pop - j) / (float)(n - j); };
    float p = 1.0f;
    for (int j = j0; j < j1; ++j) p *= quotient(j);
    product[t] = p;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
      const float before = t >= d ? product[t - d] : 1.0f;
      __syncthreads();
      product[t] *= before;
      __syncthreads();
    }
    const float before = t > 0 ? product[t - 1] : 1.0f;
    p = 1.0f;
    for (int j = j0; j < j1; ++j) {
      p *= quotient(j);
      const float a = before * p / (float)(j + 1);
      alpha[j] = a != a ? 0.0f : fminf(fmaxf(a, -3.4028234663852886e38f), 3.4028234663852886e38f);
    }
    return;
  }
  const int share = (n + parts - 1) / parts;
  const int i0 = (int)blockIdx.x * share, i1 = min(n, i0 + share);
  for (int k = 0; k < m; ++k) {
    const float r = kMetric ? ref[k * ref_stride] : 0.0f;
    float v = f[(int64_t)min(i0, n - 1) * row + k * col];
    if (kMetric) v = fabsf(v - r);
    for (int i = i0 + t; i < i1; i += 256) {
      float w = f[(int64_t)i * row + k * col];
      if (kMetric) w = fabsf(w - r);
      points_t[(int64_t)k * n + i] = w;
      v = hv_extreme<kMetric>(v, w);
    }
    v = hv_wave_extreme<kMetric>(v);
    if ((t & 63) == 0) wave_extreme[t >> 6] = v;
    __syncthreads();
    if (t == 0) {
#pragma unroll
      for (int w = 1; w < 4; ++w) v = hv_extreme<kMetric>(v, wave_extreme[w]);
      extreme[blockIdx.x * m + k] = v;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- HypE's contributions

// The number of points of [0, n) that pass the test against the lane's sample, over the steps of points that this wave
// takes: wave, wave + waves, ...; of the last step, which is moved back to end with the points, those not yet counted.
template <int M, bool kFinite>
__device__ inline int hv_count_points(const float* __restrict__ points_t, int n, int m, const float (&sv)[M], int wave, int waves) {
  constexpr int kHvStep = hv_step(M);
  int count = 0;
  const int steps = n < kHvStep ? 0 : (n + kHvStep - 1) / kHvStep;
#pragma unroll 1
  for (int step = wave; step < steps; step += waves) {
    const int i = min(step * kHvStep, n - kHvStep);
    const int counted = step * kHvStep - i;
    bool c[kHvStep];
#pragma unroll
    for (int u = 0; u < kHvStep; ++u) c[u] = u >= counted;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      if (M <= 8 || k < m) {
        const float* __restrict__ at = points_t + (int64_t)k * n + i;
#pragma unroll
        for (int u = 0; u < kHvStep; ++u) c[u] &= hv_no_worse<kFinite>(at[u], sv[k]);
      }
    }
#pragma unroll
    for (int u = 0; u < kHvStep; ++u) count += c[u] ? 1 : 0;
  }
  for (int i = wave; n < kHvStep && i < n; i += waves) {
    bool c = true;
#pragma unroll
    for (int k = 0; k < M; ++k)
      if (M <= 8 || k < m) c &= hv_no_worse<kFinite>(points_t[(int64_t)k * n + i], sv[k]);
    count += c ? 1 : 0;
  }
  return count;
}

// weight[s] = alpha[max(ds[s], 0)], ds[s] = points that cover sample s, minus one.  Up to kHvRegs objectives (M > 0) the weight
// goes behind the sample's coordinates in `packed`, hv_packed(m) floats a sample; for more (M == 0) `packed` holds the
// weights alone.
template <int M, int R>
__device__ inline void hv_store_weight(int64_t s, int m, int covered, const float (&sv)[R], const float* __restrict__ alpha,
                                       float* __restrict__ packed) {
  const float w = alpha[covered == 0 ? 0 : covered - 1];
  if constexpr (M > 0) {
    float* const at = packed + s * hv_packed(m);
#pragma unroll
    for (int k = 0; k < M; ++k)
      if (M <= 8 || k < m) at[k] = sv[k];
    at[m] = w;
  } else {
    packed[s] = w;
  }
}

// A workgroup of up to 16 waves has 64 samples and, where gridDim.y workgroups have the same ones, a share of the points:
// these add to cover[s], which must be zero, and hv_weight_kernel takes it from there.
template <int M, int kMode>
__global__ __launch_bounds__(1024) void hv_sample_weight_kernel(const float* __restrict__ points_t, HvSamples samples, int n, int m,
                                                                int n_sample, const float* __restrict__ alpha,
                                                                float* __restrict__ packed, int* __restrict__ cover) {
  __shared__ int part[64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int turn = (int)blockIdx.y * waves + wave, turns = (int)gridDim.y * waves;
  const int64_t s = (int64_t)blockIdx.x * 64 + lane;
  const int64_t sc = s < n_sample ? s : n_sample - 1;
  if (threadIdx.x < 64) part[lane] = 0;
  int count = 0;
  constexpr int R = M > 0 ? M : 1;
  float sv[R];
  if constexpr (M > 0) {
    bool finite = true;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      sv[k] = 0.0f;
      if (M <= 8 || k < m) sv[k] = hv_sample<kMode>(samples, m, sc, k);
      finite &= hv_finite(sv[k]);
    }
    count = __builtin_amdgcn_ballot_w64(!finite) == 0ull ? hv_count_points<M, true>(points_t, n, m, sv, turn, turns)
                                                         : hv_count_points<M, false>(points_t, n, m, sv, turn, turns);
  } else {
    for (int64_t i = turn; i < n; i += turns) {
      bool c = true;
      for (int k = 0; k < m; ++k) c &= hv_no_worse<false>(points_t[(int64_t)k * n + i], samples.u[sc * samples.row + k * samples.col]);
      count += c ? 1 : 0;
    }
  }
  __syncthreads();
  if (count != 0) atomicAdd(&part[lane], count);
  __syncthreads();
  if (wave != 0 || s >= n_sample) return;
  if (gridDim.y > 1) {
    if (part[lane] != 0) atomicAdd(&cover[s], part[lane]);
    return;
  }
  hv_store_weight<M>(s, m, part[lane], sv, alpha, packed);
}

// The weights of samples whose points were shared: cover[s] points cover sample s.
template <int M, int kMode>
__global__ __launch_bounds__(64) void hv_weight_kernel(HvSamples samples, int m, int n_sample, const int* __restrict__ cover,
                                                       const float* __restrict__ alpha, float* __restrict__ packed) {
  const int64_t s = (int64_t)blockIdx.x * 64 + threadIdx.x;
  const int64_t sc = s < n_sample ? s : n_sample - 1;  // (hv_sample needs every lane)
  constexpr int R = M > 0 ? M : 1;
  float sv[R];
#pragma unroll
  for (int k = 0; k < M; ++k) {
    sv[k] = 0.0f;
    if (M <= 8 || k < m) sv[k] = hv_sample<kMode>(samples, m, sc, k);
  }
  if (s < n_sample) hv_store_weight<M>(s, m, cover[s], sv, alpha, packed);
}

// The sum goes on over `count` samples of the tile, a multiple of eight (the tile is filled up with weights of zero).
template <int M, bool kFinite>
__device__ inline float hv_sum_tile(float acc, const float* tile, int count, int m, const float (&fv)[M]) {
  constexpr int kAhead = M <= 7 ? 8 : 4;  // samples whose LDS reads are in flight together
  constexpr int kPieces = (M <= 8 ? hv_packed(M) : kHvPacked) / 4;
  const int pieces = M <= 8 ? kPieces : hv_packed(m) / 4;
  const float4* at = reinterpret_cast<const float4*>(tile);
#pragma unroll 1
  for (int s = 0; s < count; s += kAhead) {
    float v[kAhead][kPieces * 4];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
#pragma unroll
      for (int q = 0; q < kPieces; ++q) {
        if (M <= 8 || q < pieces) {
          const float4 piece = at[u * pieces + q];
          v[u][4 * q] = piece.x;
          v[u][4 * q + 1] = piece.y;
          v[u][4 * q + 2] = piece.z;
          v[u][4 * q + 3] = piece.w;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      bool c = true;
#pragma unroll
      for (int k = 0; k < M; ++k)
        if (M <= 8 || k < m) c &= hv_no_worse<kFinite>(fv[k], v[u][k]);
      float w;
      if constexpr (M <= 8) {
        w = v[u][M];
      } else {
        w = tile[(s + u) * pieces * 4 + m];
      }
      acc += c ? w : 0.0f;
    }
    at += kAhead * pieces;
  }
  return acc;
}

// partial[share][i] = sum over the samples s of the share, in ascending s, of (pds[s, i] ? weight[s] : 0).  Lane = point.  grid = (point blocks, shares).
template <int M>
__global__ __launch_bounds__(256) void hv_point_partial_kernel(const float* __restrict__ points_t, const float* __restrict__ packed,
                                                               HvSamples samples, int n, int m, int n_sample, int share,
                                                               float* __restrict__ partial) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t ic = i < n ? i : n - 1;
  const int64_t s0 = (int64_t)blockIdx.y * share;
  const int64_t s1 = s0 + share < n_sample ? s0 + share : n_sample;
  float total = 0.0f;
  if constexpr (M > 0) {
    __shared__ __attribute__((aligned(16))) float tile[kHvTile * (M <= 8 ? hv_packed(M) : kHvPacked)];
    float fv[M];
    bool finite = true;
#pragma unroll
    for (int k = 0; k < M; ++k) {
      fv[k] = 0.0f;
      if (M <= 8 || k < m) fv[k] = points_t[(int64_t)k * n + ic];
      finite &= hv_finite(fv[k]);
    }
    const bool all_finite = __builtin_amdgcn_ballot_w64(!finite) == 0ull;
    const int stride = M <= 8 ? hv_packed(M) : hv_packed(m);
    for (int64_t s = s0; s < s1; s += kHvTile) {
      const int count = s1 - s < kHvTile ? (int)(s1 - s) : kHvTile;
      __syncthreads();
      // (a sample is a whole number of 16-byte pieces, and `packed` is aligned to 256 bytes)
      for (int q = threadIdx.x; q < count * (stride / 4); q += 256)
        reinterpret_cast<float4*>(tile)[q] = reinterpret_cast<const float4*>(packed + s * stride)[q];
      const int filled = (count + 7) & ~7;
      for (int q = count * stride + threadIdx.x; q < filled * stride; q += 256) tile[q] = 0.0f;
      __syncthreads();
      total = all_finite ? hv_sum_tile<M, true>(total, tile, filled, m, fv)
                         : hv_sum_tile<M, false>(total, tile, filled, m, fv);
    }
  } else {
    for (int64_t s = s0; s < s1; ++s) {
      bool c = true;
      for (int k = 0; k < m; ++k) c &= hv_no_worse<false>(points_t[(int64_t)k * n + ic], samples.u[s * samples.row + k * samples.col]);
      total += c ? packed[s] : 0.0f;
    }
  }
  if (i < n) partial[(int64_t)blockIdx.y * n + i] = total;
}

// out[i] = (sum of the partial sums of point i, in the order of the shares) * scale; in HypE's box (parts > 0) the scale is
// prod(ref - low) / n_sample.
__global__ __launch_bounds__(64) void hv_point_total_kernel(const float* __restrict__ partial, HvSamples box, int n, int m, int shares,
                                                            int n_sample, float scale, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;
  const int64_t ic = i < n ? i : n - 1;
  if (box.parts > 0) {
    scale = 1.0f;
    for (int k = 0; k < m; ++k) scale *= box.ref[k * box.ref_stride] - hv_corner<false>(box, m, k);
    scale /= (float)n_sample;
  }
  float acc = 0.0f;
  int c = 0;
  for (; c + 16 <= shares; c += 16) {  // sixteen loads in flight
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = partial[(int64_t)(c + u) * n + ic];
#pragma unroll
    for (int u = 0; u < 16; ++u) acc += v[u];
  }
  for (; c < shares; ++c) acc += partial[(int64_t)c * n + ic];
  if (i < n) out[i] = acc * scale;
}

// ---------------------------------------------------------------- the metric

// covered[b]: which of the 64 samples of workgroup b some point exceeds strictly in every objective (a NaN on either side
// compares false).  A wave stops as soon as all of its samples are covered; every kHvMeet steps the waves of the workgroup
// tell each other which are.  points_t is (m, n), row-major.  Where gridDim.y workgroups have the same samples, each with
// a share of the points, covered[b] must be zero, and one that starts late does not look for what it already holds.
template <int M, int kMode>
__global__ __launch_bounds__(1024) void hv_covered_kernel(const float* __restrict__ points_t, HvSamples samples, int n, int m,
                                                          int n_sample, unsigned long long* __restrict__ covered) {
  __shared__ unsigned long long met;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int turn = (int)blockIdx.y * waves + wave, turns = (int)gridDim.y * waves;
  const int64_t s = (int64_t)blockIdx.x * 64 + lane;
  const bool live = s < n_sample;
  const int64_t sc = live ? s : n_sample - 1;
  if (threadIdx.x == 0)
    met = gridDim.y > 1 ? __hip_atomic_load(&covered[blockIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
  __syncthreads();
  bool cov = !live || ((met >> lane) & 1ull) != 0ull;
  if constexpr (M > 0) {
    constexpr int kHvStep = hv_step(M);
    float sv[M];
#pragma unroll
    for (int k = 0; k < M; ++k) {
      sv[k] = 0.0f;
      if (M <= 8 || k < m) sv[k] = hv_sample<kMode>(samples, m, sc, k);
    }
    // (the last points once more where they are no whole step: a test may be repeated)
    const int steps = n < kHvStep || __builtin_amdgcn_ballot_w64(!cov) == 0ull ? 0 : (n + kHvStep - 1) / kHvStep;
    int since = 0;
#pragma unroll 1
    for (int step = turn; step < steps; step += turns) {
      const int i = min(step * kHvStep, n - kHvStep);
      bool c[kHvStep];
#pragma unroll
      for (int u = 0; u < kHvStep; ++u) c[u] = true;
#pragma unroll
      for (int k = 0; k < M; ++k) {
        if (M <= 8 || k < m) {
          const float* __restrict__ at = points_t + (int64_t)k * n + i;
#pragma unroll
          for (int u = 0; u < kHvStep; ++u) c[u] &= sv[k] < at[u];
        }
      }
#pragma unroll
      for (int u = 0; u < kHvStep; ++u) cov |= c[u];
      if (++since == kHvMeet) {
        since = 0;
        const unsigned long long mine = __builtin_amdgcn_ballot_w64(cov);
        unsigned long long all = 0ull;
        if (lane == 0) all = atomicOr(&met, mine);
        all = __shfl(all, 0);
        cov |= ((all >> lane) & 1ull) != 0ull;
      }
      if (__builtin_amdgcn_ballot_w64(!cov) == 0ull) break;
    }
    for (int i = turn; n < kHvStep && i < n; i += turns) {
      bool c = true;
#pragma unroll
      for (int k = 0; k < M; ++k)
        if (M <= 8 || k < m) c &= sv[k] < points_t[(int64_t)k * n + i];
      cov |= c;
    }
  } else {
    for (int64_t i = turn; i < n && __builtin_amdgcn_ballot_w64(!cov) != 0ull; i += turns) {
      bool c = true;
      for (int k = 0; k < m; ++k) c &= samples.u[sc * samples.row + k * samples.col] < points_t[(int64_t)k * n + i];
      cov |= c;
    }
  }
  const unsigned long long lives = __builtin_amdgcn_ballot_w64(live);
  const unsigned long long mine = __builtin_amdgcn_ballot_w64(cov && live);
  if (lane == 0 && mine != 0ull) atomicOr(&met, mine);
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (gridDim.y == 1)
    covered[blockIdx.x] = met & lives;
  else if ((met & lives) != 0ull)
    atomicOr(&covered[blockIdx.x], met & lives);
}

// The number of covered samples: out_count[0], or out[0] = sum / n_sample * (product of the box's sides).
template <bool kEstimate>
__global__ __launch_bounds__(1024) void hv_covered_total_kernel(const unsigned long long* __restrict__ covered, int blocks, HvSamples box,
                                                                int m, int n_sample, int64_t* __restrict__ out_count, float* __restrict__ out) {
  __shared__ int part[16];
  int acc = 0;
#pragma unroll 2
  for (int b = threadIdx.x; b < blocks; b += 1024) acc += __popcll(covered[b]);
  for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
  float volume = 1.0f;
  if (kEstimate && threadIdx.x < 64)
    for (int k = 0; k < m; ++k) volume *= hv_corner<true>(box, m, k);
  __syncthreads();
  if (threadIdx.x != 0) return;
  int64_t total = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) total += part[w];
  if (kEstimate)
    out[0] = (float)total / (float)n_sample * volume;
  else
    out_count[0] = total;
}

}  // namespace evx
