// Stand-in for the HIP runtime and the device builtins that the kernels use, for a build of the library that runs on the
// CPU under the address sanitizer (tests/emulated.py): every workgroup is a thread, every lane a fiber of it
// (emulator.cpp).  Wave operations meet in the lanes that reach the same call; the lanes of a wave run one after the
// other between them, so code that hands data from lane to lane through LDS needs a barrier here as well.
#pragma once
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <type_traits>
#include <utility>
#include <sanitizer/asan_interface.h>
#include <math.h>
#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(x) __attribute__((aligned(x)))
#define __HIP_MEMORY_SCOPE_AGENT 1
#define __HIP_MEMORY_SCOPE_SYSTEM 2
#define __HIP_MEMORY_SCOPE_WORKGROUP 3
struct dim3 { unsigned x, y, z; dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {} };
struct int2 { int x, y; }; struct alignas(16) int4 { int x, y, z, w; };
struct alignas(8) float2 { float x, y; }; struct alignas(16) float4 { float x, y, z, w; };
struct alignas(8) uint2 { unsigned x, y; }; struct alignas(16) uint4 { unsigned x, y, z, w; };
struct alignas(16) ulonglong2 { unsigned long long x, y; }; struct alignas(16) double2 { double x, y; };
inline ulonglong2 make_ulonglong2(unsigned long long a, unsigned long long b) { return {a, b}; }
inline double2 make_double2(double a, double b) { return {a, b}; }
inline int2 make_int2(int a, int b) { return {a, b}; }
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
inline uint2 make_uint2(unsigned a, unsigned b) { return {a, b}; }
inline uint4 make_uint4(unsigned a, unsigned b, unsigned c, unsigned d) { return {a, b, c, d}; }
inline float2 make_float2(float a, float b) { return {a, b}; }
inline float4 make_float4(float a, float b, float c, float d) { return {a, b, c, d}; }
using std::min; using std::max;
inline int min(int a, unsigned b) { return (int)std::min<long long>(a, b); }
inline unsigned min(unsigned a, int b) { return (unsigned)std::min<long long>(a, b); }
template <class A, class B, class = std::enable_if_t<!std::is_same_v<A, B> && std::is_integral_v<A> && std::is_integral_v<B>>>
inline std::common_type_t<A, B> min(A a, B b) { using C = std::common_type_t<A, B>; return (C)a < (C)b ? (C)a : (C)b; }
template <class A, class B, class = std::enable_if_t<!std::is_same_v<A, B> && std::is_integral_v<A> && std::is_integral_v<B>>>
inline std::common_type_t<A, B> max(A a, B b) { using C = std::common_type_t<A, B>; return (C)a > (C)b ? (C)a : (C)b; }
// ---- runtime
typedef int hipError_t; constexpr int hipSuccess = 0;
typedef void* hipStream_t;
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0 };
enum { hipDeviceAttributeMultiprocessorCount, hipFuncAttributeMaxDynamicSharedMemorySize, hipHostMallocDefault, hipMemcpyDeviceToHost };
extern int emu_cus;
inline hipError_t hipGetDevice(int* d) { *d = 0; return 0; }
inline hipError_t hipDeviceGetAttribute(int* v, int, int) { *v = emu_cus; return 0; }
inline hipError_t hipGetLastError() { return 0; }
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = hipStreamCaptureStatusNone; return 0; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { *p = malloc(n); return 0; }
inline hipError_t hipFuncSetAttribute(const void*, int, int) { return 0; }
template <class T> inline hipError_t hipGetSymbolAddress(void** p, T& s) { *p = (void*)&s; return 0; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) { memcpy(d, s, n); return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return 0; }
template <class K> inline hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* per, K, int threads, size_t lds) {
  int a = 2048 / threads, b = lds ? (int)(160 * 1024 / lds) : 32; *per = std::min(std::min(a, b), 2); return 0; }
// ---- lanes
namespace emu {
struct Lane { dim3 tid; int lane; };
extern thread_local Lane* cur; extern thread_local dim3 bid; extern dim3 bdim, gdim;
extern thread_local void* dyn;
// every wave operation: publish `v`, get all lanes' values and the mask of lanes that take part (same call site)
uint64_t wave_op(const void* site, uint64_t v, const uint64_t** all);  // -> mask
void block_op(const void* site, int v, int* any, int* all);
void yield_spin(); void load_yield();
void* shared_at(const void* key, size_t bytes);
void run(const char* name, dim3 g, dim3 b, size_t lds, const std::function<void()>& body);
}
#define threadIdx (emu::cur->tid)
#define blockIdx (emu::bid)
#define blockDim (emu::bdim)
#define gridDim (emu::gdim)
#define EMU_OP __attribute__((noinline, convergent))
#define EMU_SITE __builtin_return_address(0)
template <class T> inline uint64_t emu_bits(T v) { uint64_t b = 0; static_assert(sizeof(T) <= 8); memcpy(&b, &v, sizeof(T)); return b; }
template <class T> inline T emu_from(uint64_t b) { T v; memcpy(&v, &b, sizeof(T)); return v; }
EMU_OP uint64_t emu_ballot(bool p);
EMU_OP uint64_t emu_read(uint64_t v, int lane);
EMU_OP uint64_t emu_first(uint64_t v);
EMU_OP uint64_t emu_shfl(uint64_t v, int src, int mode);  // 0 idx, 1 up, 2 xor
EMU_OP int emu_dpp(int old, int v, int ctrl, int rowm, int bankm, bool bound);
EMU_OP void emu_sync(); EMU_OP int emu_sync_or(int); EMU_OP int emu_sync_and(int);
#define __builtin_amdgcn_ballot_w64(p) emu_ballot(p)
#define __ballot(p) emu_ballot((p) != 0)
#define __builtin_amdgcn_readlane(v, l) ((int)emu_read((uint32_t)(v), (l)))
#define __builtin_amdgcn_readfirstlane(v) ((int)emu_first((uint32_t)(v)))
#define __builtin_amdgcn_update_dpp(o, v, c, r, b, z) emu_dpp((int)(o), (int)(v), c, r, b, z)
#define __builtin_amdgcn_mov_dpp(v, c, r, b, z) emu_dpp(0, (int)(v), c, r, b, z)
#define __builtin_amdgcn_s_sleep(x) emu::yield_spin()
#define __builtin_amdgcn_fence(...) __atomic_thread_fence(__ATOMIC_SEQ_CST)
template <class T> __attribute__((always_inline)) inline T __shfl(T v, int l) { return emu_from<T>(emu_shfl(emu_bits(v), l, 0)); }
template <class T> __attribute__((always_inline)) inline T __shfl_up(T v, int l) { return emu_from<T>(emu_shfl(emu_bits(v), l, 1)); }
template <class T> __attribute__((always_inline)) inline T __shfl_xor(T v, int l) { return emu_from<T>(emu_shfl(emu_bits(v), l, 2)); }
#define __syncthreads emu_sync
#define __syncthreads_or(x) emu_sync_or(x)
#define __syncthreads_and(x) emu_sync_and(x)
// ---- atomics
template <class T, class U> inline T atomicAdd(T* p, U v) {
  if constexpr (std::is_floating_point_v<T>) { T o, n; do { __atomic_load(p, &o, __ATOMIC_RELAXED); n = o + (T)v; } while (!__atomic_compare_exchange(p, &o, &n, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST)); return o; }
  else return __atomic_fetch_add(p, (T)v, __ATOMIC_SEQ_CST); }
template <class T, class U> inline T atomicSub(T* p, U v) { return __atomic_fetch_sub(p, (T)v, __ATOMIC_SEQ_CST); }
template <class T, class U> inline T atomicOr(T* p, U v) { return __atomic_fetch_or(p, (T)v, __ATOMIC_SEQ_CST); }
template <class T, class U> inline T atomicAnd(T* p, U v) { return __atomic_fetch_and(p, (T)v, __ATOMIC_SEQ_CST); }
template <class T, class U> inline T atomicMax(T* p, U v) { T o = __atomic_load_n(p, __ATOMIC_RELAXED); while (o < (T)v && !__atomic_compare_exchange_n(p, &o, (T)v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST)) {} return o; }
template <class T, class U> inline T atomicMin(T* p, U v) { T o = __atomic_load_n(p, __ATOMIC_RELAXED); while (o > (T)v && !__atomic_compare_exchange_n(p, &o, (T)v, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST)) {} return o; }
template <class T, class U, class V> inline T atomicCAS(T* p, U a, V b) { T o = (T)a; __atomic_compare_exchange_n(p, &o, (T)b, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST); return o; }
template <class T> __attribute__((noinline)) T emu_aload(const T* p) { emu::load_yield(); T v; __atomic_load(const_cast<T*>(p), &v, __ATOMIC_SEQ_CST); return v; }
#define __hip_atomic_load(p, o, s) emu_aload(p)
int emu_error_word(const int* p, int failed);  // a look at the error word of a call; `failed`: what says that a wait ran out
// A 16-byte load of two 8-byte units, each of which arrives as a whole.
template <class V> inline void emu_load_pair(V& r, const unsigned long long* p) {
  const unsigned long long a = emu_aload(p), b = emu_aload(p + 1);
  r.x = (unsigned)a; r.y = (unsigned)(a >> 32); r.z = (unsigned)b; r.w = (unsigned)(b >> 32);
}
template <class T, class U> inline void emu_astore(T* p, U v) { T t = (T)v; __atomic_store(p, &t, __ATOMIC_SEQ_CST); }
#define __hip_atomic_store(p, v, o, s) emu_astore(p, v)
#define __hip_atomic_fetch_add(p, v, o, s) atomicAdd(p, v)
// ---- scalars
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __popc(unsigned v) { return __builtin_popcount(v); }
inline int __ffsll(unsigned long long v) { return __builtin_ffsll((long long)v); }
inline unsigned __float_as_uint(float v) { return emu_from<unsigned>(emu_bits(v)); }
inline float __uint_as_float(unsigned v) { return emu_from<float>(v); }
inline long long __double_as_longlong(double v) { return emu_from<long long>(emu_bits(v)); }
inline double __longlong_as_double(long long v) { return emu_from<double>(emu_bits(v)); }
long long wall_clock64();
// ---- launches
#include <tuple>
template <class K, class... A>
inline void emu_launch(const char* name, K k, dim3 g, dim3 b, size_t lds, hipStream_t, A... args) {
  std::tuple<A...> t(args...);
  emu::run(name, g, b, lds, [&] { auto mine = t; std::apply(k, mine); });
}
#define hipLaunchKernelGGL(kernel, g, b, lds, s, ...) emu_launch(#kernel, [&](auto&&... a_) { (kernel)(a_...); }, g, b, lds, s, ##__VA_ARGS__)
#define HIP_SYMBOL(x) x
