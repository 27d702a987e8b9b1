// Internal definitions shared by the HIP translation units of libhflmp_hip.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <type_traits>

#include "hflmp_hip.h"

// Threads per workgroup for every kernel of the library: four wave64s.
constexpr int kBlock = 256;
constexpr int kWave = 64;
// gfx950: 256 CUs in 8 XCDs, workgroups dispatched round-robin over XCDs.
constexpr int kXcds = 8;
// Upper bound on reduction partials (one per workgroup of a reduction).
constexpr int kMaxRedBlocks = 2048;  // at most twice kFinalBlock (host_sum_partials)

struct hflmp_ctx {
  int device = 0;
  int num_cus = 0;
  hipStream_t own_stream = nullptr;
  hipStream_t stream = nullptr;
  // Reduction scratch: kMaxRedBlocks partials (16 B each), a ticket
  // counter per concurrent reduction slot, result slots.
  void *red_partials = nullptr;
  unsigned int *red_counter = nullptr;
  double *red_result = nullptr;   // 64 device result slots
  void *host_pinned = nullptr;    // 4 KiB pinned host staging
  // pinned host memory for a reduction's partials (kMaxRedBlocks of 8 B),
  // and its address on the device
  void *host_partials = nullptr;
  void *host_partials_dev = nullptr;
  char last_error[512] = {0};
};

// Record an error message in the context and return the code.
inline int set_error(hflmp_ctx *ctx, int code, const char *fmt, ...) {
  if (ctx) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(ctx->last_error, sizeof(ctx->last_error), fmt, ap);
    va_end(ap);
  }
  return code;
}

#define HFLMP_HIP_CHECK(ctx, expr)                                            \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess)                                                      \
      return set_error((ctx), HFLMP_EHIP, "%s: %s (%s:%d)", #expr,            \
                       hipGetErrorString(e_), __FILE__, __LINE__);             \
  } while (0)

#define HFLMP_LAUNCH_CHECK(ctx)                                               \
  do {                                                                         \
    hipError_t e_ = hipGetLastError();                                         \
    if (e_ != hipSuccess)                                                      \
      return set_error((ctx), HFLMP_EHIP, "kernel launch: %s (%s:%d)",        \
                       hipGetErrorString(e_), __FILE__, __LINE__);             \
  } while (0)

#define HFLMP_REQUIRE(ctx, cond, ...)                                         \
  do {                                                                         \
    if (!(cond)) return set_error((ctx), HFLMP_EINVAL, __VA_ARGS__);          \
  } while (0)

inline int check_ctx(hflmp_ctx *ctx) { return ctx ? HFLMP_OK : HFLMP_EINVAL; }

// hflmp_fill_zero on a given stream (errors recorded in ctx).
int fill_zero_on(hflmp_ctx *ctx, void *dptr, size_t bytes, hipStream_t s);

// Grid for an elementwise kernel that handles `per_thread` items/thread.
inline unsigned grid_for(long long n, int per_thread) {
  long long g = (n + (long long)kBlock * per_thread - 1) / ((long long)kBlock * per_thread);
  if (g < 1) g = 1;
  if (g > 65535LL * 64) g = 65535LL * 64;
  return (unsigned)g;
}

// Number of workgroups for a grid-stride reduction over n items.
inline int red_blocks(hflmp_ctx *ctx, long long n) {
  long long g = (n + 4LL * kBlock - 1) / (4LL * kBlock);
  long long cap = ctx->num_cus > 0 ? 8LL * ctx->num_cus : 1024;
  if (cap > kMaxRedBlocks) cap = kMaxRedBlocks;
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  return (int)g;
}

// ---- device helpers --------------------------------------------------------
// v of lane (lane ^ OFF) for OFF 8, 4, 2, 1, where lanes that differ in the
// bits above OFF of a row of 16 already hold the same value (as in wave_sum):
// a rotation by 4 then reaches lane ^ 4.
template <int OFF>
__device__ __forceinline__ int dpp_xor(int v) {
  constexpr int ctrl = OFF == 8 ? 0x128 : OFF == 4 ? 0x124 : OFF == 2 ? 0x4E : 0xB1;
  return __builtin_amdgcn_update_dpp(0, v, ctrl, 0xf, 0xf, true);
}

// One step of a wave reduction: op(v, v of lane ^ OFF), on every lane.
template <int OFF, typename T, typename Op>
__device__ __forceinline__ T wave_step(T v, Op op) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "4 or 8 bytes");
  constexpr int W = sizeof(T) / 4;
  struct Words {
    int w[W];
  };
  Words a = __builtin_bit_cast(Words, v), b = a;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    if constexpr (OFF >= 16) {
      // both halves (of the wave, or of each pair of rows) hold the lower
      // half's value in a and the upper half's in b
      const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(a.w[i], a.w[i], false, false)
                               : __builtin_amdgcn_permlane16_swap(a.w[i], a.w[i], false, false);
      a.w[i] = r[0];
      b.w[i] = r[1];
    } else {
      b.w[i] = dpp_xor<OFF>(a.w[i]);
    }
  }
  return op(__builtin_bit_cast(T, a), __builtin_bit_cast(T, b));
}

template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  v = wave_step<32>(v, op);
  v = wave_step<16>(v, op);
  v = wave_step<8>(v, op);
  v = wave_step<4>(v, op);
  v = wave_step<2>(v, op);
  return wave_step<1>(v, op);
}

// Sum over the wave on every lane: pairs 32 apart first, then 16, ... 1.
// The exchanges are lane swaps and DPP moves in the vector unit: through LDS
// (__shfl_xor) each of the six dependent steps waited for two LDS round
// trips in FP64.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  return wave_reduce(v, [](T a, T b) { return a + b; });
}

// lane 0's value, uniform across the wave
template <typename T>
__device__ __forceinline__ T bcast0(T v) {
  constexpr int W = sizeof(T) / 4;
  struct Words {
    int w[W];
  };
  Words a = __builtin_bit_cast(Words, v);
#pragma unroll
  for (int i = 0; i < W; ++i) a.w[i] = __builtin_amdgcn_readfirstlane(a.w[i]);
  return __builtin_bit_cast(T, a);
}

// wave_sum of a v that is +0 on lanes `count` and above (count > 0, uniform):
// the steps that would only add those zeros are left out.
template <typename T>
__device__ __forceinline__ T wave_sum_first(T v, int count) {
  auto add = [](T a, T b) { return a + b; };
  if (count > 32) v = wave_step<32>(v, add);
  if (count > 16) v = wave_step<16>(v, add);
  if (count > 4) {  // wave_step<4> relies on <8> (dpp_xor)
    v = wave_step<8>(v, add);
    v = wave_step<4>(v, add);
  }
  if (count > 2) v = wave_step<2>(v, add);
  if (count > 1) v = wave_step<1>(v, add);
  return bcast0(v);
}

__device__ __forceinline__ int wave_min(int v) {
  return wave_reduce(v, [](int a, int b) { return a < b ? a : b; });
}

// Sum over the workgroup; the result is valid in thread 0.  `lds` must hold
// kBlock / kWave values.  Fixed order, so the result is deterministic.
template <typename T>
__device__ __forceinline__ T block_sum(T v, T *lds) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  __syncthreads();  // a previous block_sum may still be reading lds
  if (lane == 0) lds[wid] = v;
  __syncthreads();
  T s = 0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) s += lds[w];
  }
  return s;
}

// Grid-wide sums are two launches: every workgroup of the producing kernel
// stores its partial with a plain store, and a one-workgroup kernel sums
// the partials in index order.  The kernel boundary makes the partials
// visible; no device-scope fence (an L2 write-back on gfx950's per-XCD L2s)
// is issued per workgroup, and the result does not depend on timing.

// Threads of the one-workgroup kernels that sum partials.
constexpr int kFinalBlock = 1024;

// Sum of `count` strided partials src[k*stride + off] over one workgroup of
// kFinalBlock threads; valid in thread 0.  Eight independent accumulators
// keep eight loads in flight per thread (one round trip for up to 8192
// partials); the order is fixed, so the result is deterministic.  `lds` holds kFinalBlock / kWave values.
template <typename T>
__device__ __forceinline__ T sum_partials(const T *src, int count, int stride, int off, T *lds) {
  constexpr int F = 8;
  T a[F];
#pragma unroll
  for (int f = 0; f < F; ++f) a[f] = 0;
  int k = threadIdx.x;
  for (; k + (F - 1) * kFinalBlock < count; k += F * kFinalBlock) {
    T v[F];
#pragma unroll
    for (int f = 0; f < F; ++f) v[f] = src[(size_t)(k + f * kFinalBlock) * stride + off];
#pragma unroll
    for (int f = 0; f < F; ++f) a[f] += v[f];
  }
  // the remainder: up to F - 1 loads, all issued before any add
  {
    T v[F];
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const int kk = k + f * kFinalBlock;
      v[f] = kk < count ? src[(size_t)kk * stride + off] : T(0);
    }
#pragma unroll
    for (int f = 0; f < F; ++f) a[f] += v[f];
  }
  T v = wave_sum(((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7])));
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  __syncthreads();  // a previous call may still be reading lds
  if (lane == 0) lds[wid] = v;
  __syncthreads();
  T s = 0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 0; w < kFinalBlock / kWave; ++w) s += lds[w];
  }
  return s;
}

// XCD-aware tile index: workgroup b runs on XCD b % 8; give each XCD a
// contiguous range of tiles so neighbouring tiles share that XCD's L2.
__device__ __forceinline__ long long xcd_tile(long long b, long long nblocks) {
  const long long per = (nblocks + kXcds - 1) / kXcds;
  return (b % kXcds) * per + b / kXcds;
}

template <typename T>
__device__ __forceinline__ T ld_stream(const T *p) {
  return __builtin_nontemporal_load(p);
}
template <bool NT, typename T>
__device__ __forceinline__ T ld_entry(const T *p) {
  return NT ? __builtin_nontemporal_load(p) : *p;
}

// How much of a matrix products load through the caches, for the next product
// to find in the Infinity Cache (256 MB): `cached` of every kCachedParts
// slices, tiles or blocks (interleaved, so that each XCD has its share), the
// rest past the caches.  All of it where it about fits with the vectors that
// are used between two products; else as much as leaves room for those and
// for what streams through (216 MB in all), since a matrix that is too large
// would sweep itself and them out.  Jacobi-CG on 3D Q1 in FP64 (SELL-64, offset
// form), MB of matrix + vectors, ms a solve with none, part and all of the
// matrix through the caches: 96^3, 197 + 44, 15.6 - 12.4; 100^3, 223 + 49, 17.7
// 15.5 14.8; 104^3, 250 + 56, 20.1 17.2 18.8; 112^3, 312 + 69, 26.3 22.6 27.2;
// 128^3, 464 + 103, 36.9 34.5 38.6.
constexpr int kCachedParts = 64;
inline int entries_cached(long long entries, size_t entry_bytes, size_t vector_bytes) {
  constexpr size_t kAll = (size_t)264 << 20, kPart = (size_t)216 << 20;
  const size_t bytes = (size_t)entries * entry_bytes;
  if (bytes + vector_bytes <= kAll) return kCachedParts;
  return vector_bytes < kPart && bytes > 0
             ? (int)std::min<size_t>(kCachedParts, kCachedParts * (kPart - vector_bytes) / bytes)
             : 0;
}
// Vectors that an iteration of the solvers uses between two products: x, r,
// z, p, A p, D^-1.
constexpr size_t kCgVectors = 6;

// The same for a product by itself, which cannot know what comes before the
// next one: all of a matrix that takes a third of the cache with x and y, else
// none.  Of three 3D Q1 matrices in turn, us a product past and through the
// caches: 64^3 (60 MB) 15.7 and 12.3, 96^3 (197 MB) 44.5 and 45.9, 128^3 in
// FP32 (232 MB) 43.4 and 48.4.  (A product right after a kernel that has
// written 1 GB waits for the cache to write that back: 64^3 19.0 past and 27.9
// through the caches, after one that has read 1 GB 18.7 and 16.3.)
inline int entries_cached_once(long long entries, size_t entry_bytes, size_t vector_bytes) {
  return (size_t)entries * entry_bytes + vector_bytes <= ((size_t)88 << 20) ? kCachedParts : 0;
}
// Whether part `i` is loaded past the caches.
__device__ __forceinline__ bool past_caches(long long i, int cached) {
  return (int)(i & (kCachedParts - 1)) >= cached;
}

// Buffer descriptor word 3 for raw (untyped) buffer access on gfx9-family
// GPUs (gfx950 included).
constexpr int kRsrcWord3 = 0x00020000;

template <typename T>
__device__ __forceinline__ T buffer_load(__amdgpu_buffer_rsrc_t r, unsigned off);
template <>
__device__ __forceinline__ double buffer_load<double>(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}
template <>
__device__ __forceinline__ float buffer_load<float>(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
