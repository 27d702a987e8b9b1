// SELL-64 execution layout of a CSR matrix: device-side build from the CSR
// arrays, value refresh, and SpMV.  The layout is described in
// hflmp_sell.hpp.  It is an execution format of the HIP platform for a
// matrix the caller holds in CSR (lmatrix_formats.h:51-56), in the role of
// the reference's ELL format slot (la_global.h:56, MATRIX_FORMAT::ELL): the
// products y = A x and y += A x are those of CPU_CSR_lMatrix::VectorMult /
// VectorMultAdd (CPUsimple_csr_lmatrix.cc:76-111, lmatrix_csr_cpu.cc:
// 1424-1450), bit for bit.
#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>

#include "hflmp_sell.hpp"

namespace {

enum SellMode { kSellAssign = 0, kSellAdd = 1 };

struct SellStats {
  int long_rows;           // not 0: a row has more than 255 entries
  unsigned int bad16;      // entries whose offset from the slice start needs more than 16 bits
  int sample;              // above 0: the offset form would be far too large
  int bad_off;             // not 0: that, or a slice that the offset form cannot hold
  int bad16_off;           // bad16 as the offset count saw it (all of it if bad_off is 0)
  int max_off;             // the largest |offset|
  long long entries;       // of the form with columns
  long long kentries;      // of the offset form
};

// The offset form is taken where its bytes are below this part of the
// columns' (offset_form_smaller).
constexpr double kOffsetGain = 0.95;

__host__ __device__ inline double offset_form_bytes(double entries, int vb) {
  return entries * (vb + 12.0 / kSellRows);
}
__host__ __device__ inline double column_form_bytes(double entries, double rows, int vb,
                                                    int col_bytes) {
  return entries * (vb + col_bytes) + rows;
}

// Row lengths (a byte each) and, per slice, the longest row (m; where its
// entries sit is sell_pos's business).
// Threads walk rows in whole waves, so a wave is always one slice.
__global__ void __launch_bounds__(kBlock)
    sell_lengths_kernel(int nrow, int nslice, const int *__restrict__ rp,
                        unsigned char *__restrict__ rlen, int *__restrict__ slen) {
  const long long total = (long long)nslice * kSellRows;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < total;
       i += (long long)gridDim.x * kBlock) {
    int len = 0;
    if (i < nrow) {
      len = rp[i + 1] - rp[i];
      rlen[i] = (unsigned char)(len > 255 ? 255 : len);
    }
    int m = len;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
      const int other = __shfl_xor(m, o);
      m = other > m ? other : m;
    }
    if ((threadIdx.x & (kWave - 1)) == 0) slen[i / kSellRows] = m;
  }
}

// What the offset count leaves for a slice.
struct SliceOffsets {
  int len;   // distinct offsets; -1: the form cannot hold the slice
  int most;  // the largest |offset|, or kFar if a column is beyond int16
};
constexpr int kFar = INT_MAX;

__device__ __forceinline__ int slice_len(int v) { return v; }
__device__ __forceinline__ int slice_len(SliceOffsets v) { return v.len > 0 ? v.len : 0; }

// soff[s] = sum over t < s of 64 slen[t]; soff[nslice] = all, the entries.
// S = int (the longest rows) starts *stats, S = SliceOffsets adds what the
// slices' counts say together.  One workgroup, eight consecutive slices a
// thread and step (33,000 slices: 14 us; with one run of slices a thread 56).
template <typename S>
__global__ void __launch_bounds__(kFinalBlock)
    sell_scan_kernel(int nslice, const S *__restrict__ slen, long long *__restrict__ soff,
                     SellStats *stats) {
  constexpr int U = 8, kWaves = kFinalBlock / kWave;
  constexpr bool OFFS = std::is_same<S, SliceOffsets>::value;
  __shared__ int tot[kWaves];  // (a step has at most 8192 x 255 entries a row)
  int most = 0;
  bool far = false, bad = false;
  const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
  long long run = 0;  // entries before the step's slices
  S next[U];
  auto load = [&](long long s0) {
    const long long s = s0 + (long long)t * U;
    if (s + U <= nslice) {
      __builtin_memcpy(next, __builtin_assume_aligned(slen + s, 16), sizeof(next));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) next[u] = s + u < nslice ? slen[s + u] : S{};
    }
  };
  load(0);
  for (long long s0 = 0; s0 < nslice; s0 += (long long)kFinalBlock * U) {
    int m[U], sum = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      m[u] = slice_len(next[u]);
      sum += m[u];
      if constexpr (OFFS) {
        bad = bad || next[u].len < 0;
        far = far || next[u].most == kFar;
        most = next[u].most > most ? next[u].most : most;
      } else {
        bad = bad || m[u] > 255;
      }
    }
    load(s0 + (long long)kFinalBlock * U);
    int incl = sum;  // over the wave's lanes up to this one
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int v = __shfl_up(incl, o);
      if (lane >= o) incl += v;
    }
    if (lane == kWave - 1) tot[wid] = incl;
    __syncthreads();
    int before = incl - sum, all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w < wid) before += tot[w];
      all += tot[w];
    }
    long long at[U];
    at[0] = run + (long long)kSellRows * before;
#pragma unroll
    for (int u = 1; u < U; ++u) at[u] = at[u - 1] + (long long)kSellRows * m[u - 1];
    const long long s = s0 + (long long)t * U;
    if (s + U <= nslice) {
      __builtin_memcpy(__builtin_assume_aligned(soff + s, 16), at, sizeof(at));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + u < nslice) soff[s + u] = at[u];
    }
    run += (long long)kSellRows * all;
    __syncthreads();
  }
  const int any_bad = __syncthreads_or(bad);
  if constexpr (OFFS) {
    const int any_far = __syncthreads_or(far);
    most = -wave_min(-most);
    if (lane == 0) tot[wid] = most;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) most = tot[w] > most ? tot[w] : most;
    if (t == 0) {
      stats->bad_off = any_bad;
      stats->bad16_off = any_far;
      stats->max_off = most;
      stats->kentries = run;
    }
  } else if (t == 0) {
    *stats = SellStats{};
    stats->long_rows = any_bad;
    stats->entries = run;
  }
  if (t == 0) soff[nslice] = run;
}

// Counts entries whose column is not within int16 of its slice's first row
// (AFTER_OFFSETS: unless the offset count has seen every entry).
template <bool AFTER_OFFSETS>
__global__ void __launch_bounds__(kBlock)
    sell_band_kernel(int nrow, const int *__restrict__ rp, const int *__restrict__ ci,
                     SellStats *stats) {
  if (AFTER_OFFSETS && !stats->bad_off) return;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < nrow; i += gridDim.x * kBlock) {
    const int base = (i / kSellRows) * kSellRows;
    unsigned int bad = 0;
    for (int k = rp[i]; k < rp[i + 1]; ++k) {
      const int d = ci[k] - base;
      bad += (d < -32768 || d > 32767) ? 1u : 0u;
    }
    if (bad) atomicAdd(&stats->bad16, bad);
  }
}

// Scatter of row i's entries into its lane of its slice (thread per row).
// COLS = false refreshes the values only: a row whose length differs from
// the one stored at build time (rlen) would be placed past its lane's
// entries, so it is skipped and counted in *changed instead.
template <typename T, typename IT, bool COLS>
__global__ void __launch_bounds__(kBlock)
    sell_fill_kernel(int nrow, int P, const int *__restrict__ rp, const int *__restrict__ ci,
                     const T *__restrict__ val, const long long *__restrict__ soff,
                     const int *__restrict__ slen, IT *__restrict__ col,
                     T *__restrict__ sval, const unsigned char *__restrict__ rlen,
                     unsigned int *changed) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < nrow; i += gridDim.x * kBlock) {
    const int s = i / kSellRows, lane = i % kSellRows;
    const long long off = soff[s];
    const int m = slen[s];
    const int k0 = rp[i], len = rp[i + 1] - k0;
    if (!COLS && len != (int)rlen[i]) {
      atomicAdd(changed, 1u);
      continue;
    }
    for (int j = 0; j < len; ++j) {
      const long long pos = sell_pos(off, m, P, lane, j);
      if (COLS) {
        const int c = ci[k0 + j];
        col[pos] = (IT)(std::is_same<IT, int>::value ? c : c - s * kSellRows);
      }
      sval[pos] = val[k0 + j];
    }
  }
}

// ---- offset form ------------------------------------------------------------
// A slice's entries are read from LDS where it has at most so many (28 a
// row), where one wave has copied them: a lane on its row of the arrays
// itself reads 64 lines at a time, of which little is left in the caches when
// it comes to the next entry (3D Q1 128^3 in FP64: count 0.59 -> 0.09 ms, fill
// 2.08 -> 0.33 ms; the fill of the form with columns 1.7 ms).
constexpr int kStageEntries = 28 * kSellRows;

// what the wave's lanes have written to LDS is what they read next
__device__ __forceinline__ void wave_in_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <typename V>
__device__ __forceinline__ void stage_entries(V *lds, const V *__restrict__ src, int n) {
  constexpr int U = 8;
  wave_in_order();  // (the slice before is done with)
  for (int e0 = threadIdx.x & (kWave - 1); e0 < n; e0 += U * kWave) {
    V v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e0 + u * kWave < n) v[u] = src[e0 + u * kWave];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e0 + u * kWave < n) lds[e0 + u * kWave] = v[u];
  }
  wave_in_order();
}

// The rows of slice s: this lane's CSR range [k, end) and the slice's [first,
// last).
struct SliceRows {
  int row, k, end, first, last;
};
__device__ __forceinline__ SliceRows slice_rows(int s, int nrow, const int *__restrict__ rp) {
  SliceRows r;
  r.row = s * kSellRows + (threadIdx.x & (kWave - 1));
  const int i = r.row < nrow ? r.row : nrow;
  r.k = rp[i];
  r.end = rp[r.row < nrow ? r.row + 1 : nrow];
  r.first = __builtin_amdgcn_readfirstlane(r.k);
  r.last = __builtin_amdgcn_readlane(r.end, kWave - 1);
  return r;
}

// Walks a slice (one wave, lane = row) over the distinct column offsets of
// its rows in ascending order: f(position, offset, whether this lane's row
// has the entry, its CSR index), with the columns from col(CSR index).
// Returns the number of offsets, or -1 where a row's columns do not ascend
// strictly or go_on(position) is false.
template <typename Col, typename G, typename F>
__device__ __forceinline__ int for_slice_offsets(const SliceRows &r, Col &&col, G &&go_on,
                                                 F &&f) {
  int k = r.k;
  // the row's current offset and the next one, loaded a step ahead
  int off = k < r.end ? col(k) - r.row : INT_MAX;
  int next = k + 1 < r.end ? col(k + 1) - r.row : INT_MAX;
  for (int j = 0;; ++j) {
    const int m = wave_min(off);
    if (m == INT_MAX) return j;
    if (!go_on(j)) return -1;
    const bool has = off == m;
    f(j, m, has, k);
    bool bad = false;
    if (has) {
      ++k;
      off = next;
      next = k + 1 < r.end ? col(k + 1) - r.row : INT_MAX;
      bad = off <= m;
    }
    if (__any(bad)) return -1;
  }
}

// One slice's walk with the columns staged where they fit; lds: kStageEntries.
template <typename G, typename F>
__device__ __forceinline__ int count_offsets(int s, int nrow, const int *__restrict__ rp,
                                             const int *__restrict__ ci, int *lds, G &&go_on,
                                             F &&see) {
  const SliceRows r = slice_rows(s, nrow, rp);
  if (r.last - r.first > kStageEntries)
    return for_slice_offsets(r, [&](int k) { return ci[k]; }, go_on, see);
  stage_entries(lds, ci + r.first, r.last - r.first);
  return for_slice_offsets(r, [&](int k) { return lds[k - r.first]; }, go_on, see);
}

// Positions of a slice up to which the offset form is the smaller one.
__device__ __forceinline__ int offset_share(int m, int vb) {
  return (int)(kOffsetGain * column_form_bytes((double)kSellRows * m, kSellRows, vb, 4) /
               offset_form_bytes(kSellRows, vb));
}

// A look at kSampleSlices of the slices, evenly spaced, before all are
// counted: where they take more than twice their share of positions, the
// form is out of question (an unstructured matrix takes hundreds of positions
// a slice, 0.29 ms for 512^2 2D Q1 nodes in random order; the look takes 0.01).
constexpr int kSampleSlices = 64;

__global__ void __launch_bounds__(kBlock)
    sell_offsets_sample_kernel(int nrow, int nslice, int vb, const int *__restrict__ rp,
                               const int *__restrict__ ci, const int *__restrict__ slen,
                               SellStats *stats) {
  __shared__ int cols[kSellSlicesPerBlock][kStageEntries];
  __shared__ int over;
  if (threadIdx.x == 0) over = 0;
  __syncthreads();
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int i = blockIdx.x * kSellSlicesPerBlock + wid;
  const int n = nslice < kSampleSlices ? nslice : kSampleSlices;
  if (i < n) {
    const int s = (int)((long long)i * nslice / n);
    const int share = offset_share(slen[s], vb);
    const int K = count_offsets(s, nrow, rp, ci, cols[wid],
                                [&](int j) { return j < 3 * share && j < 255; },
                                [](int, int, bool, int) {});
    if ((threadIdx.x & (kWave - 1)) == 0) atomicAdd(&over, (K < 0 ? 3 * share : K) - 2 * share);
  }
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(&stats->sample, over);
}

// The distinct offsets of each slice.
__global__ void __launch_bounds__(kBlock)
    sell_offsets_count_kernel(int nrow, int nslice, const int *__restrict__ rp,
                              const int *__restrict__ ci, SliceOffsets *__restrict__ klen,
                              const SellStats *__restrict__ stats) {
  __shared__ int cols[kSellSlicesPerBlock][kStageEntries];
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int lane = threadIdx.x & (kWave - 1);
  const bool sampled_out = stats->sample > 0;
  for (int s = blockIdx.x * kSellSlicesPerBlock + wid; s < nslice;
       s += gridDim.x * kSellSlicesPerBlock) {
    SliceOffsets out{-1, 0};
    if (!sampled_out) {
      bool far = false;
      out.len = count_offsets(
          s, nrow, rp, ci, cols[wid], [](int j) { return j < 255; },
          [&](int, int o, bool has, int) {
            far = far || (has && (o + lane < -32768 || o + lane > 32767));
            const int a = o < 0 ? -o : o;
            out.most = a > out.most ? a : out.most;
          });
      if (__any(far)) out.most = kFar;
    }
    if (lane == 0) klen[s] = out;
  }
}

// One wave a workgroup: the LDS of more would leave fewer in flight.
template <typename T>
__global__ void __launch_bounds__(kWave)
    sell_offsets_fill_kernel(int nrow, int nslice, int P, const int *__restrict__ rp,
                             const int *__restrict__ ci, const T *__restrict__ val,
                             const long long *__restrict__ koff,
                             const SliceOffsets *__restrict__ klen,
                             long long *__restrict__ soff, int *__restrict__ slen,
                             int *__restrict__ off, unsigned long long *__restrict__ mask,
                             T *__restrict__ sval) {
  __shared__ T vals[kStageEntries];
  __shared__ int cols[kStageEntries];
  const int lane = threadIdx.x;
  for (int s = blockIdx.x; s < nslice; s += gridDim.x) {
    const long long base = koff[s];
    const int K = slice_len(klen[s]);
    const SliceRows r = slice_rows(s, nrow, rp);
    if (lane == 0) {
      soff[s] = base;
      slen[s] = K;
      if (s == nslice - 1) soff[nslice] = koff[nslice];
    }
    auto walk = [&](auto col, auto value) {
      for_slice_offsets(r, col, [](int) { return true; }, [&](int j, int o, bool has, int k) {
        const unsigned long long m = __ballot(has);
        if (lane == 0) {
          off[base / kSellRows + j] = o;
          mask[base / kSellRows + j] = m;
        }
        sval[sell_pos(base, K, P, lane, j)] = has ? value(k) : T(0);
      });
    };
    const int n = r.last - r.first;
    if (n <= kStageEntries) {
      stage_entries(cols, ci + r.first, n);
      stage_entries(vals, val + r.first, n);
      walk([&](int k) { return cols[k - r.first]; }, [&](int k) { return vals[k - r.first]; });
    } else {
      walk([&](int k) { return ci[k]; }, [&](int k) { return val[k]; });
    }
  }
}

// New values for the same pattern; rows whose length changed are skipped and
// counted.  A wave a slice, its values by way of LDS as in the fill (3D Q1
// 64^3 in FP64: 52 us a call; a thread a row 142, the form with columns 125).
template <typename T>
__global__ void __launch_bounds__(kWave)
    sell_offsets_values_kernel(int nrow, int nslice, int P, const int *__restrict__ rp,
                               const T *__restrict__ val, const long long *__restrict__ koff,
                               const int *__restrict__ klen,
                               const unsigned long long *__restrict__ mask,
                               T *__restrict__ sval, const unsigned char *__restrict__ rlen,
                               unsigned int *changed) {
  __shared__ T vals[kStageEntries];
  const int lane = threadIdx.x;
  for (int s = blockIdx.x; s < nslice; s += gridDim.x) {
    const long long base = koff[s];
    const int K = klen[s];
    const SliceRows r = slice_rows(s, nrow, rp);
    const bool same = r.row < nrow && r.end - r.k == (int)rlen[r.row];
    if (r.row < nrow && !same) atomicAdd(changed, 1u);
    auto put = [&](auto value) {
      int k = r.k;
      for (int j = 0; j < K; ++j)
        if (same && ((mask[base / kSellRows + j] >> lane) & 1))
          sval[sell_pos(base, K, P, lane, j)] = value(k++);
    };
    const int n = r.last - r.first;
    if (n <= kStageEntries && __all(r.k >= r.first && r.end <= r.last)) {
      stage_entries(vals, val + r.first, n);
      put([&](int k) { return vals[k - r.first]; });
    } else {
      put([&](int k) { return val[k]; });
    }
  }
}

template <typename Op, int MODE>
__device__ __forceinline__ void sell_spmv_rows(const Op &op,
                                               const typename Op::value_type *__restrict__ x,
                                               typename Op::value_type *__restrict__ y) {
  using T = typename Op::value_type;
  const long long unit = xcd_tile(blockIdx.x, gridDim.x);
  T s = 0;
  if (MODE == kSellAdd) {
    const long long r = op.thread_row(unit);
    if (r >= 0 && r < op.nrow) s = y[r];
  }
  TileRow tr;
  s = op.row_sum(unit, x, s, tr, nullptr);
  // y is not read again by this launch: stream it past the caches
  if (tr.has_row) __builtin_nontemporal_store(s, y + tr.row);
}

template <typename Op, int MODE>
__global__ void __launch_bounds__(kBlock)
    sell_spmv_kernel(Op op, const typename Op::value_type *__restrict__ x,
                     typename Op::value_type *__restrict__ y) {
  sell_spmv_rows<Op, MODE>(op, x, y);
}

// int16 columns: the loop fits 80 VGPRs, six waves per SIMD (on 128^3 Q1
// FP64: 105 us per SpMV against 109 us at five; the int32 form would
// spill at six)
template <typename Op, int MODE>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6)))
    sell_spmv16_kernel(Op op, const typename Op::value_type *__restrict__ x,
                       typename Op::value_type *__restrict__ y) {
  sell_spmv_rows<Op, MODE>(op, x, y);
}

void sell_free(hflmp_sell *m) {
  if (!m) return;
  int cur = -1;
  (void)hipGetDevice(&cur);
  if (cur != m->device) (void)hipSetDevice(m->device);
  (void)hipFree(m->meta);
  (void)hipFree(m->data);
  if (cur >= 0 && cur != m->device) (void)hipSetDevice(cur);
  delete m;
}

template <typename T>
int sell_create(hflmp_ctx *ctx, int nrow, int ncol, int nnz, const int *rp, const int *ci,
                const T *val, int flags, hflmp_sell **out) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, out != nullptr, "sell_create: null output handle");
  *out = nullptr;
  HFLMP_REQUIRE(ctx, nrow > 0 && ncol > 0 && nnz >= 0, "sell_create: bad sizes");
  HFLMP_REQUIRE(ctx, rp && (nnz == 0 || (ci && val)), "sell_create: null pointer");
  HFLMP_REQUIRE(ctx, (flags & ~(HFLMP_SELL_COL16 | HFLMP_SELL_ANY_PADDING | kSellOffsets)) == 0,
                "sell_create: unknown flags %d", flags);
  hipStream_t s = ctx->stream;
  auto *m = new hflmp_sell();
  m->device = ctx->device;
  m->nrow = nrow;
  m->ncol = ncol;
  m->nnz = nnz;
  m->nslice = (nrow + kSellRows - 1) / kSellRows;
  m->chunk = SellChunk<T>::P;
  m->value_bytes = sizeof(T);
  m->col_bytes = 4;
  // Three allocations (each costs the host several microseconds): what the
  // layout keeps a slice and row, what only the build needs, and the entries.
  char *build = nullptr;
  int rc = HFLMP_OK;
  auto fail = [&](int code, const char *msg) {
    (void)hipFree(build);
    sell_free(m);
    return set_error(ctx, code, "sell_create: %s", msg);
  };
  size_t bytes = 0;
  auto take = [&](size_t b) {
    const size_t at = bytes;
    bytes += (b + 255) & ~size_t(255);
    return at;
  };
  auto alloc = [&](char **p) {
    const size_t b = bytes;
    bytes = 0;
    return hipMalloc(reinterpret_cast<void **>(p), b) == hipSuccess;
  };
  const size_t soff_bytes = sizeof(long long) * ((size_t)m->nslice + 1);
  const size_t slen_bytes = sizeof(int) * (size_t)m->nslice;
  const size_t o_soff = take(soff_bytes), o_slen = take(slen_bytes), o_rlen = take((size_t)nrow);
  const size_t o_check = take(sizeof(unsigned int));
  if (!alloc(&m->meta)) return fail(HFLMP_ENOMEM, "out of device memory");
  m->soff = reinterpret_cast<long long *>(m->meta + o_soff);
  m->slen = reinterpret_cast<int *>(m->meta + o_slen);
  m->rlen = reinterpret_cast<unsigned char *>(m->meta + o_rlen);
  m->check = reinterpret_cast<unsigned int *>(m->meta + o_check);
  // x is read through 32-bit byte offsets in the offset form
  const bool try_off = (flags & (HFLMP_SELL_COL16 | kSellOffsets)) && nnz > 0 &&
                       (size_t)ncol * sizeof(T) < (1ull << 31) &&
                       (size_t)nrow * sizeof(T) < (1ull << 31);
  const bool try16 = (flags & HFLMP_SELL_COL16) && nnz > 0;
  const size_t o_stats = take(sizeof(SellStats));
  const size_t o_koff = take(try_off ? soff_bytes : 0),
               o_klen = take(try_off ? sizeof(SliceOffsets) * (size_t)m->nslice : 0);
  if (!alloc(&build)) return fail(HFLMP_ENOMEM, "out of device memory");
  SellStats *stats = reinterpret_cast<SellStats *>(build + o_stats);
  long long *koff = reinterpret_cast<long long *>(build + o_koff);  // the offset form's slices
  auto *klen = reinterpret_cast<SliceOffsets *>(build + o_klen);
  const long long lanes = (long long)m->nslice * kSellRows;
  long long g = (lanes + kBlock - 1) / kBlock;
  if (g > 65536) g = 65536;
  sell_lengths_kernel<<<(unsigned)g, kBlock, 0, s>>>(nrow, m->nslice, rp, m->rlen, m->slen);
  sell_scan_kernel<int><<<1, kFinalBlock, 0, s>>>(m->nslice, m->slen, m->soff, stats);
  if (try_off) {
    sell_offsets_sample_kernel<<<kSampleSlices / kSellSlicesPerBlock, kBlock, 0, s>>>(
        nrow, m->nslice, (int)sizeof(T), rp, ci, m->slen, stats);
    sell_offsets_count_kernel<<<grid_for(lanes, 1), kBlock, 0, s>>>(nrow, m->nslice, rp, ci, klen,
                                                                    stats);
    sell_scan_kernel<SliceOffsets><<<1, kFinalBlock, 0, s>>>(m->nslice, klen, koff, stats);
    if (try16) sell_band_kernel<true><<<grid_for(nrow, 1), kBlock, 0, s>>>(nrow, rp, ci, stats);
  } else if (try16) {
    sell_band_kernel<false><<<grid_for(nrow, 1), kBlock, 0, s>>>(nrow, rp, ci, stats);
  }
  if (hipGetLastError() != hipSuccess) return fail(HFLMP_EHIP, "launch failed");
  SellStats hs;
  if (hipMemcpyAsync(ctx->host_pinned, stats, sizeof(hs), hipMemcpyDeviceToHost, s) !=
          hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return fail(HFLMP_EHIP, "HIP error while sizing");
  std::memcpy(&hs, ctx->host_pinned, sizeof(hs));
  if (hs.long_rows)
    return fail(HFLMP_EFORMAT, "a row has more than 255 entries (use the CSR kernels)");
  // Padding is never loaded (a lane stops at its row's length), but it
  // costs memory and partly-used cache lines; refuse more than twice the
  // nonzeros of it.
  if (!(flags & HFLMP_SELL_ANY_PADDING) &&
      hs.entries > 3LL * nnz + (long long)kSellRows * m->chunk)
    return fail(HFLMP_EFORMAT, "row lengths vary too much within slices (use the CSR kernels)");
  if (try16 && (try_off && !hs.bad_off ? hs.bad16_off : hs.bad16) == 0) m->col_bytes = 2;
  // The offset form where it is at least 5% smaller than the columns': the
  // product's time follows its bytes, up to that line.  3D Q1 96^3 with a
  // quarter of the entries dropped at random, FP64 (1.33 stored values an
  // entry, 10.96 B against 12.43): 44.4 us, with columns 49.6; with 40%
  // dropped, FP32 (1.64, 6.96 B against 8.16): 19.0 and 29.8 us.
  m->off_form = try_off && hs.bad_off == 0 &&
                offset_form_bytes((double)hs.kentries, sizeof(T)) <
                    kOffsetGain * column_form_bytes((double)hs.entries, nrow, sizeof(T),
                                                    m->col_bytes);
  m->entries = m->off_form ? hs.kentries : hs.entries;
  m->max_off = hs.max_off;
  const size_t ne = m->entries > 0 ? (size_t)m->entries : 1;
  const size_t np = m->off_form ? ne / kSellRows : 0;  // positions
  const size_t o_val = take(ne * sizeof(T));
  const size_t o_col = take(m->off_form ? 0 : ne * m->col_bytes);
  const size_t o_mask = take(np * sizeof(unsigned long long)), o_off = take(np * sizeof(int));
  if (!alloc(&m->data)) return fail(HFLMP_ENOMEM, "out of device memory");
  m->val = m->data + o_val;
  if (m->off_form) {
    m->mask = reinterpret_cast<unsigned long long *>(m->data + o_mask);
    m->off = reinterpret_cast<int *>(m->data + o_off);
    const int grid = std::min(m->nslice, 1 << 20);
    sell_offsets_fill_kernel<T><<<grid, kWave, 0, s>>>(
        nrow, m->nslice, m->chunk, rp, ci, val, koff, klen, m->soff, m->slen, m->off, m->mask,
        static_cast<T *>(m->val));
  } else {
    m->col = m->data + o_col;
    if ((rc = hflmp_fill_zero(ctx, m->col, ne * m->col_bytes)) != HFLMP_OK)
      return fail(rc, "fill");
    if ((rc = hflmp_fill_zero(ctx, m->val, ne * sizeof(T))) != HFLMP_OK) return fail(rc, "fill");
    if (nnz > 0) {
      if (m->col_bytes == 2)
        sell_fill_kernel<T, short, true><<<grid_for(nrow, 1), kBlock, 0, s>>>(
            nrow, m->chunk, rp, ci, val, m->soff, m->slen, static_cast<short *>(m->col),
            static_cast<T *>(m->val), nullptr, nullptr);
      else
        sell_fill_kernel<T, int, true><<<grid_for(nrow, 1), kBlock, 0, s>>>(
            nrow, m->chunk, rp, ci, val, m->soff, m->slen, static_cast<int *>(m->col),
            static_cast<T *>(m->val), nullptr, nullptr);
    }
  }
  if (hipGetLastError() != hipSuccess) return fail(HFLMP_EHIP, "launch failed");
  // the build's memory is freed only after the stream has used it
  if (hipStreamSynchronize(s) != hipSuccess) return fail(HFLMP_EHIP, "HIP error in build");
  (void)hipFree(build);
  *out = m;
  return HFLMP_OK;
}

template <typename T>
int sell_set_values(hflmp_ctx *ctx, hflmp_sell *m, const int *rp, const T *val) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, m && rp && (m->nnz == 0 || val), "sell_set_values: null pointer");
  HFLMP_REQUIRE(ctx, m->value_bytes == (int)sizeof(T), "sell_set_values: value type mismatch");
  HFLMP_REQUIRE(ctx, m->device == ctx->device, "sell_set_values: matrix on another device");
  if (m->nnz == 0) return HFLMP_OK;
  hipStream_t s = ctx->stream;
  int rc = hflmp_fill_zero(ctx, m->check, sizeof(unsigned int));
  if (rc) return rc;
  if (m->off_form)
    sell_offsets_values_kernel<T><<<std::min(m->nslice, 1 << 20), kWave, 0, s>>>(
        m->nrow, m->nslice, m->chunk, rp, val, m->soff, m->slen, m->mask,
        static_cast<T *>(m->val), m->rlen, m->check);
  else
    sell_fill_kernel<T, int, false><<<grid_for(m->nrow, 1), kBlock, 0, s>>>(
      m->nrow, m->chunk, rp, nullptr, val, m->soff, m->slen, nullptr, static_cast<T *>(m->val),
      m->rlen, m->check);
  HFLMP_LAUNCH_CHECK(ctx);
  unsigned int changed = 0;
  HFLMP_HIP_CHECK(ctx, hipMemcpyAsync(&changed, m->check, sizeof(changed),
                                      hipMemcpyDeviceToHost, s));
  HFLMP_HIP_CHECK(ctx, hipStreamSynchronize(s));
  if (changed)
    return set_error(ctx, HFLMP_EFORMAT,
                     "sell_set_values: %u rows differ in length from the pattern the layout "
                     "was built for (their values were not copied; rebuild the layout)",
                     changed);
  return HFLMP_OK;
}

template <typename T, int MODE>
int sell_spmv(hflmp_ctx *ctx, const hflmp_sell *m, const T *x, T *y) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, m && x && y, "sell_spmv: null pointer");
  HFLMP_REQUIRE(ctx, m->value_bytes == (int)sizeof(T), "sell_spmv: value type mismatch");
  HFLMP_REQUIRE(ctx, m->device == ctx->device, "sell_spmv: matrix on another device");
  const unsigned grid = sell_grid(m->nrow);
  hipStream_t s = ctx->stream;
  if (m->off_form)
    sell_spmv16_kernel<SellOffOp<T>, MODE><<<grid, kBlock, 0, s>>>(
        sell_off_view<T>(m, true), x, y);
  else if (m->col_bytes == 2)
    sell_spmv16_kernel<SellOp<T, short>, MODE><<<grid, kBlock, 0, s>>>(
        sell_view<T, short>(m, true), x, y);
  else
    sell_spmv_kernel<SellOp<T, int>, MODE><<<grid, kBlock, 0, s>>>(
        sell_view<T, int>(m, true), x, y);
  HFLMP_LAUNCH_CHECK(ctx);
  return HFLMP_OK;
}

}  // namespace

int sell_create_f64_internal(hflmp_ctx *ctx, int nrow, int ncol, int nnz, const int *rp,
                             const int *ci, const double *val, int flags, hflmp_sell **out) {
  return sell_create<double>(ctx, nrow, ncol, nnz, rp, ci, val, flags, out);
}

extern "C" {

int hflmp_sell_create_f64(hflmp_ctx *ctx, int nrow, int ncol, int nnz, const int *row_ptr,
                          const int *col, const double *val, int flags, hflmp_sell **out) {
  if (ctx && (flags & kSellOffsets))
    return set_error(ctx, HFLMP_EINVAL, "sell_create: unknown flags %d", flags);
  return sell_create<double>(ctx, nrow, ncol, nnz, row_ptr, col, val, flags, out);
}
int hflmp_sell_create_f32(hflmp_ctx *ctx, int nrow, int ncol, int nnz, const int *row_ptr,
                          const int *col, const float *val, int flags, hflmp_sell **out) {
  if (ctx && (flags & kSellOffsets))
    return set_error(ctx, HFLMP_EINVAL, "sell_create: unknown flags %d", flags);
  return sell_create<float>(ctx, nrow, ncol, nnz, row_ptr, col, val, flags, out);
}
int hflmp_sell_set_values_f64(hflmp_ctx *ctx, hflmp_sell *m, const int *row_ptr,
                              const double *val) {
  return sell_set_values<double>(ctx, m, row_ptr, val);
}
int hflmp_sell_set_values_f32(hflmp_ctx *ctx, hflmp_sell *m, const int *row_ptr,
                              const float *val) {
  return sell_set_values<float>(ctx, m, row_ptr, val);
}
int hflmp_sell_get_info(const hflmp_sell *m, hflmp_sell_info *info) {
  if (!m || !info) return HFLMP_EINVAL;
  info->nrow = m->nrow;
  info->ncol = m->ncol;
  info->nnz = m->nnz;
  info->chunk = m->chunk;
  info->col_bytes = m->col_bytes;
  info->value_bytes = m->value_bytes;
  info->entries = m->entries;
  info->device_bytes = (m->off_form ? (size_t)m->entries * m->value_bytes +
                                          (size_t)m->entries / kSellRows * 12
                                    : (size_t)m->entries * (m->col_bytes + m->value_bytes)) +
                       sizeof(long long) * ((size_t)m->nslice + 1) +
                       sizeof(int) * (size_t)m->nslice + (size_t)m->nrow;
  return HFLMP_OK;
}
void hflmp_sell_destroy(hflmp_sell *m) { sell_free(m); }

int hflmp_sell_spmv_f64(hflmp_ctx *ctx, const hflmp_sell *m, const double *x, double *y) {
  return sell_spmv<double, kSellAssign>(ctx, m, x, y);
}
int hflmp_sell_spmv_f32(hflmp_ctx *ctx, const hflmp_sell *m, const float *x, float *y) {
  return sell_spmv<float, kSellAssign>(ctx, m, x, y);
}
int hflmp_sell_spmv_add_f64(hflmp_ctx *ctx, const hflmp_sell *m, const double *x, double *y) {
  return sell_spmv<double, kSellAdd>(ctx, m, x, y);
}
int hflmp_sell_spmv_add_f32(hflmp_ctx *ctx, const hflmp_sell *m, const float *x, float *y) {
  return sell_spmv<float, kSellAdd>(ctx, m, x, y);
}

}  // extern "C"
