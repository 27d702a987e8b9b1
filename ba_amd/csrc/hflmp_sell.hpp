// Sliced-ELL execution layout of a CSR matrix (SELL-64), and the two
// "operator" views the fused solver kernels are written against.
//
// SELL-64: rows are cut into slices of 64 consecutive rows, one wave64 per
// slice and one lane per row.  Slice s stores its rows' entries padded to
// the slice's longest row (m entries), the first F = m - m mod P of them
// lane-interleaved in chunks of P consecutive entries of a row, the last
// m mod P in blocks of one entry per lane:
//     entry j < F of row 64 s + l  is at  off[s] + 64 P (j / P) + P l + (j mod P)
//     entry j >= F                 is at  off[s] + 64 j + l
// so each load instruction of a wave reads one contiguous 64 P-element
// block (FP64: P = 2, 16 B per lane; FP32: P = 4, 16 B per lane), a row of
// odd length loads no padding after its last entry, and the
// x gathers of a step j hit x at 64 neighbouring rows' j-th columns, which
// for an FE band is a nearly contiguous range.  Each lane adds its row's
// products in ascending storage order starting from zero (or from y[i] for
// y += A x), i.e. the summation order of CPUsimple_CSR_lMatrix::VectorMult
// (CPUsimple_csr_lmatrix.cc:76-111): the result is bit-identical to the
// sequential CPU loop.  A lane stops at its row's length (a byte per row),
// so only the padding inside a row's last chunk of P entries is loaded.
//
// Columns are int32, or int16 offsets from the slice's first row when the
// band fits (|col - 64 s| < 32768), which cuts a nonzero from 12 to 10 B
// (FP64) or from 8 to 6 B (FP32).
//
// Offset form: where a slice's rows have nearly the same column offsets
// (column - row), as the rows of a structured mesh's numbering do, no
// columns are stored at all.  Slice s lists the distinct offsets of its rows
// in ascending order (m of them); position j of every lane belongs to offset
// j, and a 64-bit mask per position tells which rows have that entry.
// Positions without one hold a zero that is never added.  An entry then
// costs its value (plus the padding, 12 B per 64 positions): 8 B instead of
// 10 in FP64, 4 instead of 6 in FP32, and x at offset j is 64 consecutive
// values, whose loads wait for no column load.  A row's entries are in
// ascending column order (the form is chosen only for such rows), so
// ascending offsets are its storage order and the sums the same.
// Measured (128^3 Q1, int16 columns before): FP64 SpMV 105.6 -> 91.6 us
// (471 MB of arrays; 544 MB of traffic, 5.9 TB/s), the CG's 107.5 -> 98.5 us;
// FP32, the mixed solver's, 57.6 -> 41.6 us.
#pragma once

#include "hflmp_spmv_tile.hpp"

struct hflmp_sell {
  int device;
  int nrow, ncol, nnz, nslice;
  int chunk;        // P
  int col_bytes;    // 4 (absolute int32) or 2 (int16 offset from the slice's first row)
  int value_bytes;  // 8 or 4
  long long entries;
  char *meta, *data;    // the two allocations behind the arrays below
  long long *soff;      // nslice + 1 entry offsets
  int *slen;            // longest row of each slice (m): the first m - m mod P entries of a
                        // row sit in chunks of P, the rest in one-entry-per-lane blocks
  int off_form;         // offset form: no col; slen is the slices' offsets
  int *off;             // offset of position j of slice s at soff[s] / 64 + j
  unsigned long long *mask;  // its rows
  int max_off;               // the largest |offset|
  unsigned int *check;  // device counter of rows whose length changed (set_values)
  unsigned char *rlen;  // row lengths
  void *col;
  void *val;
};

// sell_create with kSellOffsets allowed among the flags
int sell_create_f64_internal(hflmp_ctx *ctx, int nrow, int ncol, int nnz, const int *rp,
                             const int *ci, const double *val, int flags, hflmp_sell **out);

template <typename T>
struct SellChunk;
template <>
struct SellChunk<double> {
  static constexpr int P = 2;  // entries per lane load
  static constexpr int U = 7;  // lane loads in flight per step
};
template <>
struct SellChunk<float> {
  static constexpr int P = 4;
  static constexpr int U = 3;
};

template <typename T, int P>
struct VecOf {
  typedef T type __attribute__((ext_vector_type(P)));
};

constexpr int kSellRows = 64;                         // rows per slice (one wave)
constexpr int kSellSlicesPerBlock = kBlock / kWave;   // 4 slices per workgroup

// Position of entry j of lane `lane` in a slice whose entries start at
// `off` and whose longest row has m entries.
__host__ __device__ inline long long sell_pos(long long off, int m, int P, int lane, int j) {
  const int full = m / P * P;
  return j < full ? off + (long long)kSellRows * P * (j / P) + (long long)P * lane + (j % P)
                  : off + (long long)kSellRows * j + lane;
}

// Workgroups for an operator over SELL-64: 256 consecutive rows each,
// rounded up to a multiple of the XCD count.
inline int sell_grid(int nrow) {
  const long long units = ((long long)nrow + kBlock - 1) / kBlock;
  return (int)(((units + kXcds - 1) / kXcds) * kXcds);
}

// CSR row tiles (hflmp_spmv_tile.hpp): unit = tile of R rows.
template <typename T, typename IT = int>
struct CsrTileOp {
  using value_type = T;
  static constexpr int kLds = TileCap<T>::value;
  int nrow, R;
  int cached;  // entries_cached, by tiles
  const int *rp;
  const IT *ci;
  const T *val;

  __device__ __forceinline__ long long thread_row(long long unit) const {
    return threadIdx.x < (unsigned)R ? unit * R + threadIdx.x : -1;
  }
  __device__ __forceinline__ T row_sum(long long unit, const T *x, T s, TileRow &tr,
                                       T *lds) const {
    return past_caches(unit, cached)
               ? tile_row_sum<T, false, true, IT>(unit, R, nrow, rp, ci, val, x, s, tr, lds)
               : tile_row_sum<T, false, false, IT>(unit, R, nrow, rp, ci, val, x, s, tr, lds);
  }
};

// One lane's row of a SELL-64 slice whose entries start at col / val (the
// slice's first entry): s + sum of a_ij x_j over the row's len entries in
// ascending storage order (SUB: s - a_ij x_j; NODIAG: the entry whose
// column is dcol skipped).  smax: the slice's entries per lane.  The loads
// cover the row's own entries, or with LOAD_ALL every entry position of the
// slice (all allocated: 64 x smax entries), so that they need not wait for
// len; the sum is the same either way.  NT: entries are loaded past the
// caches.  U: chunk loads in flight per step.
// GATHER_ALL: x is read for every entry loaded, padding included (its
// column is 0; for an x that is cheap to read and has no limit to guard).
template <typename T, typename IT, bool SUB, bool NODIAG, bool LOAD_ALL, bool NT = true,
          int U = SellChunk<T>::U, bool GATHER_ALL = false>
__device__ __forceinline__ T sell_slice_sum(const IT *__restrict__ col, const T *__restrict__ val,
                                            int smax, int len, int lane,
                                            const T *__restrict__ x, int dcol, T s) {
#pragma clang fp contract(off)
  constexpr int P = SellChunk<T>::P;
  typedef typename VecOf<T, P>::type TV;
  typedef typename VecOf<IT, P>::type IV;
  const int full = smax / P * P;  // entries in P-chunks; the rest one per block
  const IV *__restrict__ c = reinterpret_cast<const IV *>(col) + lane;
  const TV *__restrict__ v = reinterpret_cast<const TV *>(val) + lane;
  // the row's entries past the last full chunk (at most P - 1), loaded
  // first so their latency overlaps the chunks'
  constexpr int TM = P > 1 ? P - 1 : 1;
  const int ntail = len - full;
  const int nload = LOAD_ALL ? smax - full : ntail;
  IT ct[TM];
  T vt[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    if (t < nload) {
      const long long q = (long long)kSellRows * (full + t) + lane;
      ct[t] = ld_entry<NT>(col + q);
      vt[t] = ld_entry<NT>(val + q);
    }
  }
  for (int j = 0; j < full; j += P * U) {
    IV cc[U];
    TV vv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if ((LOAD_ALL || j + u * P < len) && j + u * P < full) {
        cc[u] = ld_entry<NT>(c + (j / P + u) * kWave);
        vv[u] = ld_entry<NT>(v + (j / P + u) * kWave);
      }
    }
    T xx[U][P];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < P; ++q)
        if ((GATHER_ALL || j + u * P + q < len) && j + u * P < full) xx[u][q] = x[(int)cc[u][q]];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < P; ++q) {
        if (GATHER_ALL && !SUB && !NODIAG) {
          if (j + u * P < full) {
            const T sn = s + vv[u][q] * xx[u][q];
            s = j + u * P + q < len ? sn : s;
          }
          continue;
        }
        if (j + u * P + q < len && j + u * P < full && (!NODIAG || (int)cc[u][q] != dcol)) {
          if (SUB)
            s -= vv[u][q] * xx[u][q];
          else
            s += vv[u][q] * xx[u][q];
        }
      }
  }
  // the tail, in ascending order after the chunks
  T xt[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t)
    if (t < (GATHER_ALL ? nload : ntail)) xt[t] = x[(int)ct[t]];
#pragma unroll
  for (int t = 0; t < TM; ++t)
    if (t < ntail && (!NODIAG || (int)ct[t] != dcol)) {
      if (SUB)
        s -= vt[t] * xt[t];
      else
        s += vt[t] * xt[t];
    }
  return s;
}

// Two slices at once, A and B, each lane one row of each: the sums that
// sell_slice_sum<T, IT, false, false, true> forms for either (the same
// order within each row), with both slices' entry loads issued before
// either's gathers, so that a wave keeps twice the bytes in flight.
// smaxB = 0: no slice B (sB stays as given).  U: chunk loads in flight
// per slice and step (the order of the sums does not depend on it).
template <typename T, typename IT, bool NT, int U = SellChunk<T>::U>
__device__ __forceinline__ void sell_slice_sum2(const IT *__restrict__ colA,
                                                const T *__restrict__ valA, int smaxA, int lenA,
                                                const T *__restrict__ xA,
                                                const IT *__restrict__ colB,
                                                const T *__restrict__ valB, int smaxB, int lenB,
                                                const T *__restrict__ xB, int lane, T &sA, T &sB) {
#pragma clang fp contract(off)
  constexpr int P = SellChunk<T>::P;
  typedef typename VecOf<T, P>::type TV;
  typedef typename VecOf<IT, P>::type IV;
  const int fullA = smaxA / P * P, fullB = smaxB / P * P;
  const IV *__restrict__ cA = reinterpret_cast<const IV *>(colA) + lane;
  const TV *__restrict__ vA = reinterpret_cast<const TV *>(valA) + lane;
  const IV *__restrict__ cB = reinterpret_cast<const IV *>(colB) + lane;
  const TV *__restrict__ vB = reinterpret_cast<const TV *>(valB) + lane;
  constexpr int TM = P > 1 ? P - 1 : 1;
  const int ntA = lenA - fullA, ntB = lenB - fullB;
  const int nlA = smaxA - fullA, nlB = smaxB - fullB;
  IT ctA[TM], ctB[TM];
  T vtA[TM], vtB[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    if (t < nlA) {
      const long long q = (long long)kSellRows * (fullA + t) + lane;
      ctA[t] = ld_entry<NT>(colA + q);
      vtA[t] = ld_entry<NT>(valA + q);
    }
    if (t < nlB) {
      const long long q = (long long)kSellRows * (fullB + t) + lane;
      ctB[t] = ld_entry<NT>(colB + q);
      vtB[t] = ld_entry<NT>(valB + q);
    }
  }
  const int full = fullA > fullB ? fullA : fullB;
  for (int j = 0; j < full; j += P * U) {
    IV ccA[U], ccB[U];
    TV vvA[U], vvB[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j + u * P < fullA) {
        ccA[u] = ld_entry<NT>(cA + (j / P + u) * kWave);
        vvA[u] = ld_entry<NT>(vA + (j / P + u) * kWave);
      }
      if (j + u * P < fullB) {
        ccB[u] = ld_entry<NT>(cB + (j / P + u) * kWave);
        vvB[u] = ld_entry<NT>(vB + (j / P + u) * kWave);
      }
    }
    T xxA[U][P], xxB[U][P];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < P; ++q) {
        if (j + u * P + q < lenA && j + u * P < fullA) xxA[u][q] = xA[(int)ccA[u][q]];
        if (j + u * P + q < lenB && j + u * P < fullB) xxB[u][q] = xB[(int)ccB[u][q]];
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < P; ++q)
        if (j + u * P + q < lenA && j + u * P < fullA) sA += vvA[u][q] * xxA[u][q];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < P; ++q)
        if (j + u * P + q < lenB && j + u * P < fullB) sB += vvB[u][q] * xxB[u][q];
  }
  T xtA[TM], xtB[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    if (t < ntA) xtA[t] = xA[(int)ctA[t]];
    if (t < ntB) xtB[t] = xB[(int)ctB[t]];
  }
#pragma unroll
  for (int t = 0; t < TM; ++t)
    if (t < ntA) sA += vtA[t] * xtA[t];
#pragma unroll
  for (int t = 0; t < TM; ++t)
    if (t < ntB) sB += vtB[t] * xtB[t];
}

// SELL-64: unit = four slices (256 consecutive rows), wave w of the
// workgroup runs slice 4 unit + w.  No LDS and no barrier.
template <typename T, typename IT = int>
struct SellOp {
  using value_type = T;
  static constexpr int kLds = 1;
  static constexpr int P = SellChunk<T>::P;
  static constexpr int U = SellChunk<T>::U;
  int nrow, nslice;
  int cached;  // entries_cached, by slices
  const long long *soff;
  const int *slen;
  const unsigned char *rlen;
  const IT *col;
  const T *val;

  __device__ __forceinline__ long long thread_row(long long unit) const {
    return unit * kBlock + threadIdx.x;
  }
  // s + sum of a_ij x_j over the row in ascending storage order; SUB:
  // s - a_ij x_j instead; NODIAG: the diagonal entry (column == row) skipped.
  template <bool SUB = false, bool NODIAG = false>
  __device__ __forceinline__ T row_sum(long long unit, const T *x_in, T s, TileRow &tr,
                                       T *) const {
    tr.has_row = false;
    tr.row = 0;
    const long long sl = unit * kSellSlicesPerBlock + (threadIdx.x >> 6);
    if (sl >= nslice) return s;  // uniform across the wave
    const int sid = __builtin_amdgcn_readfirstlane((int)sl);
    const int lane = threadIdx.x & (kWave - 1);
    const int row = sid * kSellRows + lane;
    tr.row = row;
    tr.has_row = row < nrow;
    const int len = tr.has_row ? (int)rlen[row] : 0;
    const long long base = soff[sid];
    const int smax = slen[sid];
    // int16 columns are offsets from the slice's first row
    const T *__restrict__ x = std::is_same<IT, int>::value ? x_in : x_in + sid * kSellRows;
    const int dcol = std::is_same<IT, int>::value ? row : lane;
    return past_caches(sid, cached)
               ? sell_slice_sum<T, IT, SUB, NODIAG, false, true>(col + base, val + base, smax, len,
                                                                 lane, x, dcol, s)
               : sell_slice_sum<T, IT, SUB, NODIAG, false, false>(col + base, val + base, smax,
                                                                  len, lane, x, dcol, s);
  }
};

// Arrays that no kernel writes while a product runs: read through the
// scalar cache wherever the address is uniform.
template <typename V>
using ScalarPtr = const __attribute__((address_space(4))) V *;
template <typename V>
__device__ __forceinline__ ScalarPtr<V> scalar_ptr(const V *p) {
  return (ScalarPtr<V>)p;
}

// One lane's row of a slice in the offset form: s + sum of a_ij x_j (SUB: s -
// a_ij x_j; NODIAG: offset 0 skipped) over the K positions in order, those
// of the lane's row only.  xf(c) reads x at column c; it is called for every
// position, present or not, and must accept any c.
// Blocks of UB (or kSmall) chunks have all their loads in flight at once, with no
// branch between them (a branch would wait for the loads before it): chunks
// past the last one read the last one again and add nothing.  Two block
// sizes, so that rows of 27 entries are 7 + 7 chunks of 2 (6 of 4 in FP32)
// and rows of 9 one block of 4 (3).
template <typename T>
struct OffBlock {
  static constexpr int kBig = sizeof(T) == 8 ? 7 : 6;
  static constexpr int kSmall = sizeof(T) == 8 ? 4 : 3;
};

template <typename T, bool SUB, bool NODIAG, bool NT, int UB = OffBlock<T>::kBig, typename XF>
__device__ __forceinline__ T sell_offset_sum(const T *__restrict__ val, ScalarPtr<int> off,
                                             ScalarPtr<unsigned long long> mask, int K, int row,
                                             int lane, XF &&xf, T s) {
#pragma clang fp contract(off)
  constexpr int P = SellChunk<T>::P;
  typedef typename VecOf<T, P>::type TV;
  if (K == 0) return s;
  const int nch = K / P, full = nch * P;
  const TV *__restrict__ v = reinterpret_cast<const TV *>(val) + lane;
  // the positions past the last full chunk, loaded first (none: the last
  // position, not added)
  constexpr int TM = P > 1 ? P - 1 : 1;
  T vt[TM], xt[TM];
  unsigned long long mt[TM];
  int ot[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int j = full + t < K ? full + t : K - 1;
    const unsigned long long m = mask[j];
    ot[t] = off[j];
    mt[t] = full + t < K ? m : 0;
    vt[t] = ld_entry<NT>(val + kSellRows * j + lane);
    xt[t] = xf(row + ot[t]);
  }
  auto add = [&](T a, T x, unsigned long long m, int o) {
    if (NODIAG) m = o == 0 ? 0 : m;
    const T sn = SUB ? s - a * x : s + a * x;
    s = __builtin_amdgcn_inverse_ballot_w64(m) ? sn : s;
  };
  auto block = [&](auto chunks, int c0) {
    constexpr int NB = decltype(chunks)::value;
    TV vv[NB];
    T xx[NB][P];
    int oo[NB][P];
    unsigned long long mm[NB][P];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int c = c0 + u < nch ? c0 + u : nch - 1;
      vv[u] = ld_entry<NT>(v + c * kWave);
#pragma unroll
      for (int q = 0; q < P; ++q) {
        const unsigned long long m = mask[c * P + q];
        oo[u][q] = off[c * P + q];
        mm[u][q] = c0 + u < nch ? m : 0;
      }
    }
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int q = 0; q < P; ++q) xx[u][q] = xf(row + oo[u][q]);
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int q = 0; q < P; ++q) add(vv[u][q], xx[u][q], mm[u][q], oo[u][q]);
  };
  constexpr int US = OffBlock<T>::kSmall;
  int c = 0;
  for (; nch - c > US; c += UB) block(std::integral_constant<int, UB>(), c);
  if (c < nch) block(std::integral_constant<int, US>(), c);
#pragma unroll
  for (int t = 0; t < TM; ++t) add(vt[t], xt[t], mt[t], ot[t]);
  return s;
}

// The offset form as an operator: the rows and units of SellOp.
template <typename T>
struct SellOffOp {
  using value_type = T;
  static constexpr int kLds = 1;
  int nrow, ncol, nslice, max_off;
  int cached;  // entries_cached, by slices
  const long long *soff;
  const int *slen;
  const int *off;
  const unsigned long long *mask;
  const T *val;

  __device__ __forceinline__ long long thread_row(long long unit) const {
    return unit * kBlock + threadIdx.x;
  }
  template <bool SUB = false, bool NODIAG = false>
  __device__ __forceinline__ T row_sum(long long unit, const T *x, T s, TileRow &tr, T *) const {
    tr.has_row = false;
    tr.row = 0;
    const long long sl = unit * kSellSlicesPerBlock + (threadIdx.x >> 6);
    if (sl >= nslice) return s;  // uniform across the wave
    const int sid = __builtin_amdgcn_readfirstlane((int)sl);
    const int lane = threadIdx.x & (kWave - 1);
    const int row = sid * kSellRows + lane;
    tr.row = row;
    tr.has_row = row < nrow;
    const long long base = scalar_ptr(soff)[sid];
    const int K = scalar_ptr(slen)[sid];
    // a column outside x (positions of rows without that entry) reads 0: as
    // a byte offset it is past the range, also where it is negative (x is
    // below 2 GiB)
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T *>(x), 0, ncol * (int)sizeof(T), kRsrcWord3);
    auto sum = [&](auto nt) {
      return sell_offset_sum<T, SUB, NODIAG, decltype(nt)::value>(
          val + base, scalar_ptr(off) + base / kSellRows, scalar_ptr(mask) + base / kSellRows, K,
          row, lane, [&](int c) { return buffer_load<T>(xr, (unsigned)c * (unsigned)sizeof(T)); },
          s);
    };
    return past_caches(sid, cached) ? sum(std::true_type()) : sum(std::false_type());
  }
  // The row's sum over beta p + z in place of x (each rounded as one fused
  // multiply-add).
  __device__ __forceinline__ T direction_sum(long long unit, const T *p, const T *z,
                                             T beta) const {
    const long long sl = unit * kSellSlicesPerBlock + (threadIdx.x >> 6);
    if (sl >= nslice) return T(0);
    const int sid = __builtin_amdgcn_readfirstlane((int)sl);
    const int lane = threadIdx.x & (kWave - 1);
    const long long base = scalar_ptr(soff)[sid];
    const int K = scalar_ptr(slen)[sid];
    const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T *>(p), 0, ncol * (int)sizeof(T), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t zr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T *>(z), 0, ncol * (int)sizeof(T), kRsrcWord3);
    return sell_offset_sum<T, false, false, false>(
        val + base, scalar_ptr(off) + base / kSellRows, scalar_ptr(mask) + base / kSellRows, K,
        sid * kSellRows + lane, lane,
        [&](int c) {
          const unsigned o = (unsigned)c * (unsigned)sizeof(T);
          return __builtin_elementwise_fma(beta, buffer_load<T>(pr, o), buffer_load<T>(zr, o));
        },
        T(0));
  }
};

// once: for a product by itself, not an iteration's
inline int sell_cached(const hflmp_sell *m, size_t entry_bytes, size_t vb, bool once) {
  return once ? entries_cached_once(m->entries, entry_bytes, vb * ((size_t)m->nrow + m->ncol))
              : entries_cached(m->entries, entry_bytes, kCgVectors * vb * m->nrow);
}

template <typename T>
inline SellOffOp<T> sell_off_view(const hflmp_sell *m, bool once = false) {
  SellOffOp<T> op;
  op.nrow = m->nrow;
  op.ncol = m->ncol;
  op.nslice = m->nslice;
  op.max_off = m->max_off;
  op.cached = sell_cached(m, sizeof(T), sizeof(T), once);
  op.soff = m->soff;
  op.slen = m->slen;
  op.off = m->off;
  op.mask = m->mask;
  op.val = static_cast<const T *>(m->val);
  return op;
}

// An internal flag of sell_create: the offset form where it fits, else
// int32 columns.
constexpr int kSellOffsets = 0x100;

template <typename T, typename IT>
inline SellOp<T, IT> sell_view(const hflmp_sell *m, bool once = false) {
  SellOp<T, IT> op;
  op.nrow = m->nrow;
  op.nslice = m->nslice;
  op.soff = m->soff;
  op.slen = m->slen;
  op.rlen = m->rlen;
  op.col = static_cast<const IT *>(m->col);
  op.val = static_cast<const T *>(m->val);
  op.cached = sell_cached(m, sizeof(T) + sizeof(IT), sizeof(T), once);
  return op;
}

template <typename T>
inline CsrTileOp<T, int> csr_view(int nrow, int nnz, const int *rp, const int *ci,
                                  const T *val) {
  CsrTileOp<T, int> op;
  op.nrow = nrow;
  op.R = tile_rows(nrow, nnz, TileCap<T>::value);
  op.cached = entries_cached(nnz, sizeof(T) + sizeof(int), kCgVectors * sizeof(T) * nrow);
  op.rp = rp;
  op.ci = ci;
  op.val = val;
  return op;
}

template <typename T, typename IT>
inline int op_grid(const CsrTileOp<T, IT> &op) {
  return tile_grid(((long long)op.nrow + op.R - 1) / op.R);
}

template <typename T, typename IT>
inline int op_grid(const SellOp<T, IT> &op) {
  return sell_grid(op.nrow);
}

template <typename T>
inline int op_grid(const SellOffOp<T> &op) {
  return sell_grid(op.nrow);
}

// fn(the operator view of a SELL-64 matrix's form)
template <typename T, typename Fn>
inline auto sell_dispatch(const hflmp_sell *m, Fn &&fn) {
  if (m->off_form) return fn(sell_off_view<T>(m));
  if (m->col_bytes == 2) return fn(sell_view<T, short>(m));
  return fn(sell_view<T, int>(m));
}
