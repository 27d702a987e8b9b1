// Jacobi-PCG of a small SELL-64 system in one workgroup.
//
// A system of a few thousand rows spends its iteration in launches: the
// three kernels of hflmp_cg3.hpp take 3.3 + 3.4 + 3.0 us and the gaps between
// them 3 us on 1,089 rows, whatever the rows cost (12.9 us an iteration).
// Here one workgroup runs the iterations with p in LDS, x, r and D^-1 in
// registers and the matrix read from LDS where it fits, else from L2; the
// grid-wide sums become three barriers.  2D Q1 32^2 with log-normal
// diffusivity to 1e-8: 1.70 -> 0.33 ms, 3.3 us an iteration (2.8 on 289
// rows, 7.6 on 3,969), which is the latency of one chain through the
// products, three wave sums, two quotients and a root.
//
// The iterates are the three-launch form's, bit for bit, so that a system
// gives the same result whichever form runs it: every sum is formed from
// the same terms in the same order (per 256-row unit as its workgroups do,
// the unit's partials in the launch's workgroup order, the update's
// partials by its workgroups of 256 threads and four elements each), and
// every product and sum is rounded as there.
#pragma once

#include <algorithm>

#include "hflmp_cg3.hpp"

namespace {

constexpr int kSmallRows = 8192;           // two sets of 4 elements for 1024 threads
constexpr int kSmallOffRows = 4096;        // one set
constexpr size_t kSmallLds = 152 * 1024;
// Entries' bytes beyond which the L2 of one CU is slower than three launches
// (64 B a clock: about 150 GB/s).
constexpr size_t kSmallBytes = 768 * 1024;
constexpr int kSmallIters = 512;           // iterations of one launch, at most

// Bytes of a stored column of an operator over SELL-64.
template <typename Op>
struct ColBytes;
template <typename T, typename IT>
struct ColBytes<SellOp<T, IT>> {
  static constexpr size_t value = sizeof(IT);
};
template <typename T>
struct ColBytes<SellOffOp<T>> {
  static constexpr size_t value = 0;
};

struct CgSmallArgs {
  int vgrid, g2;  // units and update workgroups of the three-launch form
  int entries;    // stored entries of the operator
};

// LDS: p (with its margins), Ap | wave sums of p.Ap (one a slice) | wave sums of r.r and r.z
// (four an update workgroup) | MLDS: values | slices' first entries and
// lengths | verdict | MLDS: columns | row lengths.
constexpr int kSmallSlices = kSmallRows / kSellRows;
constexpr int kSmallSums = kSmallSlices + 2 * 4 * (kSmallRows / (4 * kBlock));
// Values before and after p that the offset form may read (and drop) for
// rows without an entry.
template <typename T, typename IT>
__host__ __device__ inline int small_margin(const SellOp<T, IT> &) {
  return 0;
}
template <typename T>
__host__ __device__ inline int small_margin(const SellOffOp<T> &op) {
  return (op.max_off + 3) / 4 * 4;  // keeps the LDS areas 16-byte aligned
}
// Rows up to which one workgroup is the faster form.  The offset form's two
// launches (hflmp_cg3.hpp) overtake two sets of elements (2D Q1 FP64, us an
// iteration, here and there: 4,761 rows 10.7 and 11.3, 5,929 rows 13.0 and
// 11.3, 7,225 rows 15.1 and 11.5), the three launches of the column form do
// not (5,929 rows 11.4 and 15.2, 7,921 rows 15.1 and 15.4).
template <typename T, typename IT>
inline int small_rows(const SellOp<T, IT> &) {
  return kSmallRows;
}
template <typename T>
inline int small_rows(const SellOffOp<T> &) {
  return kSmallOffRows;
}
template <typename Op>
inline size_t small_lds_bytes(const Op &op, long long entries, bool mlds) {
  const size_t vb = sizeof(typename Op::value_type);
  const size_t nr = (size_t)op.nslice * kSellRows;
  return (2 * nr + 2 * (size_t)small_margin(op) + kSmallSums) * vb + 8 * (size_t)kSmallSlices +
         nr + 16 + (mlds ? (size_t)entries * (vb + ColBytes<Op>::value) : 0);
}

// The product of one slice (one wave, its row's sum) from the small kernel's
// LDS: the slice's entries start at base of val / col (LDS copies or the
// operator's arrays), m the longest row or the offsets.
template <typename T, typename IT>
__device__ __forceinline__ T small_slice(const SellOp<T, IT> &, const T *val, const IT *col,
                                         int base, int m, int len, int sl, int, int lane,
                                         const T *ps) {
  constexpr int U = sizeof(T) == 8 ? 4 : 3;  // fits the 128 registers of 1024 threads
  const T *x = std::is_same<IT, int>::value ? ps : ps + sl * kSellRows;
  return sell_slice_sum<T, IT, false, false, true, false, U, true>(col + base, val + base, m, len,
                                                                   lane, x, 0, T(0));
}
template <typename T>
__device__ __forceinline__ T small_slice(const SellOffOp<T> &op, const T *val, const char *,
                                         int base, int m, int, int, int row, int lane,
                                         const T *ps) {
  return sell_offset_sum<T, false, false, false, OffBlock<T>::kSmall>(
      val + base, scalar_ptr(op.off) + base / kSellRows, scalar_ptr(op.mask) + base / kSellRows,
      m, row, lane, [&](int c) { return ps[c]; }, T(0));
}
template <typename T, typename IT>
__device__ __forceinline__ const IT *small_cols(const SellOp<T, IT> &op) {
  return op.col;
}
template <typename T>
__device__ __forceinline__ const char *small_cols(const SellOffOp<T> &) {
  return nullptr;
}
template <typename T, typename IT>
__device__ __forceinline__ int small_len(const SellOp<T, IT> &op, unsigned i) {
  return op.rlen[i];
}
template <typename T>
__device__ __forceinline__ int small_len(const SellOffOp<T> &, unsigned) {
  return 0;
}

// The update's elements are its workgroups': vthread v (workgroup v / 256,
// thread v % 256, v = j 1024 + thread of this workgroup) has elements v + q
// g2 256, q < 4, in registers.  The product walks the slices by wave and
// passes Ap through LDS.
template <typename Op, int J, bool MLDS, typename T = typename Op::value_type>
__global__ void __launch_bounds__(kFinalBlock)
    cg_small_kernel(Op op, CgSmallArgs a, const T *__restrict__ invd,
                    T *__restrict__ xg, T *__restrict__ rg, T *__restrict__ pg,
                    CgState<T> *st) {
#pragma clang fp contract(off)
  constexpr bool COLS = ColBytes<Op>::value > 0;
  using IT = std::remove_cv_t<std::remove_pointer_t<decltype(small_cols(op))>>;
  extern __shared__ __align__(16) unsigned char small_lds[];
  if (st->status != kIterate) return;
  const unsigned n = op.nrow, nr = op.nslice * kSellRows;
  const int margin = small_margin(op);
  T *ps = reinterpret_cast<T *>(small_lds) + margin;
  T *aps = ps + nr + margin;
  T *sumA = aps + nr;
  T *sumB = sumA + kSmallSlices;
  T *vals = sumA + kSmallSums;
  int *soff = reinterpret_cast<int *>(vals + (MLDS ? a.entries : 0));
  int *slen = soff + kSmallSlices;
  int *verdict = slen + kSmallSlices;  // the stopping test's, for waves without elements
  IT *cols = reinterpret_cast<IT *>(verdict + 4);
  unsigned char *rlen =
      reinterpret_cast<unsigned char *>(cols + (MLDS && COLS ? a.entries : 0));
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(t / kWave);
  const int nwave = blockDim.x / kWave;
  const unsigned stride = a.g2 * kBlock;
  // Waves beyond the update's threads only take slices of the product: the
  // scalars, which every updating wave forms for itself, would keep the
  // vector units from the others.
  const bool mine = (unsigned)wid * kWave < stride;
  if (MLDS) {
    for (int e = t; e < a.entries; e += blockDim.x) {
      vals[e] = op.val[e];
      if constexpr (COLS) cols[e] = op.col[e];
    }
  }
  for (unsigned i = t; i < nr; i += blockDim.x) rlen[i] = i < n ? small_len(op, i) : 0;
  if (t < op.nslice) {
    soff[t] = (int)op.soff[t];
    slen[t] = op.slen[t];
  }
  T x[J][4], r[J][4], d[J][4];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned v = j * kFinalBlock + t, i = v + q * stride;
      const bool ok = v < stride && i < n;
      x[j][q] = ok ? xg[i] : T(0);
      r[j][q] = ok ? rg[i] : T(0);
      d[j][q] = ok ? invd[i] : T(0);
      if (ok) ps[i] = pg[i];
    }
  T rz = st->rz;
  const double res0 = (double)st->res0, atol = st->atol, rtol = st->rtol, dtol = st->dtol;
  const int maxit = st->maxit;
  int iter = st->iter, status = kIterate;
  T pAp = 0, alpha = 0, rr = 0, res = st->res, beta = st->beta;
  __syncthreads();
  // where the wave's next slice lies, one slice ahead
  const int sl0 = wid < op.nslice ? wid : 0;
  int nlen = rlen[sl0 * kSellRows + lane], nbase = soff[sl0], nmax = slen[sl0];
  for (int k = 0; k < kSmallIters; ++k) {
    // Ap = A p and the waves' sums of p.Ap
#pragma unroll 1
    for (int sl = wid; sl < op.nslice; sl += nwave) {
      const unsigned row = sl * kSellRows + lane;
      const int len = nlen;
      const int base = __builtin_amdgcn_readfirstlane(nbase);
      const int smax = __builtin_amdgcn_readfirstlane(nmax);
      const int next = sl + nwave < op.nslice ? sl + nwave : wid;
      nlen = rlen[next * kSellRows + lane];
      nbase = soff[next];
      nmax = slen[next];
      const T s = MLDS ? small_slice(op, vals, cols, base, smax, len, sl, row, lane, ps)
                       : small_slice(op, op.val, small_cols(op), base, smax, len, sl, row, lane,
                                     ps);
      T acc = T(0);
      if (row < n) {
        aps[row] = s;
        acc = __builtin_elementwise_fma(s, ps[row], T(0));
      }
      acc = wave_sum(acc);
      if (lane == 0) sumA[sl] = acc;
    }
    __syncthreads();
    // read while alpha is formed, where there are registers for it
    constexpr bool EARLY = J == 1 && !COLS;
    T p[J][4], ap[J][4];
    if (mine) {
      if (EARLY)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const unsigned i = t + q * stride, in = i < nr ? i : 0;
          p[0][q] = ps[in];
          ap[0][q] = aps[in];
        }
      // partial of workgroup b: unit xcd_tile(b)'s four waves in order
      const int unit = (int)xcd_tile(lane, a.vgrid);
      T part = T(0);
      if (lane < a.vgrid) {
#pragma unroll
        for (int w = 0; w < 4; ++w)
          part += unit * 4 + w < op.nslice ? sumA[unit * 4 + w] : T(0);
      }
      pAp = T(0) + wave_sum_first(part, a.vgrid);
      if (pAp == T(0) || !(pAp == pAp)) status = kBreakdown;
    }
    if (mine && status == kIterate) {
      alpha = rz / pAp;
      const T malpha = -alpha;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const unsigned v = j * kFinalBlock + t;
        if (__builtin_amdgcn_readfirstlane(v) >= stride) continue;
        T arr = 0, arz = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const unsigned i = v + q * stride;
          if (i < n) {
            if (!EARLY) p[j][q] = ps[i], ap[j][q] = aps[i];
            x[j][q] = __builtin_elementwise_fma(alpha, p[j][q], x[j][q]);
            r[j][q] = __builtin_elementwise_fma(malpha, ap[j][q], r[j][q]);
            const T z = r[j][q] * d[j][q];
            arr = __builtin_elementwise_fma(r[j][q], r[j][q], arr);
            arz = __builtin_elementwise_fma(r[j][q], z, arz);
          }
        }
        arr = wave_sum(arr);
        arz = wave_sum(arz);
        if (lane == 0) {
          sumB[2 * (v / kWave)] = arr;
          sumB[2 * (v / kWave) + 1] = arz;
        }
      }
    }
    __syncthreads();
    if (mine && status == kIterate) {
      T prr = T(0), prz = T(0);
      if (lane < a.g2) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          prr += sumB[2 * (4 * lane + w)];
          prz += sumB[2 * (4 * lane + w) + 1];
        }
      }
      rr = T(0) + wave_sum_first(prr, a.g2);
      const T rzn = T(0) + wave_sum_first(prz, a.g2);
      const T ratio = rzn / rz;  // the quotient and the root need not wait for each other
      ++iter;
      res = sqrt(rr);
      status = check_state(iter, (double)res, res0, maxit, atol, rtol, dtol);
      if (status == kIterate) {
        beta = ratio;
        rz = rzn;
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const unsigned v = j * kFinalBlock + t, i = v + q * stride;
            if (v < stride && i < n) {
              const T z = r[j][q] * d[j][q];
              ps[i] = __builtin_elementwise_fma(beta, EARLY ? p[j][q] : ps[i], z);
            }
          }
      }
    }
    if (t == 0) *verdict = status;
    __syncthreads();
    if (!mine) status = *verdict;
    if (status != kIterate) break;
  }
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned v = j * kFinalBlock + t, i = v + q * stride;
      if (v < stride && i < n) {
        xg[i] = x[j][q];
        rg[i] = r[j][q];
        pg[i] = ps[i];
      }
    }
  if (t == 0) {
    st->rz = rz;
    st->pAp = pAp;
    st->alpha = alpha;
    st->beta = beta;
    st->rr = rr;
    st->res = res;
    st->iter = iter;
    st->status = status;
  }
}

// Whether the one-workgroup form runs this system in place of launches with
// the grids G over vgrid units, and how.  The unit partials are summed by
// one wave (vgrid <= 64) in the order of launches of one unit a workgroup
// (G.g1 == vgrid).
template <typename Op>
bool small_fits(const Op &op, long long entries, int vgrid, const Cg3Grids &G) {
  return op.nrow <= small_rows(op) && vgrid <= kWave && G.g1 == vgrid && G.g2 * 4 * kBlock >= op.nrow &&
         G.g2 <= kSmallRows / (4 * kBlock) &&
         (size_t)entries * (sizeof(typename Op::value_type) + ColBytes<Op>::value) <= kSmallBytes &&
         small_lds_bytes(op, entries, false) <= kSmallLds;
}

template <typename Op, typename T = typename Op::value_type>
void small_launch(hipStream_t s, const Op &op, long long entries, int vgrid, const Cg3Grids &G,
                  const T *invd, T *x, T *r, T *p, CgState<T> *st) {
  const CgSmallArgs a{vgrid, G.g2, (int)entries};
  const bool mlds = small_lds_bytes(op, entries, true) <= kSmallLds;
  const size_t lds = small_lds_bytes(op, entries, mlds);
  // a wave a slice, and those of the update's threads (all when it has two sets)
  const int waves = std::max(std::min(op.nslice, kFinalBlock / kWave),
                             std::min(4 * G.g2, kFinalBlock / kWave));
  const int threads = G.g2 <= 4 ? waves * kWave : kFinalBlock;
  auto go = [&](auto kern) { kern<<<1, threads, lds, s>>>(op, a, invd, x, r, p, st); };
  if (G.g2 <= 4)
    mlds ? go(cg_small_kernel<Op, 1, true>) : go(cg_small_kernel<Op, 1, false>);
  else if constexpr (ColBytes<Op>::value > 0)
    mlds ? go(cg_small_kernel<Op, 2, true>) : go(cg_small_kernel<Op, 2, false>);
}

}  // namespace
