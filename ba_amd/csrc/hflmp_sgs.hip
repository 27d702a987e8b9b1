// Symmetric Gauss-Seidel in the sequential row order of the CPU path:
// z = M^-1 r, M = (D + L) D^-1 (D + U), as CPU_CSR_lMatrix::Psgauss_seidel
// (lmatrix_csr_cpu.cc:495-565) computes it, and its block form
// BlocksPsgauss_seidel (lmatrix_csr_cpu.cc:568-641; the CUDA platform's
// GPUscalar_CSR_lMatrix::BlocksPsgauss_seidel, cuda/GPUscalar_csr_lmatrix.cu:
// 314-363, kernel_BlockPsgauss_seidel, cuda/cuda_spmv_kernel_csr_scalar.h:
// 65-143): num_blocks row ranges of nrow / num_blocks rows (the last takes
// the rest), each swept on its own over the entries whose column lies in
// the range.
//
// Per row the operations and their order are the reference's:
//   forward (rows ascending)   t = r_i; over the row in storage order up to
//                              the first diagonal entry: t -= z_c a_ij for
//                              c < i; z_i = t / a_ii
//   D                          z_i *= a_ii (first diagonal entry)
//   backward (rows descending) over the whole row: t -= z_c a_ij for c > i;
//                              z_i = t / a_ii (last diagonal entry)
// The reference runs the sweeps one row at a time (the CUDA kernel one
// thread per block).  Here the rows are grouped by dependency level: a
// row's forward level is one more than the highest level among the rows it
// reads, so every row of a level reads only values that earlier levels have
// finished.  Each level is one launch over its rows, or, for runs of levels
// of at most kSmallLevel rows, one workgroup that walks the levels with a
// barrier between them.  The values every row reads are the ones the
// sequential sweep reads, so z is bit-identical to it.  The D scaling is
// applied by each row's backward step before its first subtraction, which
// is where the sequential sweep's separate D pass leaves the value (no row
// reads another row's scaled value before that row's backward step).
#include <algorithm>
#include <vector>

#include "hflmp_internal.hpp"

namespace {

constexpr int kSmallLevel = kFinalBlock;  // rows of a level one workgroup takes

// Row range [lo, hi) of row i's block (BlockPsgauss_seidel's start_i/end_i).
struct Blocks {
  int nrow, nb, step;
  __host__ __device__ __forceinline__ void range(int i, int &lo, int &hi) const {
    if (step == 0) {  // every block but the last is empty; the last is all rows
      lo = 0;
      hi = nrow;
      return;
    }
    int b = i / step;
    if (b > nb - 1) b = nb - 1;
    lo = b * step;
    hi = b == nb - 1 ? nrow : lo + step;
  }
};

template <typename T>
struct SgsArgs {
  const int *rp, *ci;
  const T *val;
  const T *r;
  T *z;
  Blocks blk;
};

template <typename T>
__device__ __forceinline__ void forward_row(const SgsArgs<T> &a, int i) {
#pragma clang fp contract(off)
  int lo, hi;
  a.blk.range(i, lo, hi);
  T t = a.r[i];
  int dj = -1;
  for (int j = a.rp[i]; j < a.rp[i + 1]; ++j) {
    const int c = a.ci[j];
    if (c >= lo && c < hi) {
      if (c < i) t -= a.z[c] * a.val[j];
      if (c == i) {
        dj = j;
        break;
      }
    }
  }
  // the build refused rows without a diagonal entry, so dj >= 0
  a.z[i] = t / a.val[dj];
}

template <typename T>
__device__ __forceinline__ void backward_row(const SgsArgs<T> &a, int i) {
#pragma clang fp contract(off)
  int lo, hi;
  a.blk.range(i, lo, hi);
  const int j0 = a.rp[i], j1 = a.rp[i + 1];
  int dfirst = -1;
  for (int j = j0; j < j1; ++j)
    if (a.ci[j] == i) {
      dfirst = j;
      break;
    }
  T t = a.z[i] * a.val[dfirst];  // the D pass
  int dlast = dfirst;
  for (int j = j0; j < j1; ++j) {
    const int c = a.ci[j];
    if (c >= lo && c < hi) {
      if (c == i) dlast = j;
      if (c > i) t -= a.z[c] * a.val[j];
    }
  }
  a.z[i] = t / a.val[dlast];
}

// One level: rows perm[k0 .. k1), one thread each.
template <typename T, bool FWD>
__global__ void __launch_bounds__(kBlock)
    sgs_level_kernel(SgsArgs<T> a, const int *__restrict__ perm, int k0, int k1) {
  const int k = k0 + blockIdx.x * kBlock + threadIdx.x;
  if (k >= k1) return;
  const int i = perm[k];
  if (FWD)
    forward_row(a, i);
  else
    backward_row(a, i);
}

// Levels l0 .. l1 - 1 (each at most kSmallLevel rows) in one workgroup; the
// barrier between levels orders each level's stores before the next
// level's loads (all waves share the CU's caches).
template <typename T, bool FWD>
__global__ void __launch_bounds__(kFinalBlock)
    sgs_levels_kernel(SgsArgs<T> a, const int *__restrict__ perm, const int *__restrict__ loff,
                      int l0, int l1) {
  for (int l = l0; l < l1; ++l) {
    const int k = loff[l] + threadIdx.x;
    if (k < loff[l + 1]) {
      const int i = perm[k];
      if (FWD)
        forward_row(a, i);
      else
        backward_row(a, i);
    }
    __syncthreads();
  }
}

// ---- sweeps of narrow levels, from a level-ordered copy of the pattern ----
// Where every level of a sweep has at most kPackRows rows, the whole sweep is
// one workgroup and its time is the latency of its levels one after another
// (2D Q1 96^2: 289 levels of at most 49 rows).  Walking the CSR rows, a level
// costs the chain level offset -> row -> row_ptr -> column -> value, z: 2.0 us
// (forward) to 2.9 us (backward) a level there.  So the pattern is laid out
// in level order when the schedule is made (slot l W + t is row t of level
// l, its entries E apart), which makes every address but z's known in
// advance: the descriptions of level l + 2 D and the values, right-hand side
// and diagonals of level l + D are loaded while level l is computed.  The
// values are still read from the caller's array at each apply, through the
// entries' positions in it.  z is kept in LDS where it fits, so that a level
// waits for LDS reads, its ordered sum, one division and a barrier only.
// (CG with this preconditioner through the solver templates, 2D Q1 96^2,
// 130 iterations: 194.1 -> 33.3 ms.)
constexpr int kPackRows = 512;
constexpr int kPackMaxE = 16;             // entries a row takes part with in a sweep
constexpr size_t kPackLds = 144 * 1024;   // z in LDS up to this size

// Entries per slot and prefetch distance for rows of at most e entries:
// about the same registers for each (fewer than 256 at 512 threads).
inline int pack_width(int e) { return e <= 4 ? 4 : e <= 8 ? 8 : 16; }

struct PackView {
  int nlev, W;
  const int4 *rows;  // {row, entries, first diagonal position, last}; row < 0: no row
  const int2 *ent;   // {position in val, column} at (l E + e) W + t
};

template <typename T, bool FWD, int E, int D, bool ZLDS>
__global__ void __launch_bounds__(kPackRows)
    sgs_packed_kernel(PackView pk, int nrow, const T *__restrict__ val, const T *r, T *z) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) unsigned char sgs_lds[];
  T *zs = reinterpret_cast<T *>(sgs_lds);
  const int t = threadIdx.x, W = pk.W;
  if (ZLDS && !FWD) {
    for (int i = t; i < nrow; i += W) zs[i] = z[i];
    __syncthreads();
  }
  // level l: its description in slot l mod 2 D, its values in slot l mod D
  int4 di[2 * D];
  int2 de[2 * D][E];
  T v[D][E], rhs[D], dg0[D], dg1[D];
  auto load_desc = [&](int u, int l) {
    di[u] = pk.rows[(size_t)l * W + t];
#pragma unroll
    for (int e = 0; e < E; ++e) de[u][e] = pk.ent[((size_t)l * E + e) * W + t];
  };
  auto load_vals = [&](int u, int w) {
#pragma unroll
    for (int e = 0; e < E; ++e) v[w][e] = val[de[u][e].x];
    dg1[w] = val[di[u].w];
    if (FWD)
      rhs[w] = r[di[u].x < 0 ? 0 : di[u].x];
    else
      dg0[w] = val[di[u].z];
  };
  // (4 D levels of empty slots follow the last one)
  // the order of the loop's loads, so that its waits fit the first pass too
#pragma unroll
  for (int u = 0; u < D; ++u) load_desc(u, u);
#pragma unroll
  for (int u = 0; u < D; ++u) {
    load_vals(u, u);
    load_desc(D + u, D + u);
  }
  for (int l0 = 0; l0 < pk.nlev; l0 += 2 * D) {
#pragma unroll
    for (int u = 0; u < 2 * D; ++u) {
      const int w = u % D;
      // empty slots and the entries past a row's last read row 0 and val[0]
      // and are dropped
      const int i = di[u].x, len = di[u].y;
      const T *zz = ZLDS ? zs : z;
      T x[E];
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = zz[de[u][e].y];
      T s = FWD ? rhs[w] : zz[i < 0 ? 0 : i] * dg0[w];  // backward: the D pass
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const T sn = s - x[e] * v[w][e];
        s = e < len ? sn : s;
      }
      s = s / dg1[w];
      if (i >= 0) {
        if (ZLDS) zs[i] = s;
        z[i] = s;
      }
      load_vals((u + D) % (2 * D), w);
      load_desc(u, l0 + u + 2 * D);
      __syncthreads();
    }
  }
}

// The level-ordered copy: a thread a slot (lv levels of W, those past the
// last one empty), slot l W + t from row t of level l: the entries that the
// sweep subtracts, in storage order, and the first and last diagonal positions.
template <bool FWD>
__global__ void __launch_bounds__(kBlock)
    sgs_pack_kernel(Blocks blk, const int *__restrict__ rp, const int *__restrict__ ci,
                    const int *__restrict__ perm, const int *__restrict__ loff, int nlev,
                    long long lv, int W, int E, int4 *__restrict__ rows, int2 *__restrict__ ent) {
  for (long long k = (long long)blockIdx.x * kBlock + threadIdx.x; k < lv * W;
       k += (long long)gridDim.x * kBlock) {
    const long long l = k / W;
    const int t = (int)(k - l * W);
    int2 *mine = ent + l * E * W + t;
    int4 d = make_int4(-1, 0, 0, 0);
    if (l < nlev && t < loff[l + 1] - loff[l]) {
      const int i = perm[loff[l] + t];
      int lo, hi;
      blk.range(i, lo, hi);
      d = make_int4(i, 0, -1, -1);
      for (int j = rp[i]; j < rp[i + 1]; ++j) {
        const int c = ci[j];
        if (c == i) {
          if (d.z < 0) d.z = j;
          d.w = j;
          if (FWD) break;
        } else if (FWD ? (c >= lo && c < i) : (c > i && c < hi)) {
          mine[(long long)d.y++ * W] = make_int2(j, c);
        }
      }
    }
    for (int e = d.y; e < E; ++e) mine[(long long)e * W] = make_int2(0, 0);
    rows[k] = d;
  }
}

// A sweep's launches: a single level (rows k0..k1) or a run of small levels.
struct Segment {
  bool small;
  int a, b;  // small: levels [a, b); else rows [a, b) of the permutation
};

struct Sweep {
  int levels = 0;
  int *perm = nullptr;  // rows sorted by level (DEVICE)
  int *loff = nullptr;  // level offsets into perm, levels + 1 (behind perm)
  std::vector<Segment> seg;
  // level-ordered copy of the pattern (packW = 0: none, the segments run)
  int packW = 0, packE = 0;
  int4 *prow = nullptr;
  int2 *pent = nullptr;
  int launches() const { return packW ? 1 : (int)seg.size(); }
};

}  // namespace

struct hflmp_sgs {
  int device = 0;
  int nrow = 0, nnz = 0, value_bytes = 0;
  Blocks blk{};
  const int *rp = nullptr, *ci = nullptr;
  const void *val = nullptr;
  Sweep fwd, bwd;
};

namespace {

void sweep_free(Sweep &s) {
  (void)hipFree(s.perm);
  (void)hipFree(s.prow);
  s.perm = s.loff = nullptr;
  s.prow = nullptr;
  s.pent = nullptr;
  s.packW = 0;
}

void sgs_free(hflmp_sgs *m) {
  if (!m) return;
  sweep_free(m->fwd);
  sweep_free(m->bwd);
  delete m;
}

// Bytes that a sweep's copy may take: what the pattern and FP64 values take
// four times over, or 16 MB where that is more, and at most 1 GB.  (The copy of 2D Q1 96^2 takes 0.9 of the CSR arrays, of 3D Q1
// 32^3 as well; eight slots a row with 16 entries each are 1.2 KB a row,
// where a row may have few entries.)
inline size_t pack_limit(size_t nnz, size_t n) {
  return std::min<size_t>(std::max<size_t>(4 * (12 * nnz + 4 * n), 16 << 20), 1 << 30);
}

// The pattern on the device, for the build: the caller's arrays where it was
// downloaded from them, else a copy of the host's on first use (the caller's
// device arrays need not hold it yet).
struct DevicePattern {
  int nrow, nnz;
  const int *rp, *ci;      // the caller's, or null
  const int *h_rp, *h_ci;
  int *copy = nullptr;
  ~DevicePattern() { (void)hipFree(copy); }
  int get(hflmp_ctx *ctx) {
    if (rp) return HFLMP_OK;
    if (hipMalloc(&copy, sizeof(int) * ((size_t)nrow + 1 + nnz)) != hipSuccess) {
      (void)hipGetLastError();
      return HFLMP_ENOMEM;
    }
    HFLMP_HIP_CHECK(ctx, hipMemcpy(copy, h_rp, sizeof(int) * ((size_t)nrow + 1),
                                   hipMemcpyHostToDevice));
    HFLMP_HIP_CHECK(ctx, hipMemcpy(copy + nrow + 1, h_ci, sizeof(int) * (size_t)nnz,
                                   hipMemcpyHostToDevice));
    rp = copy;
    ci = copy + nrow + 1;
    return HFLMP_OK;
  }
};

// The level-ordered copy (see sgs_packed_kernel) where it fits: levels of at
// most kPackRows rows, at most kPackMaxE entries a row (most), no more than
// about eight slots a row (levels of very uneven width would waste the rest),
// and within pack_limit.  off: the level offsets; perm and loff are on the
// device already.  Without room for it the segments run.
template <bool FWD>
int build_packed(hflmp_ctx *ctx, const Blocks &blk, DevicePattern &pat,
                 const std::vector<int> &off, int most, Sweep &s) {
  const int n = blk.nrow, nlev = s.levels;
  int widest = 0;
  for (int l = 0; l < nlev; ++l) widest = std::max(widest, off[l + 1] - off[l]);
  const int W = (widest + kWave - 1) / kWave * kWave;
  if (W > kPackRows || (long long)nlev * W > 8LL * n + 65536 || most > kPackMaxE) return HFLMP_OK;
  const int E = pack_width(most);
  const int D = kPackMaxE / E;
  const size_t lv = (size_t)nlev + 4 * (size_t)D;  // empty levels at the end
  const size_t row_bytes = lv * W * sizeof(int4), ent_bytes = lv * W * E * sizeof(int2);
  if (row_bytes + ent_bytes > pack_limit(pat.nnz, n)) return HFLMP_OK;
  const int rc = pat.get(ctx);
  if (rc) return rc == HFLMP_ENOMEM ? HFLMP_OK : rc;
  char *copy = nullptr;
  if (hipMalloc(reinterpret_cast<void **>(&copy), row_bytes + ent_bytes) != hipSuccess) {
    (void)hipGetLastError();
    return HFLMP_OK;
  }
  s.prow = reinterpret_cast<int4 *>(copy);
  s.pent = reinterpret_cast<int2 *>(copy + row_bytes);
  sgs_pack_kernel<FWD><<<grid_for((long long)(lv * W), 1), kBlock, 0, ctx->stream>>>(
      blk, pat.rp, pat.ci, s.perm, s.loff, nlev, (long long)lv, W, E, s.prow, s.pent);
  HFLMP_LAUNCH_CHECK(ctx);
  HFLMP_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  (void)hipFree(s.perm);
  s.perm = s.loff = nullptr;
  s.packW = W;
  s.packE = E;
  return HFLMP_OK;
}

// Counting sort of the rows by level, its upload, and the copy or the launch
// segments.  most: entries that a row takes part with.
template <bool FWD>
int build_sweep(hflmp_ctx *ctx, const std::vector<int> &level, int nlev, const Blocks &blk,
                DevicePattern &pat, int most, Sweep &s) {
  const int n = (int)level.size();
  // perm, then off
  std::vector<int> host((size_t)n + nlev + 1), off((size_t)nlev + 1, 0);
  for (int i = 0; i < n; ++i) ++off[level[i] + 1];
  for (int l = 0; l < nlev; ++l) off[l + 1] += off[l];
  std::copy(off.begin(), off.end(), host.begin() + n);
  std::vector<int> fill(off.begin(), off.end() - 1);
  for (int i = 0; i < n; ++i) host[fill[level[i]]++] = i;  // ascending rows within a level
  s.levels = nlev;
  s.seg.clear();
  if (hipMalloc(&s.perm, sizeof(int) * host.size()) != hipSuccess)
    return set_error(ctx, HFLMP_ENOMEM, "sgs_create: out of device memory");
  s.loff = s.perm + n;
  HFLMP_HIP_CHECK(ctx, hipMemcpy(s.perm, host.data(), sizeof(int) * host.size(),
                                 hipMemcpyHostToDevice));
  const int rc = build_packed<FWD>(ctx, blk, pat, off, most, s);
  if (rc || s.packW) return rc;
  for (int l = 0; l < nlev;) {
    if (off[l + 1] - off[l] > kSmallLevel) {
      s.seg.push_back({false, off[l], off[l + 1]});
      ++l;
      continue;
    }
    int e = l;
    while (e < nlev && off[e + 1] - off[e] <= kSmallLevel) ++e;
    s.seg.push_back({true, l, e});
    l = e;
  }
  return HFLMP_OK;
}

int sgs_create(hflmp_ctx *ctx, int nrow, int nnz, const int *rp, const int *ci,
               const void *val, int value_bytes, const int *h_rp, const int *h_ci,
               int num_blocks, hflmp_sgs **out) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, out != nullptr, "sgs_create: null output handle");
  *out = nullptr;
  HFLMP_REQUIRE(ctx, nrow > 0 && nnz > 0 && num_blocks >= 1,
                "sgs_create: need nrow > 0, nnz > 0, num_blocks >= 1");
  HFLMP_REQUIRE(ctx, rp && ci && val, "sgs_create: null device array");
  HFLMP_REQUIRE(ctx, (h_rp == nullptr) == (h_ci == nullptr),
                "sgs_create: give both host pattern arrays or neither");
  std::vector<int> hrp, hci;
  if (!h_rp) {
    hrp.resize((size_t)nrow + 1);
    hci.resize((size_t)nnz);
    HFLMP_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    HFLMP_HIP_CHECK(ctx, hipMemcpy(hrp.data(), rp, sizeof(int) * ((size_t)nrow + 1),
                                   hipMemcpyDeviceToHost));
    HFLMP_HIP_CHECK(ctx, hipMemcpy(hci.data(), ci, sizeof(int) * (size_t)nnz,
                                   hipMemcpyDeviceToHost));
    h_rp = hrp.data();
    h_ci = hci.data();
  }
  HFLMP_REQUIRE(ctx, h_rp[0] == 0 && h_rp[nrow] == nnz, "sgs_create: row_ptr does not span nnz");
  for (int i = 0; i < nrow; ++i) {
    HFLMP_REQUIRE(ctx, h_rp[i + 1] >= h_rp[i], "sgs_create: row_ptr decreases at row %d", i);
    for (int j = h_rp[i]; j < h_rp[i + 1]; ++j)
      HFLMP_REQUIRE(ctx, h_ci[j] >= 0 && h_ci[j] < nrow,
                    "sgs_create: column %d out of range in row %d", h_ci[j], i);
  }
  Blocks blk{nrow, num_blocks, nrow / num_blocks};
  // forward levels (rows ascending): entries up to the first diagonal one
  std::vector<int> lev(nrow);
  int nf = 0, most_f = 0, most_b = 0;  // levels, and the entries of a row
  for (int i = 0; i < nrow; ++i) {
    int lo, hi;
    blk.range(i, lo, hi);
    int l = 0, cnt = 0;
    bool diag = false;
    for (int j = h_rp[i]; j < h_rp[i + 1]; ++j) {
      const int c = h_ci[j];
      if (c >= lo && c < hi) {
        if (c < i) {
          l = std::max(l, lev[c] + 1);
          ++cnt;
        }
        if (c == i) {
          diag = true;
          break;
        }
      }
    }
    if (!diag)
      return set_error(ctx, HFLMP_EFORMAT, "sgs_create: row %d has no diagonal entry", i);
    lev[i] = l;
    nf = std::max(nf, l + 1);
    most_f = std::max(most_f, cnt);
  }
  auto *m = new hflmp_sgs();
  m->device = ctx->device;
  m->nrow = nrow;
  m->nnz = nnz;
  m->value_bytes = value_bytes;
  m->blk = blk;
  m->rp = rp;
  m->ci = ci;
  m->val = val;
  DevicePattern pat{nrow, nnz, hrp.empty() ? nullptr : rp, hrp.empty() ? nullptr : ci, h_rp, h_ci};
  int rc = build_sweep<true>(ctx, lev, nf, blk, pat, most_f, m->fwd);
  if (rc) {
    sgs_free(m);
    return rc;
  }
  // backward levels (rows descending): every upper entry of the range
  int nbk = 0;
  for (int i = nrow - 1; i >= 0; --i) {
    int lo, hi;
    blk.range(i, lo, hi);
    int l = 0, cnt = 0;
    for (int j = h_rp[i]; j < h_rp[i + 1]; ++j) {
      const int c = h_ci[j];
      if (c > i && c < hi) {
        l = std::max(l, lev[c] + 1);
        ++cnt;
      }
    }
    most_b = std::max(most_b, cnt);
    lev[i] = l;  // rows above i already hold their backward levels
    nbk = std::max(nbk, l + 1);
  }
  rc = build_sweep<false>(ctx, lev, nbk, blk, pat, most_b, m->bwd);
  if (rc) {
    sgs_free(m);
    return rc;
  }
  *out = m;
  return HFLMP_OK;
}

template <typename T, bool FWD, int E>
void launch_packed(const Sweep &s, const SgsArgs<T> &a, hipStream_t st) {
  constexpr int D = kPackMaxE / E;
  const PackView pk{s.levels, s.packW, s.prow, s.pent};
  const size_t lds = sizeof(T) * (size_t)a.blk.nrow;
  if (lds <= kPackLds)
    sgs_packed_kernel<T, FWD, E, D, true>
        <<<1, s.packW, lds, st>>>(pk, a.blk.nrow, a.val, a.r, a.z);
  else
    sgs_packed_kernel<T, FWD, E, D, false>
        <<<1, s.packW, 0, st>>>(pk, a.blk.nrow, a.val, a.r, a.z);
}

template <typename T, bool FWD>
void launch_sweep(const Sweep &s, const SgsArgs<T> &a, hipStream_t st) {
  if (s.packW) {
    if (s.packE == 4)
      launch_packed<T, FWD, 4>(s, a, st);
    else if (s.packE == 8)
      launch_packed<T, FWD, 8>(s, a, st);
    else
      launch_packed<T, FWD, 16>(s, a, st);
    return;
  }
  for (const Segment &g : s.seg) {
    if (g.small) {
      sgs_levels_kernel<T, FWD><<<1, kFinalBlock, 0, st>>>(a, s.perm, s.loff, g.a, g.b);
    } else {
      const unsigned grid = (unsigned)((g.b - g.a + kBlock - 1) / kBlock);
      sgs_level_kernel<T, FWD><<<grid, kBlock, 0, st>>>(a, s.perm, g.a, g.b);
    }
  }
}

template <typename T>
int sgs_apply(hflmp_ctx *ctx, const hflmp_sgs *m, const T *r, T *z) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, m && r && z, "sgs_apply: null pointer");
  HFLMP_REQUIRE(ctx, m->value_bytes == (int)sizeof(T), "sgs_apply: value type mismatch");
  HFLMP_REQUIRE(ctx, m->device == ctx->device, "sgs_apply: object on another device");
  SgsArgs<T> a{m->rp, m->ci, static_cast<const T *>(m->val), r, z, m->blk};
  launch_sweep<T, true>(m->fwd, a, ctx->stream);
  launch_sweep<T, false>(m->bwd, a, ctx->stream);
  HFLMP_LAUNCH_CHECK(ctx);
  return HFLMP_OK;
}

}  // namespace

extern "C" {

int hflmp_sgs_create_f64(hflmp_ctx *ctx, int nrow, int nnz, const int *row_ptr, const int *col,
                         const double *val, const int *h_row_ptr, const int *h_col,
                         int num_blocks, hflmp_sgs **out) {
  return sgs_create(ctx, nrow, nnz, row_ptr, col, val, 8, h_row_ptr, h_col, num_blocks, out);
}
int hflmp_sgs_create_f32(hflmp_ctx *ctx, int nrow, int nnz, const int *row_ptr, const int *col,
                         const float *val, const int *h_row_ptr, const int *h_col,
                         int num_blocks, hflmp_sgs **out) {
  return sgs_create(ctx, nrow, nnz, row_ptr, col, val, 4, h_row_ptr, h_col, num_blocks, out);
}
int hflmp_sgs_apply_f64(hflmp_ctx *ctx, const hflmp_sgs *m, const double *r, double *z) {
  return sgs_apply<double>(ctx, m, r, z);
}
int hflmp_sgs_apply_f32(hflmp_ctx *ctx, const hflmp_sgs *m, const float *r, float *z) {
  return sgs_apply<float>(ctx, m, r, z);
}
int hflmp_sgs_get_info(const hflmp_sgs *m, hflmp_sgs_info *info) {
  if (!m || !info) return HFLMP_EINVAL;
  info->nrow = m->nrow;
  info->num_blocks = m->blk.nb;
  info->levels_forward = m->fwd.levels;
  info->levels_backward = m->bwd.levels;
  info->launches = m->fwd.launches() + m->bwd.launches();
  return HFLMP_OK;
}
void hflmp_sgs_destroy(hflmp_sgs *m) {
  if (!m) return;
  int cur = -1;
  (void)hipGetDevice(&cur);
  if (cur != m->device) (void)hipSetDevice(m->device);
  const int dev = m->device;
  sgs_free(m);
  if (cur >= 0 && cur != dev) (void)hipSetDevice(cur);
}

}  // extern "C"
