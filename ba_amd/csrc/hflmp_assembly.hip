// Finite-element assembly into CSR on the device, for any mesh given as a
// cell -> dof table.  The reference assembles on the host: the pattern
// holds every pair of dofs that share a cell, columns ascending
// (compute_sparsity_structure, assembly/assembly_utils.cc:144, then
// coo_2_csr, lmp/lmatrix_formats.h:320-456), and the values are added cell
// by cell in ascending cell order (add_values, lmp/lmatrix_csr_cpu.cc:
// 1102-1153) to a zeroed matrix.
//
// Here a node -> cell incidence list, sorted by cell, gives a row's cells
// in ascending order; the row's columns are the sorted distinct dofs of
// those cells (one wave a row); the row's values are summed from 0 in
// ascending cell order, one term f_c E[a][b] (or the cell's own matrix
// entry) per cell (a group of lanes a row, lane b on local column b), so
// every value is bit-identical to the cell loop.  No atomics touch the
// values.
#include "hflmp_internal.hpp"

#include <climits>
#include <cstring>

struct hflmp_fe_mesh {
  int device;
  char *block;        // the one allocation behind the arrays below
  int nnode, ncell, nloc;
  int *dofs;          // ncell * nloc (own copy)
  int *inc_off;       // nnode + 1
  long long *inc;     // ncell * nloc keys: cell * 32 + local index, sorted per node
  int *row_len;       // nnode pattern row lengths
  long long *tile_sum; // scan workspace, one value per kScanTile nodes
  long long nnz;
  bool repeated;      // some cell has a dof twice
};

namespace {

constexpr int kMaxLoc = 32;

// Cells per node; bad[0]: dofs outside the mesh, bad[1]: dofs that an
// earlier local index of their cell holds too.
__global__ void __launch_bounds__(kBlock)
    fe_count_kernel(int n, int nnode, int nloc, const int *__restrict__ dofs,
                    int *__restrict__ cnt, unsigned int *bad) {
  for (long long kl = blockIdx.x * (long long)kBlock + threadIdx.x; kl < n;
       kl += (long long)gridDim.x * kBlock) {
    const int k = (int)kl, b = k % nloc;
    const int d = dofs[k];
    bool rep = false;
    for (int q = k - b; q < k; ++q) rep = rep || dofs[q] == d;
    if (rep) atomicAdd(bad + 1, 1u);
    if (d < 0 || d >= nnode) {
      atomicAdd(bad, 1u);
      continue;
    }
    atomicAdd(cnt + d, 1);
  }
}

// Exclusive scan of cnt[0..n) into off[0..n] (off[n] = total), in three
// launches: per-tile sums (kScanTile values per workgroup), a one-workgroup
// scan of the tile sums, and a rescan of each tile from its offset.
constexpr int kScanPer = 16;                    // values per thread
constexpr int kScanTile = kBlock * kScanPer;    // values per workgroup

__global__ void __launch_bounds__(kBlock)
    scan_tiles_kernel(int n, const int *__restrict__ cnt, long long *__restrict__ tile_sum) {
  __shared__ long long lds[kBlock / kWave];
  const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanPer;
  long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k)
    if (base + k < n) s += cnt[base + k];
  const long long t = block_sum(s, lds);
  if (threadIdx.x == 0) tile_sum[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kFinalBlock)
    scan_offsets_kernel(int ntiles, long long *__restrict__ tile_sum, long long *total) {
  __shared__ long long tot[kFinalBlock];
  const int t = threadIdx.x;
  const int per = (ntiles + kFinalBlock - 1) / kFinalBlock;
  const int lo = t * per < ntiles ? t * per : ntiles;
  const int hi = lo + per < ntiles ? lo + per : ntiles;
  long long s = 0;
  for (int k = lo; k < hi; ++k) s += tile_sum[k];
  tot[t] = s;
  __syncthreads();
  for (int o = 1; o < kFinalBlock; o <<= 1) {
    const long long add = t >= o ? tot[t - o] : 0;
    __syncthreads();
    tot[t] += add;
    __syncthreads();
  }
  long long run = tot[t] - s;
  for (int k = lo; k < hi; ++k) {
    const long long v = tile_sum[k];
    tile_sum[k] = run;  // exclusive offset of tile k
    run += v;
  }
  if (t == kFinalBlock - 1 && total) *total = tot[t];
}

__global__ void __launch_bounds__(kBlock)
    scan_write_kernel(int n, const int *__restrict__ cnt, const long long *__restrict__ tile_off,
                      int *__restrict__ off) {
  __shared__ long long part[kBlock];
  const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanPer;
  long long s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k)
    if (base + k < n) s += cnt[base + k];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int o = 1; o < kBlock; o <<= 1) {
    const long long add = threadIdx.x >= (unsigned)o ? part[threadIdx.x - o] : 0;
    __syncthreads();
    part[threadIdx.x] += add;
    __syncthreads();
  }
  long long run = tile_off[blockIdx.x] + part[threadIdx.x] - s;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k)
    if (base + k < n) {
      off[base + k] = (int)run;
      run += cnt[base + k];
    }
  if (base + kScanPer >= n && base < n) off[n] = (int)run;  // the last value's thread
}

// tile_sum (ceil(n / kScanTile) values) = the tiles' exclusive offsets,
// *total (device, optional) = the sum of cnt
void scan_tile_offsets(hipStream_t s, int n, const int *cnt, long long *tile_sum,
                       long long *total) {
  const int ntiles = (n + kScanTile - 1) / kScanTile;
  scan_tiles_kernel<<<ntiles, kBlock, 0, s>>>(n, cnt, tile_sum);
  scan_offsets_kernel<<<1, kFinalBlock, 0, s>>>(ntiles, tile_sum, total);
}

// off[0..n] = exclusive scan of cnt
void scan_exclusive(hipStream_t s, int n, const int *cnt, int *off, long long *tile_sum) {
  scan_tile_offsets(s, n, cnt, tile_sum, nullptr);
  scan_write_kernel<<<(n + kScanTile - 1) / kScanTile, kBlock, 0, s>>>(n, cnt, tile_sum, off);
}

__global__ void __launch_bounds__(kBlock)
    fe_incidence_kernel(long long n, int nloc, const int *__restrict__ dofs,
                        const int *__restrict__ off, int *__restrict__ cursor,
                        long long *__restrict__ inc) {
  for (long long k = blockIdx.x * (long long)kBlock + threadIdx.x; k < n;
       k += (long long)gridDim.x * kBlock) {
    const int d = dofs[k];
    const int p = off[d] + atomicAdd(cursor + d, 1);
    inc[p] = (k / nloc) * kMaxLoc + (k % nloc);
  }
}

// sort each node's incidence keys (ascending cell, then local index)
__global__ void __launch_bounds__(kBlock)
    fe_sort_kernel(int nnode, const int *__restrict__ off, long long *__restrict__ inc) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < nnode; i += gridDim.x * kBlock) {
    const int lo = off[i], hi = off[i + 1];
    for (int k = lo + 1; k < hi; ++k) {
      const long long v = inc[k];
      int m = k - 1;
      while (m >= lo && inc[m] > v) {
        inc[m + 1] = inc[m];
        --m;
      }
      inc[m + 1] = v;
    }
  }
}

// Ascending bitonic sort of V values a lane across the wave: value u of a
// lane has index 64 u + lane.
template <int V>
__device__ __forceinline__ void wave_sort(int (&v)[V]) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int k = 2; k <= V * kWave; k <<= 1)
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1)
#pragma unroll
      for (int u = 0; u < V; ++u) {
        if (j < kWave) {
          const int w = __shfl_xor(v[u], j);
          const bool up = ((u * kWave + lane) & k) == 0;
          v[u] = up == ((lane & j) == 0) ? (w < v[u] ? w : v[u]) : (w > v[u] ? w : v[u]);
        } else if ((u & (j / kWave)) == 0) {  // both values are this lane's
          const int q = u | (j / kWave), x = v[u], y = v[q];
          const bool up = ((u * kWave) & k) == 0;
          v[u] = up == (x < y) ? x : y;
          v[q] = up == (x < y) ? y : x;
        }
      }
}

// Distinct dofs of a row's m cells (incidences from lo) in ascending order,
// at most 64 V candidates: their number; WRITE stores them at out.
template <bool WRITE, int V>
__device__ __forceinline__ int fe_row_sorted(int lo, int m, int nloc, int lk, int lb,
                                             const int *__restrict__ dofs,
                                             const long long *__restrict__ inc,
                                             int kstep, int bstep, int *__restrict__ out) {
  const int lane = threadIdx.x & (kWave - 1);
  int d[V];
#pragma unroll
  for (int u = 0; u < V; ++u) {
    d[u] = INT_MAX;
    if (lk < m) d[u] = dofs[(inc[lo + lk] / kMaxLoc) * nloc + lb];
    lk += kstep;
    lb += bstep;
    if (lb >= nloc) {
      lb -= nloc;
      ++lk;
    }
  }
  wave_sort(d);
  int n = 0, last = 0;
#pragma unroll
  for (int u = 0; u < V; ++u) {
    int before = __shfl_up(d[u], 1);
    if (lane == 0) before = last;
    last = __builtin_amdgcn_readlane(d[u], kWave - 1);
    const bool first = d[u] != INT_MAX && ((u == 0 && lane == 0) || d[u] != before);
    const unsigned long long firsts = __ballot(first);
    if (WRITE && first) out[n + __popcll(firsts & ((1ull << lane) - 1))] = d[u];
    n += __popcll(firsts);
  }
  return n;
}

// Distinct dofs of row i's cells in ascending order: WRITE = false counts
// them into len[i], WRITE = true stores them at col + row_ptr[i].
// One wave a row.  Its candidates (every local dof of every cell, 64 for 3D
// Q1, up to 216 for 3D Q2) are loaded at once and sorted across the wave; a
// candidate that differs from its lower neighbour is a column.  On 96^3 Q1
// cells (912,673 rows) the passes take 0.26 and 0.28 ms; one thread a row
// with a repeated search for the next smallest dof (27 x 64 loads, each lane
// elsewhere) took 3.4 ms, and broadcasting the candidates in turn instead of
// the sort 0.9 and 1.4 ms.  Rows of more than 512 candidates search for the
// next smallest with the whole wave.  32^3 Q2 cells (274,625 rows, 17.0 M
// entries): 0.20 ms a pass; with that search for all rows of more than 64
// candidates 4.0 ms, with one thread a row 3.7.
template <bool WRITE>
__global__ void __launch_bounds__(kBlock)
    fe_pattern_kernel(int nnode, int nloc, const int *__restrict__ dofs,
                      const int *__restrict__ off, const long long *__restrict__ inc,
                      int *__restrict__ len, const int *__restrict__ row_ptr,
                      int *__restrict__ col) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  // candidate of this lane, and the way to the one 64 on
  const int lk = lane / nloc, lb = lane - lk * nloc;
  const int kstep = kWave / nloc, bstep = kWave - kstep * nloc;
  const int nwave = gridDim.x * (kBlock / kWave);
  // two passes over the wave's rows, so that the sort of 64, which most meshes
  // need alone, keeps its lane masks in registers (one pass for all: 5% slower
  // on 3D Q1 cells, 13 to 20% on 2D ones)
  bool more = false;
  for (int i = blockIdx.x * (kBlock / kWave) + wid; i < nnode; i += nwave) {
    const int lo = off[i], m = off[i + 1] - lo;
    if ((long long)m * nloc > kWave) {
      more = true;
      continue;
    }
    const int n = fe_row_sorted<WRITE, 1>(lo, m, nloc, lk, lb, dofs, inc, kstep, bstep,
                                          WRITE ? col + row_ptr[i] : nullptr);
    if (!WRITE && lane == 0) len[i] = n;
  }
  if (!more) return;
  for (int i = blockIdx.x * (kBlock / kWave) + wid; i < nnode; i += nwave) {
    const int lo = off[i], m = off[i + 1] - lo;
    const long long cand = (long long)m * nloc;
    if (cand <= kWave) continue;
    int *out = WRITE ? col + row_ptr[i] : nullptr;
    int n = 0;
    if (cand <= 2 * kWave) {
      n = fe_row_sorted<WRITE, 2>(lo, m, nloc, lk, lb, dofs, inc, kstep, bstep, out);
    } else if (cand <= 4 * kWave) {
      n = fe_row_sorted<WRITE, 4>(lo, m, nloc, lk, lb, dofs, inc, kstep, bstep, out);
    } else if (cand <= 8 * kWave) {
      n = fe_row_sorted<WRITE, 8>(lo, m, nloc, lk, lb, dofs, inc, kstep, bstep, out);
    } else {
      int last = -1;
      for (;;) {
        int next = INT_MAX;
        for (long long e = lane; e < cand; e += kWave) {
          const int k = (int)(e / nloc), b = (int)(e - (long long)k * nloc);
          const int d = dofs[(inc[lo + k] / kMaxLoc) * nloc + b];
          if (d > last && d < next) next = d;
        }
        next = wave_min(next);
        if (next == INT_MAX) break;
        if (WRITE && lane == 0) out[n] = next;
        ++n;
        last = next;
      }
    }
    if (!WRITE && lane == 0) len[i] = n;
  }
}

// Row i's values: zero, then for each (cell, local index a) of the node in
// ascending order and each local column b, val[(i, dof b)] += term.  One
// thread a row.
template <typename T>
__global__ void __launch_bounds__(kBlock)
    fe_values_kernel(int nnode, int nloc, const int *__restrict__ dofs,
                     const int *__restrict__ off, const long long *__restrict__ inc,
                     const T *__restrict__ cell_mats, const T *__restrict__ E,
                     const T *__restrict__ factor, const int *__restrict__ row_ptr,
                     const int *__restrict__ col, T *__restrict__ val) {
#pragma clang fp contract(off)
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < nnode; i += gridDim.x * kBlock) {
    const int r0 = row_ptr[i], r1 = row_ptr[i + 1];
    for (int p = r0; p < r1; ++p) val[p] = T(0);
    for (int k = off[i]; k < off[i + 1]; ++k) {
      const long long c = inc[k] / kMaxLoc;
      const int a = (int)(inc[k] % kMaxLoc);
      const int *cd = dofs + c * nloc;
      const T f = factor ? factor[c] : T(1);
      const T *Er = cell_mats ? cell_mats + (c * nloc + a) * nloc : E + a * nloc;
      for (int b = 0; b < nloc; ++b) {
        const int j = cd[b];
        int lo = r0, hi = r1 - 1;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (col[mid] < j) lo = mid + 1;
          else hi = mid;
        }
        const T term = cell_mats ? Er[b] : f * Er[b];
        val[lo] += term;
      }
    }
  }
}

// The same with G >= nloc lanes a row, lane b on local column b, the row's
// columns and sums in LDS: a cell's terms go to different columns (no cell
// repeats a dof: the caller checks), so they are added side by side, and
// cell after cell keeps each column's order.  With one thread a row every add
// was a read and a write of memory behind a search through memory: 4.88 ms on
// 96^3 Q1 cells (24.1 M values), 0.22 ms with groups of 8.
// LDS holds kFeRow entries of a row: as elements of more nodes have longer
// rows, it follows the group (27 entries for 3D Q1, 49 for 2D Q3, 125 for 3D
// Q2).  The group adds a longer row's terms in memory, a search and an add a
// lane and cell.  32^3 3D Q2 cells (17.0 M values): 2.07 ms with one thread a
// row, 3.81 with 32 entries in LDS and one lane for longer rows, 0.138 here;
// 128^2 2D Q3 cells (3.7 M values) 0.20, 0.226, 0.027 ms.
template <int G>
constexpr int kFeRow = G <= 8 ? 32 : 4 * G;

template <typename T, int G>
__global__ void __launch_bounds__(kBlock)
    fe_values_group_kernel(int nnode, int nloc, const int *__restrict__ dofs,
                           const int *__restrict__ off, const long long *__restrict__ inc,
                           const T *__restrict__ cell_mats, const T *__restrict__ E,
                           const T *__restrict__ factor, const int *__restrict__ row_ptr,
                           const int *__restrict__ col, T *val) {
#pragma clang fp contract(off)
  constexpr int R = kBlock / G;  // rows of a workgroup
  constexpr int W = kFeRow<G>;
  __shared__ T acc[R][W + 1];
  __shared__ int cols[R][W + 1];
  const int g = threadIdx.x / G, b = threadIdx.x % G;
  // what the group's lanes have written is what they read next
  auto in_order = []() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // whole waves leave the loop together: a group's lanes are in one wave
  for (long long i0 = (long long)blockIdx.x * R; i0 < nnode; i0 += (long long)gridDim.x * R) {
    const long long il = i0 + g;
    const int i = (int)(il < nnode ? il : nnode - 1);
    const int r0 = row_ptr[i];
    const int n = il < nnode ? row_ptr[i + 1] - r0 : 0;
    const int k0 = off[i], k1 = il < nnode ? off[i + 1] : k0;
    // add(j, term) for each cell in turn, lane b's column and term
    auto cells = [&](auto add) {
      for (int k = k0; k < k1; ++k) {
        if (b < nloc) {
          const long long key = inc[k];
          const long long c = key / kMaxLoc;
          const int a = (int)(key % kMaxLoc);
          const int j = dofs[c * nloc + b];
          add(j, cell_mats ? cell_mats[(c * nloc + a) * nloc + b]
                           : (factor ? factor[c] : T(1)) * E[a * nloc + b]);
        }
        in_order();
      }
    };
    if (n > W) {
      for (int p = b; p < n; p += G) val[r0 + p] = T(0);
      in_order();
      cells([&](int j, T term) {
        int lo = r0, hi = r0 + n - 1;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (col[mid] < j) lo = mid + 1;
          else hi = mid;
        }
        val[lo] += term;
      });
    } else {
      for (int p = b; p < n; p += G) {
        cols[g][p] = col[r0 + p];
        acc[g][p] = T(0);
      }
      in_order();
      auto sum = [&](auto top) {
        cells([&](int j, T term) {
          // the last column not above j is j itself
          int p = 0;
#pragma unroll
          for (int s = decltype(top)::value; s > 0; s >>= 1)
            if (p + s < n && cols[g][p + s] <= j) p += s;
          acc[g][p] += term;
        });
      };
      // a wave without longer rows searches in five steps
      if (W > 32 && __any(n > 32))
        sum(std::integral_constant<int, W / 2>());
      else
        sum(std::integral_constant<int, 16>());
      for (int p = b; p < n; p += G) val[r0 + p] = acc[g][p];
      in_order();
    }
  }
}

unsigned grid_n(long long n) {
  long long g = (n + kBlock - 1) / kBlock;
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return (unsigned)g;
}

void mesh_free(hflmp_fe_mesh *m) {
  if (!m) return;
  int cur = -1;
  (void)hipGetDevice(&cur);
  if (cur != m->device) (void)hipSetDevice(m->device);
  (void)hipFree(m->block);
  if (cur >= 0 && cur != m->device) (void)hipSetDevice(cur);
  delete m;
}

template <typename T>
int fe_assemble(hflmp_ctx *ctx, const hflmp_fe_mesh *m, const T *cell_mats, const T *E,
                const T *factor, const int *row_ptr, const int *col, T *val) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, m && row_ptr && (m->nnz == 0 || (col && val)) && (cell_mats || E),
                "fe_assemble: null pointer (cell_mats or E is needed)");
  HFLMP_REQUIRE(ctx, m->device == ctx->device, "fe_assemble: mesh on another device");
  auto group = [&](auto g) {
    constexpr int G = decltype(g)::value;
    fe_values_group_kernel<T, G><<<grid_n((long long)m->nnode * G), kBlock, 0, ctx->stream>>>(
        m->nnode, m->nloc, m->dofs, m->inc_off, m->inc, cell_mats, E, factor, row_ptr, col, val);
  };
  if (m->repeated)  // a column gets two terms of one cell: in local order, one thread a row
    fe_values_kernel<T><<<grid_n(m->nnode), kBlock, 0, ctx->stream>>>(
        m->nnode, m->nloc, m->dofs, m->inc_off, m->inc, cell_mats, E, factor, row_ptr, col, val);
  else if (m->nloc <= 4)
    group(std::integral_constant<int, 4>());
  else if (m->nloc <= 8)
    group(std::integral_constant<int, 8>());
  else if (m->nloc <= 16)
    group(std::integral_constant<int, 16>());
  else
    group(std::integral_constant<int, 32>());
  HFLMP_LAUNCH_CHECK(ctx);
  return HFLMP_OK;
}

}  // namespace

extern "C" {

int hflmp_fe_mesh_create(hflmp_ctx *ctx, int nnode, int ncell, int nloc, const int *cell_dofs,
                         hflmp_fe_mesh **out) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, out && cell_dofs, "fe_mesh_create: null pointer");
  *out = nullptr;
  HFLMP_REQUIRE(ctx, nnode > 0 && ncell > 0 && nloc >= 1 && nloc <= kMaxLoc,
                "fe_mesh_create: need nnode > 0, ncell > 0, 1 <= nloc <= %d", kMaxLoc);
  const long long n = (long long)ncell * nloc;
  HFLMP_REQUIRE(ctx, n < 0x7fffffffLL, "fe_mesh_create: more than 2^31-1 cell dofs");
  auto *m = new hflmp_fe_mesh();
  m->device = ctx->device;
  m->nnode = nnode;
  m->ncell = ncell;
  m->nloc = nloc;
  auto fail = [&](int code, const char *msg) {
    mesh_free(m);
    return set_error(ctx, code, "fe_mesh_create: %s", msg);
  };
  // one allocation (each costs the host about as long as these kernels
  // run); the counts of the build lie where the row lengths will
  const size_t ntile = ((size_t)nnode + kScanTile - 1) / kScanTile;
  size_t bytes = 0;
  auto take = [&](size_t b) {
    const size_t at = bytes;
    bytes += (b + 255) & ~size_t(255);
    return at;
  };
  const size_t o_dofs = take(sizeof(int) * (size_t)n);
  const size_t o_off = take(sizeof(int) * ((size_t)nnode + 1));
  const size_t o_inc = take(sizeof(long long) * (size_t)n);
  const size_t o_len = take(sizeof(int) * (size_t)nnode);
  const size_t o_tile = take(sizeof(long long) * ntile);
  const size_t o_total = take(sizeof(long long));
  if (hipMalloc(reinterpret_cast<void **>(&m->block), bytes) != hipSuccess)
    return fail(HFLMP_ENOMEM, "out of device memory");
  m->dofs = reinterpret_cast<int *>(m->block + o_dofs);
  m->inc_off = reinterpret_cast<int *>(m->block + o_off);
  m->inc = reinterpret_cast<long long *>(m->block + o_inc);
  m->row_len = reinterpret_cast<int *>(m->block + o_len);
  m->tile_sum = reinterpret_cast<long long *>(m->block + o_tile);
  int *cnt = m->row_len;
  long long *total = reinterpret_cast<long long *>(m->block + o_total);
  hipStream_t s = ctx->stream;
  unsigned int *bad = ctx->red_counter + 32;
  int rc;
  if ((rc = hflmp_fill_zero(ctx, cnt, sizeof(int) * (size_t)nnode)) != HFLMP_OK ||
      (rc = hflmp_fill_zero(ctx, bad, 2 * sizeof(unsigned int))) != HFLMP_OK)
    return fail(rc, "fill");
  if (hipMemcpyAsync(m->dofs, cell_dofs, sizeof(int) * (size_t)n, hipMemcpyDeviceToDevice, s) !=
      hipSuccess)
    return fail(HFLMP_EHIP, "copy failed");
  fe_count_kernel<<<grid_n(n), kBlock, 0, s>>>((int)n, nnode, nloc, m->dofs, cnt, bad);
  unsigned int hbad[2] = {0, 0};  // dofs out of range, dofs repeated in a cell
  if (hipGetLastError() != hipSuccess ||
      hipMemcpyAsync(ctx->host_pinned, bad, sizeof(hbad), hipMemcpyDeviceToHost, s) !=
          hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return fail(HFLMP_EHIP, "HIP error while counting");
  std::memcpy(hbad, ctx->host_pinned, sizeof(hbad));
  m->repeated = hbad[1] != 0;
  if (hbad[0]) return fail(HFLMP_EINVAL, "a cell dof is outside [0, nnode)");
  scan_exclusive(s, nnode, cnt, m->inc_off, m->tile_sum);
  if ((rc = hflmp_fill_zero(ctx, cnt, sizeof(int) * (size_t)nnode)) != HFLMP_OK)
    return fail(rc, "fill");
  fe_incidence_kernel<<<grid_n(n), kBlock, 0, s>>>(n, nloc, m->dofs, m->inc_off, cnt, m->inc);
  fe_sort_kernel<<<grid_n(nnode), kBlock, 0, s>>>(nnode, m->inc_off, m->inc);
  fe_pattern_kernel<false><<<grid_n((long long)nnode * kWave), kBlock, 0, s>>>(
      nnode, nloc, m->dofs, m->inc_off, m->inc, m->row_len, nullptr, nullptr);
  // total pattern entries
  scan_tile_offsets(s, nnode, m->row_len, m->tile_sum, total);
  long long nnz = 0;
  const bool ok = hipGetLastError() == hipSuccess &&
                  hipMemcpyAsync(&nnz, total, sizeof(nnz), hipMemcpyDeviceToHost, s) ==
                      hipSuccess &&
                  hipStreamSynchronize(s) == hipSuccess;
  if (!ok) return fail(HFLMP_EHIP, "HIP error while building the pattern");
  if (nnz > 0x7fffffffLL) return fail(HFLMP_EINVAL, "pattern has more than 2^31-1 entries");
  m->nnz = nnz;
  *out = m;
  return HFLMP_OK;
}

int hflmp_fe_mesh_nnz(const hflmp_fe_mesh *m, long long *nnz) {
  if (!m || !nnz) return HFLMP_EINVAL;
  *nnz = m->nnz;
  return HFLMP_OK;
}

int hflmp_fe_mesh_pattern(hflmp_ctx *ctx, const hflmp_fe_mesh *m, int *row_ptr, int *col) {
  if (!ctx) return HFLMP_EINVAL;
  HFLMP_REQUIRE(ctx, m && row_ptr && (m->nnz == 0 || col), "fe_mesh_pattern: null pointer");
  HFLMP_REQUIRE(ctx, m->device == ctx->device, "fe_mesh_pattern: mesh on another device");
  hipStream_t s = ctx->stream;
  scan_exclusive(s, m->nnode, m->row_len, row_ptr, m->tile_sum);
  fe_pattern_kernel<true><<<grid_n((long long)m->nnode * kWave), kBlock, 0, s>>>(
      m->nnode, m->nloc, m->dofs, m->inc_off, m->inc, nullptr, row_ptr, col);
  HFLMP_LAUNCH_CHECK(ctx);
  return HFLMP_OK;
}

int hflmp_fe_assemble_f64(hflmp_ctx *ctx, const hflmp_fe_mesh *m, const double *cell_mats,
                          const double *E, const double *factor, const int *row_ptr,
                          const int *col, double *val) {
  return fe_assemble<double>(ctx, m, cell_mats, E, factor, row_ptr, col, val);
}

int hflmp_fe_assemble_f32(hflmp_ctx *ctx, const hflmp_fe_mesh *m, const float *cell_mats,
                          const float *E, const float *factor, const int *row_ptr,
                          const int *col, float *val) {
  return fe_assemble<float>(ctx, m, cell_mats, E, factor, row_ptr, col, val);
}

void hflmp_fe_mesh_destroy(hflmp_fe_mesh *m) { mesh_free(m); }

}  // extern "C"
