// Row-block layout for Y = A X over a row-major block of k <= 64 vectors,
// and the device walk that applies it.
//
// Rows are grouped into blocks, each the rows of up to 8 runs of
// consecutive rows taken from consecutive "lines" of L rows: block b of
// line group g (lines g nl .. g nl + nl - 1) and segment c holds, from each
// of its nl lines, the rows at positions c a .. c a + a - 1.  With L the
// line length of a structured mesh's numbering this is an a x nl patch of
// the mesh; with nl = 1 and L = nrow it is a run of a consecutive rows.
// For each block the distinct columns of its entries are listed once, in
// ascending order (ucol[uoff[b] .. uoff[b+1])), and every entry j of the
// CSR arrays gets the position of its column in that list (lidx[j]).  A
// workgroup loads a block's X rows into LDS once -- each a contiguous run
// of k values -- and every entry of the block then reads its X row from
// LDS.  A 4 x 4 patch of the 2D Q2 pattern has 16 rows over at most 64
// distinct columns (4 staged X rows per row), where a run of 8 consecutive
// rows has about 55 (7 per row); neighbouring blocks are walked in order
// by one XCD, so the X rows they share stay in its L2.
//
// Each column c of a row is summed in ascending storage order from zero
// (s += a_ij * x_j, no contraction), the order of the single-vector CSR
// loop (CPUsimple_csr_lmatrix.cc:76-111), so column c of the product is
// bit-identical to A times column c.  The layout shares row_ptr and the
// values with the CSR matrix; lidx replaces the column array.
#pragma once

#include <type_traits>

#include "hflmp_internal.hpp"

// Limits of the pipelined walk: distinct columns and entries of one block.
// A wave holds the next block's X rows in registers: 20 of them in FP64,
// 32 in FP32.
__host__ __device__ constexpr int plan_max_cols(int vb) { return vb == 8 ? 80 : 128; }
constexpr int kPlanMaxEntries = 1024;  // 4 per thread that loads
// Threads of the walk: kBlock that compute and kBlock that load.
constexpr int kPlanThreads = 2 * kBlock;

// Block geometry: lines of L rows, blocks of nl runs (one per line) of at
// most a rows; nseg blocks per line group.
struct PlanGeom {
  int nrow, L, a, nl, nseg;
};

constexpr int kPlanMaxRuns = 8;

inline PlanGeom plan_geom(int nrow, int L, int a, int nl) {
  return PlanGeom{nrow, L, a, nl, (L + a - 1) / a};
}
inline int plan_nblk(const PlanGeom &g) {
  const long long lines = ((long long)g.nrow + g.L - 1) / g.L;
  return (int)((lines + g.nl - 1) / g.nl * g.nseg);
}

// Run t (< nl) of block b: rows [r0, r0 + n), clipped to the matrix.
struct PlanRun {
  int r0, n;
};
__host__ __device__ __forceinline__ PlanRun plan_run(const PlanGeom &g, int b, int t) {
  const int grp = b / g.nseg, c = b - grp * g.nseg;
  const long long s = ((long long)grp * g.nl + t) * g.L + (long long)c * g.a;
  const int w = g.a < g.L - c * g.a ? g.a : g.L - c * g.a;
  const long long lo = s < g.nrow ? s : g.nrow;
  const long long hi = s + w < g.nrow ? s + w : g.nrow;
  return PlanRun{(int)lo, (int)(hi - lo)};
}

struct hflmp_spmm_plan {
  int device;
  int nrow, ncol, nnz;
  int L, a, nl;     // block geometry (PlanGeom)
  int R;            // rows per block, at most (a nl)
  int nblk;
  int umax;         // most distinct columns of one block
  int emax;         // most entries of one block
  int nrhs, value_bytes;  // the products the block size was chosen for
  long long nuniq;  // total of the per-block column lists
  int *uoff;        // nblk + 1 offsets into ucol
  int *ucol;        // each block's distinct columns, ascending
  int *lidx;        // per entry: position of its column in its block's list
  int2 *rows;       // R per block, longest first: global row (-1: none), plan_row_pack
};

// A row within its block's entries: first entry and length.
__host__ __device__ constexpr int plan_row_pack(int first, int len) { return first << 16 | len; }

struct PlanView {
  PlanGeom g;
  int nnz, R, nblk, umax, emax;
  const int *__restrict__ uoff;
  const int *__restrict__ ucol;
  const int *__restrict__ lidx;
  const int2 *__restrict__ rows;
  int cached;  // entries_cached, by blocks
};

inline PlanView plan_view(const hflmp_spmm_plan *p, int cached) {
  return PlanView{plan_geom(p->nrow, p->L, p->a, p->nl), p->nnz, p->R, p->nblk, p->umax,
                  p->emax, p->uoff, p->ucol, p->lidx, p->rows,
                  cached};
}

// LDS of the walk: the X rows of one block, then two buffers of the
// block's description: entries (values, column positions), column list,
// local row pointers and global row numbers.
__host__ __device__ inline size_t plan_meta_bytes(int R, int umax, int emax, int vb) {
  const size_t b =
      (size_t)emax * (4 + vb) + (size_t)umax * 4 + (size_t)(R + 1) * 4 + (size_t)R * 4;
  return (b + 15) & ~size_t(15);
}
__host__ __device__ inline size_t plan_lds_bytes(int R, int umax, int emax, int k, int vb) {
  const size_t x = ((size_t)umax * k * vb + 15) & ~size_t(15);
  return x + 2 * plan_meta_bytes(R, umax, emax, vb);
}

// Workgroups of a walk: as many as are resident at once on the CUs (the
// kernel's occupancy with `lds` dynamic bytes on top of its static LDS and
// registers; at most 8 per CU), a multiple of the XCD count, and no more
// than the blocks rounded up to that multiple.  A grid beyond what is
// resident would run a second partial round of workgroups.
inline int plan_grid(hflmp_ctx *ctx, const void *kern, int nblk, size_t lds) {
  const int cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kPlanThreads, lds) != hipSuccess)
    per_cu = lds > 0 ? (int)(160 * 1024 / lds) : 8;
  if (per_cu > 8) per_cu = 8;
  if (per_cu < 1) per_cu = 1;
  long long g = (long long)per_cu * cus / kXcds * kXcds;
  const long long gb = ((long long)nblk + kXcds - 1) / kXcds * kXcds;
  if (g > gb) g = gb;
  if (g < kXcds) g = kXcds;
  return (int)g;
}

// One block's description in LDS.
template <typename T>
struct PlanMeta {
  int *li;  // entries' column positions
  T *v;     // entries' values
  int *uc;  // distinct columns
  int *gr;  // global row of each of the block's rows (R), -1 past its last
  int *se;  // their plan_row_pack
};

template <typename T>
__device__ __forceinline__ PlanMeta<T> plan_meta_at(unsigned char *base, const PlanView &pv) {
  PlanMeta<T> m;
  m.v = reinterpret_cast<T *>(base);
  m.li = reinterpret_cast<int *>(base + (size_t)pv.emax * sizeof(T));
  m.uc = m.li + pv.emax;
  m.gr = m.uc + pv.umax;
  m.se = m.gr + pv.R;
  return m;
}

// A block's header, one register: lane t < 8 holds rp at the start of run
// t, lane 8 + t rp at its end (runs t >= nl: rp[0] twice), lanes 16 and 17
// uoff[b] and uoff[b + 1].  Loaded a stage before the block's description,
// as a vector load, so that nothing waits on it in the stage that issues it.
__device__ __forceinline__ int plan_hdr_load(int b, const PlanView &pv,
                                             const int *__restrict__ rp) {
  const int lane = threadIdx.x & (kWave - 1);
  const int t = lane & 7;
  const int *p = rp;
  if (lane < 16 && t < pv.g.nl) {
    const PlanRun run = plan_run(pv.g, b, t);
    p = rp + run.r0 + (lane < 8 ? 0 : run.n);
  } else if (lane == 16 || lane == 17) {
    p = pv.uoff + b + (lane - 16);
  }
  return *p;
}

// The uniform values of a block: its number, entries and column list.
struct PlanHdr {
  int b, hreg, ne, u0, U;
};

__device__ __forceinline__ PlanHdr plan_hdr(int hreg, int b, const PlanView &pv) {
  PlanHdr h;
  h.b = b;
  h.hreg = hreg;
  int ne = 0;
  for (int t = 0; t < pv.g.nl; ++t)
    ne += __builtin_amdgcn_readlane(hreg, 8 + t) - __builtin_amdgcn_readlane(hreg, t);
  h.ne = ne;
  h.u0 = __builtin_amdgcn_readlane(hreg, 16);
  h.U = __builtin_amdgcn_readlane(hreg, 17) - h.u0;
  return h;
}

// A block's description on its way from memory to LDS: thread t holds
// entries t, t+256, ... (at most 4) of the block's runs laid end to end,
// column t of the list and row t.  Every load is issued (addresses past the
// block's end are clamped into it), so the number of loads in flight does
// not depend on the block.
template <typename T>
struct PlanMetaRegs {
  int li[4];
  T v[4];
  int uc;
  int2 row;
};

template <typename T>
__device__ __forceinline__ void plan_meta_load(PlanMetaRegs<T> &m, const PlanHdr &h,
                                               const PlanView &pv, const T *__restrict__ val) {
  const int t = threadIdx.x & (kBlock - 1);
  // Local entry e lies in the last run that starts at or before it, and has
  // CSR index e + base for that run's base.  (Runs are in row order, and an
  // empty run starts where the next one does.)
  int base[4] = {0, 0, 0, 0};
  int eacc = 0;
  for (int r = 0; r < pv.g.nl; ++r) {
    const int j = __builtin_amdgcn_readlane(h.hreg, r);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (t + q * kBlock >= eacc) base[q] = j - eacc;
    eacc += __builtin_amdgcn_readlane(h.hreg, 8 + r) - j;
  }
  m.row = pv.rows[(size_t)h.b * pv.R + (t < pv.R ? t : pv.R - 1)];
  m.uc = pv.ucol[h.u0 + (t < h.U ? t : (h.U > 0 ? h.U - 1 : 0))];
  // entries past the block's last read its first run's first entry
  const int j0 = __builtin_amdgcn_readlane(h.hreg, 0);
  const int jpad = j0 < pv.nnz ? j0 : pv.nnz - 1;
  int j[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) j[q] = t + q * kBlock < h.ne ? t + q * kBlock + base[q] : jpad;
  if (past_caches(h.b, pv.cached)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      m.li[q] = __builtin_nontemporal_load(pv.lidx + j[q]);
      m.v[q] = __builtin_nontemporal_load(val + j[q]);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      m.li[q] = pv.lidx[j[q]];
      m.v[q] = val[j[q]];
    }
  }
}

template <typename T>
__device__ __forceinline__ void plan_meta_store(const PlanMetaRegs<T> &m, const PlanHdr &h,
                                                const PlanView &pv, const PlanMeta<T> &d) {
  const int t = threadIdx.x & (kBlock - 1);
  if (t < pv.R) {
    d.gr[t] = m.row.x;
    d.se[t] = m.row.y;
  }
  if (t < h.U) d.uc[t] = m.uc;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = t + q * kBlock;
    if (e < h.ne) {
      d.li[e] = m.li[q];
      d.v[e] = m.v[q];
    }
  }
}

// v of lane Q of the lane's row of 16.
template <int Q, typename T>
__device__ __forceinline__ T row_bcast(T v) {
  constexpr int W = sizeof(T) / 4;
  struct Words {
    int w[W];
  };
  Words a = __builtin_bit_cast(Words, v);
#pragma unroll
  for (int i = 0; i < W; ++i)
    a.w[i] = __builtin_amdgcn_update_dpp(0, a.w[i], 0x150 + Q, 0xf, 0xf, true);
  return __builtin_bit_cast(T, a);
}

// The columns of a lane.  Four rows are computed side by side, 16 lanes
// each; lane i of 16 holds CV of the k columns: i, i + 16, ... or, of 64
// (FULL), runs of 16 bytes, 16 lanes apart, so that LDS and memory are read
// and written 16 bytes a lane.  Columns past k - 1 are read (from what lies
// behind the X row in LDS: the next one, or the descriptions, which are
// longer than the 15 values) and dropped.
template <typename T, int CV, bool FULL>
struct PlanCols {
  static constexpr int kRun = FULL ? 16 / (int)sizeof(T) : 1;  // columns a piece
  static constexpr int kPieces = CV / kRun;
  typedef T Piece __attribute__((ext_vector_type(kRun), aligned(sizeof(T))));
  // first column of piece p of lane i of 16
  __device__ __forceinline__ static int first(int i, int p) { return (p * 16 + i) * kRun; }
  template <typename F>
  __device__ __forceinline__ static void each(F &&f) {
#pragma unroll
    for (int p = 0; p < kPieces; ++p) f(p);
  }
  __device__ __forceinline__ static void load(T *x, const T *src, int i, int k) {
    each([&](int p) {
      const int c = first(i, p);
      const Piece v = *reinterpret_cast<const Piece *>(src + (FULL || c < k ? c : 0));
      __builtin_memcpy(x + p * kRun, &v, sizeof(v));
    });
  }
  // STREAM: past the caches
  template <bool STREAM>
  __device__ __forceinline__ static void store(T *dst, const T *x, int i, int k) {
    each([&](int p) {
      const int c = first(i, p);
      Piece v;
      __builtin_memcpy(&v, x + p * kRun, sizeof(v));
      if (!FULL && c >= k) return;
      if (STREAM)
        __builtin_nontemporal_store(v, reinterpret_cast<Piece *>(dst + c));
      else
        *reinterpret_cast<Piece *>(dst + c) = v;
    });
  }
};

// s += the first n of 16 entries, in order: lane i of 16 holds the value v
// and the byte offset pos in LDS of the X row of entry i, xl is the lane's
// place in X row 0.  nmin <= n <= nmax <= 4 NG over the wave's rows.  The
// X values of the next E entries (2 or 4) are read while E are added.
constexpr int kPlanStrip = 16;

template <typename T, int CV, bool FULL, int E, int NG>
struct PlanStripSum {
  using Cols = PlanCols<T, CV, FULL>;
  template <int Q>
  __device__ __forceinline__ static void read(T (*x)[CV], const unsigned char *xl, int pos) {
    const unsigned char *at = xl + row_bcast<Q>(pos);
    Cols::each([&](int p) {
      typedef T Piece __attribute__((ext_vector_type(Cols::kRun)));
      const Piece v = *reinterpret_cast<const Piece *>(at + p * 16 * Cols::kRun * sizeof(T));
      __builtin_memcpy(&x[Q % E][p * Cols::kRun], &v, sizeof(v));
    });
    if constexpr (Q % E < E - 1) read<Q + 1>(x, xl, pos);
  }
  template <int Q>
  __device__ __forceinline__ static void add(T *s, const T (*x)[CV], T v, int n, bool all) {
#pragma clang fp contract(off)
    const T vq = row_bcast<Q>(v);
    if (all || Q < n)
#pragma unroll
      for (int j = 0; j < CV; ++j) s[j] += vq * x[Q % E][j];
    if constexpr (Q % E < E - 1) add<Q + 1>(s, x, v, n, all);
  }
  // entries Q on, Q's group being in x[Q / E % 2]
  template <int Q>
  __device__ __forceinline__ static void group(T *s, T (*x)[E][CV], const unsigned char *xl,
                                               int pos, T v, int n, int nmin) {
    if constexpr (Q + E < 4 * NG) read<Q + E>(x[(Q / E + 1) % 2], xl, pos);
    if (nmin >= Q + E)
      add<Q>(s, x[Q / E % 2], v, n, true);
    else
      add<Q>(s, x[Q / E % 2], v, n, false);
    if constexpr (Q + E < 4 * NG) group<Q + E>(s, x, xl, pos, v, n, nmin);
  }
  __device__ __forceinline__ static void run(T *s, const unsigned char *xl, int pos, T v, int n,
                                             int nmin) {
    T x[2][E][CV];
    read<0>(x[0], xl, pos);
    group<0>(s, x, xl, pos, v, n, nmin);
  }
};

template <typename T, int CV, bool FULL, int E>
__device__ __forceinline__ void plan_strip(T *s, const unsigned char *xl, int pos, T v, int n,
                                           int nmin, int nmax) {
  if (nmax > 12)
    PlanStripSum<T, CV, FULL, E, 4>::run(s, xl, pos, v, n, nmin);
  else if (nmax > 8)
    PlanStripSum<T, CV, FULL, E, 3>::run(s, xl, pos, v, n, nmin);
  else if (nmax > 4)
    PlanStripSum<T, CV, FULL, E, 2>::run(s, xl, pos, v, n, nmin);
  else if (nmax > 0)
    PlanStripSum<T, CV, FULL, E, 1>::run(s, xl, pos, v, n, nmin);
}

// The walk.  XCD x (workgroups b with b % 8 == x) takes the contiguous band
// of blocks [x band, (x+1) band) and its workgroups stride over it, so the
// workgroups of one XCD are on neighbouring blocks at any time.
//
// The first four waves of a workgroup compute block m from LDS while the
// last four have the next blocks on their way: the X rows of block m+1, the
// description of block m+2 and the header of block m+3 in registers, stored
// to LDS between two barriers after waiting for loads issued a whole step
// before.  A wave that loads and stores Y as well waits, with its loads, for
// the stores of the step (one counter), and spends its issue slots on both.
//
// The computing waves are bound by their instructions: a product and a sum
// per entry and column (the CSR loop's rounding, so not fused), and the
// entry's value and position for every lane.  So a wave computes four rows
// side by side, 16 lanes each with up to four columns a lane; lane i of a
// row's 16 holds entry i and the others take it as a DPP row broadcast, once
// for all the lane's columns.  The rows of a block are in order of length,
// so that the four are about as long (2D Q2 has rows of 25, 15 and 9), and
// a wave's turns alternate between the longer and the shorter.  The first 32
// entries of rows are read a turn ahead.
// 2D Q2 512^2 (1,050,625 rows, 16.8 M entries), FP64, 64 vectors: 520 us
// with a row a wave and its entries read from LDS by all lanes, 463 with
// broadcasts, 412 with the roles apart, 303 with four rows (16 vectors: 449
// with broadcasts, 390, 155; FP32, 64 vectors: 345, 298, 200).
// Blocks of fewer than 16 rows give only R / 4 waves a turn, and are still
// faster than a row a wave: 3D Q1 48^3 (blocks of 8 rows in FP64), us, a row a
// wave and now: 64 vectors 136 and 100, 16 vectors 135 and 49; blocks of 4
// rows of 75 entries, the most work for one wave, 64 vectors 56 and 57, 16
// vectors 55 and 27.
// The code is long (28 to 37 KB for four columns a lane) and entries of up to
// 88 MB are loaded through the caches, so repeated products gain more than one
// after other work; one call between two waits of the host, the caches swept
// in between: 2D Q1 64^2, 64 vectors, FP64 27.2 -> 20.9 us (repeated 18.3 -> 11.4),
// 400^2 83.8 -> 75.6 (64.7 -> 42.6).
//
// pre(i, u) leaves CV values for row i before its sums (what the epilogue
// needs, loaded early); epi(i, s, u) gets row i's sums of the lane's columns
// (PlanCols) on the lanes that have a row.  E: the entries read ahead.
template <typename T, int CV, bool FULL, int E, typename Pre, typename Epi>
__device__ __forceinline__ void plan_walk(const PlanView &pv, int k_arg,
                                          const int *__restrict__ rp, const T *__restrict__ val,
                                          const T *__restrict__ X, unsigned char *lds,
                                          Pre &&pre, Epi &&epi) {
  const int k = FULL ? 64 : k_arg;
  constexpr int nw = kBlock / kWave;
  // X rows a load of one wave brings, and its loads
  constexpr int SUB = CV == 1 ? 4 : CV == 2 ? 2 : 1;
  constexpr int PFX = plan_max_cols((int)sizeof(T)) / (nw * SUB);
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int wid = wave % nw;
  const int per = gridDim.x / kXcds;
  const int xcd = blockIdx.x % kXcds, bx = blockIdx.x / kXcds;
  const int band = (pv.nblk + kXcds - 1) / kXcds;
  const int b_beg = xcd * band + bx;
  const int b_end = (xcd + 1) * band < pv.nblk ? (xcd + 1) * band : pv.nblk;
  if (b_beg >= b_end) return;
  const int nb = (b_end - b_beg + per - 1) / per;  // blocks of this workgroup
  // block m of this workgroup; past the last one, the last one again (its
  // loads are issued and never used)
  auto blk = [&](int m) { return b_beg + (m < nb ? m : nb - 1) * per; };

  T *xs = reinterpret_cast<T *>(lds);
  unsigned char *mb = lds + (((size_t)pv.umax * k * sizeof(T) + 15) & ~size_t(15));
  const size_t msz = plan_meta_bytes(pv.R, pv.umax, pv.emax, (int)sizeof(T));
  // buffer `i` of the descriptions, recomputed from the LDS base each time
  // (an array of the two pointers would hide that they point into LDS)
  auto meta = [&](int i) { return plan_meta_at<T>(mb + (size_t)i * msz, pv); };

  // Both roles pass the same barriers: one, and two a block.  (The role is
  // uniform across a wave; two loops keep one's registers out of the other's.)
  if (wave >= nw) {
    PlanMetaRegs<T> mr;
    T xr[PFX];
    // Load q brings X rows (wid + nw q) SUB + sub of the block's list, lane l
    // value l % k of row sub = l / k.  Past the last row the last one again,
    // so that no branch lies between the loads.
    const int sub = SUB == 1 ? 0 : lane / k < SUB ? lane / k : SUB - 1;
    const int col = SUB == 1 ? (lane < k ? lane : k - 1) : lane % k;
    const bool mine = lane < SUB * k;
    auto load_x = [&](const PlanMeta<T> &m, int U) {
      // SUB == 1: lane q holds the column of load q (a read of the list per
      // load would wait for LDS before it)
      const int ul = wid + lane * nw;
      const int uc = SUB == 1 && U > 0 ? m.uc[ul < U ? ul : U - 1] : 0;
      int c[PFX];
#pragma unroll
      for (int q = 0; q < PFX; ++q) {
        const int u = (wid + q * nw) * SUB + sub;
        c[q] = SUB == 1 ? __builtin_amdgcn_readlane(uc, q)
                        : U > 0 ? m.uc[u < U ? u : U - 1] : 0;
      }
#pragma unroll
      for (int q = 0; q < PFX; ++q) xr[q] = X[(size_t)c[q] * k + col];
    };
    auto store_x = [&](int U) {
      if (mine && U > 0) {
#pragma unroll
        for (int q = 0; q < PFX; ++q) {
          const int u = (wid + q * nw) * SUB + sub;
          xs[(u < U ? u : U - 1) * k + col] = xr[q];
        }
      }
    };
    // prologue: block 0's description in buffer 0, block 1's in registers,
    // block 0's X rows and block 2's header in flight
    const int h0 = plan_hdr_load(blk(0), pv, rp);
    const int h1 = plan_hdr_load(blk(1), pv, rp);
    PlanHdr H0 = plan_hdr(h0, blk(0), pv);
    plan_meta_load(mr, H0, pv, val);
    plan_meta_store(mr, H0, pv, meta(0));
    PlanHdr H1 = plan_hdr(h1, blk(1), pv);
    plan_meta_load(mr, H1, pv, val);
    __syncthreads();
    load_x(meta(0), H0.U);
    int hn = plan_hdr_load(blk(2), pv, rp);  // header of block m+2
    for (int m = 0; m < nb; ++m) {
      const int buf = m & 1;
      // loads of the previous step: X rows of m, description of m+1, header of m+2
      store_x(H0.U);
      plan_meta_store(mr, H1, pv, meta(buf ^ 1));
      const PlanHdr H2 = plan_hdr(hn, blk(m + 2), pv);
      __syncthreads();
      // this step's loads
      hn = plan_hdr_load(blk(m + 3), pv, rp);
      plan_meta_load(mr, H2, pv, val);
      load_x(meta(buf ^ 1), H1.U);
      __syncthreads();
      H0 = H1;
      H1 = H2;
    }
    return;
  }

  // Four rows on their way through a wave: the lane's row, its length and
  // first two strips, and the wave's longest and shortest.
  struct Rows {
    int gi, a, n, nmin, nmax, pos[2];
    T v[2];
  };
  const int li = lane & 15;
  const unsigned char *xl =
      lds + (size_t)PlanCols<T, CV, FULL>::first(li, 0) * sizeof(T);
  auto strip = [&](const PlanMeta<T> &md, int j, int e, int &pos, T &v) {
    const int je = j + li < e ? j + li : e - 1;
    const int jl = je > 0 ? je : 0;
    pos = md.li[jl] * (k * (int)sizeof(T));
    v = md.v[jl];
  };
  const int turns = pv.R / 4;  // R is a multiple of 4
  auto compute = [&](const PlanMeta<T> &md) {
    auto rows = [&](int j) {
      const int t = j * nw + (j & 1 ? nw - 1 - wid : wid);
      const int r = 4 * (t < turns ? t : turns - 1) + lane / 16;
      Rows w;
      const int se = md.se[r];
      w.gi = t < turns ? md.gr[r] : -1;
      w.a = se >> 16;
      w.n = w.gi >= 0 ? se & 0xffff : 0;
      w.nmax = __builtin_amdgcn_readlane(w.n, 0);
      w.nmin = __builtin_amdgcn_readlane(w.n, 48);
      strip(md, w.a, w.a + w.n, w.pos[0], w.v[0]);
      strip(md, w.a + kPlanStrip, w.a + w.n, w.pos[1], w.v[1]);
      return w;
    };
    Rows w = rows(0);
    for (int j = 0; j * nw < turns; ++j) {
      const Rows next = rows(j + 1);
      T s[CV], u[CV];
      pre(w.gi >= 0 ? w.gi : 0, u);
#pragma unroll
      for (int c = 0; c < CV; ++c) s[c] = 0;
      plan_strip<T, CV, FULL, E>(s, xl, w.pos[0], w.v[0], w.n, w.nmin, w.nmax);
      if (w.nmax > kPlanStrip) {
        plan_strip<T, CV, FULL, E>(s, xl, w.pos[1], w.v[1], w.n - kPlanStrip, w.nmin - kPlanStrip,
                                w.nmax - kPlanStrip);
        for (int d = 2 * kPlanStrip; d < w.nmax; d += kPlanStrip) {
          int pos;
          T v;
          strip(md, w.a + d, w.a + w.n, pos, v);
          plan_strip<T, CV, FULL, E>(s, xl, pos, v, w.n - d, w.nmin - d, w.nmax - d);
        }
      }
      if (w.gi >= 0) epi(w.gi, s, u);
      w = next;
    }
  };
  __syncthreads();
  for (int m = 0; m < nb; ++m) {
    __syncthreads();
    compute(meta(m & 1));
    __syncthreads();
  }
}

// f with the kernel's column template for k vectors: f(CV, FULL) as
// integral constants.
template <typename F>
inline auto plan_dispatch(int k, F &&f) {
  using std::integral_constant;
  if (k == 64) return f(integral_constant<int, 4>(), std::true_type());
  if (k > 48) return f(integral_constant<int, 4>(), std::false_type());
  if (k > 32) return f(integral_constant<int, 3>(), std::false_type());
  if (k > 16) return f(integral_constant<int, 2>(), std::false_type());
  return f(integral_constant<int, 1>(), std::false_type());
}
