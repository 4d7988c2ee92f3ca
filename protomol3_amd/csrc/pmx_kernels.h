// HIP kernels for the ProtoMol nonbonded hot path on gfx950 (CDNA4).
//
// Data layout in HBM (per system):
//   xorig  double[3N]  positions as the caller hands them (AoS, original order)
//   permp  int[Npad]   sorted slot -> original atom (-1 for padding slots)
//   slot   int[N]      original atom -> sorted slot
//   xs     R4[Npad]    coordinates relative to the slot's supercluster origin
//                      + scaled charge, sorted (R = double for the FP64 form,
//                      float for the mixed form)
//   sorg   float4[Nsuper]  supercluster origins (multiples of 1/16 A)
//   ts     int[Npad]   LJ type per sorted slot (-1 padding)
//   facc   Acc[3Npad]  force accumulators in sorted order (double, or int64
//                      fixed point 2^-32 for the mixed form)
// Superclusters are 64 slots (one wavefront): up to 64 atoms of one x-y
// column of the box, consecutive in z, split by x, then y, then z into 8
// clusters of 8 slots.  Padding slots fill the last supercluster of a column.
#pragma once
#include <type_traits>

#include "pmx_common.h"

namespace pmx {

// ---------------------------------------------------------------------------
// helpers

template <class T>
struct Real4;
template <>
struct Real4<double> {
  using type = double4;
};
template <>
struct Real4<float> {
  using type = float4;
};

// Reference minimal image in FP64 with the reference's operation order and
// no FMA contraction (PeriodicBoundaryConditions.h:72-110).  Returns d^2.
__device__ inline double exact_d2(const double *__restrict__ x, int a, int b, const Box &bx) {
#pragma clang fp contract(off)
  double d[3] = {x[3 * b] - x[3 * a], x[3 * b + 1] - x[3 * a + 1], x[3 * b + 2] - x[3 * a + 2]};
  double d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  if (d2 > bx.D) {
    for (int k = 0; k < 3; ++k) {
      if (d[k] < -bx.H2[k])
        d[k] += bx.H[k];
      else if (d[k] > bx.H2[k])
        d[k] -= bx.H[k];
    }
    d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    if (d2 > bx.D) {
      for (int k = 0; k < 3; ++k) d[k] -= bx.L[k] * rint(bx.Lr[k] * d[k]);
      d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    }
  }
  return d2;
}

// Reference minimalPosition (PeriodicBoundaryConditions.h:113-147), FP64, no contraction.
__device__ inline void exact_minpos(const double *p, const Box &bx, double *out) {
#pragma clang fp contract(off)
  double d[3] = {p[0] - bx.o[0], p[1] - bx.o[1], p[2] - bx.o[2]};
  if (d[0] * d[0] + d[1] * d[1] + d[2] * d[2] <= bx.D) {
    out[0] = d[0];
    out[1] = d[1];
    out[2] = d[2];
    return;
  }
  for (int k = 0; k < 3; ++k) {
    if (d[k] < -bx.H2[k])
      d[k] += bx.H[k];
    else if (d[k] > bx.H2[k])
      d[k] -= bx.H[k];
  }
  if (d[0] * d[0] + d[1] * d[1] + d[2] * d[2] <= bx.D) {
    out[0] = d[0];
    out[1] = d[1];
    out[2] = d[2];
    return;
  }
  for (int k = 0; k < 3; ++k) out[k] = d[k] - bx.L[k] * rint(bx.Lr[k] * d[k]);
}

template <class T>
__device__ inline T wave_sum(T v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}
__device__ inline int wave_max(int v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = max(v, __shfl_xor(v, m));
  return v;
}

// inclusive prefix over the wave
__device__ inline int wave_prefix(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int y = __shfl_up(v, off);
    if (lane >= off) v += y;
  }
  return v;
}

struct PmeParams {
  int nx, ny, nz, nzh, order;
  double hxr, hyr, hzr;   // K/L per axis (Grid.h:520-522)
  int offx, offy, offz;   // -(p-1)/2 + K (Grid.h:509-511)
  int tx, ty;             // lines of a tile along x (even) and y, powers of two
  int ntx, nty;           // tiles per axis
  int ncy, ncx;           // x-y columns of the sort
};

// An atom's place on the grid, per sorted slot: fractional offsets and charge
// (pmw), base indices x | y << 16 and z (pmb; x = kNoGrid for slots without a
// charge).  Written by the sort and by every drift.
constexpr int kNoGrid = -1;
template <class R>
struct PmeSlots {
  typename Real4<R>::type *w;
  int2 *b;
};

// Grid index of base + offset for base in [0, K), offset < K.
__host__ __device__ inline int wrap_grid(int v, int K) { return v >= K ? v - K : v; }

// Grid coordinate of one axis: u = x K/L wrapped to [0, K) (Grid.h:111-120);
// the base is wrapped too.  Far from the box whole periods are taken off at
// once, exactly (their number times K is below 2^53); from 2^40 points on (a run
// that blew up, infinity) no fraction is left and the place is 0.  One period at
// a time would take up to 2^40 turns of the loop there, or never end.
__host__ __device__ inline void grid_coord(double x, double hr, int K, int off, int &base, double &w) {
  double u = x * hr;
  if (fabs(u) >= 1024.0 * K) u = fabs(u) < 0x1p40 ? u - K * floor(u / K) : 0.0;
  while (u < 0.0) u += K;
  while (u >= K) u -= K;
  const int iu = (int)u;
  base = wrap_grid(iu + off, K);
  w = u - iu;
}

// The grid record of slot s for an atom of charge q at x (a < 0: no atom).
template <class R>
__device__ inline void pme_record(const PmeParams &p, const PmeSlots<R> &rec, int s, bool atom, const double x[3],
                                  double q) {
  int b[3] = {kNoGrid, 0, 0};
  double w[3] = {0, 0, 0};
  if (atom && (R)q != (R)0) {
    grid_coord(x[0], p.hxr, p.nx, p.offx, b[0], w[0]);
    grid_coord(x[1], p.hyr, p.ny, p.offy, b[1], w[1]);
    grid_coord(x[2], p.hzr, p.nz, p.offz, b[2], w[2]);
  }
  typename Real4<R>::type v;
  v.x = (R)w[0];
  v.y = (R)w[1];
  v.z = (R)w[2];
  v.w = (R)q;
  rec.w[s] = v;
  rec.b[s] = make_int2(b[0] < 0 ? kNoGrid : (b[0] | (b[1] << 16)), b[2]);
}

// ---------------------------------------------------------------------------
// 1. Binning: wrapped coordinates, column x z-bin sort key, reference cell.
struct BinParams {
  Box box;
  int ncx, ncy, nzb;  // column grid in x-y, z bins per column (sort key)
  double cxinv, cyinv, zinv;  // ncx / Lx, ncy / Ly, nzb / Lz
  int rc_n[3];        // reference cell grid
  double rc_inv[3];   // 1 / reference cell edge
  double delta[3];    // origin - min
};

// Block number for work laid out in order: the hardware deals consecutive
// blocks of a launch to the 8 XCDs in turn, so this renumbering gives the
// blocks of one XCD one contiguous range of the work (block bx runs on XCD
// bx mod 8; XCD x's ranks 0, 1, ... map to the x-th of 8 consecutive ranges,
// the first nb mod 8 of them one block longer), and neighbouring work shares
// that XCD's L2.  A bijection on [0, nb).
__device__ inline int xcd_block(int bx, int nb) {
  const int x = bx & 7, q = nb >> 3, r = nb & 7;
  return x * q + min(x, r) + (bx >> 3);
}

__device__ __forceinline__ void bin_body(const int bid_, const int nbk_, int n, const double *__restrict__ xorig,
                                         BinParams p, uint32_t *__restrict__ key, double *__restrict__ xwrap,
                                         int *__restrict__ refcell, uint32_t *__restrict__ hist, int *clear) {
  int a = bid_ * blockDim.x + threadIdx.x;
  if (clear && a < 2) clear[a] = 0;  // the overflow flag of the pass that begins here
  if (a >= n) return;
  double w[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double x = xorig[3 * a + k];
    double v = x - p.box.L[k] * floor(x * p.box.Linv[k]);
    if (v >= p.box.L[k]) v -= p.box.L[k];
    if (v < 0.0) v = 0.0;
    w[k] = v;
  }
  // key: x-y column, then z bin
  const int cx = min((int)(w[0] * p.cxinv), p.ncx - 1), cy = min((int)(w[1] * p.cyinv), p.ncy - 1);
  const int zb = min((int)(w[2] * p.zinv), p.nzb - 1);
  const uint32_t kb = (uint32_t)((cx * p.ncy + cy) * p.nzb + zb);
  key[a] = kb;
  atomicAdd(&hist[kb], 1u);  // the scan clears hist after reading it
  xwrap[3 * a] = w[0];
  xwrap[3 * a + 1] = w[1];
  xwrap[3 * a + 2] = w[2];
  // Reference cell: findCell(delta + minimalPosition(x)) (Topology.h:64-66,
  // CubicCellManager.cpp:40-44), an upper-face index wrapped to its image.
  double mp[3];
  exact_minpos(&xorig[3 * a], p.box, mp);
  int c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double t;
    {
#pragma clang fp contract(off)
      t = (p.delta[k] + mp[k]) * p.rc_inv[k];
    }
    int ci = (int)floor(t);
    ci %= p.rc_n[k];
    if (ci < 0) ci += p.rc_n[k];
    c[k] = ci;
  }
  refcell[a] = (c[0] * p.rc_n[1] + c[1]) * p.rc_n[2] + c[2];
}

static __global__ void k_bin(int n, const double *__restrict__ xorig, BinParams p, uint32_t *__restrict__ key,
                      double *__restrict__ xwrap, int *__restrict__ refcell, uint32_t *__restrict__ hist, int *clear) {
  bin_body(blockIdx.x, gridDim.x, n, xorig, p, key, xwrap, refcell, hist, clear);
}

// Counting sort by key (one radix digit spanning the key range): histogram,
// exclusive scan, scatter; the split takes each bin's atoms in index order, so
// the result is deterministic.
static __global__ void k_fill_u32(uint32_t *p, uint32_t v, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
static __global__ void k_fill_i32(int *p, int v, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
static __global__ void k_fill_u64(unsigned long long *p, unsigned long long v, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Exclusive scan of m uint32 in 3 launches: per-block sums, scan of sums in
// one block, then per-block rescan with the block offset.
constexpr int kScanBlock = 1024;
static __global__ void k_scan_blocksums(const uint32_t *__restrict__ in, long long m, uint32_t *__restrict__ sums) {
  __shared__ uint32_t s[kScanBlock / kWave];
  long long i = (long long)blockIdx.x * kScanBlock + threadIdx.x;
  uint32_t v = i < m ? in[i] : 0u;
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < kScanBlock / kWave; ++w) t += s[w];
    sums[blockIdx.x] = t;
  }
}
static __global__ void k_scan_sums(uint32_t *sums, int nb) {
  // single block: serial over chunks of 1024 with a block-wide scan
  __shared__ uint32_t s[kScanBlock];
  uint32_t carry = 0;
  for (int base = 0; base < nb; base += kScanBlock) {
    int i = base + threadIdx.x;
    uint32_t v = i < nb ? sums[i] : 0u;
    s[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < kScanBlock; off <<= 1) {
      uint32_t t = threadIdx.x >= off ? s[threadIdx.x - off] : 0u;
      __syncthreads();
      s[threadIdx.x] += t;
      __syncthreads();
    }
    if (i < nb) sums[i] = carry + s[threadIdx.x] - v;  // exclusive
    __syncthreads();
    carry += s[kScanBlock - 1];
    __syncthreads();
  }
}
// Exclusive scan result to out and to out2 (the scatter cursors).
static __global__ void k_scan_final(uint32_t *__restrict__ in, long long m, const uint32_t *__restrict__ sums,
                             uint32_t *__restrict__ out, uint32_t *__restrict__ out2) {
  __shared__ uint32_t s[kScanBlock];
  long long i = (long long)blockIdx.x * kScanBlock + threadIdx.x;
  uint32_t v = i < m ? in[i] : 0u;
  s[threadIdx.x] = v;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {
    uint32_t t = threadIdx.x >= off ? s[threadIdx.x - off] : 0u;
    __syncthreads();
    s[threadIdx.x] += t;
    __syncthreads();
  }
  if (i < m) {
    const uint32_t r = sums[blockIdx.x] + s[threadIdx.x] - v;
    out[i] = r;
    out2[i] = r;
    in[i] = 0u;  // cleared for the next histogram
  }
}

// Superclusters of each column: sc_info[sc] = (first sorted position, atom
// count) and sc_col[sc] = its column for sc < total, (0, 0) and -1 beyond;
// colsc[col] = first supercluster of column col, colsc[ncols] = total.  One
// block of 1,024 takes the columns in chunks with a running offset.
__device__ __forceinline__ void columns_block(int ncols, int nzb, int n, const uint32_t *start, int nsuper_max,
                                              int2 *__restrict__ sc_info, int *__restrict__ sc_col,
                                              int *__restrict__ colsc) {
  __shared__ int s_w[kScanBlock / kWave];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int carry = 0;
  for (int base = 0; base < ncols; base += kScanBlock) {
    const int col = base + threadIdx.x;
    int cs = 0, cnt = 0;
    if (col < ncols) {
      cs = (int)start[(size_t)col * nzb];
      const int ce = col + 1 < ncols ? (int)start[(size_t)(col + 1) * nzb] : n;
      cnt = ce - cs;
    }
    const int nsc = (cnt + kSuperSize - 1) / kSuperSize;
    const int incl = wave_prefix(nsc);
    if (lane == kWave - 1) s_w[wv] = incl;
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < kScanBlock / kWave; ++w) {
      const int v = s_w[w];
      before += w < wv ? v : 0;
      all += v;
    }
    const int first = carry + before + incl - nsc;
    if (col < ncols) colsc[col] = first;
    for (int q = 0; q < nsc && first + q < nsuper_max; ++q) {
      sc_info[first + q] = make_int2(cs + q * kSuperSize, min(kSuperSize, cnt - q * kSuperSize));
      sc_col[first + q] = col;
    }
    carry += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) colsc[ncols] = carry;
  for (int sc = carry + threadIdx.x; sc < nsuper_max; sc += kScanBlock) {
    sc_info[sc] = make_int2(0, 0);
    sc_col[sc] = -1;
  }
}

static __global__ void __launch_bounds__(kScanBlock) k_columns(int ncols, int nzb, int n, const uint32_t *start,
                                                               int nsuper_max, int2 *__restrict__ sc_info,
                                                               int *__restrict__ sc_col, int *__restrict__ colsc) {
  columns_block(ncols, nzb, n, start, nsuper_max, sc_info, sc_col, colsc);
}

// Exclusive scan of m <= kScanSingleMax counts and the columns'
// superclusters, in one block: bound by latency, so each wave owns a
// contiguous segment, four counts a lane and round, and every round is loaded
// before the first is summed; segment totals are combined across the block (13,000
// bins: 12.3 and 4.8 us in two launches, 6.5 in one).
// Counts and starts are padded to whole groups of four.  The counts are cleared for the next histogram.
constexpr long long kScanSingleMax = 1 << 16;
__device__ __forceinline__ void scan_columns_body(uint32_t *__restrict__ in, int m, uint32_t *out,
                                                  uint32_t *__restrict__ out2, int ncols, int nzb, int n,
                                                  int nsuper_max, int2 *__restrict__ sc_info,
                                                  int *__restrict__ sc_col, int *__restrict__ colsc) {
  constexpr int NW = kScanBlock / kWave, ROUND = 4 * kWave;
  constexpr int RMAX = (int)(kScanSingleMax / (NW * ROUND));
  __shared__ uint32_t s_tot[NW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int seg = ((m + NW - 1) / NW + ROUND - 1) / ROUND * ROUND;  // at most RMAX rounds
  const int b = w * seg;
  uint4 v[RMAX];
#pragma unroll
  for (int r = 0; r < RMAX; ++r) {
    v[r] = make_uint4(0, 0, 0, 0);
    const int i = b + r * ROUND + 4 * lane;
    if (r * ROUND < seg && i < m) v[r] = *reinterpret_cast<const uint4 *>(in + i);  // (m is padded)
  }
  uint32_t t = 0;
#pragma unroll
  for (int r = 0; r < RMAX; ++r) t += v[r].x + v[r].y + v[r].z + v[r].w;
  t = wave_sum(t);
  if (lane == 0) s_tot[w] = t;
  __syncthreads();
  uint32_t base = 0;
  for (int k = 0; k < w; ++k) base += s_tot[k];
#pragma unroll
  for (int r = 0; r < RMAX; ++r) {
    if (r * ROUND >= seg) break;
    const uint32_t own = v[r].x + v[r].y + v[r].z + v[r].w;
    const uint32_t incl = (uint32_t)wave_prefix((int)own);
    const int i = b + r * ROUND + 4 * lane;
    uint4 at;
    at.x = base + incl - own;
    at.y = at.x + v[r].x;
    at.z = at.y + v[r].y;
    at.w = at.z + v[r].z;
    if (i < m) {
      *reinterpret_cast<uint4 *>(out + i) = at;
      *reinterpret_cast<uint4 *>(out2 + i) = at;
      *reinterpret_cast<uint4 *>(in + i) = make_uint4(0, 0, 0, 0);
    }
    base += (uint32_t)__shfl((int)incl, kWave - 1);
  }
  __syncthreads();
  columns_block(ncols, nzb, n, out, nsuper_max, sc_info, sc_col, colsc);
}

static __global__ void __launch_bounds__(kScanBlock) k_scan_columns(uint32_t *__restrict__ in, int m, uint32_t *out,
                                                                    uint32_t *__restrict__ out2, int ncols, int nzb,
                                                                    int n, int nsuper_max, int2 *__restrict__ sc_info,
                                                                    int *__restrict__ sc_col,
                                                                    int *__restrict__ colsc) {
  scan_columns_body(in, m, out, out2, ncols, nzb, n, nsuper_max, sc_info, sc_col, colsc);
}

__device__ __forceinline__ void scatter_body(const int bid_, const int nbk_, int n, const uint32_t *__restrict__ key,
                                             uint32_t *__restrict__ cursor, int *__restrict__ perm) {
  int a = bid_ * blockDim.x + threadIdx.x;
  if (a < n) perm[atomicAdd(&cursor[key[a]], 1u)] = a;
}

static __global__ void k_scatter(int n, const uint32_t *__restrict__ key, uint32_t *__restrict__ cursor,
                          int *__restrict__ perm) {
  scatter_body(blockIdx.x, gridDim.x, n, key, cursor, perm);
}

// The atoms of bin [s0, s1) that belong at positions [p0, p1) when the bin is
// ordered by atom index (the scatter leaves a bin's atoms in any order), one
// wave; bins hold a handful of atoms.
__device__ inline void ranked_bin(const int *__restrict__ in, int s0, int s1, int p0, int p1, int *out) {
  for (int q = s0 + (int)(threadIdx.x & 63); q < s1; q += kWave) {
    const int a = in[q];
    int p = s0;
    for (int r = s0; r < s1; ++r) p += in[r] < a;
    if (p >= p0 && p < p1) out[p - p0] = a;
  }
}

// Ascending bitonic sort of (key, idx) within aligned segments of SEG lanes.
template <int SEG>
__device__ inline void wave_sort(double &key, int &idx) {
  const int lane = threadIdx.x & 63, loc = lane & (SEG - 1);
#pragma unroll
  for (int kk = 2; kk <= SEG; kk <<= 1) {
#pragma unroll
    for (int j = kk >> 1; j > 0; j >>= 1) {
      const double ok = __shfl_xor(key, j);
      const int oi = __shfl_xor(idx, j);
      const bool up = (loc & kk) == 0;
      const bool lower = (lane & j) == 0;
      const bool less = ok < key || (ok == key && oi < idx);
      if ((lower == up) ? less : !less) {
        key = ok;
        idx = oi;
      }
    }
  }
}


// Supercluster boxes are widened by this slack (A) beyond the union of their
// cluster boxes, so that FP32 rounding keeps every cluster box inside.
constexpr float kScSlack = 1e-3f;

// One wave per supercluster (the atoms of sc_info[sc], in z order within
// their column):
//  - split: its atoms (lanes, padding last) are sorted by x, halves by y,
//    quarters by z, so slots 8c..8c+7 form compact clusters; permp (slot ->
//    atom, -1 padding) and slot (atom -> slot) are written;
//  - sorted SoA: coordinates relative to the supercluster origin (the
//    position of the first slot's atom rounded to 1/16 A, in sorg) + charge
//    times qpair (0 when the pair pass carries no Coulomb term),
//    FP64 copy in xs64, LJ type (padding: type -1); xbuild (MD only, else
//    null) receives the positions the list is built from and the inverse masses;
//  - with PME, the atoms' grid records (rec);
//  - bounding boxes (FP32, list building only): per cluster (8-lane groups;
//    ctr.w = real atoms, empty clusters get negative half extents), and per
//    supercluster (the whole wave, widened by kScSlack).
// Thread 0 also clears the mask slot counter for the list build that follows.
// The atoms by bin (in any order within a bin) and the bins' first positions.
struct SortedBins {
  int n;
  long long nbins;
  const uint32_t *key, *start;
  const int *order;
  __device__ int end(uint32_t b) const { return (long long)b + 1 < nbins ? (int)start[b + 1] : n; }
};

template <class R>
__device__ __forceinline__ void split_fill_body(const int bid_, const int nbk_, int nsuper_max,
                                                const int2 *__restrict__ sc_info, const SortedBins &sb,
                                                const double *__restrict__ xwrap, int *__restrict__ permp,
                                                int *__restrict__ slot, const double *__restrict__ q,
                                                const int *__restrict__ type, typename Real4<R>::type *__restrict__ xs,
                                                double4 *__restrict__ xs64, int *__restrict__ ts,
                                                const double *__restrict__ xorig, const double *__restrict__ minv,
                                                double4 *__restrict__ xbuild,
                                                float4 *__restrict__ sorg, float4 *__restrict__ ctr,
                                                float4 *__restrict__ half, float4 *__restrict__ sctr,
                                                float4 *__restrict__ shalf, int *__restrict__ nmaskwork, double qpair,
                                                const PmeParams &pme, PmeSlots<R> rec) {
  const int sc = (bid_ * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (bid_ == 0 && threadIdx.x == 0) *nmaskwork = 0;
  if (sc >= nsuper_max) return;  // whole waves
  const int2 info = sc_info[sc];
  // The sort below orders the supercluster's atoms whatever order they come
  // in; which of a bin's atoms they are matters only for a bin that
  // continues in the previous or the next supercluster.
  __shared__ int s_order[256 / kWave][kSuperSize];
  int *const so = s_order[threadIdx.x >> 6];
  int a = lane < info.y ? sb.order[info.x + lane] : -1;
  if (info.y > 0) {
    const int end = info.x + info.y;
    const uint32_t b = a >= 0 ? sb.key[a] : 0u;
    const uint32_t b0 = __shfl(b, 0), b1 = __shfl(b, info.y - 1);
    so[lane] = a;
    __builtin_amdgcn_wave_barrier();
    const int f0 = (int)sb.start[b0], f1 = sb.end(b0), l0 = (int)sb.start[b1], l1 = sb.end(b1);
    if (f0 < info.x || f1 > end) ranked_bin(sb.order, f0, f1, info.x, end, so);
    if (b1 != b0 && l1 > end) ranked_bin(sb.order, l0, l1, info.x, end, so);
    __builtin_amdgcn_wave_barrier();
    a = so[lane];
  }
  int idx = a < 0 ? 0x7fffffff : a;
  double key = a < 0 ? 1.0e300 : xwrap[3 * a];
  wave_sort<64>(key, idx);
  key = idx == 0x7fffffff ? 1.0e300 : xwrap[3 * idx + 1];
  wave_sort<32>(key, idx);
  key = idx == 0x7fffffff ? 1.0e300 : xwrap[3 * idx + 2];
  wave_sort<16>(key, idx);
  const int s = sc * kSuperSize + lane;
  a = idx == 0x7fffffff ? -1 : idx;
  permp[s] = a;
  if (a >= 0) slot[a] = s;
  // sorted SoA
  double p[3] = {0.0, 0.0, 0.0};
  if (a >= 0)
    for (int k = 0; k < 3; ++k) p[k] = xwrap[3 * a + k];
  const int a0 = __shfl(a, 0);
  double o[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double p0 = __shfl(p[k], 0);
    o[k] = a0 >= 0 ? origin_round(p0) : 0.0;
  }
  if (lane == 0) sorg[sc] = make_float4((float)o[0], (float)o[1], (float)o[2], 0.f);
  typename Real4<R>::type v;
  if (a >= 0) {
    if (xbuild) xbuild[s] = make_double4(xorig[3 * a], xorig[3 * a + 1], xorig[3 * a + 2], minv[a]);
    v.x = (R)(p[0] - o[0]);
    v.y = (R)(p[1] - o[1]);
    v.z = (R)(p[2] - o[2]);
    v.w = (R)(q[a] * qpair);
    ts[s] = type[a];
    xs64[s] = make_double4(p[0], p[1], p[2], q[a]);
  } else {
    v.x = v.y = v.z = v.w = (R)0;
    ts[s] = -1;
    xs64[s] = make_double4(0, 0, 0, 0);
  }
  xs[s] = v;
  if (rec.w) pme_record<R>(pme, rec, s, a >= 0, p, a >= 0 ? q[a] : 0.0);
  // boxes: clusters (8-lane groups), then the supercluster (the wave)
  double lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    lo[k] = a >= 0 ? p[k] : 1e300;
    hi[k] = a >= 0 ? p[k] : -1e300;
  }
  int cnt = a >= 0 ? 1 : 0;
#pragma unroll
  for (int m = 1; m < kClusterSize; m <<= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], m));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], m));
    }
    cnt += __shfl_xor(cnt, m);
  }
  if ((lane & (kClusterSize - 1)) == 0) {
    const int c = s / kClusterSize;
    if (cnt == 0) {
      ctr[c] = make_float4(0, 0, 0, 0);
      half[c] = make_float4(-1, -1, -1, 0);  // empty
    } else {
      ctr[c] = make_float4((float)(0.5 * (lo[0] + hi[0])), (float)(0.5 * (lo[1] + hi[1])),
                           (float)(0.5 * (lo[2] + hi[2])), (float)cnt);
      half[c] = make_float4((float)(0.5 * (hi[0] - lo[0])) * 1.0000005f + 1e-6f,
                            (float)(0.5 * (hi[1] - lo[1])) * 1.0000005f + 1e-6f,
                            (float)(0.5 * (hi[2] - lo[2])) * 1.0000005f + 1e-6f, 0.f);
    }
  }
#pragma unroll
  for (int m = kClusterSize; m < kWave; m <<= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], m));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], m));
    }
    cnt += __shfl_xor(cnt, m);
  }
  if (lane == 0) {
    if (cnt == 0) {
      sctr[sc] = make_float4(0, 0, 0, 0);
      shalf[sc] = make_float4(-1, -1, -1, 0);
    } else {
      sctr[sc] = make_float4((float)(0.5 * (lo[0] + hi[0])), (float)(0.5 * (lo[1] + hi[1])),
                             (float)(0.5 * (lo[2] + hi[2])), (float)cnt);
      shalf[sc] = make_float4((float)(0.5 * (hi[0] - lo[0])) + kScSlack, (float)(0.5 * (hi[1] - lo[1])) + kScSlack,
                              (float)(0.5 * (hi[2] - lo[2])) + kScSlack, 0.f);
    }
  }
}

template <class R>
__global__ void __launch_bounds__(256) k_split_fill(int nsuper_max, const int2 *__restrict__ sc_info,
                                                    SortedBins sb, const double *__restrict__ xwrap,
                                                    int *__restrict__ permp, int *__restrict__ slot,
                                                    const double *__restrict__ q, const int *__restrict__ type,
                                                    typename Real4<R>::type *__restrict__ xs,
                                                    double4 *__restrict__ xs64, int *__restrict__ ts,
                                                    const double *__restrict__ xorig, const double *__restrict__ minv,
                                                double4 *__restrict__ xbuild,
                                                    float4 *__restrict__ sorg, float4 *__restrict__ ctr,
                                                    float4 *__restrict__ half, float4 *__restrict__ sctr,
                                                    float4 *__restrict__ shalf, int *__restrict__ nmaskwork,
                                                    double qpair, PmeParams pme, PmeSlots<R> rec) {
  split_fill_body<R>(blockIdx.x, gridDim.x, nsuper_max, sc_info, sb, xwrap, permp, slot, q, type, xs, xs64, ts,
                     xorig, minv, xbuild, sorg, ctr, half, sctr, shalf, nmaskwork, qpair, pme, rec);
}


// ---------------------------------------------------------------------------
// 2. The cluster list, from the cluster and supercluster boxes.

__device__ inline float bbox_dist2(float4 ca, float4 ha, float4 cb, float4 hb, const float *L) {
  float d2 = 0.f;
  float dc[3] = {fabsf(ca.x - cb.x), fabsf(ca.y - cb.y), fabsf(ca.z - cb.z)};
  float hs[3] = {ha.x + hb.x, ha.y + hb.y, ha.z + hb.z};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float d = fminf(dc[k], L[k] - dc[k]);
    float g = fmaxf(0.f, d - hs[k]);
    d2 += g * g;
  }
  return d2;
}

// Largest squared distance between points of two boxes (minimum image of
// the centers).
__device__ inline float bbox_far2(float4 ca, float4 ha, float4 cb, float4 hb, const float *L) {
  float d2 = 0.f;
  float dc[3] = {fabsf(ca.x - cb.x), fabsf(ca.y - cb.y), fabsf(ca.z - cb.z)};
  float hs[3] = {ha.x + hb.x, ha.y + hb.y, ha.z + hb.z};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float g = fminf(dc[k], L[k] - dc[k]) + hs[k];
    d2 += g * g;
  }
  return d2;
}

// Image shift of a cluster pair: per axis s in {-1, 0, 1} with the j-center
// + s L nearest the i-center, coded (sx+1) | (sy+1) << 2 | (sz+1) << 4.
// bad is set when j-atoms shifted by s could be more than L/2 from an
// i-atom on some axis, allowing each atom to move by up to skin/2 before the
// next build (then the shift is not the minimum image of every pair and the
// pair kernel takes the per-pair image instead).
constexpr int kShiftPerPair = 64;
__device__ inline int entry_shift(float4 ci, float4 hi, float4 cj, float4 hj, const float *L, const float *Linv,
                                  float skin, bool &bad) {
  const float dc[3] = {cj.x - ci.x, cj.y - ci.y, cj.z - ci.z};
  const float hs[3] = {hi.x + hj.x, hi.y + hj.y, hi.z + hj.z};
  int code = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float s = -rintf(dc[k] * Linv[k]);
    const float d = dc[k] + s * L[k];
    bad |= fabsf(d) + hs[k] + skin >= 0.5f * L[k] * 0.999f;
    code |= ((int)s + 1) << (2 * k);
  }
  return code;
}

struct ListParams {
  float L[3];
  float Linv[3];
  float skin;        // MD pair-list buffer (0 outside MD)
  float rlist2;      // (rc_max + margin)^2
  float rlist2_sc;   // supercluster pruning radius^2 (rlist plus slack)
  float rc;          // largest cutoff (work estimate of an entry)
  int ncl;           // clusters
  int nsuper;
  int cap;           // entries per supercluster
  int ncx, ncy;      // x-y column grid of the sort
  int kx, ky;        // column reach: columns within +-kx, +-ky can hold a j-cluster in range
};

// Contiguous runs of the column window c-k..c+k on a ring of n, ascending:
// returns the number of runs (1 or 2) in r.
__device__ inline int col_runs(int c, int k, int n, int r[2][2]) {
  if (2 * k + 1 >= n) {
    r[0][0] = 0;
    r[0][1] = n - 1;
    return 1;
  }
  const int lo = c - k, hi = c + k;
  if (lo < 0) {
    r[0][0] = 0;
    r[0][1] = hi;
    r[1][0] = lo + n;
    r[1][1] = n - 1;
    return 2;
  }
  if (hi >= n) {
    r[0][0] = 0;
    r[0][1] = hi - n;
    r[1][0] = lo;
    r[1][1] = n - 1;
    return 2;
  }
  r[0][0] = lo;
  r[0][1] = hi;
  return 1;
}

// Tests j-cluster cj (< 0: none) against the eight i-clusters of S and
// appends a list entry when at least one is within the list radius.  Called
// by every thread of the block with cj ascending over threads; a block-wide
// prefix count keeps the entries sorted by cj.  Diagonal entries and entries
// with a partial cluster are flagged in s_need (explicit pair masks).
constexpr int kListBlock = 256;
// Work estimate of a list entry for cutting the list into runs, in units of
// about 35 ns of one pair-kernel wave (fitted to per-wave times): kCpCost per
// cluster pair (its 64 candidates: membership and force passes), kMemCost
// times the estimated member fraction of the cluster pair (evaluation; the
// fraction is linear in the cutoff between the boxes' nearest and farthest
// distances), kEntryCost per entry (its dependent loads, the last partial
// batch, j-force sums and atomics), kTileCost on the first entry of a
// supercluster (a wave whose run crosses into it loads its i-atoms and adds
// their forces once more).
constexpr int kCpCost = 8, kMemCost = 9, kEntryCost = 14, kTileCost = 80;

__device__ inline void list_append(const ListParams &q, int S, const float4 *ic, const float4 *ih, int cj,
                                   float4 jc, float4 jh, int4 *__restrict__ entries, unsigned *s_need,
                                   int *__restrict__ overflow, int *s_cnt, int *s_cost, int *__restrict__ ecost, int &total, int &ctotal) {
  constexpr int NW = kListBlock / kWave;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint32_t imask = 0;
  int mc = kEntryCost;  // work estimate of this entry
  bool need = false;
  int shift = -1;         // image shift code of the entry (see entry_shift)
  bool per_pair = false;  // no single shift is the minimum image for every pair
  if (cj >= 0 && jh.x >= 0.f) {
    const bool jpartial = jc.w < (float)kClusterSize;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int ci = S * 8 + c;
      if (ih[c].x < 0.f || ci > cj) continue;
      const float d2 = bbox_dist2(ic[c], ih[c], jc, jh, q.L);
      if (d2 <= q.rlist2) {
        imask |= 1u << c;
        {
          const float dn = sqrtf(d2), df = sqrtf(bbox_far2(ic[c], ih[c], jc, jh, q.L));
          const float frac = fminf(1.f, fmaxf(0.f, (q.rc - dn) / fmaxf(df - dn, 1e-3f)));
          mc += kCpCost + (int)(kMemCost * frac + 0.5f);
        }
        const bool ipartial = ic[c].w < (float)kClusterSize;
        if (ci == cj || ipartial || jpartial) need = true;
        const int code = entry_shift(ic[c], ih[c], jc, jh, q.L, q.Linv, q.skin, per_pair);
        if (shift < 0) shift = code;
        per_pair |= code != shift;
      }
    }
  }
  const unsigned long long act = __ballot(imask != 0);
  // inclusive prefix of the work over this call's entries (lanes in order)
  int wc = imask != 0 ? mc : 0;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int v = __shfl_up(wc, off);
    if (lane >= off) wc += v;
  }
  if (lane == 0) s_cnt[wv] = __popcll(act);
  if (lane == kWave - 1) s_cost[wv] = wc;
  __syncthreads();
  int before = 0, all = 0, cbefore = 0, call = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const int c = s_cnt[w], k = s_cost[w];
    before += w < wv ? c : 0;
    all += c;
    cbefore += w < wv ? k : 0;
    call += k;
  }
  __syncthreads();
  const int e = total + before + __popcll(act & ((1ull << lane) - 1ull));
  if (imask != 0) {
    if (e < q.cap) {
      if (need) atomicOr(&s_need[e >> 5], 1u << (e & 31));
      entries[(size_t)S * q.cap + e] = make_int4(cj, (int)imask, -1, per_pair ? kShiftPerPair : shift);
      ecost[(size_t)S * q.cap + e] = kTileCost + ctotal + cbefore + wc;  // the tile cost counts from entry 0
    } else {
      atomicExch(overflow, 1);
    }
  }
  total += all;
  ctotal += call;
}

// Masks of one supercluster made together, in LDS.
constexpr int kMaskBatch = 64;
struct MaskArgs {
  const int *perm, *slot, *eptr;
  const int2 *elist;
  unsigned short *masks;
  int maxmaskwork;
};
inline size_t list_lds_bytes(int cap) { return 8 * (size_t)((cap + 31) / 32); }

// Cluster-pair list of supercluster S (one block each).  Superclusters are
// numbered column by column (x-major, then y, then z inside a column), so the
// j-superclusters of the columns within the column reach of S's column form
// at most four ascending index ranges per column row x.  Each range is
// pruned by supercluster boxes (a conservative test: a cluster box lies in
// its supercluster box), the survivors' clusters are tested against the
// eight i-clusters of S, and entries are appended in ascending cj.  Only
// cj >= 8S is listed, so each cluster pair appears once.  The work per S is
// bounded by the neighbourhood, independent of the system size.
//
// The block then gives the entries of S that need them their explicit masks
// (diagonal entries, entries with a partial cluster or an excluded or scaled
// pair).  Mask slot w holds one 16-bit word per lane l = tj*8 + ti of the
// pair kernel: bit c set when i = slot 8ci+ti (ci = 8S + c, c in the entry's
// mask) and j = slot 8cj+tj are real atoms, i precedes j within a shared
// cluster, and the pair is not FULL-excluded; bit 8 + c marks MODIFIED.  The
// entry's mask field becomes w.  The excluded pairs of the supercluster's
// atoms look up their entry (sorted by j-cluster); a pair whose clusters are
// not listed is beyond the list radius and never evaluated.  Bound by the
// chains of dependent loads of a block, of which eight fit a CU.  With the
// masks in launches of their own (a thread per excluded pair that claimed its
// entry by compare-and-swap, a wave per mask that searched every pair's
// exclusions) 26,000 atoms took 30 + 12 + 20 us and 1,000,000 atoms 283 + 174 +
// 387; in one 36 to 45 and 287.
__device__ __forceinline__ void build_list_body(const int bid_, const int nbk_, const ListParams &q,
                                                const int *__restrict__ sc_col, const int *__restrict__ colsc,
                                                const float4 *__restrict__ sctr, const float4 *__restrict__ shalf,
                                                const float4 *__restrict__ ctr, const float4 *__restrict__ half,
                                                int4 *entries, int *__restrict__ count, int *ecost,
                                                int *__restrict__ cost_out, const MaskArgs &ma,
                                                int *__restrict__ nmaskwork, int *__restrict__ overflow) {
  // bit e: entry e needs a mask; flags before each word (list_lds_bytes)
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int words = (q.cap + 31) / 32;
  unsigned *const s_need = reinterpret_cast<unsigned *>(smem_raw);
  int *const s_pre = reinterpret_cast<int *>(smem_raw) + words;
  __shared__ unsigned s_mask[kMaskBatch][kWave / 2];  // two 16-bit words each
  __shared__ int2 s_ent[kMaskBatch];                  // j-cluster, i-clusters
  __shared__ int s_wbase, s_nmask;
  constexpr int NW = kListBlock / kWave;
  constexpr int kScPerBatch = kListBlock / kClusterSize;
  __shared__ int s_cnt[NW];
  __shared__ int s_cost[NW];
  __shared__ int s_sc[kListBlock];
  __shared__ int s_ra[kWave], s_rpre[kWave], s_rtot;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int S = bid_;
  const int col = sc_col[S];
  if (col < 0) {  // past the last occupied supercluster: no atoms
    if (threadIdx.x == 0) {
      count[S] = 0;
      cost_out[S] = 0;
    }
    return;
  }
  // the boxes of S in LDS (read by every lane at once): as scalars they spill
  __shared__ float4 ic[8], ih[8];
  if (threadIdx.x < 8) ic[threadIdx.x] = ctr[S * 8 + threadIdx.x];
  if (threadIdx.x >= 64 && threadIdx.x < 72) ih[threadIdx.x - 64] = half[S * 8 + threadIdx.x - 64];
  const float4 Sc = sctr[S], Sh = shalf[S];
  int xr[2][2], yr[2][2];
  const int cx = col / q.ncy, cy = col - cx * q.ncy;
  const int nxr = col_runs(cx, q.kx, q.ncx, xr), nyr = col_runs(cy, q.ky, q.ncy, yr);
  // the candidate j-superclusters form index ranges, one per (x, y run) in
  // ascending order; they are enumerated as one flat sequence (64 ranges at
  // a time) so that each pass of 256 threads tests 256 candidates
  const int nx0 = xr[0][1] - xr[0][0] + 1, nxt = nx0 + (nxr > 1 ? xr[1][1] - xr[1][0] + 1 : 0);
  const int R = nxt * nyr;
  for (int w = threadIdx.x; w < words; w += kListBlock) s_need[w] = 0u;
  int total = 0;   // block-uniform
  int ctotal = 0;  // block-uniform work of the entries so far
  for (int g0 = 0; g0 < R; g0 += kWave) {
    const int nrg = min(kWave, R - g0);
    __syncthreads();  // every thread has read the previous group's ranges
    if (threadIdx.x < kWave) {
      const int r = g0 + lane;
      int a = 0, len = 0;
      if (r < R) {
        const int xi = r / nyr, ry = r - xi * nyr;
        const int x = xi < nx0 ? xr[0][0] + xi : xr[1][0] + (xi - nx0);
        a = max(S, colsc[x * q.ncy + (ry ? yr[1][0] : yr[0][0])]);
        len = max(0, colsc[x * q.ncy + (ry ? yr[1][1] : yr[0][1]) + 1] - a);
      }
      int incl = len;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const int y = __shfl_up(incl, off);
        if (lane >= off) incl += y;
      }
      s_ra[lane] = a;
      s_rpre[lane] = incl - len;
      if (lane == kWave - 1) s_rtot = incl;
    }
    __syncthreads();
    const int T = s_rtot;
    for (int base = 0; base < T; base += kListBlock) {
      const int k = base + threadIdx.x;
      bool pass = false;
      int sc = 0;
      if (k < T) {
        // range of candidate k: the last range starting at or before k
        int lo = 0, hi = nrg - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (s_rpre[mid] <= k)
            lo = mid;
          else
            hi = mid - 1;
        }
        sc = s_ra[lo] + (k - s_rpre[lo]);
        const float4 jh = shalf[sc];
        pass = jh.x >= 0.f && bbox_dist2(Sc, Sh, sctr[sc], jh, q.L) <= q.rlist2_sc;
      }
      const unsigned long long act = __ballot(pass);
      if (lane == 0) s_cnt[wv] = __popcll(act);
      __syncthreads();
      int before = 0, npass = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const int c = s_cnt[w];
        before += w < wv ? c : 0;
        npass += c;
      }
      if (pass) s_sc[before + __popcll(act & ((1ull << lane) - 1ull))] = sc;
      __syncthreads();
      for (int k0 = 0; k0 < npass; k0 += kScPerBatch) {
        const int kk = k0 + (int)(threadIdx.x / kClusterSize);
        int cj = -1;
        float4 jc = make_float4(0, 0, 0, 0), jh = make_float4(-1, -1, -1, 0);
        if (kk < npass) {
          cj = s_sc[kk] * kClusterSize + (int)(threadIdx.x & (kClusterSize - 1));
          jc = ctr[cj];
          jh = half[cj];
        }
        list_append(q, S, ic, ih, cj, jc, jh, entries, s_need, overflow, s_cnt, s_cost, ecost, total, ctotal);
      }
      __syncthreads();  // s_sc and s_cnt are rewritten by the next pass
    }
  }
  __syncthreads();  // entries, costs and flags of every thread
  const int n = total < q.cap ? total : q.cap;
  int4 *const ep = entries + (size_t)S * q.cap;
  if (threadIdx.x == 0) {
    count[S] = n;
    cost_out[S] = n > 0 ? ecost[(size_t)S * q.cap + n - 1] : 0;
  }
  // excluded pairs, four threads an atom: the entry (-1: none, or another
  // supercluster's pair), the j-slot and the class of the thread's pair k
  constexpr int TPA = kListBlock / kSuperSize, KEPT = 2;
  const int si = S * kSuperSize + (int)threadIdx.x / TPA;
  const int ai = ma.perm[si];
  const int x0 = (ai >= 0 ? ma.eptr[ai] : 0) + (int)threadIdx.x % TPA, x1 = ai >= 0 ? ma.eptr[ai + 1] : 0;
  auto excluded = [&](int k) {
    const int2 x = k < x1 ? ma.elist[k] : make_int2(-1, 0);
    if (x.x < 0) return make_int3(-1, 0, 0);
    const int sj = ma.slot[x.x];
    const int ci = si / kClusterSize, cj = sj / kClusterSize;
    if (cj < ci || (cj == ci && sj < si)) return make_int3(-1, 0, 0);
    int lo = 0, hi = n - 1;
    while (lo <= hi) {
      const int m = (lo + hi) >> 1;
      const int v = ep[m].x;
      if (v == cj) return make_int3(m, sj, x.y);
      if (v < cj)
        lo = m + 1;
      else
        hi = m - 1;
    }
    return make_int3(-1, 0, 0);
  };
  int3 kept[KEPT];  // most atoms have no more
#pragma unroll
  for (int u = 0; u < KEPT; ++u) kept[u] = excluded(x0 + u * TPA);
  auto each_excluded = [&](auto f) {
#pragma unroll
    for (int u = 0; u < KEPT; ++u)
      if (kept[u].x >= 0) f(kept[u]);
    for (int k = x0 + KEPT * TPA; k < x1; k += TPA) {
      const int3 v = excluded(k);
      if (v.x >= 0) f(v);
    }
  };
  each_excluded([&](int3 v) { atomicOr(&s_need[v.x >> 5], 1u << (v.x & 31)); });
  __syncthreads();
  // mask slots in entry order
  if (wv == 0) {
    int carry = 0;
    for (int w0 = 0; w0 * 32 < n; w0 += kWave) {
      const int c = (w0 + lane) * 32 < n ? __popc(s_need[w0 + lane]) : 0;
      const int incl = wave_prefix(c);
      if (w0 + lane < words) s_pre[w0 + lane] = carry + incl - c;
      carry += __shfl(incl, kWave - 1);
    }
    if (lane == 0) {
      const int w0 = carry ? atomicAdd(nmaskwork, carry) : 0;
      const bool fits = w0 + carry <= ma.maxmaskwork;
      if (!fits) atomicExch(overflow, 1);
      s_wbase = w0;
      s_nmask = fits ? carry : 0;
    }
  }
  __syncthreads();
  const int nmask = s_nmask;
  auto rank = [&](int e) { return s_pre[e >> 5] + __popc(s_need[e >> 5] & ((1u << (e & 31)) - 1u)); };
  const int ti = lane & 7, tj = lane >> 3;
  unsigned ireal = 0;  // i-atoms 8 c + ti
#pragma unroll
  for (int c = 0; c < 8; ++c) ireal |= ma.perm[S * kSuperSize + c * kClusterSize + ti] >= 0 ? 1u << c : 0u;
  for (int m0 = 0; m0 < nmask; m0 += kMaskBatch) {
    const int mn = min(kMaskBatch, nmask - m0);
    for (int e = threadIdx.x; e < n; e += kListBlock) {
      if (!(s_need[e >> 5] >> (e & 31) & 1u)) continue;
      const int k = rank(e) - m0;
      if (k < 0 || k >= mn) continue;
      s_ent[k] = make_int2(ep[e].x, ep[e].y);
      ep[e].z = s_wbase + m0 + k;
    }
    __syncthreads();
    // without exclusions
    for (int k = wv; k < mn; k += NW) {
      const int cj = s_ent[k].x, d = cj - S * 8;  // (only clusters from 8 S on are listed)
      unsigned bits = s_ent[k].y & ireal;
      if (ma.perm[cj * kClusterSize + tj] < 0) bits = 0;
      if (d < 8 && ti >= tj) bits &= ~(1u << d);
      const unsigned other = __shfl_xor(bits, 1);
      if (!(lane & 1)) s_mask[k][lane >> 1] = bits | other << 16;
    }
    __syncthreads();
    each_excluded([&](int3 v) {
      const int k = rank(v.x) - m0;
      if (k < 0 || k >= mn) return;
      const int c = (si / kClusterSize) & 7, l = (v.y & 7) * 8 + (si & 7), sh = 16 * (l & 1);
      if (v.z == 1)
        atomicAnd(&s_mask[k][l >> 1], ~((1u << c) << sh));
      else if (v.z == 2 && (s_ent[k].y & (1 << c)))
        atomicOr(&s_mask[k][l >> 1], (256u << c) << sh);
    });
    __syncthreads();
    unsigned *const out = reinterpret_cast<unsigned *>(ma.masks) + (size_t)(s_wbase + m0) * (kWave / 2);
    for (int k = threadIdx.x; k < mn * (kWave / 2); k += kListBlock) out[k] = (&s_mask[0][0])[k];
    __syncthreads();  // the next batch overwrites s_mask and s_ent
  }
}

static __global__ void __launch_bounds__(kListBlock) k_build_list(ListParams q, const int *__restrict__ sc_col,
                                                           const int *__restrict__ colsc,
                                                           const float4 *__restrict__ sctr,
                                                           const float4 *__restrict__ shalf,
                                                           const float4 *__restrict__ ctr,
                                                           const float4 *__restrict__ half, int4 *entries,
                                                           int *__restrict__ count, int *ecost,
                                                           int *__restrict__ cost_out, MaskArgs ma,
                                                           int *__restrict__ nmaskwork, int *__restrict__ overflow) {
  build_list_body(blockIdx.x, gridDim.x, q, sc_col, colsc, sctr, shalf, ctr, half, entries, count, ecost, cost_out,
                  ma, nmaskwork, overflow);
}

// Binary search of b in the sorted exclusion partners of a (original indices).
__device__ inline int excl_class(const int *__restrict__ eptr, const int2 *__restrict__ elist, int a, int b) {
  int lo = eptr[a], hi = eptr[a + 1] - 1;
  while (lo <= hi) {
    int mid = (lo + hi) >> 1;
    int v = elist[mid].x;
    if (v == b) return elist[mid].y;
    if (v < b)
      lo = mid + 1;
    else
      hi = mid - 1;
  }
  return 0;
}

// Run schedule: the list entries of all superclusters, in supercluster
// order, are cut into nruns contiguous runs of equal estimated work (the
// work estimates of k_build_list: per supercluster, and as an inclusive
// prefix over its entries); nruns, a multiple of cut.min_runs set by C, the
// total, or fewer (RunCut), depends only on the list.  Run w starts in supercluster runs[w].x
// at entry runs[w].y, where the global work prefix first exceeds b_w = floor(w C / nruns), and ends where
// run w + 1 starts; runs[nruns] is the end of the last supercluster with
// entries.  The tile of run w in supercluster S, which may be empty at the
// run's end, is number w + S: numbers rise by one from tile to tile, also from a
// run's last to the next run's first.
// One launch: each block adds up the work ahead of its superclusters and in
// total for itself (a table of 4 bytes per supercluster), its waves take one
// supercluster after the other, and each entry places the run boundaries
// that fall in its work interval.  26,000 atoms 23 us in three launches (two of
// them one block), 9.7 in one; 1,000,000 atoms 130 and 28.
constexpr int kRunsBlock = 1024;
__device__ __forceinline__ void runs_body(const int bid_, const int nbk_, int nsuper, const int *__restrict__ count,
                                          const int *__restrict__ cost, const int *__restrict__ ecost, int cap,
                                          RunCut cut, int2 *__restrict__ runs,
                                          int *__restrict__ ntiles) {
  constexpr int NW = kRunsBlock / kWave;
  __shared__ long long s_c[2][NW];
  __shared__ int s_last[NW];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int c0 = (int)((long long)bid_ * nsuper / nbk_), c1 = (int)((long long)(bid_ + 1) * nsuper / nbk_);
  long long before = 0, C = 0;
  int last = -1;
  for (int S = threadIdx.x; S < nsuper; S += kRunsBlock) {
    const int c = cost[S];
    C += c;
    before += S < c0 ? c : 0;
    if (c > 0) last = S;
  }
  before = wave_sum(before);
  C = wave_sum(C);
  last = wave_max(last);
  if (lane == 0) {
    s_c[0][wv] = before;
    s_c[1][wv] = C;
    s_last[wv] = last;
  }
  __syncthreads();
  before = C = 0;
  for (int k = 0; k < NW; ++k) {
    before += s_c[0][k];
    C += s_c[1][k];
    last = max(last, s_last[k]);
  }
  const int min_runs = cut.min_runs;
  const long long per = (long long)min_runs * kRunCost;
  const long long k = (C + per - 1) / per;
  int nruns = min_runs * (int)(k < 1 ? 1 : (k > kMaxRuns / min_runs ? kMaxRuns / min_runs : k));
  {
    // whole waves' worth of 64 runs of at least cut.least units
    long long r = (C + cut.least - 1) / cut.least;
    if (r > cut.few) r = max((long long)cut.few, (C + cut.least_many - 1) / cut.least_many);
    nruns = (int)min((long long)nruns, max(64ll, (r + 63) / 64 * 64));
  }
  if (bid_ == 0) {
    // an empty list: every run is empty
    for (int w = C > 0 ? nruns + threadIdx.x : threadIdx.x; w < nruns; w += kRunsBlock) runs[w] = make_int2(0, 0);
    if (threadIdx.x == 0) {
      runs[0] = make_int2(0, 0);
      runs[nruns] = make_int2(last + 1, 0);
      ntiles[0] = nruns + last + 1;
      ntiles[2] = nruns;
    }
  }
  if (C <= 0) return;
  const int w0 = c0 + (int)((long long)wv * (c1 - c0) / NW), w1 = c0 + (int)((long long)(wv + 1) * (c1 - c0) / NW);
  long long base = 0;
  for (int S = c0 + lane; S < w0; S += kWave) base += cost[S];
  base = before + wave_sum(base);
  const double inv = 1.0 / (double)C;
  // first run w with floor(w C / nruns) >= x, i.e. ceil(x nruns / C)
  auto first_run = [&](long long x) {
    // q is off by one at most (the product stays below 2^53)
    const long long y = x * nruns, q = (long long)((double)y * inv), r = y - q * C;
    return (int)min(q + (r > 0 ? 1 : 0) + (r > C ? 1 : 0) - (r <= -C ? 1 : 0), (long long)nruns);
  };
  for (int S = w0; S < w1; ++S) {
    const int n = count[S];
    const int *ec = ecost + (size_t)S * cap;
    int carry = first_run(base);
    constexpr int AHEAD = 8;  // rounds whose loads are in flight together
    for (int e0 = 0; e0 < n; e0 += AHEAD * kWave) {
      int hi[AHEAD];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int e = e0 + u * kWave + lane;
        hi[u] = e < n ? ec[e] : 0;
      }
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int e = e0 + u * kWave + lane;
        if (e0 + u * kWave >= n) break;
        const int rb = first_run(base + hi[u]);
        int ra = __shfl_up(rb, 1);
        if (lane == 0) ra = carry;
        carry = __shfl(rb, kWave - 1);
        // runs w in [1, nruns) with lo <= floor(w C / nruns) < hi
        if (e < n)
          for (int w = max(ra, 1); w < rb; ++w) runs[w] = make_int2(S, e);
      }
    }
    base += cost[S];
  }
}

static __global__ void __launch_bounds__(kRunsBlock) k_runs(int nsuper, const int *__restrict__ count,
                                                            const int *__restrict__ cost,
                                                            const int *__restrict__ ecost, int cap, RunCut cut,
                                                            int2 *__restrict__ runs, int *__restrict__ ntiles) {
  runs_body(blockIdx.x, gridDim.x, nsuper, count, cost, ecost, cap, cut, runs, ntiles);
}

// ---------------------------------------------------------------------------
// 3. Pair kernel: LJ + Coulomb (cutoff or PME real space) with switching.
//
// Wavefront layout: lane = 8*tj + ti.  A work tile is the part of a run in
// one i-supercluster S.  Each entry names one j-cluster (8 atoms,
// lane tj holds atom tj) and an 8-bit mask of the i-clusters of S it is in
// range of; for every set i-cluster c the 64 lanes evaluate the 8x8 atom
// pairs (8c+ti, tj).  i-forces stay in registers for the whole tile, j-forces
// are summed over the 8 i-lanes with DPP and added once per entry.
//
// Membership is decided exactly: a pair whose FP32/FP64 r^2 lies within
// `guard` of a cutoff^2 is not evaluated here but recorded, and the
// boundary-pair pass of k_fixups re-tests it in FP64 with the reference's
// operation order on the original coordinates before evaluating it.

__device__ inline float fast_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
// FP64: the unit's estimate (about 23 bits) and one step of third order, the
// rounding of x y included.  Errors over 4 M arguments from 2^-8 to 2^8, in
// units of the last place (1 / sqrt(x), 1 / x and exp in brackets): 0.5005
// (1.4907), fast_rcp 0.5000 (0.5000), fast_exp 0.880 (0.879).  With the three
// 26,000 atoms took 221 -> 210 us a launch, 93,000 with cutoffs 375 -> 364.
__device__ inline double fast_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double h = x * y, l = fma(x, y, -h);
  const double e = fma(-l, y, fma(-h, y, 1.0));
  const double r = fma(y * e, fma(0.375, e, 0.5), y);
  return x > 0.0 ? r : y;  // (coincident atoms: infinite, as before)
}
__device__ inline float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ inline double fast_rcp(double x) {  // 0 < x < infinity, normal
  const double y = __builtin_amdgcn_rcp(x), e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}
__device__ inline float fast_exp(float x) { return __expf(x); }
// x <= 0: x = n ln 2 + r (Cody and Waite's reduction), the Taylor series of
// e^r to r^13 (|r| <= 0.35: the rest is below 5e-18), scaled by 2^n.
__device__ inline double fast_exp(double x) {
  const double n = rint(x * 1.4426950408889634);
  double r = fma(n, -0x1.62e42fefa39efp-1, x);
  r = fma(n, -0x1.abc9e3b39803fp-56, r);
  double p = 1.0 / 6227020800.0;
  p = fma(p, r, 1.0 / 479001600.0);
  p = fma(p, r, 1.0 / 39916800.0);
  p = fma(p, r, 1.0 / 3628800.0);
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return ldexp(p, (int)n);
}
__device__ inline float fast_rint(float x) { return rintf(x); }
__device__ inline double fast_rint(double x) { return rint(x); }

template <class R>
__device__ inline R poly5(R ar) {
  // Abramowitz & Stegun 7.1.26 (reference: protomol/base/MathUtilities.cpp:39-49)
  const R E1 = (R)0.254829592, E2 = (R)-0.284496736, E3 = (R)1.421413741, E4 = (R)-1.453152027,
          E5 = (R)1.061405429, PP = (R)0.3275911;
  R t = fast_rcp((R)1 + PP * ar);
  return t * (E1 + t * (E2 + t * (E3 + t * (E4 + t * E5))));
}

template <bool MIXED>
struct AccT;
template <>
struct AccT<false> {
  using type = double;
  __device__ static void add(double *p, double v) { unsafeAtomicAdd(p, v); }
};
template <>
struct AccT<true> {
  using type = unsigned long long;
  __device__ static void add(unsigned long long *p, float v) {
    long long q = __float2ll_rn(v * 4294967296.0f);
    atomicAdd(p, (unsigned long long)q);
  }
  __device__ static void add(unsigned long long *p, double v) {
    long long q = __double2ll_rn(v * kForceScale);
    atomicAdd(p, (unsigned long long)q);
  }
};

// Switching function value and (1/r) dS/dr at r2 (in range), branch-free.
// KIND = SW_ANY selects at run time from `kind`.
constexpr int SW_ANY = 9;
template <int KIND, class R>
__device__ inline void switch_val(int kind, const SwR<R> &s, R r2, R rinv, R &val, R &der) {
  const int k = KIND == SW_ANY ? kind : KIND;
  if (k == SW_C2) {
    // C2SwitchingFunction.h:42-53: 1 below r_on, polynomial on [r_on, rc]
    R c2 = s.rc2 - r2;
    c2 = c2 > (R)0 ? c2 : (R)0;
    const R c4 = c2 * (s.s2 + (R)2 * r2);
    const bool on = r2 >= s.on2;
    val = on ? s.s1 * (c2 * c4) : (R)1;
    der = on ? s.s3 * (c2 * c2 - c4) : (R)0;
  } else if (k == SW_C1) {
    // C1SwitchingFunction.h:41-50
    const R dist = r2 * rinv;
    val = (R)1 - dist * (s.c15_1 - r2 * s.c05_3);
    der = -s.c15_1 * rinv + dist * s.c15_3;
  } else {
    val = (R)1;
    der = (R)0;
  }
}

// One pair's energies and scalar force (F = f * d), given membership flags.
template <int COUL, int LJSW, int CSW, class R>
__device__ inline void pair_eval(const PairParams &pp, const SwR<R> &sl, const SwR<R> &sc, R alpha, R a2pi, R csf,
                                 R r2, R qq, R A, R B, bool in_lj, bool in_c, R &elj, R &eco, R &fr) {
  const R r2s = (in_lj || in_c) ? r2 : (R)1;
  const R rinv = fast_rsqrt(r2s);
  const R rinv2 = rinv * rinv;
  fr = (R)0;
  elj = (R)0;
  eco = (R)0;
  if (LJSW != SW_NONE) {
    // LennardJonesForce.h:28-60
    const R r6 = rinv2 * rinv2 * rinv2;
    const R r6B = B * r6, r12A = A * r6 * r6;
    R e = r12A - r6B;
    R f = ((R)12 * r12A - (R)6 * r6B) * rinv2;
    R sv, sd;
    switch_val<LJSW, R>(pp.lj.kind, sl, r2s, rinv, sv, sd);
    f = f * sv - e * sd;
    e = e * sv;
    elj = in_lj ? e : (R)0;
    fr += in_lj ? f : (R)0;
  }
  if (COUL == COUL_CUTOFF) {
    // CoulombForce.h:29-40
    R e = qq * rinv;
    R f = e * rinv2;
    if constexpr (CSW != SW_CUTOFF) {  // a plain cutoff switches nothing (1 and 0)
      R sv, sd;
      switch_val<CSW, R>(pp.co.kind, sc, r2s, rinv, sv, sd);
      f = f * sv - e * sd;
      e = e * sv;
    }
    eco = in_c ? e : (R)0;
    fr += in_c ? f : (R)0;
  } else if (COUL == COUL_PME) {
    // NonbondedPMEwaldSystemForce.h:657-683 (poly5 form)
    const R r = r2s * rinv;
    const R ar = alpha * r;
    const R ex = qq * fast_exp(-ar * ar);
    R e = poly5<R>(ar) * ex * rinv;
    R f = (e + a2pi * ex) * rinv2;
    if constexpr (CSW != SW_CUTOFF) {
      R sv, sd;
      switch_val<CSW, R>(pp.co.kind, sc, r2s, rinv, sv, sd);
      f = f * sv - e * sd;
      e = e * sv;
    }
    eco = in_c ? e : (R)0;
    fr += in_c ? f : (R)0;
  }
}

// Sum over the 8 lanes of a cluster group (lanes differing in bits 0..2).
__device__ inline float group8_sum(float v) {
  // quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));
  return v;
}
template <int CTRL>
__device__ inline double dpp_of(double v) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true),
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true));
}
__device__ inline double group8_sum(double v) {
  v += dpp_of<0xB1>(v);
  v += dpp_of<0x4E>(v);
  v += dpp_of<0x141>(v);
  return v;
}
struct PairOut {
  double *energy;            // [2 * ntiles]: per tile (coulomb, lj); int64 fixed point 2^-32 in the mixed form
  long long *npairs;         // [ntiles] when stats
  unsigned long long *hash;  // [ntiles]
  int2 *border;              // recorded boundary pairs (sorted slots i, j)
  int *nborder;
  int maxborder;
  int *overflow;
  unsigned long long *border_acc;  // [4] boundary-pair energies and stats, cleared here
  __device__ void clear(int t, bool stats) const {
    energy[2 * t] = energy[2 * t + 1] = 0.0;
    if (stats) {
      npairs[t] = 0;
      hash[t] = 0;
    }
  }
};

// A wave's way through runs w .. wstop - 1, tile by tile (wave-uniform).
struct RunWalk {
  int w, wstop, t = 0;    // next run; the tile's number
  int S = 0, e0 = 0;      // the tile: supercluster, first entry
  int Send = -1, eend = 0;  // the run's end
  __device__ RunWalk(int r0, int r1) : w(r0), wstop(r1) {}
  __device__ bool run_done() const { return S > Send; }
  __device__ void next_run(const int2 *__restrict__ runs) {
    const int2 a = runs[w], b = runs[w + 1];
    S = __builtin_amdgcn_readfirstlane(a.x);
    e0 = __builtin_amdgcn_readfirstlane(a.y);
    Send = __builtin_amdgcn_readfirstlane(b.x);
    eend = __builtin_amdgcn_readfirstlane(b.y);
    t = w + S;
    ++w;
  }
  __device__ int tile_end(const int *__restrict__ count) const {
    return S == Send ? eend : __builtin_amdgcn_readfirstlane(count[S]);
  }
  __device__ void next_tile() {
    ++S;
    ++t;
    e0 = 0;
  }
};

// r^2 given to an excluded candidate pair: beyond every cutoff, band and
// list radius
template <class R>
constexpr R kFarR2 = (R)1e30;
constexpr int kPairPlain = 0, kPairPrune = 1, kPairStats = 2;  // k_pair MODE

// Fixed-point (mixed form) or FP64 sums of a wave's own i-atom forces and of
// its pair energies.
template <bool MIXED>
struct WaveAcc;
template <>
struct WaveAcc<true> {
  using T = long long;
  __device__ static T of(float v) { return __float2ll_rn(v * 4294967296.0f); }
  __device__ static void add(unsigned long long *p, T v) { atomicAdd(p, (unsigned long long)v); }
  __device__ static double energy_bits(T v) { return __longlong_as_double(v); }
};
template <>
struct WaveAcc<false> {
  using T = double;
  __device__ static T of(double v) { return v; }
  __device__ static void add(double *p, T v) { unsafeAtomicAdd(p, v); }
  __device__ static double energy_bits(T v) { return v; }
};

// Box edges in the kernel's type, split as hi + lo (see PairParams::Lhi).
template <class R>
struct EdgesR {
  R hi[3], lo[3], inv[3];
  __device__ void load(const PairParams &pp) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      hi[k] = (R)pp.Lhi[k];
      lo[k] = (R)pp.Llo[k];
      inv[k] = (R)pp.box.Linv[k];
    }
  }
  // image k of a difference: d - k (hi + lo), hi exact
  __device__ R image(R d, int ax) const {
    const R k = fast_rint(d * inv[ax]);
    return (d - k * hi[ax]) - k * lo[ax];
  }
};

// Cluster-pair kernel.  Every lane of a cluster pair (i = 8c+ti of the
// supercluster, j = lane tj of the entry's j-cluster) computes r^2 and its
// membership; where any lane is a member all are evaluated and the others'
// results selected away: no queue, no force slots.  A tile's i-atoms sit in
// LDS, its i-forces in registers, the constants in scalar registers; the
// j-forces are summed over the 8 i-lanes with DPP and added once per entry.
// Deterministic sums: a tile (a run's part of one supercluster's list) is the
// same whichever wave takes it, and at its end lane 8 c + ti sums its i-atom's
// eight partials in a fixed order and adds the sum to the force array, in
// fixed point in the mixed form, whose FP32 pair energies of a tile go to
// fixed point too.  So the mixed form's forces and energies do not depend on
// the schedule, the grid or the device.
//
// MODE kPairPrune (the first pass after a list build): cluster pairs without
// a candidate pair inside the list radius are dropped from the entries'
// masks (through entries_w, which aliases entries; each entry is read and
// written by the one wave that takes it).  MODE kPairStats: the pass also
// counts the in-cutoff pairs and sums their hashes.
//
// Bound by VALU issue.  Before, the member pairs (about two fifths of the lanes)
// were packed into an LDS queue and evaluated in full batches, which cost as
// much issue time as it saved, and LDS round trips and scalar work on top; in
// FP64 its 59 KB of LDS a block also left two waves per SIMD.
// One launch alone, before and after, skin 1.5 / 1.0 / 1.2 A.  Mixed: 26,000
// atoms 78.8 -> 60.1 us (VALU instructions 29.0 -> 26.6 M, scalar 16.0 -> 6.7 M,
// LDS 3.0 -> 0.9 M), 9,400 atoms 31.0 -> 27.3, 1,000,000 atoms 1.63 -> 1.07 ms;
// unequal cutoffs, 46,000 atoms 126 -> 97 us.  FP64: 26,000 atoms
// with PME 210 -> 109 us, 93,000 with cutoffs 364 -> 173; three blocks per CU
// (151 VGPRs; at 128 the PME form spills 118), with cutoffs four.
// Mixed, 72 VGPRs and 8 KB of LDS a block would take six blocks per CU (55.7 us
// and 0.93 ms alone), but then the PME passes beside it starve and a step takes
// longer (26,000 atoms 124 -> 136 us): four, which leave them half the
// registers.

// e^(-alpha^2 r^2) from DirectC::ke r^2.
__device__ inline float gauss(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ inline double gauss(double x) { return fast_exp(x); }

// Energies and scalar force (F = f d) of one member pair; il, ic: in range of
// the LJ and the Coulomb cutoff.
template <int COUL, int LJSW, int CSW, class R>
__device__ __forceinline__ void direct_eval(const DirectC<R> &k, R r2, R qq, R A, R B, R &elj, R &eco, R &flj,
                                            R &fco) {
  const R rinv = fast_rsqrt(r2);
  const R rinv2 = rinv * rinv;
  if (LJSW != SW_NONE) {
    // LennardJonesForce.h:28-60
    const R r6 = rinv2 * rinv2 * rinv2;
    const R t = A * r6 - B;
    R e = t * r6;                               // A r^-12 - B r^-6
    R f = (A * r6 + t) * (r6 * ((R)6 * rinv2));  // (12 A r^-12 - 6 B r^-6) / r^2
    if (LJSW == SW_C2) {
      // C2SwitchingFunction.h:42-53: 1 below r_on, the polynomial up to rc
      const bool on = r2 >= k.lj.on2;
      if (__builtin_amdgcn_ballot_w64(on)) {
        const R c2 = k.lj.rc2 - r2, c4 = c2 * (k.lj.s2 + (R)2 * r2);
        const R sv = k.lj.s1 * (c2 * c4);
        const R fs = f * sv - e * (k.lj.s3 * (c2 * c2 - c4)), es = e * sv;
        f = on ? fs : f;
        e = on ? es : e;
      }
    } else {
      R sv, sd;
      switch_val<LJSW, R>(k.ljkind, k.lj, r2, rinv, sv, sd);
      f = f * sv - e * sd;
      e = e * sv;
    }
    flj = f;
    elj = e;
  }
  if (COUL != COUL_NONE) {
    R e, f;
    if (COUL == COUL_CUTOFF) {
      // CoulombForce.h:29-40
      e = qq * rinv;
      f = e * rinv2;
    } else {
      // NonbondedPMEwaldSystemForce.h:657-683 (poly5 form)
      const R t = fast_rcp((R)1 + k.pa * (r2 * rinv));
      const R ex = qq * gauss(k.ke * r2);
      const R p = t * ((R)0.254829592 +
                           t * ((R)-0.284496736 + t * ((R)1.421413741 + t * ((R)-1.453152027 + t * (R)1.061405429))));
      e = p * ex * rinv;
      f = (e + k.a2pi * ex) * rinv2;
    }
    if constexpr (CSW != SW_CUTOFF) {
      R sv, sd;
      switch_val<CSW, R>(k.cokind, k.co, r2, rinv, sv, sd);
      f = f * sv - e * sd;
      e = e * sv;
    }
    fco = f;
    eco = e;
  }
}

// a over lane l and lane l ^ 32 in the lower half wave, b in the upper.
__device__ inline float swap32_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// The same over lane l ^ 16: a in even rows of 16 lanes, b in odd ones.
__device__ inline float swap16_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// The same over lane l ^ 8: a in lanes with bit 3 clear, b in the others.
__device__ inline float swap8_sum(float a, float b, bool hi) {
  const float keep = hi ? b : a, give = hi ? a : b;
  return keep + __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, __float_as_int(give), 0x128, 0xF, 0xF, true));
}

__device__ inline double double_of(unsigned lo, unsigned hi) { return __hiloint2double((int)hi, (int)lo); }
__device__ inline double swap32_sum(double a, double b) {
  const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return double_of(l[0], h[0]) + double_of(l[1], h[1]);
}
__device__ inline double swap16_sum(double a, double b) {
  const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  return double_of(l[0], h[0]) + double_of(l[1], h[1]);
}
__device__ inline double swap8_sum(double a, double b, bool hi) {
  const double keep = hi ? b : a, give = hi ? a : b;
  return keep + double_of((unsigned)__builtin_amdgcn_update_dpp(0, __double2loint(give), 0x128, 0xF, 0xF, true),
                          (unsigned)__builtin_amdgcn_update_dpp(0, __double2hiint(give), 0x128, 0xF, 0xF, true));
}

template <bool MIXED, int COUL, int LJSW, int CSW, bool BIGLJ, int MODE>
__device__ __forceinline__ void pair_body(
    const int bid_, const int nbk_, const PairParams &pp, int dynamic, const int2 *__restrict__ runs,
    const int *__restrict__ ntiles_p, const int *__restrict__ count, int *__restrict__ tile_counter,
    const int4 *__restrict__ entries, int4 *entries_w, int cap, const unsigned short *__restrict__ masks,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ xs,
    const float4 *__restrict__ sorg, const int *__restrict__ ts, const int *__restrict__ perm,
    const double *__restrict__ ljtab,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ ljt,
    typename AccT<MIXED>::type *__restrict__ facc, PairOut out) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using R2 = typename std::conditional<MIXED, float2, double2>::type;
  using R4 = typename Real4<R>::type;
  using WA = WaveAcc<MIXED>;
  constexpr int W = kPairBlock / kWave;
  constexpr bool PRUNE = MODE == kPairPrune, STATS = MODE == kPairStats;
  constexpr bool LJ = LJSW != SW_NONE;
  // {A, B} of the plain and of the 1-4 pairs
  __shared__ R2 s_lj[2][kMaxTypes * kMaxTypes];
  __shared__ R4 s_i[W][kSuperSize];  // the tile's i-atoms
  const int nt = pp.ntypes;
  for (int k = threadIdx.x; LJ && !BIGLJ && k < nt * nt; k += blockDim.x) {
    s_lj[0][k] = R2{(R)ljtab[4 * k], (R)ljtab[4 * k + 1]};
    s_lj[1][k] = R2{(R)ljtab[4 * k + 2], (R)ljtab[4 * k + 3]};
  }
  __syncthreads();

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int ti = lane & 7, tj = lane >> 3;
  const DirectC<R> &kc = direct_of(pp, R());
  const bool same_cut = !LJ || COUL == COUL_NONE || kc.lj.rc2 == kc.co.rc2;
  // the boundary-pair sums are filled after this kernel (same stream)
  if (bid_ == 0 && threadIdx.x < 4) out.border_acc[threadIdx.x] = 0ull;

  // Runs (the grid holds the waves that fit on the device at once): wave w
  // takes the contiguous runs [w nruns / nwaves, (w + 1) nruns / nwaves)
  // (dynamic == 0), or run w and then runs in order from a device-wide counter
  // (dynamic == 1).  A tile is the part of a run in one supercluster.  Which
  // wave takes a run changes no result.
  const int nwaves = nbk_ * W;
  const int gw = bid_ * W + wv;
  const int nruns = ntiles_p[2];
  const int r0 = dynamic ? gw : (int)((long long)gw * nruns / nwaves);
  const int r1 = dynamic ? min(gw + 1, nruns) : (int)((long long)(gw + 1) * nruns / nwaves);
  RunWalk walk(r0, r1);
  while (true) {
    if (walk.run_done()) {
      if (walk.w >= walk.wstop) {
        if (!dynamic) break;
        int rn = 0;
        if (lane == 0) rn = nwaves + atomicAdd(tile_counter, 1);
        const int r = __builtin_amdgcn_readfirstlane(__shfl(rn, 0));
        if (r >= nruns) break;
        walk = RunWalk(r, r + 1);
      }
      walk.next_run(runs);
    }
    const int S = walk.S, t = walk.t, e0 = walk.e0, e1 = walk.tile_end(count);
    walk.next_tile();
    if (e0 >= e1) {
      if (lane == 0) out.clear(t, STATS);
      continue;
    }
    const float4 oS = sorg[S];
    // i-atoms, and the rows of the LJ table of this lane's (8 c + ti), 8 bits each
    __builtin_amdgcn_wave_barrier();
    s_i[wv][lane] = xs[S * kSuperSize + lane];
    __builtin_amdgcn_wave_barrier();
    unsigned irow[2] = {0, 0};
#pragma unroll
    for (int c = 0; LJ && !BIGLJ && c < 8; ++c)
      irow[c >> 2] |= (unsigned)(max(0, ts[S * kSuperSize + c * kClusterSize + ti]) * nt) << (8 * (c & 3));
    R fi[8][3];
#pragma unroll
    for (int c = 0; c < 8; ++c) fi[c][0] = fi[c][1] = fi[c][2] = (R)0;
    R elT = 0, ecT = 0;  // this lane's pair energies over the tile
    int npair = 0;
    unsigned long long hsum = 0;

    const int4 *const ep = entries + (size_t)S * cap;
    // the next entry is read while the current one is evaluated
    auto entry = [&](int e) {
      int4 v = ep[min(e, e1 - 1)];
      v.x = __builtin_amdgcn_readfirstlane(v.x);
      v.y = __builtin_amdgcn_readfirstlane(v.y);
      v.z = __builtin_amdgcn_readfirstlane(v.z);
      v.w = __builtin_amdgcn_readfirstlane(v.w);
      return v;
    };
    auto mask_of = [&](const int4 &v) {
      return v.z >= 0 ? (unsigned)masks[(size_t)v.z * kWave + lane] : 0xffu;
    };
    int4 nent = entry(e0);
    for (int e = e0; e < e1; ++e) {
      const int4 ent = nent;
      const int sj = ent.x * kClusterSize + tj;
      const unsigned em = ent.y & 0xff;
      const int sh = ent.w, masked = ent.z >= 0;
      R4 xj = xs[sj];
      const int tyj = ts[sj];
      const float4 oJ = sorg[ent.x / (kSuperSize / kClusterSize)];
      const unsigned mb = mask_of(ent);
      nent = entry(e + 1);
      // j-cluster into the frame of S: origin difference (exact) plus the
      // entry's image shift (hi part exact, lo part rounded once)
      {
        R ox = (R)(oJ.x - oS.x), oy = (R)(oJ.y - oS.y), oz = (R)(oJ.z - oS.z);
        if (!(sh & kShiftPerPair) && sh != 21) {  // 21: no shift
          const R sx = (R)((sh & 3) - 1), sy = (R)(((sh >> 2) & 3) - 1), sz = (R)(((sh >> 4) & 3) - 1);
          ox = (ox + sx * kc.hi[0]) + sx * kc.lo[0];
          oy = (oy + sy * kc.hi[1]) + sy * kc.lo[1];
          oz = (oz + sz * kc.hi[2]) + sz * kc.lo[2];
        }
        xj.x += ox;
        xj.y += oy;
        xj.z += oz;
      }
      const int tyc = max(0, tyj);
      if (LJ && !BIGLJ) asm volatile("" : "+v"(irow[0]), "+v"(irow[1]));  // unpacked where used, not ahead of the loop
      R fj0 = 0, fj1 = 0, fj2 = 0;
      unsigned used = 0, kept = 0;  // cluster pairs with a member; with a candidate within the list radius

      // GENERAL: the entry carries an exclusion mask or takes the per-pair
      // image; SAME: one cutoff for both kinds.
      auto scan = [&](auto same, auto general) {
        constexpr bool SAME = decltype(same)::value, GENERAL = decltype(general)::value;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          if (!(em & (1u << c))) continue;
          const R4 xi = s_i[wv][c * kClusterSize + ti];
          R dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
          if (GENERAL && (sh & kShiftPerPair)) {
            dx = kc.image(dx, 0);
            dy = kc.image(dy, 1);
            dz = kc.image(dz, 2);
          }
          R r2 = dx * dx + dy * dy + dz * dz;
          if (GENERAL && !(mb & (1u << c))) r2 = kFarR2<R>;
          if (PRUNE && __builtin_amdgcn_ballot_w64(r2 <= kc.prune_r2)) kept |= 1u << c;
          const bool near = r2 <= kc.near2;
          const unsigned long long nm = __builtin_amdgcn_ballot_w64(near);
          if (!nm) continue;
          // a pair within the guard band of a cutoff is left to the FP64
          // boundary pass; a member is in range of a cutoff and outside
          // every band
          bool in, border;
          if (SAME) {
            in = r2 < kc.in2;
            border = near && !in;
          } else {
            const R d = fmin(fabs(r2 - kc.lj.rc2), fabs(r2 - kc.co.rc2));
            in = r2 <= kc.rmax2 && d > kc.guard;
            border = near && d <= kc.guard;
          }
          if (__builtin_expect(
                  SAME ? nm != __builtin_amdgcn_ballot_w64(in) : __builtin_amdgcn_ballot_w64(border) != 0, 0)) {
            if (border) {
              const int b = atomicAdd(out.nborder, 1);
              int si = ti;
              asm volatile("" : "+v"(si));  // rare: nothing of it is worth a register outside
              if (b < out.maxborder)
                out.border[b] = make_int2(S * kSuperSize + c * kClusterSize + si, sj);
              else
                atomicExch(out.overflow, 1);
            }
          }
          if (STATS && in) {
            const int ai = perm[S * kSuperSize + c * kClusterSize + ti], aj = perm[sj];
            ++npair;
            hsum += pair_hash(ai < aj ? ai : aj, ai < aj ? aj : ai);
          }
          // lanes without a member are evaluated too and selected away
          const bool mod = GENERAL && ((mb >> (8 + c)) & 1u);
          R A = 0, B = 0;
          if (LJ && BIGLJ) {
            const int tyi = max(0, ts[S * kSuperSize + c * kClusterSize + ti]);
            const R4 v = ljt[(size_t)tyi * nt + tyc];
            A = mod ? v.z : v.x;
            B = mod ? v.w : v.y;
          } else if (LJ) {
            const R2 v = s_lj[GENERAL ? (mod ? 1 : 0) : 0][((irow[c >> 2] >> (8 * (c & 3))) & 255u) + tyc];
            A = v.x;
            B = v.y;
          }
          R qq = xi.w * xj.w;
          if (GENERAL && mod) qq *= kc.csf;
          R el = 0, ec = 0, fl = 0, fc = 0, f;
          direct_eval<COUL, LJSW, CSW, R>(kc, r2, qq, A, B, el, ec, fl, fc);
          if (SAME) {
            f = in ? fl + fc : (R)0;
            elT += in ? el : (R)0;
            ecT += in ? ec : (R)0;
          } else {
            const bool il = in && r2 <= kc.lj.rc2, ic = in && r2 <= kc.co.rc2;
            f = (il ? fl : (R)0) + (ic ? fc : (R)0);
            elT += il ? el : (R)0;
            ecT += ic ? ec : (R)0;
          }
          fi[c][0] += f * dx;  // of the opposite sign
          fi[c][1] += f * dy;
          fi[c][2] += f * dz;
          fj0 += f * dx;
          fj1 += f * dy;
          fj2 += f * dz;
          used = 1;
        }
      };
      const bool general = masked || (sh & kShiftPerPair);
      if (__builtin_expect(same_cut && !general, 1))
        scan(std::true_type{}, std::false_type{});
      else if (same_cut)
        scan(std::true_type{}, std::true_type{});
      else if (!general)
        scan(std::false_type{}, std::false_type{});
      else
        scan(std::false_type{}, std::true_type{});
      // prune pass: cluster pairs without a candidate pair inside the list
      // radius cannot have a member before the next list build (every atom
      // stays within half the skin of its build position); later passes skip
      // them.  They have no member now either, so no result changes.
      if (PRUNE && lane == 0 && kept != em) entries_w[(size_t)S * cap + e].y = (int)kept;
      if (used) {
        fj0 = group8_sum(fj0);
        fj1 = group8_sum(fj1);
        fj2 = group8_sum(fj2);
        if (ti < 3 && tyj >= 0) {
          const R v = ti == 0 ? fj0 : (ti == 1 ? fj1 : fj2);
          AccT<MIXED>::add(&facc[3 * sj + ti], v);
        }
      }
    }
    // tile end: lane 8 c + ti sums the eight partials of its i-atom
    {
      const int s = S * kSuperSize + lane;
      const bool real = ts[s] >= 0, hi8 = lane & 8;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        R a[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = swap32_sum(fi[c][k], fi[c + 4][k]);
        const R b0 = swap16_sum(a[0], a[2]), b1 = swap16_sum(a[1], a[3]);
        const R v = swap8_sum(b0, b1, hi8);
        if (real) WA::add(&facc[3 * s + k], WA::of(-v));
      }
    }
    const typename WA::T eljA = wave_sum(WA::of(elT));
    const typename WA::T ecoA = wave_sum(WA::of(ecT));
    long long np = 0;
    if (STATS) {
      np = wave_sum((long long)npair);
      hsum = wave_sum(hsum);
    }
    if (lane == 0) {
      out.energy[2 * t] = WA::energy_bits(ecoA);
      out.energy[2 * t + 1] = WA::energy_bits(eljA);
      if (STATS) {
        out.npairs[t] = np;
        out.hash[t] = hsum;
      }
    }
  }
}

template <bool MIXED, int COUL, int LJSW, int CSW, bool BIGLJ, int MODE>
__global__ void __launch_bounds__(kPairBlock, MIXED ? 4 : 3) k_pair(
    PairParams pp, int dynamic, const int2 *__restrict__ runs, const int *__restrict__ ntiles_p,
    const int *__restrict__ count, int *__restrict__ tile_counter, const int4 *__restrict__ entries, int4 *entries_w,
    int cap,
    const unsigned short *__restrict__ masks,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ xs,
    const float4 *__restrict__ sorg, const int *__restrict__ ts, const int *__restrict__ perm,
    const double *__restrict__ ljtab,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ ljt,
    typename AccT<MIXED>::type *__restrict__ facc, PairOut out) {
  // the blocks of one XCD take a contiguous range of runs
  const int bid = xcd_block(blockIdx.x, gridDim.x);
  pair_body<MIXED, COUL, LJSW, CSW, BIGLJ, MODE>(bid, gridDim.x, pp, dynamic, runs, ntiles_p, count, tile_counter,
                                                 entries, entries_w, cap, masks, xs, sorg, ts, perm, ljtab, ljt, facc,
                                                 out);
}

// Boundary pairs: exact FP64 membership on the original coordinates
// (reference operation order), then the same pair evaluation.  Energies go
// to int64 fixed point (2^-32) so the total is independent of record order.
// Blocks [0, nblocks) of the fixup launch walk the records with a grid stride.
template <bool MIXED, int COUL, int LJSW, int CSW>
__device__ void border_pairs(int blk, int nblocks, const PairParams &pp, int stats, const int2 *__restrict__ border,
                             const int *__restrict__ nborder, int maxborder,
                             const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ xs,
                             const float4 *__restrict__ sorg, const int *__restrict__ ts, const int *__restrict__ perm,
                             const double *__restrict__ xorig,
                             const double *__restrict__ ljtab, const int *__restrict__ eptr,
                             const int2 *__restrict__ elist, typename AccT<MIXED>::type *__restrict__ facc,
                             unsigned long long *__restrict__ eacc, unsigned long long *__restrict__ stat) {
  using R = typename std::conditional<MIXED, float, double>::type;
  const int nb = min(*nborder, maxborder);
  for (int b = blk * blockDim.x + threadIdx.x; b < nb; b += nblocks * blockDim.x) {
    const int2 rec = border[b];
    const int si = rec.x, sj = rec.y;
    const int ai = perm[si], aj = perm[sj];
    const int lo = ai < aj ? ai : aj, hi = ai < aj ? aj : ai;
    const double d2 = exact_d2(xorig, lo, hi, pp.box);
    const bool in_lj = LJSW != SW_NONE && d2 <= pp.lj.rc2;
    const bool in_c = COUL != COUL_NONE && d2 <= pp.co.rc2;
    if (!(in_lj || in_c)) continue;
    // exclusion class (recorded pairs already passed the FULL mask)
    const int cls = excl_class(eptr, elist, ai, aj);
    const bool modified = cls == 2;
    SwR<R> sl, sc;
    sl.load(pp.lj);
    sc.load(pp.co);
    const auto xi = xs[si], xj = xs[sj];
    const float4 oi = sorg[si / kSuperSize], oj = sorg[sj / kSuperSize];
    EdgesR<R> E;
    E.load(pp);
    R dx = (xj.x - xi.x) + (R)(oj.x - oi.x), dy = (xj.y - xi.y) + (R)(oj.y - oi.y),
      dz = (xj.z - xi.z) + (R)(oj.z - oi.z);
    dx = E.image(dx, 0);
    dy = E.image(dy, 1);
    dz = E.image(dz, 2);
    R r2 = dx * dx + dy * dy + dz * dz;
    // evaluate at the cutoff side the exact test chose
    R A = 0, B = 0;
    if (LJSW != SW_NONE) {
      const int k = 4 * (ts[si] * pp.ntypes + ts[sj]);
      A = (R)ljtab[k + (modified ? 2 : 0)];
      B = (R)ljtab[k + (modified ? 3 : 1)];
    }
    R qq = xi.w * xj.w;
    if (modified) qq *= (R)pp.csf;
    R e1, e2, fr;
    pair_eval<COUL, LJSW, CSW, R>(pp, sl, sc, (R)pp.alpha, (R)pp.a2pi, (R)pp.csf, r2, qq, A, B, in_lj, in_c, e1, e2, fr);
    AccT<MIXED>::add(&facc[3 * si], -dx * fr);
    AccT<MIXED>::add(&facc[3 * si + 1], -dy * fr);
    AccT<MIXED>::add(&facc[3 * si + 2], -dz * fr);
    AccT<MIXED>::add(&facc[3 * sj], dx * fr);
    AccT<MIXED>::add(&facc[3 * sj + 1], dy * fr);
    AccT<MIXED>::add(&facc[3 * sj + 2], dz * fr);
    atomicAdd(&eacc[0], (unsigned long long)__double2ll_rn((double)e2 * kForceScale));
    atomicAdd(&eacc[1], (unsigned long long)__double2ll_rn((double)e1 * kForceScale));
    if (stats) {
      atomicAdd(&stat[0], 1ull);
      atomicAdd(&stat[1], pair_hash(lo, hi));
    }
  }
}

// ---------------------------------------------------------------------------
// 4. PME (Grid.h:107-341): charge spread with the z transform, y and x
//    transforms with the influence function, inverse z transform with the
//    force gather.  The half spectrum is [k][j][i] (i fastest) throughout.
//
// The charge grid and the real potential never exist in memory: a block owns
// a tile of grid lines along z (tx x ty neighbouring (i, j)), sums every
// stencil contribution to them in LDS and transforms them there; the inverse
// pass transforms the tile's lines back and interpolates the forces from
// LDS.  A tile finds the atoms whose stencils touch it in the x-y columns of
// the sort (the window of the tile widened by the stencil and by half the
// skin the atoms may have moved since the sort).  With the grid in memory
// (atomics from an LDS patch per 32 atoms, a transform that read and cleared
// it, a gather that loaded patches of the potential) the reciprocal part of a
// step moved 2.7 GB on a 256^3 grid, the atomics 0.58 GB of it; here each
// pass reads and writes the half spectrum once.  Million-atom box, 216 x 240 x
// 240 points, order 6, before and after: spread + z 1.18 -> 0.30 ms alone, x
// and y 0.91 -> 0.25 ms, inverse z + gather 0.46 -> 0.35 ms (the last two
// beside the pair kernel).

// BSpline::set (mdl/interface/force/nonbonded/BSpline.cpp:55-105) for a
// compile-time order P (2..8): weights th[0..P-1] and derivatives dth.
template <int P, class R>
__device__ inline void bspline_w(R w, R *th, R *dth) {
  if constexpr (P == 2) {  // linear: the recursion starts from it
    th[0] = (R)1 - w;
    th[1] = w;
    dth[0] = (R)-1;
    dth[1] = (R)1;
    return;
  }
  th[P - 1] = 0;
  th[1] = w;
  th[0] = (R)1 - w;
#pragma unroll
  for (int k = 2; k < P - 1; k++) {
    const R div = (R)1 / (R)k;
    th[k] = div * w * th[k - 1];
#pragma unroll
    for (int j = 1; j < k; j++) th[k - j] = div * ((w + (R)j) * th[k - j - 1] + ((R)(k + 1 - j) - w) * th[k - j]);
    th[0] = div * ((R)1 - w) * th[0];
  }
  dth[0] = -th[0];
#pragma unroll
  for (int j = 1; j <= P - 1; j++) dth[j] = th[j - 1] - th[j];
  const R div = (R)1 / (R)(P - 1);
  th[P - 1] = div * w * th[P - 2];
#pragma unroll
  for (int j = 1; j < P - 1; j++)
    th[P - 1 - j] = div * ((w + (R)j) * th[P - j - 2] + ((R)(P - j) - w) * th[P - 1 - j]);
  th[0] = div * ((R)1 - w) * th[0];
}

template <class T>
struct alignas(2 * sizeof(T)) Cx {
  T x, y;
};

template <class T>
__device__ inline Cx<T> cmul(Cx<T> a, Cx<T> b) {
  return Cx<T>{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <class T>
__device__ inline Cx<T> cadd(Cx<T> a, Cx<T> b) {
  return Cx<T>{a.x + b.x, a.y + b.y};
}
template <class T>
__device__ inline Cx<T> csub(Cx<T> a, Cx<T> b) {
  return Cx<T>{a.x - b.x, a.y - b.y};
}

// Forward DFT of small radix R in registers, e^{-2 pi i rk/R}.  6 and 10 are
// prime-factor products (no twiddles), 8 and 9 two steps.
template <int R, class T>
__device__ __forceinline__ void dft_small(Cx<T> *v) {
  if constexpr (R == 2) {
    const Cx<T> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    const Cx<T> s0 = cadd(v[0], v[2]), s1 = csub(v[0], v[2]);
    const Cx<T> s2 = cadd(v[1], v[3]), s3 = csub(v[1], v[3]);
    v[0] = cadd(s0, s2);
    v[2] = csub(s0, s2);
    // -i * s3 = (s3.y, -s3.x)
    v[1] = Cx<T>{s1.x + s3.y, s1.y - s3.x};
    v[3] = Cx<T>{s1.x - s3.y, s1.y + s3.x};
  } else if constexpr (R == 3) {
    const T c = (T)-0.5, s = (T)0.86602540378443864676;
    const Cx<T> a = v[0], t = cadd(v[1], v[2]), u = csub(v[1], v[2]);
    v[0] = cadd(a, t);
    const Cx<T> m{a.x + c * t.x, a.y + c * t.y};
    // -i s u = (s u.y, -s u.x)
    v[1] = Cx<T>{m.x + s * u.y, m.y - s * u.x};
    v[2] = Cx<T>{m.x - s * u.y, m.y + s * u.x};
  } else if constexpr (R == 5) {
    const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
    const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;
    const Cx<T> a = v[0], t1 = cadd(v[1], v[4]), u1 = csub(v[1], v[4]), t2 = cadd(v[2], v[3]), u2 = csub(v[2], v[3]);
    v[0] = Cx<T>{a.x + t1.x + t2.x, a.y + t1.y + t2.y};
    const Cx<T> m1{a.x + c1 * t1.x + c2 * t2.x, a.y + c1 * t1.y + c2 * t2.y};
    const Cx<T> m2{a.x + c2 * t1.x + c1 * t2.x, a.y + c2 * t1.y + c1 * t2.y};
    // y1 = m1 - i(s1 u1 + s2 u2); y4 = m1 + i(...); y2 = m2 - i(s2 u1 - s1 u2); y3 = m2 + i(...)
    const Cx<T> n1{s1 * u1.x + s2 * u2.x, s1 * u1.y + s2 * u2.y};
    const Cx<T> n2{s2 * u1.x - s1 * u2.x, s2 * u1.y - s1 * u2.y};
    v[1] = Cx<T>{m1.x + n1.y, m1.y - n1.x};
    v[4] = Cx<T>{m1.x - n1.y, m1.y + n1.x};
    v[2] = Cx<T>{m2.x + n2.y, m2.y - n2.x};
    v[3] = Cx<T>{m2.x - n2.y, m2.y + n2.x};
  } else if constexpr (R == 6 || R == 10) {
    // element (n1, n2) is input (H n1 + 2 n2) mod R; output k has k1 = k mod 2, k2 = k mod H
    constexpr int H = R / 2;
    Cx<T> e[H], o[H];
#pragma unroll
    for (int m = 0; m < H; ++m) {
      const Cx<T> a = v[(2 * m) % R], b = v[(H + 2 * m) % R];
      e[m] = cadd(a, b);
      o[m] = csub(a, b);
    }
    dft_small<H, T>(e);
    dft_small<H, T>(o);
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = (k & 1) ? o[k % H] : e[k % H];
  } else if constexpr (R == 8) {
    const T h = (T)0.70710678118654752440;
    Cx<T> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft_small<4, T>(e);
    dft_small<4, T>(o);
    // o[k] e^{-2 pi i k/8}
    o[1] = Cx<T>{h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
    o[2] = Cx<T>{o[2].y, -o[2].x};
    o[3] = Cx<T>{h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = cadd(e[k], o[k]);
      v[k + 4] = csub(e[k], o[k]);
    }
  } else {
    static_assert(R == 9, "radix 2, 3, 4, 5, 6, 8, 9 or 10");
    const Cx<T> w1{(T)0.76604444311897803520, (T)-0.64278760968653932632};
    const Cx<T> w2{(T)0.17364817766693034885, (T)-0.98480775301220805937};
    const Cx<T> w4{(T)-0.93969262078590838405, (T)-0.34202014332566873304};
    Cx<T> a[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 3; ++n1) a[n2][n1] = v[3 * n1 + n2];
      dft_small<3, T>(a[n2]);
    }
    a[1][1] = cmul(a[1][1], w1);
    a[1][2] = cmul(a[1][2], w2);
    a[2][1] = cmul(a[2][1], w2);
    a[2][2] = cmul(a[2][2], w4);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      Cx<T> b[3] = {a[0][k1], a[1][k1], a[2][k1]};
      dft_small<3, T>(b);
#pragma unroll
      for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = b[k2];
    }
  }
}

// Division of t < 2^16 by a constant d: (t * magic) >> 32, magic =
// floor(2^32 / d) + 1 (exact for t d < 2^32; d = 1 has none).
__host__ __device__ inline unsigned div_magic(unsigned d) { return (unsigned)(0x100000000ull / d) + 1u; }
__device__ inline int div_by(int t, unsigned magic) { return (int)__umulhi((unsigned)t, magic); }

constexpr int kFftMax = 4096;       // longest ordinary transform (points), and most points of a block
constexpr int kFftPerThread = 8;    // points a thread holds in a pass, at least (8 keeps a pass within 64 VGPRs,
                                    // so that these kernels fit on a SIMD beside four pair-kernel waves)
constexpr int kPmeBlock = kFftMax / kFftPerThread;  // threads of a PME block, at most
template <class T>
constexpr int kPmeWaves = sizeof(T) == 4 ? 8 : 4;   // resident waves per SIMD to compile for
// Axes beyond kFftMax take passes of their own (LONG; a block per line, on z
// per pair of lines) with more points per thread and the twiddles read from
// memory: up to 10,125 points in the mixed form, whose FP64 charge sums of a
// line pair then fill the 160 KB of LDS, half as many in FP64, whose
// points take twice the registers.  A launch that asks for more LDS than a
// CU has ends the queue.
template <class T, bool LONG>
constexpr int kFftPoints = !LONG ? kFftPerThread : sizeof(T) == 4 ? 20 : 10;
template <class T>
constexpr int kFftMaxLong = sizeof(T) == 4 ? 10125 : kPmeBlock * kFftPoints<T, true>;
static_assert(kFftMaxLong<float> <= kPmeBlock * kFftPoints<float, true>);
struct FftPlan {
  int n;
  int nrad;
  int rad[12];
  unsigned magic[12];  // div_magic of the product of the radices before this one
  unsigned magic_n;    // div_magic(n)
};

// `lines` transforms in LDS: element e of line l at l ls + e es.  Threads
// take the lines fastest (1 << llog of them, a power of two of at least
// `lines`), so that with an odd ls (or es = 1 across odd rows) neighbouring
// lanes fall on different banks and no thread index is divided by a length.
struct FftLines {
  int llog, lines, ls, es;
};

// One Stockham pass of radix R in place: every thread holds its butterflies
// (up to PER points or the next multiple of R) in registers between the two
// barriers.  Butterfly j reads elements j + r n/R, twiddles by
// tw[k r n/(Ns R)] (k = j mod Ns), writes (j - k) R + k + r Ns.
template <int R, class T, int PER>
__device__ __forceinline__ void fft_pass(Cx<T> *buf, const FftLines &f, int n, int Ns, unsigned magic,
                                         const Cx<T> *tw) {
  constexpr int NB = (PER + R - 1) / R;
  const int line = threadIdx.x & ((1 << f.llog) - 1), tb = threadIdx.x >> f.llog, step = blockDim.x >> f.llog;
  const int nbut = n / R, tstep = n / (Ns * R);
  Cx<T> v[NB][R];
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int j = tb + m * step;
    if (line < f.lines && j < nbut) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[m][r] = buf[line * f.ls + (j + r * nbut) * f.es];
      if (Ns > 1) {
        const int k = (j - div_by(j, magic) * Ns) * tstep;
#pragma unroll
        for (int r = 1; r < R; ++r) v[m][r] = cmul(v[m][r], tw[k * r]);
      }
      dft_small<R, T>(v[m]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    const int j = tb + m * step;
    if (line < f.lines && j < nbut) {
      const int k = Ns > 1 ? j - div_by(j, magic) * Ns : 0;
      Cx<T> *d = buf + line * f.ls + ((j - k) * R + k) * f.es;
#pragma unroll
      for (int r = 0; r < R; ++r) d[r * Ns * f.es] = v[m][r];
    }
  }
  __syncthreads();
}

// Forward transforms of the lines in place (blockDim.x >> f.llog threads per
// line, at least n / PER; tw in LDS, or in memory).  All threads of the block take part;
// the data are in place before the call and after it.
template <class T, int PER = kFftPerThread>
__device__ __forceinline__ void lds_fft(Cx<T> *buf, const FftLines &f, const FftPlan &pl, const Cx<T> *tw) {
  int Ns = 1;
  for (int s = 0; s < pl.nrad; ++s) {
    const unsigned mg = pl.magic[s];
    const int R = __builtin_amdgcn_readfirstlane(pl.rad[s]);
    switch (R) {
      case 2: fft_pass<2, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
      case 3: fft_pass<3, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
      case 4: fft_pass<4, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
      case 5: fft_pass<5, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
      case 6: fft_pass<6, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
      case 8: fft_pass<8, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
      case 9: fft_pass<9, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
      default: fft_pass<10, T, PER>(buf, f, pl.n, Ns, mg, tw); break;
    }
    Ns *= R;
  }
}

template <class T>
__device__ __forceinline__ void lds_twiddles(Cx<T> *s_tw, const Cx<T> *__restrict__ tw, int n) {
  for (int t = threadIdx.x; t < n; t += blockDim.x) s_tw[t] = tw[t];
}

// Calls work(cnt, slot) for the atoms whose stencils touch the tile (i0, j0),
// up to 64 of them at a time on one wave (lanes below cnt hold a slot).
// Waves take the superclusters of the tile's columns in turn.  LONG: without
// the queue, whose LDS such lines leave no room for (cnt is 64 in the lanes
// that hold a slot and 0 in the others).
template <int P, bool LONG, class WORK>
__device__ __forceinline__ void pme_tile_atoms(const PmeParams &p, const int2 *__restrict__ tcol, int tix, int tjy,
                                               const int *__restrict__ colsc, const int2 *__restrict__ pmb,
                                               int (*s_q)[128], WORK work) {
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int i0 = tix * p.tx, j0 = tjy * p.ty;
  const int2 cx = tcol[tix], cy = tcol[p.ntx + tjy];  // first column and column count
  int *const q = LONG ? nullptr : s_q[wv];
  int qn = 0;                   // queued slots
  int r = -1;                   // range of superclusters: column a = r / 2 of the x window, part r & 1 in y
  int sc = 0, s1 = 0;           // the range's next supercluster and its end
  int turn = wv;                // superclusters until this wave's next
  bool more = true;
  while (true) {
    while (more && qn < kWave) {
      while (sc + turn >= s1) {
        turn -= s1 - sc;
        sc = s1 = 0;
        if (++r >= 2 * cx.y) {
          more = false;
          break;
        }
        const int col = wrap_grid(cx.x + (r >> 1), p.ncx) * p.ncy;
        const int y0 = (r & 1) ? 0 : cy.x, y1 = (r & 1) ? cy.x + cy.y - p.ncy : min(cy.x + cy.y, p.ncy);
        if (y1 <= y0) continue;
        sc = __builtin_amdgcn_readfirstlane(colsc[col + y0]);
        s1 = __builtin_amdgcn_readfirstlane(colsc[col + y1]);
      }
      if (!more) break;
      const int s = (sc + turn) * kSuperSize + lane;
      sc += nw;
      const int b = pmb[s].x;
      int ex = (b & 0xffff) - (i0 - P + 1), ey = (b >> 16) - (j0 - P + 1);
      ex -= ex >= p.nx ? p.nx : 0;
      ex += ex < 0 ? p.nx : 0;
      ey -= ey >= p.ny ? p.ny : 0;
      ey += ey < 0 ? p.ny : 0;
      const bool hit = b != kNoGrid && ex < p.tx + P - 1 && ey < p.ty + P - 1;
      if constexpr (LONG) {
        work(hit ? kWave : 0, s);
        continue;
      }
      const unsigned long long m = __ballot(hit);
      if (hit) q[qn + __popcll(m & ((1ull << lane) - 1ull))] = s;
      qn += __popcll(m);
    }
    if (qn == 0) break;
    const int cnt = min(qn, kWave);
    __builtin_amdgcn_wave_barrier();
    const int mine = q[lane < cnt ? lane : 0], rest = q[kWave + (lane < qn - cnt ? lane : 0)];
    __builtin_amdgcn_wave_barrier();
    if (lane < qn - cnt) q[lane] = rest;
    qn -= cnt;
    work(cnt, mine);
    __builtin_amdgcn_wave_barrier();
  }
}

// Line stride of a tile in LDS: nz points, and the p - 1 points after the
// last that the stencils of the last cells reach (copies of the first points:
// a stencil's z points then lie at fixed offsets from its first), made odd.
__host__ __device__ constexpr int pme_line(int nz, int order) { return (nz + order - 1) | 1; }

// Transforms of all of a tile's np line pairs, as many at a time as the block
// holds points for.
template <class T, bool LONG>
__device__ __forceinline__ void pme_tile_fft(Cx<T> *buf, int np, int n, int ls, const FftPlan &pl, const Cx<T> *tw) {
  if constexpr (LONG) {
    for (int l = 0; l < np; ++l) lds_fft<T, kFftPoints<T, true>>(buf + l * ls, FftLines{0, 1, ls, 1}, pl, tw);
    return;
  }
  const int need = n > kFftPerThread ? 32 - __clz((n - 1) / kFftPerThread) : 0;  // log2 of a line's threads
  const int llog = min(31 - __clz(np), 31 - __clz((int)blockDim.x) - need);
  for (int l0 = 0; l0 < np; l0 += 1 << llog)
    lds_fft<T>(buf + l0 * ls, FftLines{llog, min(1 << llog, np - l0), ls, 1}, pl, tw);
}

// Fixed-point charge sums: a double holding a multiple of 2^-40 below 2^12
// in size adds exactly, so sums of charges rounded to that grid do not depend
// on the order of the adds (an LDS ds_add_f64 instead of the conversions to
// and from int64).
constexpr double kGridRound = 6144.0;  // 1.5 2^12: its last bit is 2^-40

// Spread and z transform of one tile (see above).  Bound by VALU and LDS
// atomics: each lane takes one atom and walks the stencil rows inside the
// tile.  Two real lines share one complex transform.  On small grids the
// block's own latency bounds it: 9.5 us at 30^3 points and 1,500 atoms, where
// the spread (in the kick-drift launch) and the z transform took 7 + 5.6 us
// and a launch gap.
template <bool MIXED, int P, bool LONG = false>
__device__ __forceinline__ void pme_spread_z_body(
    const int bid_, const int nbk_, const PmeParams &p, const FftPlan &pl, const int2 *__restrict__ tcol,
    const int *__restrict__ colsc,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ pmw,
    const int2 *__restrict__ pmb, const Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ tw,
    Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ spec) {
  using T = typename std::conditional<MIXED, float, double>::type;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int s_q[LONG ? 1 : kPmeBlock / kWave][128];
  Cx<T> *const s_tw = reinterpret_cast<Cx<T> *>(smem_raw);
  // sums of lines 2 l and 2 l + 1 interleaved at l, in the order of the
  // complex lines they become
  double *const acc = reinterpret_cast<double *>(s_tw + (LONG ? 0 : (p.nz + 1) & ~1));
  Cx<T> *const buf = reinterpret_cast<Cx<T> *>(acc);
  const int nzs = pme_line(p.nz, P), lines = p.tx * p.ty;
  const int tjy = bid_ / p.ntx, tix = bid_ - tjy * p.ntx;
  const int i0 = tix * p.tx, j0 = tjy * p.ty;
  if (!LONG) lds_twiddles(s_tw, tw, p.nz);
  for (int t = threadIdx.x; t < lines * nzs; t += blockDim.x) acc[t] = 0.0;
  __syncthreads();
  pme_tile_atoms<P, LONG>(p, tcol, tix, tjy, colsc, pmb, s_q, [&](int cnt, int slot) {
    if ((int)(threadIdx.x & 63) >= cnt) return;
    const auto a = pmw[slot];
    const int2 b = pmb[slot];
    T wx[P], wy[P], wz[P], dd[P];
    bspline_w<P, T>(a.x, wx, dd);
    bspline_w<P, T>(a.y, wy, dd);
    bspline_w<P, T>(a.z, wz, dd);
    const int bx = (b.x & 0xffff), by = b.x >> 16;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int li = wrap_grid(bx + i, p.nx) - i0;
      if ((unsigned)li >= (unsigned)p.tx) continue;
      const T qx = a.w * wx[i];
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const int lj = wrap_grid(by + j, p.ny) - j0;
        if ((unsigned)lj >= (unsigned)p.ty) continue;
        const T qxy = qx * wy[j];
        const int line = lj * p.tx + li;
        double *const row = acc + ((line >> 1) * nzs + b.y) * 2 + (line & 1);
#pragma unroll
        for (int k = 0; k < P; ++k) {
          double v = (double)(qxy * wz[k]);
          if (MIXED) v = (v + kGridRound) - kGridRound;
          unsafeAtomicAdd(&row[2 * k], v);
        }
      }
    }
  });
  __syncthreads();
  // the points past the end belong to the first ones
  for (int t = threadIdx.x; t < lines * (P - 1); t += blockDim.x) {
    const int k = t / lines, line = t - k * lines, z = (line >> 1) * nzs * 2 + (line & 1);
    int g = k;  // nz may be smaller than p - 1
    while (g >= p.nz) g -= p.nz;
    unsafeAtomicAdd(&acc[z + 2 * g], acc[z + 2 * (p.nz + k)]);
  }
  __syncthreads();
  // lines 2 l and 2 l + 1 are the real and imaginary part of transform l
  const int np = lines >> 1, nplog = 31 - __clz(np);
  if (MIXED) {
    // to FP32 in place, through registers; what a round writes lies below
    // what later rounds read
    const double2 *const a2 = reinterpret_cast<const double2 *>(acc);
    for (int e0 = threadIdx.x; e0 - (int)threadIdx.x < np * nzs; e0 += 4 * blockDim.x) {
      Cx<T> v[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int e = e0 + m * blockDim.x;
        if (e < np * nzs) v[m] = Cx<T>{(T)a2[e].x, (T)a2[e].y};
      }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int e = e0 + m * blockDim.x;
        if (e < np * nzs) buf[e] = v[m];
      }
    }
    __syncthreads();
  }
  pme_tile_fft<T, LONG>(buf, np, p.nz, nzs, pl, LONG ? tw : s_tw);
  const int hlog = 31 - __clz(p.tx) - 1;  // line pairs per row of the tile: tx / 2
  for (int t = threadIdx.x; t < p.nzh << nplog; t += blockDim.x) {
    const int l = t & (np - 1), k = t >> nplog;
    const int i = i0 + 2 * (l & ((1 << hlog) - 1)), j = j0 + (l >> hlog);
    if (i >= p.nx || j >= p.ny) continue;
    const Cx<T> u = buf[l * nzs + k], v = buf[l * nzs + (k ? p.nz - k : 0)];
    Cx<T> *o = spec + ((size_t)k * p.ny + j) * p.nx + i;
    o[0] = Cx<T>{(T)0.5 * (u.x + v.x), (T)0.5 * (u.y - v.y)};
    if (i + 1 < p.nx) o[1] = Cx<T>{(T)0.5 * (u.y + v.y), (T)0.5 * (v.x - u.x)};
  }
}

template <bool MIXED, int P, bool LONG = false>
__global__ void __launch_bounds__(kPmeBlock, LONG ? 2 : MIXED ? 8 : 4) k_pme_spread_z(
    PmeParams p, FftPlan pl, const int2 *__restrict__ tcol, const int *__restrict__ colsc,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ pmw,
    const int2 *__restrict__ pmb, const Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ tw,
    Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ spec) {
  // the blocks of one XCD take a contiguous range of tiles
  pme_spread_z_body<MIXED, P, LONG>(xcd_block(blockIdx.x, gridDim.x), gridDim.x, p, pl, tcol, colsc, pmw, pmb, tw, spec);
}

// y pass of the lines (k, i0 .. i0 + (1 << llog) - 1), in place: forward, or
// inverse (conj-in / conj-out around the forward transform).  Bound by memory
// on large grids: 0.21 -> 0.058 ms for 2 x 50 MB (216 x 240 x 240, beside the
// pair kernel).
template <class T, bool LONG = false>
__device__ __forceinline__ void fft_y_body(const int bid_, const int nbk_, const PmeParams &p, const FftPlan &pl,
                                           int llog, bool inverse, const Cx<T> *__restrict__ tw,
                                           Cx<T> *__restrict__ spec) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Cx<T> *const s_tw = reinterpret_cast<Cx<T> *>(smem_raw);
  Cx<T> *const buf = LONG ? s_tw : s_tw + p.ny;
  const int it = (p.nx + (1 << llog) - 1) >> llog;
  const int k = bid_ / it, i0 = (bid_ - k * it) << llog;
  const FftLines f{llog, min(1 << llog, p.nx - i0), p.ny | 1, 1};
  Cx<T> *const g = spec + (size_t)k * p.ny * p.nx + i0;
  if (!LONG) lds_twiddles(s_tw, tw, p.ny);
  const int l = threadIdx.x & ((1 << llog) - 1);
  if (l < f.lines)
    for (int j = threadIdx.x >> llog; j < p.ny; j += blockDim.x >> llog) {
      Cx<T> v = g[(size_t)j * p.nx + l];
      if (inverse) v.y = -v.y;
      buf[l * f.ls + j] = v;
    }
  __syncthreads();
  lds_fft<T, kFftPoints<T, LONG>>(buf, f, pl, LONG ? tw : s_tw);
  if (l < f.lines)
    for (int j = threadIdx.x >> llog; j < p.ny; j += blockDim.x >> llog) {
      Cx<T> v = buf[l * f.ls + j];
      if (inverse) v.y = -v.y;
      g[(size_t)j * p.nx + l] = v;
    }
}

template <class T, bool LONG = false>
__global__ void __launch_bounds__(kPmeBlock, LONG ? 2 : kPmeWaves<T>) k_fft_y(PmeParams p, FftPlan pl, int llog, bool inverse,
                                                     const Cx<T> *__restrict__ tw, Cx<T> *__restrict__ spec) {
  fft_y_body<T, LONG>(xcd_block(blockIdx.x, gridDim.x), gridDim.x, p, pl, llog, inverse, tw, spec);
}

// Weight of plane k of the half spectrum in the energy.
__device__ inline double plane_weight(const PmeParams &p, int k) {
  return (k > 0 && ((k != p.nz / 2) || (p.nz & 1))) ? 2.0 : 1.0;
}

// The block's energy sum into epart[bid].
__device__ __forceinline__ void block_energy(double e, double *epart) {
  __shared__ double s_e[1024 / kWave];
  e = wave_sum(e);
  if ((threadIdx.x & 63) == 0) s_e[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0;
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) tot += s_e[w];
    *epart = tot;
  }
}

// Influence function on one element (Grid.h:237-341; theta [k][j][i]): the
// energy term, and the product conjugated for the inverse transform.
template <class T>
__device__ inline double convolve(Cx<T> &v, T th) {
  const double e = (double)th * ((double)v.x * (double)v.x + (double)v.y * (double)v.y);
  v = Cx<T>{v.x * th, -(v.y * th)};
  return e;
}

// x pass of the lines (k, j0 .. j0 + (1 << llog) - 1), in place: forward
// transform, influence function with the energy, inverse transform.  The
// energy is summed over `threads` threads (the block may be larger in a
// batched launch), so it does not depend on the batch.  0.49 -> 0.11 ms for
// 125 MB on that grid: radices up to 10 in registers (three passes of LDS
// instead of five), no division by a length, odd line strides.
template <class T, bool LONG = false>
__device__ __forceinline__ void fft_x_conv_body(const int bid_, const int nbk_, const PmeParams &p, const FftPlan &pl,
                                                int llog, int threads, const Cx<T> *__restrict__ tw,
                                                const T *__restrict__ theta, Cx<T> *__restrict__ spec,
                                                double *__restrict__ epart) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Cx<T> *const s_tw = reinterpret_cast<Cx<T> *>(smem_raw);
  Cx<T> *const buf = LONG ? s_tw : s_tw + p.nx;
  const int jt = (p.ny + (1 << llog) - 1) >> llog;
  const int k = bid_ / jt, j0 = (bid_ - k * jt) << llog;
  const FftLines f{llog, min(1 << llog, p.ny - j0), p.nx | 1, 1};
  const int pad = f.ls - p.nx;
  const size_t base = ((size_t)k * p.ny + j0) * p.nx;
  if (!LONG) lds_twiddles(s_tw, tw, p.nx);
  for (int t = threadIdx.x; t < f.lines * p.nx; t += blockDim.x)
    buf[t + pad * div_by(t, pl.magic_n)] = spec[base + t];
  __syncthreads();
  double e = 0.0;
  for (int back = 0; back < 2; ++back) {
    lds_fft<T, kFftPoints<T, LONG>>(buf, f, pl, LONG ? tw : s_tw);
    if (back) break;
    for (int t = threadIdx.x; (int)threadIdx.x < threads && t < f.lines * p.nx; t += threads)
      e += convolve<T>(buf[t + pad * div_by(t, pl.magic_n)], theta[base + t]);
    __syncthreads();
  }
  for (int t = threadIdx.x; t < f.lines * p.nx; t += blockDim.x) {
    Cx<T> v = buf[t + pad * div_by(t, pl.magic_n)];
    v.y = -v.y;
    spec[base + t] = v;
  }
  block_energy(plane_weight(p, k) * e, &epart[bid_]);
}

template <class T, bool LONG = false>
__global__ void __launch_bounds__(kPmeBlock, LONG ? 2 : kPmeWaves<T>) k_fft_x_conv(PmeParams p, FftPlan pl, int llog,
                                                          const Cx<T> *__restrict__ tw, const T *__restrict__ theta,
                                                          Cx<T> *__restrict__ spec, double *__restrict__ epart) {
  fft_x_conv_body<T, LONG>(xcd_block(blockIdx.x, gridDim.x), gridDim.x, p, pl, llog, blockDim.x, tw, theta, spec, epart);
}

// The y pass, the x pass with the convolution and the inverse y pass of one
// plane k in one block (for planes of at most kFftPlanePoints): the plane
// stays in LDS, rows of odd length, so both directions are transformed in
// place without a transpose.  18 -> 13 us at 30 x 30 points alone.  The conj-out of the inverse x transform and the
// conj-in of the inverse y transform cancel, so only the last conj remains.
constexpr int kFftPlanePoints = kFftMax;
template <class T>
__device__ __forceinline__ void fft_plane_conv_body(const int bid_, const int nbk_, const PmeParams &p,
                                                    const FftPlan &ply, const FftPlan &plx, int threads,
                                                    const Cx<T> *__restrict__ twy, const Cx<T> *__restrict__ twx,
                                                    const T *__restrict__ theta, Cx<T> *__restrict__ spec,
                                                    double *__restrict__ epart) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  Cx<T> *const s_twx = reinterpret_cast<Cx<T> *>(smem_raw);
  Cx<T> *const s_twy = s_twx + p.nx;
  Cx<T> *const buf = s_twy + p.ny;
  const int k = bid_, nxy = p.nx * p.ny, row = p.nx | 1, pad = row - p.nx;
  const size_t base = (size_t)k * nxy;
  lds_twiddles(s_twx, twx, p.nx);
  lds_twiddles(s_twy, twy, p.ny);
  for (int t = threadIdx.x; t < nxy; t += blockDim.x) buf[t + pad * div_by(t, plx.magic_n)] = spec[base + t];
  __shared__ FftPlan s_pl[2];  // read by index: y, x
  if (threadIdx.x == 0) {
    s_pl[0] = ply;
    s_pl[1] = plx;
  }
  __syncthreads();
  const int blog = 31 - __clz((int)blockDim.x);
  double e = 0.0;
  // y, x, (influence function) x, y
  for (int turn = 0; turn < 4; ++turn) {
    const bool y = turn == 0 || turn == 3;
    const FftPlan &pl = s_pl[y ? 0 : 1];
    const int n = y ? p.ny : p.nx, nlines = y ? p.nx : p.ny;
    // as many lines at a time as leave n / kFftPerThread threads or more for each
    const int nlog = nlines > 1 ? 32 - __clz(nlines - 1) : 0;
    const int need = n > kFftPerThread ? 32 - __clz((n - 1) / kFftPerThread) : 0;
    const int llog = min(nlog, blog - need);
    if (turn == 2) {
      for (int t = threadIdx.x; (int)threadIdx.x < threads && t < nxy; t += threads)
        e += convolve<T>(buf[t + pad * div_by(t, plx.magic_n)], theta[base + t]);
      __syncthreads();
    }
    for (int l0 = 0; l0 < nlines; l0 += 1 << llog)
      lds_fft<T>(buf + l0 * (y ? 1 : row), FftLines{llog, min(1 << llog, nlines - l0), y ? 1 : row, y ? row : 1}, pl,
                 y ? s_twy : s_twx);
  }
  for (int t = threadIdx.x; t < nxy; t += blockDim.x) {
    Cx<T> v = buf[t + pad * div_by(t, plx.magic_n)];
    v.y = -v.y;
    spec[base + t] = v;
  }
  block_energy(plane_weight(p, k) * e, &epart[k]);
}

template <class T>
__global__ void __launch_bounds__(kPmeBlock, kPmeWaves<T>) k_fft_plane_conv(
    PmeParams p, FftPlan ply, FftPlan plx, const Cx<T> *__restrict__ twy, const Cx<T> *__restrict__ twx,
    const T *__restrict__ theta, Cx<T> *__restrict__ spec, double *__restrict__ epart) {
  fft_plane_conv_body<T>(blockIdx.x, gridDim.x, p, ply, plx, blockDim.x, twy, twx, theta, spec, epart);
}

// Inverse z transform and force gather of one tile (Grid.h:159-189): the
// potential of lines 2 l and 2 l + 1 is the real and the (negated) imaginary
// part of transform l; each lane takes one atom, sums the stencil rows
// inside the tile and adds the atom's force.
template <bool MIXED, int P, bool LONG = false>
__device__ __forceinline__ void pme_z_gather_body(
    const int bid_, const int nbk_, const PmeParams &p, const FftPlan &pl, const int2 *__restrict__ tcol,
    const int *__restrict__ colsc,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ pmw,
    const int2 *__restrict__ pmb, const Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ tw,
    const Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ spec,
    typename AccT<MIXED>::type *__restrict__ facc) {
  using T = typename std::conditional<MIXED, float, double>::type;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int s_q[LONG ? 1 : kPmeBlock / kWave][128];
  Cx<T> *const s_tw = reinterpret_cast<Cx<T> *>(smem_raw);
  Cx<T> *const buf = LONG ? s_tw : s_tw + p.nz;
  const int nzs = pme_line(p.nz, P), lines = p.tx * p.ty;
  const int tjy = bid_ / p.ntx, tix = bid_ - tjy * p.ntx;
  const int i0 = tix * p.tx, j0 = tjy * p.ty;
  if (!LONG) lds_twiddles(s_tw, tw, p.nz);
  const int np = lines >> 1, nplog = 31 - __clz(np), hlog = 31 - __clz(p.tx) - 1;
  for (int t = threadIdx.x; t < p.nzh << nplog; t += blockDim.x) {
    const int l = t & (np - 1), k = t >> nplog;
    const int i = i0 + 2 * (l & ((1 << hlog) - 1)), j = j0 + (l >> hlog);
    Cx<T> a{(T)0, (T)0}, b{(T)0, (T)0};
    if (i < p.nx && j < p.ny) {
      const Cx<T> *o = spec + ((size_t)k * p.ny + j) * p.nx + i;
      a = o[0];
      if (i + 1 < p.nx) b = o[1];
    }
    // the lines are real: k = 0 and the middle of an even line have no
    // imaginary part
    const bool self = k == 0 || 2 * k == p.nz;
    if (self) a.y = b.y = (T)0;
    // conj-in of a + i b, and of its Hermitian completion at nz - k
    buf[l * nzs + k] = Cx<T>{a.x - b.y, -(a.y + b.x)};
    if (!self) buf[l * nzs + p.nz - k] = Cx<T>{a.x + b.y, a.y - b.x};
  }
  __syncthreads();
  pme_tile_fft<T, LONG>(buf, np, p.nz, nzs, pl, LONG ? tw : s_tw);
  for (int t = threadIdx.x; t < np * (P - 1); t += blockDim.x) {
    const int l = t & (np - 1), k = t >> nplog;
    int g = k;
    while (g >= p.nz) g -= p.nz;
    buf[l * nzs + p.nz + k] = buf[l * nzs + g];
  }
  __syncthreads();
  const T *const pot = reinterpret_cast<const T *>(buf);
  pme_tile_atoms<P, LONG>(p, tcol, tix, tjy, colsc, pmb, s_q, [&](int cnt, int slot) {
    if ((int)(threadIdx.x & 63) >= cnt) return;
    const auto a = pmw[slot];
    const int2 b = pmb[slot];
    T wx[P], wy[P], wz[P], dx[P], dy[P], dz[P];
    bspline_w<P, T>(a.x, wx, dx);
    bspline_w<P, T>(a.y, wy, dy);
    bspline_w<P, T>(a.z, wz, dz);
    const int bx = (b.x & 0xffff), by = b.x >> 16;
    T fx = 0, fy = 0, fz = 0;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int li = wrap_grid(bx + i, p.nx) - i0;
      if ((unsigned)li >= (unsigned)p.tx) continue;
      T gx = 0, gy = 0, gz = 0;  // this x row of the stencil, without its x weights
#pragma unroll
      for (int j = 0; j < P; ++j) {
        const int lj = wrap_grid(by + j, p.ny) - j0;
        if ((unsigned)lj >= (unsigned)p.ty) continue;
        const int line = lj * p.tx + li;
        const T *const r = pot + ((line >> 1) * nzs + b.y) * 2 + (line & 1);
        T s = 0, d = 0;
#pragma unroll
        for (int k = 0; k < P; ++k) {
          const T v = r[2 * k];
          s += v * wz[k];
          d += v * dz[k];
        }
        gx += wy[j] * s;
        gy += dy[j] * s;
        gz += wy[j] * d;
      }
      // odd lines hold the negated potential
      const T w = (li & 1) ? -wx[i] : wx[i], v = (li & 1) ? -dx[i] : dx[i];
      fx -= v * gx;
      fy -= w * gy;
      fz -= w * gz;
    }
    AccT<MIXED>::add(&facc[3 * slot], fx * (T)p.hxr * a.w);
    AccT<MIXED>::add(&facc[3 * slot + 1], fy * (T)p.hyr * a.w);
    AccT<MIXED>::add(&facc[3 * slot + 2], fz * (T)p.hzr * a.w);
  });
}

template <bool MIXED, int P, bool LONG = false>
__global__ void __launch_bounds__(kPmeBlock, LONG ? 2 : MIXED ? 8 : 4) k_pme_z_gather(
    PmeParams p, FftPlan pl, const int2 *__restrict__ tcol, const int *__restrict__ colsc,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ pmw,
    const int2 *__restrict__ pmb, const Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ tw,
    const Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ spec,
    typename AccT<MIXED>::type *__restrict__ facc) {
  pme_z_gather_body<MIXED, P, LONG>(xcd_block(blockIdx.x, gridDim.x), gridDim.x, p, pl, tcol, colsc, pmw, pmb, tw, spec,
                              facc);
}

// ---------------------------------------------------------------------------
// 6. Finalize: sorted accumulators -> caller's AoS order, FP64.
// The accumulators are cleared as they are read, and so are the pair
// kernel's tile counter and the boundary-pair count, so the next force pass
// starts from zero without a separate clearing launch (padding slots are
// never accumulated into).
// What the last pass of a chunk of MD steps hands to the host: the chunk's
// displacement record (at most 256 steps) and the overflow flag, both complete
// by then, into pinned memory.
struct ChunkEnd {
  const unsigned *record;
  int steps;  // 0: none
  const int *overflow;
  unsigned *host_record, *host_overflow;
};

template <bool MIXED>
__device__ __forceinline__ void unsort_forces_body(const int bid_, const int nbk_, int n, const int *__restrict__ slot,
                                                   typename AccT<MIXED>::type *__restrict__ facc,
                                                   double *__restrict__ fout, int *__restrict__ tilectr,
                                                   int *__restrict__ nborder, const ChunkEnd &end = {}) {
  int a = bid_ * blockDim.x + threadIdx.x;
  if (a == 0) {
    *tilectr = 0;
    *nborder = 0;
  }
  if (a < end.steps) {
    end.host_record[a] = end.record[a];
    if (a == 0) *end.host_overflow = (unsigned)*end.overflow;
    __threadfence_system();
  }
  if (a >= n) return;
  const int s = slot[a];
  for (int k = 0; k < 3; ++k) {
    if (MIXED)
      fout[3 * a + k] = (double)(long long)facc[3 * s + k] * (1.0 / kForceScale);
    else
      fout[3 * a + k] = ((const double *)facc)[3 * s + k];
    facc[3 * s + k] = 0;
  }
}

template <bool MIXED>
__global__ void k_unsort_forces(int n, const int *__restrict__ slot, typename AccT<MIXED>::type *__restrict__ facc,
                                double *__restrict__ fout, int *__restrict__ tilectr, int *__restrict__ nborder,
                                ChunkEnd end) {
  unsort_forces_body<MIXED>(blockIdx.x, gridDim.x, n, slot, facc, fout, tilectr, nborder, end);
}

// Deterministic energy/pair-stat reduction in one block, in index order.
// Pair energies per tile are int64 fixed point (2^-32) when pair_fixed (the
// mixed form: their sum is exact, whatever tiles the schedule made), FP64
// otherwise.
struct EnergyArgs {
  int ntiles_cap;
  const int *ntiles;
  const double *pair_e;
  int pair_fixed, nrecip;
  const double *recip_e;
  int ncorr;
  const double *corr_e;
  const long long *npairs;
  const unsigned long long *hash;
  int stats;
  const unsigned long long *border_e, *border_stat;
  double *out;
  long long *out_np;
  unsigned long long *out_hash;
};

__device__ __forceinline__ void reduce_energy_body(const EnergyArgs &a) {
  __shared__ double sd[4][1024 / kWave];
  __shared__ long long sn[1024 / kWave];
  __shared__ unsigned long long sh[1024 / kWave];
  __shared__ long long sf[2][1024 / kWave];
  const int nt = min(*a.ntiles, a.ntiles_cap);
  double c = 0, l = 0, r = 0, k = 0;
  long long np = 0, cf = 0, lf = 0;
  unsigned long long h = 0;
  for (int i = threadIdx.x; i < nt; i += blockDim.x) {
    if (a.pair_fixed) {
      cf += __double_as_longlong(a.pair_e[2 * i]);
      lf += __double_as_longlong(a.pair_e[2 * i + 1]);
    } else {
      c += a.pair_e[2 * i];
      l += a.pair_e[2 * i + 1];
    }
    if (a.stats) {
      np += a.npairs[i];
      h += a.hash[i];
    }
  }
  for (int i = threadIdx.x; i < a.nrecip; i += blockDim.x) r += a.recip_e[i];
  for (int i = threadIdx.x; i < a.ncorr; i += blockDim.x) k += a.corr_e[i];
  c = wave_sum(c);
  l = wave_sum(l);
  cf = wave_sum(cf);
  lf = wave_sum(lf);
  r = wave_sum(r);
  k = wave_sum(k);
  np = wave_sum(np);
  h = wave_sum(h);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sd[0][w] = c;
    sd[1][w] = l;
    sd[2][w] = r;
    sd[3][w] = k;
    sn[w] = np;
    sh[w] = h;
    sf[0][w] = cf;
    sf[1][w] = lf;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double C = 0, Lj = 0, Rr = 0, K = 0;
    long long N = 0, CF = 0, LF = 0;
    unsigned long long H = 0;
    for (int i = 0; i < (int)(blockDim.x / kWave); ++i) {
      CF += sf[0][i];
      LF += sf[1][i];
      C += sd[0][i];
      Lj += sd[1][i];
      Rr += sd[2][i];
      K += sd[3][i];
      N += sn[i];
      H += sh[i];
    }
    a.out[0] = C + (double)(CF + (long long)a.border_e[0]) * (1.0 / kForceScale);
    a.out[1] = Lj + (double)(LF + (long long)a.border_e[1]) * (1.0 / kForceScale);
    a.out[2] = 0.5 * Rr;
    a.out[3] = K;
    *a.out_np = N + (long long)a.border_stat[0];
    *a.out_hash = H + a.border_stat[1];
  }
}

static __global__ void k_reduce_energy(EnergyArgs a) { reduce_energy_body(a); }

// The end of a pass whose energies are wanted: block 0 reduces them, the others
// bring the forces into the caller's order (the two in turn took 6 + 11 us at
// 26,000 atoms, and a launch).
constexpr int kEndBlock = 1024;
template <bool MIXED>
__device__ __forceinline__ void unsort_energy_body(const int bid_, int n, const int *__restrict__ slot,
                                                   typename AccT<MIXED>::type *__restrict__ facc,
                                                   double *__restrict__ fout, int *__restrict__ tilectr,
                                                   int *__restrict__ nborder, const EnergyArgs &a) {
  if (bid_ == 0)
    reduce_energy_body(a);
  else
    unsort_forces_body<MIXED>(bid_ - 1, 0, n, slot, facc, fout, tilectr, nborder);
}

template <bool MIXED>
__global__ void __launch_bounds__(kEndBlock) k_unsort_energy(int n, const int *__restrict__ slot,
                                                             typename AccT<MIXED>::type *__restrict__ facc,
                                                             double *__restrict__ fout, int *__restrict__ tilectr,
                                                             int *__restrict__ nborder, EnergyArgs a) {
  unsort_energy_body<MIXED>(blockIdx.x, n, slot, facc, fout, tilectr, nborder, a);
}

// Results to the host: up to five arrays of 8-byte words one after the other
// into pinned memory, in one launch instead of a copy each.
struct OutArgs {
  const unsigned long long *src[5];
  long long end[5];  // running ends (unused: the last end again)
  unsigned long long *dst;
};
__device__ __forceinline__ void out_body(int bid, int nbk, const OutArgs &a) {
  for (long long i = (long long)bid * blockDim.x + threadIdx.x; i < a.end[4]; i += (long long)nbk * blockDim.x) {
    const unsigned long long *p = a.src[0] + i;
#pragma unroll
    for (int k = 1; k < 5; ++k)
      if (i >= a.end[k - 1]) p = a.src[k] + (i - a.end[k - 1]);
    a.dst[i] = *p;
  }
}
static __global__ void __launch_bounds__(256) k_out(OutArgs a) { out_body(blockIdx.x, gridDim.x, a); }

// ---------------------------------------------------------------------------
// 7. Device-resident MD: bonded terms, leapfrog kick/drift, kinetic energy.

// Zeroes up to 8 ranges of 64-bit words in one launch (blockIdx.y = range).
struct ZeroRanges {
  unsigned long long *p[8];
  long long n[8];
};
static __global__ void k_zero(ZeroRanges z) {
  const int r = blockIdx.y;
  unsigned long long *p = z.p[r];
  const long long n = z.n[r];
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = 0ull;
}

// Reference minimalDifference(c1, c2) = c2 - c1 folded to the minimal image.
__device__ inline void min_diff(const double *x, int c1, int c2, const Box &bx, double *d) {
  double d2;
  for (int k = 0; k < 3; ++k) d[k] = x[3 * c2 + k] - x[3 * c1 + k];
  d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  if (d2 > bx.D) {
    for (int k = 0; k < 3; ++k) {
      if (d[k] < -bx.H2[k])
        d[k] += bx.H[k];
      else if (d[k] > bx.H2[k])
        d[k] -= bx.H[k];
    }
    d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    if (d2 > bx.D)
      for (int k = 0; k < 3; ++k) d[k] -= bx.L[k] * rint(bx.Lr[k] * d[k]);
  }
}

// The terms of one atom, by atom: exclusion corrections (partner, class),
// bonds (partner; k, r0) and angles (first, vertex, third atom, the atom's
// place in it; k, theta0).  Each term is listed once for every atom it acts on.
struct AtomTerms {
  const int *eptr;        // [n + 1] (null: no corrections)
  const int2 *excl;
  const int2 *mptr;       // [n + 1] first bond and first angle (null: none)
  const int *bond;
  const double2 *bpar;
  const int4 *angle;
  const double2 *apar;
};

// Exclusion correction (NonbondedPMEwaldSystemForce.h:874-911, exact erf),
// harmonic bonds (BondSystemForce.h:97-118) and angles without Urey-Bradley
// (AngleSystemForce.h:95-147), FP64.  One thread per sorted slot sums its
// atom's terms and adds the atom's force once: a term is evaluated for each
// of its atoms, but the 15 to 33 scattered adds of a water molecule (which
// bound the pass that took a term per thread: each is a memory-side atomic)
// become 9 in slot order.  A million atoms 0.51 -> 0.11 ms beside the pair
// kernel, 26,000 atoms 17 -> 12 us.  Energies are counted by the atom of the
// lower index, the first atom of a bond, the vertex of an angle.
template <bool MIXED>
__device__ __forceinline__ void atom_terms_block(int blk, int npad, const int *__restrict__ perm,
                                                 const double *__restrict__ x, const double *__restrict__ q,
                                                 const Box &box, double alpha, double csf, const AtomTerms &at,
                                                 typename AccT<MIXED>::type *__restrict__ facc,
                                                 double *__restrict__ corr_e, double *__restrict__ bond_e) {
  __shared__ double s_e[3][kPairBlock / kWave];
  const int s = blk * blockDim.x + threadIdx.x;
  const int a = s < npad ? perm[s] : -1;
  double en = 0.0, eb = 0.0, ea = 0.0;
  if (a >= 0) {
    double f[3] = {0, 0, 0};
    if (at.eptr) {
      const double qa = q[a];
      const int t1 = at.eptr[a + 1];
      for (int t = at.eptr[a]; t < t1; ++t) {
        const int2 e = at.excl[t];
        double d[3];
        min_diff(x, a, e.x, box, d);
        const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        double qq = qa * q[e.x];
        if (e.y == 2) qq *= 1 - csf;
        const double r = sqrt(r2), rr = 1.0 / r;
        const double ee = erf(alpha * r) * rr;
        if (a < e.x) en -= qq * ee;
        const double fr = qq * (2.0 * alpha / sqrt(M_PI) * exp(-alpha * alpha * r2) - ee) * rr * rr;
        for (int k = 0; k < 3; ++k) f[k] -= d[k] * fr;
      }
    }
    if (at.mptr) {
      const int2 m0 = at.mptr[a], m1 = at.mptr[a + 1];
      for (int t = m0.x; t < m1.x; ++t) {
        const int b = at.bond[t];
        const double2 p = at.bpar[t];
        double r12[3];
        min_diff(x, b, a, box, r12);
        const double r = sqrt(r12[0] * r12[0] + r12[1] * r12[1] + r12[2] * r12[2]);
        const double c = -2.0 * p.x * (r - p.y) / r;
        for (int k = 0; k < 3; ++k) f[k] += r12[k] * c;
        if (a < b) eb += p.x * (r - p.y) * (r - p.y);
      }
      for (int t = m0.y; t < m1.y; ++t) {
        const int4 g = at.angle[t];
        const double2 p = at.apar[t];
        double r12[3], r32[3];
        min_diff(x, g.y, g.x, box, r12);  // atom1 - atom2
        min_diff(x, g.y, g.z, box, r32);  // atom3 - atom2
        const double d12 = sqrt(r12[0] * r12[0] + r12[1] * r12[1] + r12[2] * r12[2]);
        const double d32 = sqrt(r32[0] * r32[0] + r32[1] * r32[1] + r32[2] * r32[2]);
        const double cx = r12[1] * r32[2] - r12[2] * r32[1], cy = r12[2] * r32[0] - r12[0] * r32[2],
                     cz = r12[0] * r32[1] - r12[1] * r32[0];
        const double theta =
            atan2(sqrt(cx * cx + cy * cy + cz * cz), r12[0] * r32[0] + r12[1] * r32[1] + r12[2] * r32[2]);
        const double st = sin(theta), ct = cos(theta);
        const double dpot = 2.0 * p.x * (theta - p.y);
        const double g1 = -dpot / (st * d12), g3 = -dpot / (st * d32);
        for (int k = 0; k < 3; ++k) {
          const double u1 = r12[k] / d12, u3 = r32[k] / d32;
          const double f1 = (u1 * ct - u3) * g1, f3 = (u3 * ct - u1) * g3;
          f[k] += g.w == 0 ? f1 : (g.w == 1 ? -f1 - f3 : f3);
        }
        if (g.w == 1) ea += p.x * (theta - p.y) * (theta - p.y);
      }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) AccT<MIXED>::add(&facc[3 * s + k], f[k]);
  }
  en = wave_sum(en);
  eb = wave_sum(eb);
  ea = wave_sum(ea);
  if ((threadIdx.x & 63) == 0) {
    s_e[0][threadIdx.x >> 6] = en;
    s_e[1][threadIdx.x >> 6] = eb;
    s_e[2][threadIdx.x >> 6] = ea;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double c = 0, b = 0, g = 0;
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) {
      c += s_e[0][w];
      b += s_e[1][w];
      g += s_e[2][w];
    }
    corr_e[blk] = c;
    if (at.mptr) {
      bond_e[2 * blk] = b;
      bond_e[2 * blk + 1] = g;
    }
  }
}

// The small FP64 passes that follow the pair and PME kernels, in one launch
// of 256-thread blocks: [0, border) boundary pairs, then the atoms' exclusion
// corrections and bonded terms.
template <bool MIXED>
struct FixupArgs {
  using R4 = typename Real4<typename std::conditional<MIXED, float, double>::type>::type;
  int border_blocks;
  // boundary pairs
  PairParams pp;
  int stats;
  const int2 *border;
  const int *nborder;
  int maxborder;
  const R4 *xs;
  const float4 *sorg;
  const int *ts, *perm;
  const double *xorig, *ljtab;
  const int *eptr;
  const int2 *elist;
  unsigned long long *border_e, *border_stat;
  // terms of single atoms
  AtomTerms at;
  int npad;
  const double *q;
  double alpha, csf;
  double *corr_e, *bond_e;
  typename AccT<MIXED>::type *facc;
};

template <bool MIXED, int COUL, int LJSW, int CSW>
__device__ __forceinline__ void fixups_body(const int bid_, const int nbk_, FixupArgs<MIXED> a) {
  int b = bid_;
  if (b < a.border_blocks) {
    border_pairs<MIXED, COUL, LJSW, CSW>(b, a.border_blocks, a.pp, a.stats, a.border, a.nborder, a.maxborder, a.xs,
                                         a.sorg, a.ts, a.perm, a.xorig, a.ljtab, a.eptr, a.elist, a.facc, a.border_e,
                                         a.border_stat);
    return;
  }
  atom_terms_block<MIXED>(b - a.border_blocks, a.npad, a.perm, a.xorig, a.q, a.pp.box, a.alpha, a.csf, a.at, a.facc,
                          a.corr_e, a.bond_e);
}

template <bool MIXED, int COUL, int LJSW, int CSW>
__global__ void __launch_bounds__(256) k_fixups(FixupArgs<MIXED> a) {
  fixups_body<MIXED, COUL, LJSW, CSW>(blockIdx.x, gridDim.x, a);
}

// Charge spread and the atoms' terms in one launch, where the spread has the
// device to itself: its blocks leave most CUs idle, and the terms, a chain of
// dependent FP64 operations of 9 us, no longer follow the pair kernel.  A step of
// 1,500 atoms 61.6 -> 60.2 us, 9,400 atoms 81.7 -> 80.5.
template <bool MIXED, int P>
__global__ void __launch_bounds__(kPmeBlock, 4) k_pme_spread_terms(
    PmeParams p, FftPlan pl, const int2 *__restrict__ tcol, const int *__restrict__ colsc,
    const typename Real4<typename std::conditional<MIXED, float, double>::type>::type *__restrict__ pmw,
    const int2 *__restrict__ pmb, const Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ tw,
    Cx<typename std::conditional<MIXED, float, double>::type> *__restrict__ spec, FixupArgs<MIXED> a) {
  const int tiles = p.ntx * p.nty, b = blockIdx.x;
  if (b < tiles)
    pme_spread_z_body<MIXED, P>(xcd_block(b, tiles), tiles, p, pl, tcol, colsc, pmw, pmb, tw, spec);
  else
    atom_terms_block<MIXED>(b - tiles, a.npad, a.perm, a.xorig, a.q, a.pp.box, a.alpha, a.csf, a.at, a.facc, a.corr_e,
                            a.bond_e);
}

// Velocity kicks of one leapfrog step.  Leapfrog (LeapfrogIntegrator.cpp):
// v += F h_kick / m.  Langevin leapfrog (LangevinLeapfrogIntegrator.cpp:
// 44-71): nhalf half kicks v = v vdt + F fdt / m + g sqrt(fc / m) ndt, g a
// standard normal triple for (atom, global half-kick index).
// One kick: h_kick = fraction of the step times h; Langevin half kicks
// numbered half0, half0 + 1 (plus 2 x *step_dev when step_dev is set: a
// captured chunk reads its first step index from device memory, half0 then
// being relative to it, modulo 2^64).
struct Kick {
  double h_kick;
  int langevin, nhalf;
  unsigned long long half0, seed;
  double vdt, fdt, ndt, fc;
  const unsigned long long *step_dev;
};

__device__ inline void apply_kick(const Kick &kk, int a, const double f[3], double minv, double v[3]) {
  if (!kk.langevin) {
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] += f[k] * kk.h_kick * minv;
    return;
  }
  const double sfm = sqrt(kk.fc * minv) * kk.ndt;
  const unsigned long long h0 = kk.half0 + (kk.step_dev ? 2ull * *kk.step_dev : 0ull);
  for (int hh = 0; hh < kk.nhalf; ++hh) {
    double g[3];
    langevin_gauss3(kk.seed, h0 + hh, (uint32_t)a, g);
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = v[k] * kk.vdt + f[k] * kk.fdt * minv + g[k] * sfm;
  }
}

// The largest of a block's values (>= 0) folded into *dmax: one atomic a block.
// Adds to one address take about 12 ns each whatever the grid; one per wave
// bound the kick and drift: 1,000,000 atoms 185 -> 55 us, 26,000 atoms 8.1 -> 5.1.
__device__ __forceinline__ void record_max(float d, unsigned *__restrict__ dmax) {
  __shared__ float s_d[256 / kWave];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) d = fmaxf(d, __shfl_xor(d, m));
  if ((threadIdx.x & 63) == 0) s_d[threadIdx.x >> 6] = d;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 256 / kWave; ++w) d = fmaxf(d, s_d[w]);
    if (d > 0.f) atomicMax(dmax, __float_as_uint(d));
  }
}

// Kick (v += F kick h / m) and drift (x += v h) of every atom, FP64
// (LeapfrogIntegrator.cpp:33-87).  The pair kernel's sorted coordinates then
// follow each atom continuously from its wrapped position at the last list
// build (xs64), since list entries carry a fixed image shift, and the largest
// squared displacement since that build is folded into dmax (float bits).
template <class R>
__device__ __forceinline__ void kick_drift_body(const int bid_, const int nbk_, int n, Kick kk, double h,
                                                const int *__restrict__ perm, const double *__restrict__ fout,
                                                double *__restrict__ v, double *__restrict__ x,
                                                const double4 *__restrict__ xbuild,
                                                typename Real4<R>::type *__restrict__ xs,
                                                const double4 *__restrict__ xs64, const float4 *__restrict__ sorg,
                                                unsigned int *__restrict__ dmax, const PmeParams &pme,
                                                PmeSlots<R> rec) {
  const int s = bid_ * blockDim.x + threadIdx.x;
  float d2f = 0.f;
  const int a = s < n ? perm[s] : -1;  // n counts slots; padding slots have a < 0
  if (a >= 0) {
    double dd[3], xn[3], vv[3] = {v[3 * a], v[3 * a + 1], v[3 * a + 2]};
    const double ff[3] = {fout[3 * a], fout[3 * a + 1], fout[3 * a + 2]};
    const double4 xb = xbuild[s];
    apply_kick(kk, a, ff, xb.w, vv);
    double d2 = 0;
    for (int k = 0; k < 3; ++k) {
      v[3 * a + k] = vv[k];
      const double xk = x[3 * a + k] + vv[k] * h;
      x[3 * a + k] = xn[k] = xk;
      dd[k] = xk - (k == 0 ? xb.x : k == 1 ? xb.y : xb.z);
      d2 += dd[k] * dd[k];
    }
    d2f = (float)d2;
    const double4 b = xs64[s];
    const float4 o = sorg[s / kSuperSize];
    typename Real4<R>::type r = xs[s];
    r.x = (R)((b.x + dd[0]) - (double)o.x);
    r.y = (R)((b.y + dd[1]) - (double)o.y);
    r.z = (R)((b.z + dd[2]) - (double)o.z);
    xs[s] = r;
    if (rec.w) pme_record<R>(pme, rec, s, true, xn, b.w);
  }
  record_max(d2f, dmax);
}

template <class R>
__global__ void k_kick_drift(int n, Kick kk, double h, const int *__restrict__ perm,
                             const double *__restrict__ fout, double *__restrict__ v, double *__restrict__ x,
                             const double4 *__restrict__ xbuild,
                             typename Real4<R>::type *__restrict__ xs, const double4 *__restrict__ xs64,
                             const float4 *__restrict__ sorg, unsigned int *__restrict__ dmax, PmeParams pme,
                             PmeSlots<R> rec) {
  kick_drift_body<R>(blockIdx.x, gridDim.x, n, kk, h, perm, fout, v, x, xbuild, xs, xs64, sorg, dmax, pme,
                     rec);
}

// The end of one MD step and the start of the next in one pass over the
// sorted slots: the step's forces leave the accumulators (cleared, with the
// pass counters) for the next step's kick and drift (the force array is
// written only where a chunk of steps ends).  Bound by memory: positions and
// velocities are in the caller's order, each 24 bytes of one or two lines;
// build positions and inverse masses lie by slot.
template <bool MIXED, class R>
__device__ __forceinline__ void unsort_kick_drift_body(const int bid_, const int nbk_, int n, const Kick &kk, double h,
                                                       const int *__restrict__ perm,
                                                       typename AccT<MIXED>::type *__restrict__ facc,
                                                       int *__restrict__ tilectr, int *__restrict__ nborder,
                                                       double *__restrict__ v, double *__restrict__ x,
                                                       const double4 *__restrict__ xbuild,
                                                       typename Real4<R>::type *__restrict__ xs,
                                                       const double4 *__restrict__ xs64,
                                                       const float4 *__restrict__ sorg,
                                                       unsigned int *__restrict__ dmax, const PmeParams &pme,
                                                       PmeSlots<R> rec) {
  const int s = bid_ * blockDim.x + threadIdx.x;
  if (s == 0) {
    *tilectr = 0;
    *nborder = 0;
  }
  float d2f = 0.f;
  const int a = s < n ? perm[s] : -1;  // n counts slots; padding slots have a < 0
  if (a >= 0) {
    double ff[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (MIXED)
        ff[k] = (double)(long long)facc[3 * s + k] * (1.0 / kForceScale);
      else
        ff[k] = ((const double *)facc)[3 * s + k];
      facc[3 * s + k] = 0;
    }
    double dd[3], xn[3], vv[3] = {v[3 * a], v[3 * a + 1], v[3 * a + 2]};
    const double4 xb = xbuild[s];
    apply_kick(kk, a, ff, xb.w, vv);
    double d2 = 0;
    for (int k = 0; k < 3; ++k) {
      v[3 * a + k] = vv[k];
      const double xk = x[3 * a + k] + vv[k] * h;
      x[3 * a + k] = xn[k] = xk;
      dd[k] = xk - (k == 0 ? xb.x : k == 1 ? xb.y : xb.z);
      d2 += dd[k] * dd[k];
    }
    d2f = (float)d2;
    const double4 b = xs64[s];
    const float4 o = sorg[s / kSuperSize];
    typename Real4<R>::type r = xs[s];
    r.x = (R)((b.x + dd[0]) - (double)o.x);
    r.y = (R)((b.y + dd[1]) - (double)o.y);
    r.z = (R)((b.z + dd[2]) - (double)o.z);
    xs[s] = r;
    if (rec.w) pme_record<R>(pme, rec, s, true, xn, b.w);
  }
  record_max(d2f, dmax);
}

template <bool MIXED, class R>
__global__ void k_unsort_kick_drift(int n, Kick kk, double h, const int *__restrict__ perm,
                                    typename AccT<MIXED>::type *__restrict__ facc, int *__restrict__ tilectr,
                                    int *__restrict__ nborder, double *__restrict__ v, double *__restrict__ x, const double4 *__restrict__ xbuild,
                                    typename Real4<R>::type *__restrict__ xs, const double4 *__restrict__ xs64,
                                    const float4 *__restrict__ sorg, unsigned int *__restrict__ dmax, PmeParams pme,
                                    PmeSlots<R> rec) {
  unsort_kick_drift_body<MIXED, R>(blockIdx.x, gridDim.x, n, kk, h, perm, facc, tilectr, nborder, v, x,
                                   xbuild, xs, xs64, sorg, dmax, pme, rec);
}

// Start of an MD chunk in one launch: the committed state (x, v, f: m3 =
// 3N doubles each) is backed up for a rollback, the overflow flags (2) and
// the chunk's displacement record (nrec) are cleared.
__device__ __forceinline__ void chunk_begin_body(const int bid_, const int nbk_, long long m3,
                                                 const double *__restrict__ x, const double *__restrict__ v,
                                                 const double *__restrict__ f, double *__restrict__ xbak,
                                                 double *__restrict__ vbak, double *__restrict__ fbak,
                                                 int *__restrict__ overflow, unsigned *__restrict__ dmax, int nrec) {
  const long long i = (long long)bid_ * blockDim.x + threadIdx.x;
  if (i < m3) {
    xbak[i] = x[i];
    vbak[i] = v[i];
    fbak[i] = f[i];
  }
  if (i < 2) overflow[i] = 0;
  if (i < nrec) dmax[i] = 0u;
}

static __global__ void k_chunk_begin(long long m3, const double *__restrict__ x, const double *__restrict__ v,
                              const double *__restrict__ f, double *__restrict__ xbak, double *__restrict__ vbak,
                              double *__restrict__ fbak, int *__restrict__ overflow, unsigned *__restrict__ dmax,
                              int nrec) {
  chunk_begin_body(blockIdx.x, gridDim.x, m3, x, v, f, xbak, vbak, fbak, overflow, dmax, nrec);
}

static __global__ void k_set_u64(unsigned long long *p, unsigned long long v) { *p = v; }

__device__ __forceinline__ void half_kick_body(const int bid_, const int nbk_, int n, Kick kk,
                                               const double *__restrict__ fout, const double *__restrict__ minv,
                                               double *__restrict__ v) {
  const int a = bid_ * blockDim.x + threadIdx.x;
  if (a >= n) return;
  double vv[3] = {v[3 * a], v[3 * a + 1], v[3 * a + 2]};
  const double ff[3] = {fout[3 * a], fout[3 * a + 1], fout[3 * a + 2]};
  apply_kick(kk, a, ff, minv[a], vv);
  for (int k = 0; k < 3; ++k) v[3 * a + k] = vv[k];
}

static __global__ void k_half_kick(int n, Kick kk, const double *__restrict__ fout, const double *__restrict__ minv,
                            double *__restrict__ v) {
  half_kick_body(blockIdx.x, gridDim.x, n, kk, fout, minv, v);
}

// Kinetic energy 0.5 sum m v^2 into per-block partials.
static __global__ void k_kinetic(int n, const double *__restrict__ v, const double *__restrict__ minv,
                          double *__restrict__ epart) {
  __shared__ double s_e[kPairBlock / kWave];
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  double e = 0.0;
  if (a < n) e = 0.5 * (v[3 * a] * v[3 * a] + v[3 * a + 1] * v[3 * a + 1] + v[3 * a + 2] * v[3 * a + 2]) / minv[a];
  e = wave_sum(e);
  if ((threadIdx.x & 63) == 0) s_e[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0;
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) t += s_e[w];
    epart[blockIdx.x] = t;
  }
}

}  // namespace pmx
