// rsg_batch.hip -- batched phylogenetic null: simulate, score and fit many alignments of
// uneven size in one pass on the device.
//
// Per alignment this is R-scape's per-replicate work (null_rscape, src/R-scape.c:1615-1724
// with the cov_GenerateAlignment simulator, src/cov_simulate.c:60-190): cov_Calculate of the
// replicate (corr_Probs + statistic + APC/ASC, src/covariation.c:63-306), the histogram width
// of calculate_width_histo (src/R-scape.c:1280-1371), the rank histogram
// (src/covariation.c:414-432) and the tail fit (cov_NullFitExponential / Gamma,
// :1914-1975 with cov_histogram_pmass :2483-2506).
//
// Layout: every alignment ("item") owns slices of a few large buffers, described by an
// int64 descriptor (RSG_BDESC fields, see rsg_internal.h).  Each kernel below covers all
// items in one launch; a block reads its item from a per-kernel block map (k_block_map).  No host synchronisation happens between the launches, so the whole batch can
// be recorded once as a hipGraph and replayed; buffers are cleared by fill kernels, not
// memset nodes.
#include "rsg_device.h"
#include <algorithm>
#include <cfloat>
#include <chrono>
#include <climits>
#include <cstring>
#include <numeric>
#include <type_traits>

// Histogram geometry, bins and E-values are rounded exactly as the host computes them.
#pragma clang fp contract(off)

enum { D_N = 0, D_L, D_NPAD, D_LPAD, D_XT, D_CNT, D_COV, D_PM, D_ROWS, D_HIST, D_LEAF, D_BPACK,
       D_BSTAT, D_BEL, D_NB32, D_GROUP, D_BHIST, D_PMP, D_BCOL16, D_BROW };
#define STAT_TAB_LDS (54 << 10)   // the largest logarithm table kept in LDS (bytes): up to 6911 sequences
#define NBPOOL 16384         // bins of the shared bin pool per group (a group may take more)

// The per-kernel block maps: item of block b of kernel `field` is map[d[field] + b] of its section
// (one dependent load per block in place of a binary search over the descriptors: ten loads one
// after another for 1000 items).  Blocks past the items make the table of logarithms of counts up to
// NM, and the first one clears the error flags: launches of their own took 5 us each.
enum { M_PACK = 0, M_COL16, M_STAT, M_ROW, M_EL, M_HIST, M_N };
struct BlockMap { int *m; int64_t off[M_N + 1]; };          // section s: off[s] .. off[s + 1] - 1
__global__ void __launch_bounds__(256) k_block_map(const int64_t *__restrict__ desc, int n, BlockMap B, int64_t NM,
                                                   double *__restrict__ lgc, int *__restrict__ flags)
{
  if (blockIdx.x == 0 && threadIdx.x < 16) flags[threadIdx.x] = 0;
  if ((int)blockIdx.x >= n) {
    const int64_t k = (int64_t)(blockIdx.x - n) * 256 + threadIdx.x;
    if (k <= NM) log_entry(NM, k, lgc);
    return;
  }
  constexpr int field[M_N] = {D_BPACK, D_BCOL16, D_BSTAT, D_BROW, D_BEL, D_BHIST};
  const int it = blockIdx.x;
  const int64_t *d = desc + (int64_t)it * RSG_BDESC;
#pragma unroll
  for (int s = 0; s < M_N; s++) {
    const int64_t b0 = d[field[s]], b1 = (it + 1 < n) ? d[RSG_BDESC + field[s]] : B.off[s + 1] - B.off[s];
    for (int64_t b = b0 + threadIdx.x; b < b1; b += 256) B.m[B.off[s] + b] = it;
  }
}

// Pairs i < j of an item as row pairs p (rows p and L - 1 - p, L - 1 elements together): element
// e of row pair p is (p, p + 1 + e) while e < L - 1 - p, else (L - 1 - p, e + 1); the middle row of an
// odd L stands alone.
// row pairs per work group of k_minmax_b: about `target` pairs, one to four row pairs per wave
__host__ __device__ __forceinline__ int64_t el_rp(int64_t L, int64_t target)
{
  const int64_t r = (target + 4 * (L - 1) - 1) / (4 * (L - 1)) * 4;
  return r < 4 ? 4 : r > 16 ? 16 : r;
}
// row pairs per work group of k_hist_b: about `target` pairs, at least one row pair per wave
__host__ __device__ __forceinline__ int64_t hist_rp(int64_t L, int64_t target)
{
  const int64_t r = (target + L - 2) / (L - 1);
  return r < 16 ? 16 : r;
}
// the APC (or ASC) corrected score; without a correction (actype < 0) the score itself
__device__ __forceinline__ double corrected(double v, double xi, double xj, double avg, int actype)
{
  if (actype == RSG_APC) return (avg != 0.0) ? v - xi * xj / avg : 0.0;
  if (actype == RSG_ASC) return v - (xi + xj - avg);
  return v;
}
// fn(x) on the corrected scores of row pair p, one wave: four loads of scores and row means in flight
template <class F>
__device__ __forceinline__ void row_pair(const double *__restrict__ C, const double *__restrict__ R, int64_t L, int64_t p, int lane,
                                         int actype, F fn)
{
  const int64_t n0 = L - 1 - p, tot = (2 * p == L - 1) ? n0 : L - 1;
  const double *r0 = C + p * L + p + 1, *r1 = C + (L - 1 - p) * L + 1, *m0 = R + p + 1, *m1 = R + 1;
  const double xp = (actype >= 0) ? R[p] : 0., xq = (actype >= 0) ? R[L - 1 - p] : 0., avg = (actype >= 0) ? R[2 * L] : 0.;
  for (int64_t e0 = lane; e0 < tot; e0 += 256) {
    double v[4], x[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int64_t e = min(e0 + 64 * q, tot - 1);
      v[q] = (e < n0) ? r0[e] : r1[e];
      x[q] = (actype < 0) ? 0. : (e < n0) ? m0[e] : m1[e];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int64_t e = e0 + 64 * q;
      if (e < tot) fn(corrected(v[q], (e < n0) ? xp : xq, x[q], avg, actype));
    }
  }
}

// leaves (N x L, row-major) -> one-hot FP4 operands (pack_block)
__global__ void __launch_bounds__(256)
k_pack_b(const int64_t *__restrict__ desc, const int *__restrict__ map, const uint8_t *__restrict__ leaves,
         uint8_t *__restrict__ x4)
{
  const int it = map[blockIdx.x];
  const int64_t *d = desc + it * RSG_BDESC;
  const int64_t Lpad = d[D_LPAD];
  const int64_t local = blockIdx.x - d[D_BPACK], nbx = (Lpad + 127) / 128;
  pack_block<PACK_X4>(leaves + d[D_LEAF], d[D_N], d[D_L], d[D_NPAD], Lpad, (local / nbx) * 128, (local % nbx) * 128, nullptr,
                      nullptr, x4 + d[D_XT]);
}

// corr_Marginals per item from the 32 x 32 block partials the batched Gram leaves (the
// single-alignment path's layout, order and reduction: a replicate's marginals match its
// rsg_corr_Probs bit for bit)
__global__ void __launch_bounds__(256)
k_pm_reduce_b(const int64_t *__restrict__ desc, const int *__restrict__ map, const double *__restrict__ part, double *__restrict__ pm,
              double tol, int *__restrict__ flag)
{
  const int it = map[blockIdx.x];
  const int64_t *d = desc + it * RSG_BDESC;
  const int64_t L = d[D_L], nb32 = d[D_NB32];
  const int64_t col = (blockIdx.x - d[D_BCOL16]) * 16 + (threadIdx.x >> 4);
  if (col >= L) return;
  const double *pi = part + d[D_PMP];
  pm32_reduce_col(pi, pi + pm32_n(nb32), (int)nb32, L, col, threadIdx.x & 15, tol, pm + d[D_PM], pm + d[D_PM] + 4 * L, flag);
}

__device__ __forceinline__ StatArgs item_stat(const StatArgs &A0, const int64_t *d, const uint16_t *cnt, const double *pm, double *cov)
{
  StatArgs A = A0;
  A.L = d[D_L];
  A.cnt = cnt + d[D_CNT]; A.pm = pm + d[D_PM]; A.lpm = pm + d[D_PM] + 4 * A.L;
  A.wsum = (double)d[D_N]; A.cov = cov + d[D_COV];
  return A;
}

// The statistic of the items of class CLS (others are left to the other class's launch), a 32 x 32
// pair tile per work group.
template <int TYPE, int CLS>
__global__ void __launch_bounds__(256)
k_stat_b(const int64_t *__restrict__ desc, const int *__restrict__ map, StatArgs A0, const uint16_t *__restrict__ cnt,
         const double *__restrict__ pm, double *__restrict__ cov, const int *__restrict__ cls)
{
  const int it = map[blockIdx.x];
  if (cls[it] != CLS) return;
  const int64_t *d = desc + (int64_t)it * RSG_BDESC;
  int bi, bj;
  tri_tile(blockIdx.x - d[D_BSTAT], bi, bj);      // tiles on or above the diagonal only
  stat_tile<double, CNT_U16, true, TYPE, CLS>(item_stat(A0, d, cnt, pm, cov), bi, bj, (int64_t)blockIdx.x);
}

// Class C16 statistics with logarithms: persistent work groups (as many as fit the device) with the
// table (c + 1e-10) ln(c + 1e-10), c = 0 .. nmax, in LDS, each taking every gridDim-th tile.  Sixteen
// table reads per pair: from LDS they cost its bank cycles, from global memory the L1's
// address processing of 64 lanes each, which bound this pass (and its 169 registers held it at two
// waves per SIMD): 1470 us for 1000 uneven alignments, 482 us for 20 of N = 5000 x L = 1500.
// Block min / max only where they are wanted (A0.part).
template <int TYPE>
__global__ void __launch_bounds__(512)
k_stat_tab_b(const int64_t *__restrict__ desc, const int *__restrict__ map, int64_t ntiles, StatArgs A0,
             const uint16_t *__restrict__ cnt, const double *__restrict__ pm, double *__restrict__ cov,
             const int *__restrict__ cls)
{
  extern __shared__ double xln[];
  __shared__ double tile[32][33];
  for (int64_t k = threadIdx.x; k <= A0.N; k += 512) xln[k] = A0.lgc[2 * (A0.N + 1) + k];
  __syncthreads();
  // the next tile's records load while this one's statistics are formed, and the tile after
  // that one's descriptor, so no load waits on another within a tile
  struct Tile { int bi, bj, on; StatArgs A; };
  auto describe = [&](int64_t t) {
    Tile T;
    const int it = map[min(t, ntiles - 1)];
    const int64_t *d = desc + (int64_t)it * RSG_BDESC;
    T.on = t < ntiles && cls[it] == RSG_C16;
    T.A = item_stat(A0, d, cnt, pm, cov);
    tri_tile(min(t, ntiles - 1) - d[D_BSTAT], T.bi, T.bj);
    return T;
  };
  const int64_t g = gridDim.x;
  Tile cur = describe(blockIdx.x), nxt = describe(blockIdx.x + g);
  TabTile wc, wn;
  tab_tile_load(cur.A, cur.bi, cur.bj, wc);
  for (int64_t t = blockIdx.x; t < ntiles; t += g) {
    tab_tile_load(nxt.A, nxt.bi, nxt.bj, wn);
    const Tile aft = describe(t + 2 * g);
    if (cur.on) {
      double lmin = INFINITY, lmax = -INFINITY;
      tab_tile_stat<TYPE>(cur.A, cur.bi, cur.bj, wc, tile, [&](unsigned c) { return xln[c]; }, lmin, lmax);
      if (A0.part) {
        block_minmax512(lmin, lmax, &tile[0][0]);
        if (threadIdx.x == 0) { A0.part[2 * t] = lmin; A0.part[2 * t + 1] = lmax; }
      }
    }
    cur = nxt; nxt = aft; wc = wn;
  }
}

// raw row sums of COV (diagonal excluded): one wave per row, four rows per block.  Lane l
// keeps the partials of the single path's threads l, l + 64, l + 128, l + 192 (k_rowsum's
// 256-strided sums) and combines them in block_sum_tree256's order, so every row sum equals
// the single path's bit for bit.  The four partials' loads are in flight together.
__global__ void __launch_bounds__(256)
k_rowsum_b(const int64_t *__restrict__ desc, const int *__restrict__ map, const double *__restrict__ cov, double *__restrict__ rows)
{
  const int64_t *d = desc + (int64_t)map[blockIdx.x] * RSG_BDESC;
  const int64_t L = d[D_L], i = (blockIdx.x - d[D_BROW]) * 4 + (threadIdx.x >> 6);
  if (i >= L) return;
  const int lane = threadIdx.x & 63;
  const double *C = cov + d[D_COV] + i * L;
  double p[4] = {0., 0., 0., 0.};
  for (int64_t j0 = lane; j0 < L; j0 += 256) {
    double v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = C[min(j0 + 64 * q, L - 1)];
#pragma unroll
    for (int q = 0; q < 4; q++) if (j0 + 64 * q < L && j0 + 64 * q != i) p[q] += v[q];
  }
  double x = (p[0] + p[2]) + (p[1] + p[3]);
#pragma unroll
  for (int st = 32; st > 0; st >>= 1) x += __shfl_down(x, st, 64);
  if (lane == 0) rows[d[D_ROWS] + L + i] = x;
}

__global__ void __launch_bounds__(256)
k_rowmean_b(const int64_t *__restrict__ desc, double *__restrict__ rows)
{
  __shared__ double red[256];
  const int64_t *d = desc + blockIdx.x * RSG_BDESC;
  const int64_t L = d[D_L];
  double *R = rows + d[D_ROWS];
  double s = 0.;
  for (int64_t i = threadIdx.x; i < L; i += 256) { double r = R[L + i]; s += r; R[i] = (L > 1) ? r / ((double)L - 1.) : r; }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) { if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st]; __syncthreads(); }
  if (threadIdx.x == 0) R[2 * L] = (L > 1) ? red[0] / ((double)L * ((double)L - 1.)) : red[0];
}

// min / max of the APC / ASC corrected scores (block min / max to part[blockIdx]) and the NaN flag.  The
// corrected matrix itself is not an output: the histogram pass forms the scores again, so both
// passes read the upper triangle and none writes (correcting in place read and wrote both
// triangles: 462 us for 1000 uneven alignments, 147 us for 20 of L = 1500; this takes 161 and
// 48 us).  A thousand work groups where the batch has the rows: 16 row pairs each left one replicate of
// L = 1500 on 47 of them (27 us, 8.7 now).
__global__ void __launch_bounds__(256)
k_minmax_b(const int64_t *__restrict__ desc, const int *__restrict__ map, const double *__restrict__ cov,
           const double *__restrict__ rows, int actype, int64_t target, int *__restrict__ flag, double *__restrict__ part)
{
  const int64_t *d = desc + (int64_t)map[blockIdx.x] * RSG_BDESC;
  const int64_t L = d[D_L], rp = el_rp(L, target), p0 = (blockIdx.x - d[D_BEL]) * rp;
  double a = INFINITY, b = -INFINITY;
  bool bad = false;
  for (int64_t p = p0 + (threadIdx.x >> 6); p < min(p0 + rp, (L + 1) / 2); p += 4)
    row_pair(cov + d[D_COV], rows + d[D_ROWS], L, p, threadIdx.x & 63, actype, [&](double r) {
      bad |= isnan(r);
      a = fmin(a, r); b = fmax(b, r);
    });
  if (bad) atomicOr(flag, 1);
  block_minmax(a, b, part, (int64_t)blockIdx.x);
}

// per item: reduce block partials [p0, p1) to (min, max)
__global__ void __launch_bounds__(256)
k_item_minmax(const int64_t *__restrict__ desc, int field, int64_t nblk_total, int n, const double *__restrict__ part,
              double *__restrict__ mm)
{
  __shared__ double rmin[256], rmax[256];
  const int it = blockIdx.x;
  const int64_t p0 = desc[it * RSG_BDESC + field];
  const int64_t p1 = (it + 1 < n) ? desc[(it + 1) * RSG_BDESC + field] : nblk_total;
  double a = INFINITY, b = -INFINITY;
  for (int64_t k = p0 + threadIdx.x; k < p1; k += 256) { a = fmin(a, part[2 * k]); b = fmax(b, part[2 * k + 1]); }
  rmin[threadIdx.x] = a; rmax[threadIdx.x] = b;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) { rmin[threadIdx.x] = fmin(rmin[threadIdx.x], rmin[threadIdx.x + s]); rmax[threadIdx.x] = fmax(rmax[threadIdx.x], rmax[threadIdx.x + s]); }
    __syncthreads();
  }
  if (threadIdx.x == 0) { mm[2 * it] = rmin[0]; mm[2 * it + 1] = rmax[0]; }
}

// Histogram geometry per null (group of replicates): the width comes from the group's first
// replicate (calculate_width_histo runs on the first null replicate, src/R-scape.c:1353);
// the bounds cover every replicate, as the cumulative histogram grows to do
// (null_add2cumranklist, src/R-scape.c:1564-1612).
struct HGeo { double w, bmax, xmin, xmax, npairs, mn, mx; int64_t off; int nb, imin, imax, ok; };

__device__ __forceinline__ HGeo group_geo(int g, const int *__restrict__ gfirst, const int64_t *__restrict__ desc,
                                          const double *__restrict__ mm, double bmin, double w0, int hpts, double tol)
{
  const int j0 = gfirst[g], j1 = gfirst[g + 1];
  HGeo G; G.ok = 0;
  const double lo = fmax(bmin, mm[2 * j0]);
  double w = fmin(w0, (mm[2 * j0 + 1] - lo) / (double)hpts);
  if (w < tol) w = 0.;
  double mn = INFINITY, mx = -INFINITY, np = 0.;
  for (int j = j0; j < j1; j += 8) {                   // eight replicates' loads in flight
    double2 e[8];
    int64_t L[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int k = min(j + q, j1 - 1);
      e[q] = ((const double2 *)mm)[k]; L[q] = desc[(int64_t)k * RSG_BDESC + D_L];
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
      mn = fmin(mn, e[q].x); mx = fmax(mx, e[q].y);
      if (j + q < j1) np += (double)(L[q] * (L[q] - 1) / 2);
    }
  }
  G.w = w; G.bmax = 0.; G.xmin = G.xmax = 0.; G.nb = 0; G.imin = 0; G.imax = -1; G.off = 0;
  G.npairs = np; G.mn = mn; G.mx = mx;
  if (w > 0. && mx > bmin) {
    double bmax = mx + 5 * w;
    while (fabs(bmax - bmin) < tol) bmax += w;
    const double nbd = (bmax - bmin) / w;
    if (nbd < (double)INT_MAX) {
      G.nb = (int)nbd; G.bmax = bmax;
      G.xmin = fmax(mn, bmin + w); G.xmax = fmax(mx, bmin + w);
      G.imin = (int)ceil((G.xmin - bmin) / w - 1.); G.imax = (int)ceil((G.xmax - bmin) / w - 1.);
      G.ok = (G.imin >= 0 && G.imax < G.nb) ? 1 : 0;
    }
  }
  return G;
}
__global__ void k_width_b(int ng, const int *__restrict__ gfirst, const int64_t *__restrict__ desc,
                          const double *__restrict__ mm, double bmin, double w0, int hpts, double tol,
                          HGeo *__restrict__ geo)
{
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < ng) geo[g] = group_geo(g, gfirst, desc, mm, bmin, w0, hpts, tol);
}

// Bins of every group in one pool: offsets by an exclusive scan over the groups (one block,
// fixed order); a group that does not fit in the pool's cap bins is marked failed (its fit is
// NaN, as for a group without a histogram).  Up to 1024 groups, one per thread, the geometry is
// formed here: a launch of 5 us less.  (The bins of a few groups cleared here as well took the time
// their launch takes, those of 32 and 200 groups 13 and 80 us more.)
__global__ void __launch_bounds__(1024) k_hist_layout(int ng, HGeo *__restrict__ geo, int64_t cap,
                                                      const int *__restrict__ gfirst, const int64_t *__restrict__ desc,
                                                      const double *__restrict__ mm, double bmin, double w0, int hpts,
                                                      double tol)
{
  __shared__ int64_t sh[1024];
  const int T = 1024, tid = threadIdx.x;
  if (ng <= T && tid < ng) geo[tid] = group_geo(tid, gfirst, desc, mm, bmin, w0, hpts, tol);
  const int chunk = (ng + T - 1) / T, g0 = tid * chunk, g1 = min(g0 + chunk, ng);
  int64_t own = 0;
  for (int g = g0; g < g1; g++) own += geo[g].ok ? (int64_t)geo[g].nb : 0;
  sh[tid] = own;
  __syncthreads();
  for (int o = 1; o < T; o <<= 1) {                 // inclusive Hillis-Steele scan
    const int64_t add = (tid >= o) ? sh[tid - o] : 0;
    __syncthreads();
    sh[tid] += add;
    __syncthreads();
  }
  int64_t off = sh[tid] - own;
  for (int g = g0; g < g1; g++) {
    if (!geo[g].ok) continue;
    geo[g].off = off;
    off += geo[g].nb;
    if (off > cap) geo[g].ok = 0;
  }
}

// clear the bins of every group (blocks take groups round-robin)
__global__ void __launch_bounds__(256) k_clear_bins(int ng, const HGeo *__restrict__ geo, unsigned long long *__restrict__ hist)
{
  for (int g = blockIdx.x; g < ng; g += gridDim.x) {
    const HGeo G = geo[g];
    if (!G.ok) continue;
    for (int64_t b = threadIdx.x; b < G.nb; b += 256) hist[G.off + b] = 0ull;
  }
}

// Rank histogram of every item's corrected scores into its group's bins: a work group counts the
// HB_WIN bins from the group's smallest score in LDS (a null's scores span a few thousand bins at
// most) and adds the nonzero ones to the group's; scores past them go there directly.  As many
// work groups as fill the device, since each adds ~300 bins that all of a group share.  Bound by the
// divisions (two per score, in FP64); with bins for 16384 in LDS (two work groups of four waves
// per CU) and both triangles read it took 1155 us for 1000 uneven alignments, 208 us for 20 of
// L = 1500; this takes 300 and 66 us.
#define HB_WIN 4096
__global__ void __launch_bounds__(1024)
k_hist_b(const int64_t *__restrict__ desc, const int *__restrict__ map, const double *__restrict__ cov,
         const double *__restrict__ rows, int actype, const HGeo *__restrict__ geo, double bmin, int64_t target,
         unsigned long long *__restrict__ hist)
{
  __shared__ unsigned int lh[HB_WIN];
  const int64_t *d = desc + (int64_t)map[blockIdx.x] * RSG_BDESC;
  const HGeo g = geo[d[D_GROUP]];
  if (!g.ok) return;
  const int win = min(g.nb - g.imin, HB_WIN);
  unsigned long long *H = hist + g.off;
  for (int b = threadIdx.x; b < win; b += 1024) lh[b] = 0u;
  __syncthreads();
  const int64_t L = d[D_L], rp = hist_rp(L, target), p0 = (blockIdx.x - d[D_BHIST]) * rp;
  const double fl = bmin + g.w;
  for (int64_t p = p0 + (threadIdx.x >> 6); p < min(p0 + rp, (L + 1) / 2); p += 16)
    row_pair(cov + d[D_COV], rows + d[D_ROWS], L, p, threadIdx.x & 63, actype, [&](double x) {
      const double add = (x > fl) ? x : fl;
      int b = (int)ceil(((add - bmin) / g.w) - 1.);
      b = (b < 0) ? 0 : ((b >= g.nb) ? g.nb - 1 : b);
      const unsigned k = (unsigned)(b - g.imin);
      if (k < (unsigned)win) atomicAdd(&lh[k], 1u);
      else                   atomicAdd(&H[b], 1ull);
    });
  __syncthreads();
  for (int b = threadIdx.x; b < win; b += 1024)
    if (lh[b]) atomicAdd(&H[g.imin + b], (unsigned long long)lh[b]);
}

// tail fit per null (one 1024-thread block per group): see rsg_rank.hip for the method
__global__ void __launch_bounds__(1024)
k_fit_b(const HGeo *__restrict__ geo, const unsigned long long *__restrict__ hist, double bmin, double pmass, double fracfit, int doexp,
        double *__restrict__ fits)
{
  const int g = blockIdx.x;
  const HGeo G = geo[g];
  double *o = fits + g * 8;
  if (threadIdx.x == 0) { o[6] = G.mn; o[7] = G.mx; }
  if (!G.ok) {
    if (threadIdx.x == 0) { o[0] = NAN; o[1] = INFINITY; o[2] = 0.; o[3] = 0.; o[4] = NAN; o[5] = G.w; }
    return;
  }
  nullfit_body(hist + G.off, G.nb, G.imin, G.imax, G.npairs, G.npairs, bmin, G.w, pmass, fracfit, doexp,
               nullptr, o);
  if (threadIdx.x == 0) { o[5] = G.w; o[6] = G.mn; o[7] = G.mx; }
}

// ------------------------------------------------------------------------------- host side
namespace {
// Bump allocation over a base pointer (256-byte aligned slices); with base == nullptr it only
// measures.
struct Arena {
  uint8_t *base = nullptr;
  size_t off = 0;
  template <typename T> T *get(size_t count)
  {
    T *p = base ? (T *)(base + off) : nullptr;
    off += (std::max<size_t>(count, 1) * sizeof(T) + 255) & ~(size_t)255;
    return p;
  }
};
}

// The bytes that fix a batch's launch geometry, kept to compare a call with the cached graph's
struct GeoSig {
  std::vector<uint8_t> b;
  void add(const void *p, size_t n)
  {
    const uint64_t len = n;
    b.insert(b.end(), (const uint8_t *)&len, (const uint8_t *)&len + sizeof(len));
    if (n) b.insert(b.end(), (const uint8_t *)p, (const uint8_t *)p + n);
  }
};

// The batch; with fp != nullptr the null alignments are R-scape's nulls of one alignment fax
// (Fitch + shuffle, rsg_fitch.hip), one per job (all jobs of that alignment's size, seeds from the
// jobs), in place of the simulation.
static int null_batch_impl(rsg_ctx *c, const rsg_null_job *jobs, int nj, int covtype, double bmin, double pmass,
                           double fracfit, int doexpfit, rsg_hist **hists, double *fits, float *feats, int use_graph,
                           const uint8_t *fax, const FitchPlan *fp, char *errbuf)
{
  HIPCHK(hipSetDevice(c->device));
  if (nj < 1) return rsg_fail(errbuf, "empty batch");
  const int base = covtype - covtype % 3, corr = covtype % 3;
  auto clk = std::chrono::steady_clock::now;
  auto since = [](std::chrono::steady_clock::time_point a) {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - a).count();
  };
  auto h0 = clk();
  // groups: contiguous, ascending from 0
  std::vector<int> gfirst;
  for (int k = 0; k < nj; k++) {
    const int g = jobs[k].group;
    if (k == 0 ? g != 0 : (g != jobs[k - 1].group && g != jobs[k - 1].group + 1))
      return rsg_fail(errbuf, "job %d: group ids must start at 0 and be contiguous and ascending", k);
    if (k == 0 || g != jobs[k - 1].group) gfirst.push_back(k);
  }
  const int ng = (int)gfirst.size();
  gfirst.push_back(nj);
  if (base == RSG_RAF || base == RSG_RAFS || base == RSG_CCF)
    return rsg_fail(errbuf, "batched null supports CHI/GT/MI/MIr/MIg/OMES statistics");
  // ---- layout
  std::vector<int64_t> desc((size_t)nj * RSG_BDESC, 0);
  std::vector<SimItem> sim((size_t)nj);
  std::vector<int> cls((size_t)nj);
  int nc2 = 0;                                   // items of class C2
  int64_t o_xt = 0, o_cnt = 0, o_cov = 0, o_pm = 0, o_rows = 0, o_leaf = 0, nodes = 0, seqs = 0;
  int64_t b_pack = 0, b_stat = 0, b_el = 0, b_sim = 0, b_hist = 0, nmax = 1, npairs = 0;
  for (int k = 0; k < nj; k++) npairs += jobs[k].alen * (jobs[k].alen - 1) / 2;
  // pairs per work group of the histogram (two per CU) and of the extremes (four)
  const int64_t htarget = npairs / 512, etarget = npairs / 1024;
  int64_t b_col16 = 0, o_pmp = 0, b_row = 0;
  std::vector<int4> tiles, btiles;        // 32 x 32-column tiles (small alignments), 64 x 32 (large)
  for (int k = 0; k < nj; k++) {
    const rsg_null_job &J = jobs[k];
    if (J.nleaf < 2 || J.alen < 2) return rsg_fail(errbuf, "job %d: needs >= 2 sequences and >= 2 columns", k);
    if (J.nleaf > RSG_U16_MAXN) return rsg_fail(errbuf, "job %d: more than %d sequences", k, RSG_U16_MAXN);
    const int64_t N = J.nleaf, L = J.alen, Npad = rsg_npad(N), Lpad = ((L + 63) / 64) * 64;
    int64_t *d = &desc[(size_t)k * RSG_BDESC];
    d[D_N] = N; d[D_L] = L; d[D_NPAD] = Npad; d[D_LPAD] = Lpad;
    d[D_XT] = o_xt; d[D_CNT] = o_cnt; d[D_COV] = o_cov; d[D_PM] = o_pm; d[D_ROWS] = o_rows;
    d[D_HIST] = 0; d[D_LEAF] = o_leaf;
    d[D_BPACK] = b_pack; d[D_BSTAT] = b_stat; d[D_BEL] = b_el; d[D_BROW] = b_row;
    const int64_t nb32 = (L + 31) / 32;
    d[D_NB32] = nb32; d[D_GROUP] = J.group; d[D_BHIST] = b_hist;
    d[D_PMP] = o_pmp; d[D_BCOL16] = b_col16;
    b_col16 += (L + 15) / 16; o_pmp += 2 * pm32_n(nb32);
    cls[(size_t)k] = (N <= 8 || L <= 50) ? RSG_C2 : RSG_C16;           // CSELECT (correlators.c:335-341)
    nc2 += cls[(size_t)k] == RSG_C2;
    SimItem &s = sim[(size_t)k];
    s.N = N; s.L = L; s.tree_off = nodes; s.seq_off = seqs; s.leaf_off = o_leaf; s.seed = J.seed; s.stream = J.stream;
    s.gapthr = (J.gapfrac <= 0.) ? 0u : (J.gapfrac >= 1. ? 0xFFFFFFFFu : (uint32_t)(J.gapfrac * 4294967296.0));
    s.col_blk0 = b_sim; s.model_off = 40 * (int64_t)k;
    o_xt += Lpad * Npad / 2; o_cnt += 16 * L * L; o_cov += L * L; o_pm += 8 * L; o_rows += 2 * L + 2; o_leaf += N * L;
    nodes += N - 1; seqs += (N - 1) * L;
    b_pack += ((Lpad + 127) / 128) * (Npad / 128); b_row += (L + 3) / 4; b_stat += nb32 * (nb32 + 1) / 2;
    b_sim += (L + 63) / 64;
    const int64_t np = (L + 1) / 2, hrp = hist_rp(L, htarget), erp = el_rp(L, etarget);
    b_el += (np + erp - 1) / erp; b_hist += (np + hrp - 1) / hrp;
    nmax = std::max(nmax, N);
  }
  rsg_thost(c, "batch_plan_layout", since(h0));
  h0 = clk();
  // Gram tiles, longest K loops first so the tail of each launch is short work: the jobs in
  // order of decreasing padded sequence count (ties in job order), each job's tiles row by row
  {
    std::vector<int> ord((size_t)nj);
    std::iota(ord.begin(), ord.end(), 0);
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) {
      return desc[(size_t)a * RSG_BDESC + D_NPAD] > desc[(size_t)b * RSG_BDESC + D_NPAD];
    });
    for (int k : ord) {
      const int64_t N = jobs[k].nleaf, L = jobs[k].alen, Lpad = desc[(size_t)k * RSG_BDESC + D_LPAD], nb32 = (L + 31) / 32;
      if (rsg_batch_big_tiles(N, L)) {
        // 64 (i) x 32 (j) columns: every tile holding a pair i < j < L
        for (int64_t bi = 0; bi < Lpad / 64; bi++)
          for (int64_t bj = 0; bj < nb32; bj++)
            if (bi * 64 < std::min((bj + 1) * 32, L) - 1) btiles.push_back(make_int4(k, (int)bi, (int)bj, 0));
      } else {
        for (int64_t bi = 0; bi < nb32; bi++)
          for (int64_t bj = bi; bj < nb32; bj++) tiles.push_back(make_int4(k, (int)bi, (int)bj, 0));
      }
    }
  }
  rsg_thost(c, "batch_plan_tiles", since(h0));
  h0 = clk();
  HostArr<double> ld, rd, models;
  SimLevels lv;
  std::vector<int> fperm;
  std::vector<uint64_t> fseed;
  if (!fp) {
    ld.alloc((size_t)nodes); rd.alloc((size_t)nodes); models.alloc((size_t)nj * 40);
    rsg_parallel_ranges(nj, nodes, [&](int k) { return jobs[k].nleaf - 1; }, [&](int k0, int k1) {
      for (int k = k0; k < k1; k++) {
        const int64_t off = sim[(size_t)k].tree_off, m1 = jobs[k].nleaf - 1;
        memcpy(&ld[(size_t)off], jobs[k].ld, sizeof(double) * m1);
        memcpy(&rd[(size_t)off], jobs[k].rd, sizeof(double) * m1);
        memcpy(&models[(size_t)k * 40], jobs[k].model, sizeof(double) * 40);
      }
    });
    rsg_thost(c, "batch_plan_trees", since(h0));
    h0 = clk();
    std::vector<const int *> lp((size_t)nj), rp((size_t)nj);
    for (int k = 0; k < nj; k++) { lp[(size_t)k] = jobs[k].left; rp[(size_t)k] = jobs[k].right; }
    if (rsg_sim_levels(sim.data(), nj, lp.data(), rp.data(), lv, errbuf) != RSG_OK) return RSG_FAIL;
    rsg_thost(c, "batch_plan_levels", since(h0));
    h0 = clk();
  } else {
    // one column permutation per replicate (for long rows; else the device makes them)
    for (int k = 0; k < nj; k++)
      if (jobs[k].nleaf != fp->N || jobs[k].alen != fp->L) return rsg_fail(errbuf, "Fitch batch: job %d has another size", k);
    const bool perm = rsg_fitch_host_perm(*fp);
    if (perm) fperm.resize((size_t)nj * fp->L);
    fseed.assign((size_t)nj + 1, 0u);                // the seeds, then the Fitch flag (0)
    for (int k = 0; k < nj; k++) {
      fseed[(size_t)k] = jobs[k].seed;
      if (perm) rsg_fitch_perm(jobs[k].seed, fp->L, &fperm[(size_t)k * fp->L]);
    }
  }
  // surrogate features of each group's first replicate
  std::vector<int64_t> fitems((size_t)ng * 6);
  int64_t fblocks = 0;
  for (int g = 0; g < ng; g++) {
    const int64_t *d0 = &desc[(size_t)gfirst[(size_t)g] * RSG_BDESC];
    int64_t *f = &fitems[(size_t)g * 6];
    f[0] = d0[D_XT]; f[1] = d0[D_N]; f[2] = d0[D_NPAD]; f[3] = d0[D_L]; f[4] = fblocks; f[5] = d0[D_LPAD];
    fblocks += (d0[D_L] + 3) / 4;
  }
  // histogram bins of all groups share one pool (a group's share is set on the device once its
  // score range is known)
  const int64_t pool = std::max<int64_t>((int64_t)ng * NBPOOL, (int64_t)1 << 21);
  // ---- device buffers: one grow-only arena of the context, carved in two passes
  int64_t *d_desc; SimItem *d_sim; int *d_cls; int4 *d_tiles, *d_btiles;
  double *d_ld, *d_rd, *d_models; int4 *d_ent; int *d_gfirst; int64_t *d_fitems; unsigned long long *d_fcnt;
  uint32_t *d_cdf; uint8_t *d_seqs, *d_leaves, *d_x4; uint16_t *d_cnt; double *d_cov, *d_pm, *d_rows, *d_lgc;
  double *d_part_s, *d_part_e, *d_mm, *d_pmp; HGeo *d_geo; unsigned long long *d_hist; double *d_fits;
  BlockMap M;
  {
    const int64_t nb[M_N] = {b_pack, b_col16, b_stat, b_row, b_el, b_hist};
    M.off[0] = 0;
    for (int s = 0; s < M_N; s++) M.off[s + 1] = M.off[s] + nb[s];
  }
  uint8_t *f_ax = nullptr, *f_mask = nullptr, *f_all = nullptr; int4 *f_ent = nullptr; int *f_perm = nullptr, *f_nsub = nullptr;
  int *f_cols = nullptr; uint64_t *f_seeds = nullptr; int *d_queue = nullptr;
  auto carve = [&](Arena &A) {
    d_desc = A.get<int64_t>(desc.size()); d_sim = A.get<SimItem>((size_t)nj); d_cls = A.get<int>((size_t)nj);
    d_tiles = A.get<int4>(tiles.size()); d_btiles = A.get<int4>(btiles.size());
    d_ld = A.get<double>((size_t)nodes); d_rd = A.get<double>((size_t)nodes);
    d_models = A.get<double>(40 * (size_t)nj); d_ent = A.get<int4>(lv.ent.size());
    d_gfirst = A.get<int>((size_t)ng + 1); d_fitems = A.get<int64_t>(fitems.size());
    d_fcnt = A.get<unsigned long long>((size_t)ng * 36);
    d_cdf = A.get<uint32_t>((size_t)nodes * 24); d_seqs = A.get<uint8_t>((size_t)seqs);
    d_leaves = A.get<uint8_t>((size_t)o_leaf); d_x4 = A.get<uint8_t>((size_t)o_xt);
    d_cnt = A.get<uint16_t>((size_t)o_cnt); d_cov = A.get<double>((size_t)o_cov); d_pm = A.get<double>((size_t)o_pm);
    d_rows = A.get<double>((size_t)o_rows); d_lgc = A.get<double>(3 * (size_t)(nmax + 1));
    d_part_s = A.get<double>(2 * (size_t)b_stat); d_part_e = A.get<double>(2 * (size_t)b_el);
    d_mm = A.get<double>(2 * (size_t)nj); d_pmp = A.get<double>((size_t)o_pmp); d_geo = A.get<HGeo>((size_t)ng);
    d_hist = A.get<unsigned long long>((size_t)pool);
    d_fits = A.get<double>((size_t)ng * 8); d_queue = A.get<int>(128);
    M.m = A.get<int>((size_t)M.off[M_N]);
    if (fp) {
      const size_t N = (size_t)fp->N, L = (size_t)fp->L, R = (size_t)nj;
      f_ax = A.get<uint8_t>(N * L); f_ent = A.get<int4>((size_t)fp->m); f_perm = A.get<int>(fperm.size());
      f_seeds = A.get<uint64_t>(R + 1); f_mask = A.get<uint8_t>(R * (N - 1) * L); f_all = A.get<uint8_t>(R * (N - 1) * L);
      f_nsub = A.get<int>(R * 2 * (size_t)fp->m * 25); f_cols = A.get<int>(R * rsg_fitch_cols(*fp));
    }
  };
  rsg_thost(c, "batch_plan_rest", since(h0));
  h0 = clk();
  size_t plan_bytes = 0;
  {
    Arena plan;
    carve(plan);
    plan_bytes = plan.off;
    if (c->arena_cap < plan.off) {
      if (c->bexec) { hipGraphExecDestroy(c->bexec); c->bexec = nullptr; c->bexec_sig.clear(); }
      if (c->d_arena) hipFree(c->d_arena);
      c->d_arena = nullptr; c->arena_cap = 0;
      if (rsg_dev_malloc(&c->d_arena, plan.off) != hipSuccess)
        return rsg_fail(errbuf, "batch: out of device memory (%zu bytes)", plan.off);
      c->arena_cap = plan.off;
    }
    Arena A; A.base = (uint8_t *)c->d_arena;
    carve(A);
  }
  HIPCHK(hipMemcpyAsync(d_desc, desc.data(), sizeof(int64_t) * desc.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(d_sim, sim.data(), sizeof(SimItem) * nj, hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(d_cls, cls.data(), sizeof(int) * nj, hipMemcpyHostToDevice, c->stream));
  if (!tiles.empty()) HIPCHK(hipMemcpyAsync(d_tiles, tiles.data(), sizeof(int4) * tiles.size(), hipMemcpyHostToDevice, c->stream));
  if (!btiles.empty()) HIPCHK(hipMemcpyAsync(d_btiles, btiles.data(), sizeof(int4) * btiles.size(), hipMemcpyHostToDevice, c->stream));
  if (!fp) {
    HIPCHK(hipMemcpyAsync(d_ld, ld.data(), sizeof(double) * nodes, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(d_rd, rd.data(), sizeof(double) * nodes, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(d_models, models.data(), sizeof(double) * models.size(), hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(d_ent, lv.ent.data(), sizeof(int4) * lv.ent.size(), hipMemcpyHostToDevice, c->stream));
  } else {
    HIPCHK(hipMemcpyAsync(f_ax, fax, (size_t)(fp->N * fp->L), hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(f_ent, fp->ent.data(), sizeof(int4) * fp->ent.size(), hipMemcpyHostToDevice, c->stream));
    if (!fperm.empty()) HIPCHK(hipMemcpyAsync(f_perm, fperm.data(), sizeof(int) * fperm.size(), hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(f_seeds, fseed.data(), sizeof(uint64_t) * fseed.size(), hipMemcpyHostToDevice, c->stream));
  }
  HIPCHK(hipMemcpyAsync(d_gfirst, gfirst.data(), sizeof(int) * gfirst.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(d_fitems, fitems.data(), sizeof(int64_t) * fitems.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  rsg_thost(c, "batch_host_upload", since(h0));
  h0 = clk();

  StatArgs A0;
  memset(&A0, 0, sizeof(A0));
  A0.lgc = d_lgc; A0.N = nmax; A0.part = d_part_s;
  for (int k = 0; k < 16; k++) {                     // WC + GU (src/R-scape.c:882-887)
    int x = k / 4, y = k % 4;
    if ((x == 0 && y == 3) || (x == 3 && y == 0) || (x == 1 && y == 2) || (x == 2 && y == 1) ||
        (x == 2 && y == 3) || (x == 3 && y == 2)) A0.allow |= 1u << k;
  }

  const int actype = (corr == 0) ? -1 : (corr == 1) ? RSG_APC : RSG_ASC;
  auto launch_all = [&]() -> int {
    if (fp) {
      const FitchDev D{f_ax, f_ent, f_perm, f_seeds, (int *)(f_seeds + nj), f_mask,
                       f_all, d_seqs, d_leaves, f_nsub, f_cols};
      if (rsg_fitch_launch(c, *fp, D, nj) != RSG_OK) return RSG_FAIL;
    } else if (rsg_sim_launch(c, d_sim, nj, nodes, b_sim, lv, d_ent, d_ld, d_rd, d_models, d_cdf, d_seqs,
                              d_leaves, nullptr, 0) != RSG_OK) return RSG_FAIL;
    hipLaunchKernelGGL(k_block_map, dim3((unsigned)(nj + (nmax + 256) / 256)), dim3(256), 0, c->stream, d_desc, nj, M, nmax, d_lgc,
                       c->d_flag);
    hipLaunchKernelGGL(k_pack_b, dim3((unsigned)b_pack), dim3(256), 0, c->stream, d_desc, M.m + M.off[M_PACK], d_leaves, d_x4);
    if (feats && rsg_feat_launch(c, d_fitems, ng, fblocks, d_x4, d_fcnt) != RSG_OK) return RSG_FAIL;
    if (rsg_gram_batch_launch(c, d_btiles, (int)btiles.size(), d_tiles, (int)tiles.size(), d_desc, d_x4, d_cnt, d_pmp,
                              (int)D_PMP, d_queue) != RSG_OK)
      return RSG_FAIL;
    hipLaunchKernelGGL(k_pm_reduce_b, dim3((unsigned)b_col16), dim3(256), 0, c->stream, d_desc, M.m + M.off[M_COL16], d_pmp, d_pm, 1e-6, c->d_flag);
    {
      const int *map = M.m + M.off[M_STAT];
      auto stat = [&](auto type) {
        constexpr int TYPE = decltype(type)::value;
        constexpr bool logs = TYPE == RSG_GT || TYPE == RSG_MI || TYPE == RSG_MIr || TYPE == RSG_MIg;
        // the table in LDS beside the 8.4 KiB tile, up to 64 KiB together (two work groups per CU)
        const size_t lds = sizeof(double) * (size_t)(nmax + 1);
        if (nc2 > 0)
          hipLaunchKernelGGL((k_stat_b<TYPE, RSG_C2>), dim3((unsigned)b_stat), dim3(256), 0, c->stream, d_desc, map, A0, d_cnt, d_pm,
                             d_cov, d_cls);
        if (nc2 == nj) return;
        if constexpr (logs)
          if (lds <= STAT_TAB_LDS) {
            StatArgs A1 = A0;
            if (corr) A1.part = nullptr;
            const int64_t fit = (int64_t)(c->ncu > 0 ? c->ncu : 256) * std::min<int64_t>(4, (160 << 10) / (int64_t)(lds + 8704));
            hipLaunchKernelGGL((k_stat_tab_b<TYPE>), dim3((unsigned)std::min(b_stat, fit)), dim3(512), lds, c->stream, d_desc, map,
                               b_stat, A1, d_cnt, d_pm, d_cov, d_cls);
            return;
          }
        hipLaunchKernelGGL((k_stat_b<TYPE, RSG_C16>), dim3((unsigned)b_stat), dim3(256), 0, c->stream, d_desc, map, A0, d_cnt, d_pm,
                           d_cov, d_cls);
      };
      switch (base) {
      case RSG_CHI:  stat(std::integral_constant<int, RSG_CHI>()); break;
      case RSG_GT:   stat(std::integral_constant<int, RSG_GT>()); break;
      case RSG_MI:   stat(std::integral_constant<int, RSG_MI>()); break;
      case RSG_MIr:  stat(std::integral_constant<int, RSG_MIr>()); break;
      case RSG_MIg:  stat(std::integral_constant<int, RSG_MIg>()); break;
      default:       stat(std::integral_constant<int, RSG_OMES>());
      }
    }
    if (corr) {
      hipLaunchKernelGGL(k_rowsum_b, dim3((unsigned)b_row), dim3(256), 0, c->stream, d_desc, M.m + M.off[M_ROW], d_cov, d_rows);
      hipLaunchKernelGGL(k_rowmean_b, dim3((unsigned)nj), dim3(256), 0, c->stream, d_desc, d_rows);
      hipLaunchKernelGGL(k_minmax_b, dim3((unsigned)b_el), dim3(256), 0, c->stream, d_desc, M.m + M.off[M_EL], d_cov, d_rows,
                         actype, etarget, c->d_flag + 1, d_part_e);
      hipLaunchKernelGGL(k_item_minmax, dim3((unsigned)nj), dim3(256), 0, c->stream, d_desc, (int)D_BEL, b_el, nj, d_part_e, d_mm);
    } else {
      hipLaunchKernelGGL(k_item_minmax, dim3((unsigned)nj), dim3(256), 0, c->stream, d_desc, (int)D_BSTAT, b_stat, nj, d_part_s, d_mm);
    }
    if (ng > 1024)
      hipLaunchKernelGGL(k_width_b, dim3((unsigned)((ng + 63) / 64)), dim3(64), 0, c->stream, ng, d_gfirst, d_desc, d_mm,
                         bmin, 0.05, 400, 1e-6, d_geo);
    hipLaunchKernelGGL(k_hist_layout, dim3(1), dim3(1024), 0, c->stream, ng, d_geo, pool, d_gfirst, d_desc, d_mm, bmin, 0.05, 400,
                       1e-6);
    hipLaunchKernelGGL(k_clear_bins, dim3((unsigned)std::min(ng, 4096)), dim3(256), 0, c->stream, ng, d_geo, d_hist);
    hipLaunchKernelGGL(k_hist_b, dim3((unsigned)b_hist), dim3(1024), 0, c->stream, d_desc, M.m + M.off[M_HIST], d_cov, d_rows, actype, d_geo,
                       bmin, htarget, d_hist);
    hipLaunchKernelGGL(k_fit_b, dim3((unsigned)ng), dim3(1024), 0, c->stream, d_geo, d_hist, bmin, pmass, fracfit, doexpfit, d_fits);
    return hipGetLastError() == hipSuccess ? RSG_OK : RSG_FAIL;
  };

  int t; rsg_tstart(c, "null_batch", &t);
  if (use_graph) {
    // The graph's nodes depend only on the launch geometry: the descriptors (sizes and offsets),
    // the tile lists, the tree levels, the scalar arguments and the arena's address.  Every
    // input that changes between calls of one geometry (seeds, trees, branch lengths, models,
    // the alignment, permutations) is read from device buffers uploaded above, outside the
    // graph, so a graph instantiated for this key is replayed as it is.
    GeoSig H;
    H.add(&nj, sizeof(nj)); H.add(&ng, sizeof(ng)); H.add(&covtype, sizeof(covtype)); H.add(&bmin, sizeof(bmin));
    H.add(&pmass, sizeof(pmass)); H.add(&fracfit, sizeof(fracfit)); H.add(&doexpfit, sizeof(doexpfit));
    const int flags2[3] = {feats != nullptr, fp != nullptr, c->batch_persistent};
    H.add(flags2, sizeof(flags2));
    H.add(desc.data(), sizeof(int64_t) * desc.size());
    H.add(tiles.data(), sizeof(int4) * tiles.size()); H.add(btiles.data(), sizeof(int4) * btiles.size());
    const int64_t sc[6] = {nodes, b_sim, fblocks, pool, nmax, (int64_t)plan_bytes};
    H.add(sc, sizeof(sc));
    H.add(lv.lev_ent0.data(), sizeof(int64_t) * lv.lev_ent0.size());
    H.add(lv.lev_blocks.data(), sizeof(int64_t) * lv.lev_blocks.size());
    H.add(lv.lev_maxl.data(), sizeof(int64_t) * lv.lev_maxl.size());
    if (fp) {
      const int64_t fs[5] = {fp->N, fp->L, fp->m, fp->maxd, fp->maxw};
      H.add(fs, sizeof(fs)); H.add(fp->lev0.data(), sizeof(int) * fp->lev0.size());
    }
    const uintptr_t base_addr = (uintptr_t)c->d_arena;
    H.add(&base_addr, sizeof(base_addr));
    if (!c->bexec || c->bexec_sig != H.b) {
      if (c->bexec) { hipGraphExecDestroy(c->bexec); c->bexec = nullptr; c->bexec_sig.clear(); }
      hipGraph_t graph = nullptr;
      HIPCHK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
      int lr = launch_all();
      hipError_t ec = hipStreamEndCapture(c->stream, &graph);
      if (lr != RSG_OK || ec != hipSuccess) { if (graph) hipGraphDestroy(graph); return rsg_fail(errbuf, "batch graph capture failed"); }
      hipGraphExec_t exec = nullptr;
      hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      hipGraphDestroy(graph);
      if (ei != hipSuccess) return rsg_fail(errbuf, "graph instantiate failed");
      c->bexec = exec; c->bexec_sig.swap(H.b);
    } else c->bexec_hits++;
    hipError_t el = hipSuccess, es = hipSuccess;
    for (int rep = 0; rep < use_graph && el == hipSuccess && es == hipSuccess; rep++) {
      el = hipGraphLaunch(c->bexec, c->stream);             // every replay recomputes from scratch
      if (rep + 1 < use_graph) es = hipStreamSynchronize(c->stream);
    }
    rsg_tstop(c, t);
    if (es == hipSuccess) es = hipStreamSynchronize(c->stream);
    if (el != hipSuccess || es != hipSuccess) {
      hipGraphExecDestroy(c->bexec); c->bexec = nullptr; c->bexec_sig.clear();
      return rsg_fail(errbuf, "batch graph launch failed");
    }
  } else {
    if (launch_all() != RSG_OK) return rsg_fail(errbuf, "batch launch failed");
    rsg_tstop(c, t);
    HIPCHK(hipStreamSynchronize(c->stream));
  }
  rsg_thost(c, "batch_host_run", since(h0));
  int flags[2];
  HIPCHK(hipMemcpy(flags, c->d_flag, sizeof(flags), hipMemcpyDeviceToHost));
  if (flags[0]) return rsg_fail(errbuf, "pm validation failed in a batch item");
  if (flags[1]) return rsg_fail(errbuf, "bad covariation (NaN after correction) in a batch item");
  HIPCHK(hipMemcpy(fits, d_fits, sizeof(double) * 8 * ng, hipMemcpyDeviceToHost));
  if (feats) {
    std::vector<unsigned long long> cnt((size_t)ng * 36);
    HIPCHK(hipMemcpy(cnt.data(), d_fcnt, sizeof(unsigned long long) * cnt.size(), hipMemcpyDeviceToHost));
    for (int g = 0; g < ng; g++) {
      const rsg_null_job &J = jobs[gfirst[(size_t)g]];
      rsg_feat_finish(&cnt[(size_t)g * 36], J.nleaf, J.alen, J.left, J.right, J.ld, J.rd, feats + (size_t)g * RSG_NULL_NFEAT);
    }
  }
  if (hists) {
    std::vector<HGeo> geo((size_t)ng);
    HIPCHK(hipMemcpy(geo.data(), d_geo, sizeof(HGeo) * ng, hipMemcpyDeviceToHost));
    std::vector<unsigned long long> h;
    for (int k = 0; k < ng; k++) {
      hists[k] = nullptr;
      const HGeo &g = geo[(size_t)k];
      if (!g.ok) continue;
      rsg_hist *H = rsg_hist_create(bmin, g.bmax, g.w);
      if (!H) return rsg_fail(errbuf, "out of memory");
      h.resize((size_t)g.nb);
      HIPCHK(hipMemcpy(h.data(), d_hist + g.off, sizeof(unsigned long long) * g.nb, hipMemcpyDeviceToHost));
      for (int b = 0; b < g.nb; b++) H->obs[b] = h[(size_t)b];
      H->n = H->Nc = H->No = (uint64_t)g.npairs;
      H->imin = H->cmin = g.imin; H->imax = g.imax; H->xmin = g.xmin; H->xmax = g.xmax;
      hists[k] = H;
    }
  }
  return RSG_OK;
}

extern "C" int rsg_ctx_graph_reuses(const rsg_ctx *c) { return c ? c->bexec_hits : 0; }

extern "C" int rsg_null_batch(rsg_ctx *c, const rsg_null_job *jobs, int nj, int covtype, double bmin, double pmass,
                              double fracfit, int doexpfit, rsg_hist **hists, double *fits, float *feats,
                              int use_graph, char *errbuf)
{
  if (!c || !jobs || !fits) return rsg_fail(errbuf, "rsg_null_batch: bad arguments");
  return null_batch_impl(c, jobs, nj, covtype, bmin, pmass, fracfit, doexpfit, hists, fits, feats, use_graph, nullptr,
                         nullptr, errbuf);
}

extern "C" int rsg_null_batch_fitch(rsg_ctx *c, const uint8_t *ax, int64_t nseq, int64_t alen, const int *left,
                                    const int *right, const uint64_t *seeds, int nrep, int covtype, double bmin,
                                    double pmass, double fracfit, int doexpfit, rsg_hist **hist, double *fit,
                                    int use_graph, char *errbuf)
{
  if (!c || !ax || !left || !right || !seeds || nrep < 1 || !fit) return rsg_fail(errbuf, "rsg_null_batch_fitch: bad arguments");
  FitchPlan P;
  if (rsg_fitch_plan(nseq, alen, left, right, P, errbuf) != RSG_OK) return RSG_FAIL;
  std::vector<rsg_null_job> jobs((size_t)nrep);
  for (int r = 0; r < nrep; r++) {
    rsg_null_job &J = jobs[(size_t)r];
    J.nleaf = nseq; J.alen = alen; J.left = left; J.right = right; J.ld = nullptr; J.rd = nullptr; J.model = nullptr;
    J.seed = seeds[r]; J.stream = (uint32_t)r; J.gapfrac = 0.; J.group = 0;
  }
  return null_batch_impl(c, jobs.data(), nrep, covtype, bmin, pmass, fracfit, doexpfit, hist, fit, nullptr, use_graph, ax,
                         &P, errbuf);
}
