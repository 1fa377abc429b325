// rsg_fitch.hip -- R-scape's own null alignment on the device: Fitch ancestral states,
// one shuffle of all columns, per-branch substitution replay.
//
// Reference: null_rscape (src/R-scape.c:1615-1724) -> Tree_FitchAlgorithmAncenstral
// (src/msatree.c:173-229, 1700-1931) -> msamanip_ShuffleTreeSubstitutions
// (src/msamanip.c:1449-1530, 1597-1780).  Symbols 0..4 (gap = 4 is a state); a leaf with
// another code enters the Fitch pass as one random state.  Draws are Philox4x32-10 keyed by
// (seed, purpose stream, node, position, tag) in place of Easel's sequential generator, so
// results match the reference in distribution and the oracle symbol for symbol.
//
// Rows: the internal nodes' state sets, states and shuffled rows are N - 1 rows of L bytes (node v ->
// row v) per replicate; leaves are read from the alignment itself and written to `leaves`.
// Work: the Fitch passes and the replay run one launch per tree depth (children before parents
// upward, parents before children downward).  A node (Fitch) or a branch (replay) is one work
// group; rows are read and written as dwords of four columns.
#include <type_traits>
#include "rsg_internal.h"
#include <algorithm>
#include <vector>

namespace {

typedef uint32_t u32u __attribute__((aligned(1)));

// node rows are keyed in the draws as the reference's allmsa rows: leaf n -> n, internal v -> N + v
__device__ __forceinline__ int row_of(int d, int64_t N) { return d > 0 ? (int)(N + d) : -d; }

// four columns of a row at c (bytes past L read as 0; unaligned: L is any number)
__device__ __forceinline__ uint32_t load4(const uint8_t *row, int64_t c, int64_t L)
{
  if (c + 4 <= L) return *(const u32u *)(row + c);
  uint32_t v = 0;
  for (int b = 0; b < 3; b++) if (c + b < L) v |= (uint32_t)row[c + b] << (8 * b);
  return v;
}
__device__ __forceinline__ void store4(uint8_t *row, int64_t c, int64_t L, uint32_t v)
{
  if (c + 4 <= L) { *(u32u *)(row + c) = v; return; }
  for (int b = 0; b < 3; b++) if (c + b < L) row[c + b] = (uint8_t)(v >> (8 * b));
}
// 0xFF in the bytes of v (each <= 0x7F) that are not 0
__device__ __forceinline__ uint32_t nonzero4(uint32_t v)
{
  const uint32_t n = (v + 0x7F7F7F7Fu) & 0x80808080u;
  return n | (n - (n >> 7));
}
// 1 << code for the codes 0..4 of four bytes, 0 for others (byte permute from a table)
__device__ __forceinline__ uint32_t bits4(uint32_t codes)
{
  const uint32_t big = (((codes >> 3) & 0x1F1F1F1Fu) + 0x7F7F7F7Fu) & 0x80808080u;      // code > 7
  return __builtin_amdgcn_perm(0x00000010u, 0x08040201u, (codes & 0x07070707u) | (big >> 5) | (big >> 6) | (big >> 7));
}

// inclusive sum over the lanes of a wave (DPP row shifts, then the row totals broadcast upward)
__device__ __forceinline__ uint32_t wave_scan(uint32_t x)
{
  x += __builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, false);
  x += __builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);      // row 0 -> 1, 2 -> 3
  x += __builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);      // lane 31 -> rows 2, 3
  return x;
}

// flag |= the alignment holds a code > 4: such a leaf enters the Fitch pass as one random state of
// its own in every replicate; without one the state sets are the same in all replicates and are
// formed once
__global__ void __launch_bounds__(256) k_fitch_scan(const uint8_t *__restrict__ ax, int64_t n, int *__restrict__ flag)
{
  uint32_t any = 0;
  const int64_t n4 = n / 4;
  for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n4; k += (int64_t)gridDim.x * 256) {
    const uint32_t v = ((const uint32_t *)ax)[k];
    any |= (v & 0xF8F8F8F8u) | (((v & 0x07070707u) + 0x03030303u) & 0x08080808u);      // > 7, or 5..7
  }
  if (blockIdx.x == 0 && threadIdx.x < (unsigned)(n & 3) && ax[n4 * 4 + threadIdx.x] > 4) any = 1;
  if (any) atomicOr(flag, 1);
}

// a child's state sets for four columns from its row's bytes there: an internal node's are the sets, a
// leaf's are codes: their bits, one random state for any other code
__device__ __forceinline__ uint32_t child_set(int d, uint32_t v, int64_t c, int64_t L, uint64_t seed)
{
  if (d > 0) return v;
  const uint32_t s = bits4(v);
  uint32_t other = ~nonzero4(s);
  if (c + 4 > L) other &= (1u << (8 * (int)(L - c))) - 1u;
  uint32_t r = s;
  while (other) {                                        // each lane its own byte: one round in most waves
    const int b = (__ffs(other) - 1) & ~7;
    other &= ~(0xFFu << b);
    r |= (1u << (int)(((uint64_t)rsg_philox(seed, 1u, (uint32_t)(-d), (uint32_t)(c + (b >> 3)), 1u) * 5u) >> 32)) << b;
  }
  return r;
}
// S_v = S_l & S_r, or the residues of S_l | S_r when the intersection is empty, for four columns; both
// children's bytes are asked for before either is looked at
__device__ __forceinline__ void up4(const int4 en, int64_t c, int64_t L, const uint8_t *ax, uint8_t *M, uint64_t seed)
{
  const uint8_t *pl = en.y > 0 ? M + (int64_t)en.y * L : ax + (int64_t)(-en.y) * L;
  const uint8_t *pr = en.z > 0 ? M + (int64_t)en.z * L : ax + (int64_t)(-en.z) * L;
  uint32_t vl, vr;
  if (c + 4 <= L) { vl = *(const u32u *)(pl + c); vr = *(const u32u *)(pr + c); }
  else            { vl = load4(pl, c, L); vr = load4(pr, c, L); }
  const uint32_t sl = child_set(en.y, vl, c, L, seed), sr = child_set(en.z, vr, c, L, seed), in = sl & sr;
  store4(M + (int64_t)en.x * L, c, L, in | (~nonzero4(in) & (sl | sr) & 0x0F0F0F0Fu));
}

// upward pass over the internal nodes of one depth (work group x: node, y: replicates y, y + grid.y,
// ..., replicate 0 only where all share it).  Bound by HBM and launch latency: 548 us for 20 replicates of
// N = 5000 x L = 1500 with a byte per thread and every replicate on its own, 96 us with a launch per
// depth, 66 us now (48 here for the depths of more than 64 nodes, 18 in k_fitch_up_run).
template <int NT>
__global__ void __launch_bounds__(NT) k_fitch_up(const int4 *__restrict__ ent, int64_t L, const uint8_t *__restrict__ ax,
                                                 const uint64_t *__restrict__ seeds, const int *__restrict__ flag, int R,
                                                 uint8_t *__restrict__ mask, int64_t rs)
{
  const int Ru = *flag ? R : 1;
  if ((int)blockIdx.y >= Ru) return;
  const int4 en = ent[blockIdx.x];
  for (int r = blockIdx.y; r < Ru; r += gridDim.y) {
    const uint64_t seed = seeds[r];
    for (int64_t c = 4 * threadIdx.x; c < L; c += 4 * NT) up4(en, c, L, ax, mask + r * rs, seed);
  }
}

// upward pass over several depths of no more than FITCH_RUN_W internal nodes each, the deepest first, depth d
// of the run being the entries U.lev[d] .. U.lev[d + 1).  A column needs only itself, so a work group takes
// 64 columns of all depths, 16 threads a node -- as many nodes as its threads hold at once: a wider
// depth would go round on a few CUs -- and the depths follow each other behind its own barriers.
// Bound by latency (a child's bytes, then the barrier): 1.4 us a depth, 25 us for 18 depths of 400
// sequences of 203 columns, which took 66 with a launch each.  (Runs of 32 depths at most: of 8 a null of 20
// replicates on a chain of 400 takes 2495 us in place of 2438, of 64 it takes 2426 with more kernel arguments.)
#define FITCH_RUN_W 64
#define FITCH_RUN_D 32
struct UpRun { int n, lev[FITCH_RUN_D + 1]; };
__global__ void __launch_bounds__(16 * FITCH_RUN_W)
k_fitch_up_run(const int4 *__restrict__ ent, UpRun U, int64_t L, const uint8_t *__restrict__ ax, const uint64_t *__restrict__ seeds,
               const int *__restrict__ flag, int R, uint8_t *mask, int64_t rs)
{
  const int Ru = *flag ? R : 1, node = threadIdx.x >> 4;
  const int64_t c = 64 * (int64_t)blockIdx.x + 4 * (threadIdx.x & 15);
  for (int r = blockIdx.y; r < Ru; r += gridDim.y) {
    uint8_t *M = mask + r * rs;
    const uint64_t seed = seeds[r];
    int4 en = ent[min(U.lev[U.n - 1] + node, U.lev[U.n] - 1)];
    for (int d = U.n - 1; d >= 0; d--) {
      const int4 nx = ent[d ? min(U.lev[d - 1] + node, U.lev[d] - 1) : 0];      // asked for ahead of the barrier
      if (U.lev[d] + node < U.lev[d + 1] && c < L) up4(en, c, L, ax, M, seed);
      en = nx;
      __syncthreads();
    }
  }
}

// downward pass over the internal nodes of one depth (work group x: node, y: replicate): keep the
// parent's state when the set holds it, else a uniform member.  Only sets of more than one member
// draw: they are gathered in LDS (a few per cent of the columns), so the draws run in full
// waves.  With nsub the branches' substitution counts nsub[2 v + side][old * 5 + new], old != new,
// are taken on the way: of the branch above the node, and of those to its leaves.  706 us (and
// 296 us for the counts, 197 us for copies of the leaves) at 20 x 5000 x 1500 with a draw per
// column and passes of their own.
template <int NT>
__device__ __forceinline__ void down_block(const int4 en, int64_t N, int64_t L, const uint8_t *__restrict__ ax,
                                           const uint64_t *__restrict__ seeds, const int *__restrict__ flag,
                                           const uint8_t *__restrict__ mask, uint8_t *__restrict__ all, int64_t rs,
                                           int *__restrict__ nsub)
{
  __shared__ uint32_t row[NT], queue[4 * NT];
  __shared__ int hist[3][25], nq;
  const int tid = threadIdx.x, v = en.x, dl = en.y, dr = en.z, pv = en.w >> 1;
  const int64_t r = blockIdx.y;
  const uint64_t seed = seeds[r];
  const uint8_t *M = mask + (*flag ? r * rs : 0) + (int64_t)v * L;
  uint8_t *A = all + r * rs;
  for (int k = tid; k < 75; k += NT) hist[k / 25][k % 25] = 0;
  // counts of the columns where two rows differ, a -> x, codes past 4 left out
  auto count = [&](int *h, uint32_t a, uint32_t x, int64_t c) {
    uint32_t diff = a ^ x;
    if (c + 4 > L) diff &= (1u << (8 * (int)(L - c))) - 1u;
    for (; diff; ) {
      const int b = (__ffs(diff) - 1) & ~7;
      diff &= ~(0xFFu << b);
      const unsigned xo = (a >> b) & 0xFFu, xn = (x >> b) & 0xFFu;
      if (xn <= 4u) atomicAdd(&h[xo * 5 + xn], 1);
    }
  };
  for (int64_t c0 = 0; c0 < L; c0 += 4 * NT) {
    const int64_t c = c0 + 4 * tid;
    if (tid == 0) nq = 0;
    __syncthreads();
    uint32_t S = 0, pa = 0, xl = 0, xr = 0;
    if (c < L) {
      S = load4(M, c, L);
      if (nsub && dl <= 0) xl = load4(ax + (int64_t)(-dl) * L, c, L);
      if (nsub && dr <= 0) xr = load4(ax + (int64_t)(-dr) * L, c, L);
      if (v > 0) {
        pa = load4(A + (int64_t)pv * L, c, L);
        const uint32_t keep = S & bits4(pa);
        S = keep | (S & ~nonzero4(keep));
      }
      uint32_t st = 0;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const uint32_t s = (S >> (8 * b)) & 0xFFu;
        if (s & (s - 1u)) queue[atomicAdd(&nq, 1)] = (uint32_t)(4 * tid + b) | (s << 16);
        else if (s) st |= (uint32_t)(__ffs(s) - 1) << (8 * b);
      }
      row[tid] = st;
    }
    __syncthreads();
    for (int k = tid; k < nq; k += NT) {
      const uint32_t e = queue[k], s = e >> 16, col = e & 0xFFFFu;
      const uint32_t u = rsg_philox(seed, 2u, (uint32_t)v, (uint32_t)(c0 + col), 2u);
      unsigned idx = (unsigned)(((uint64_t)u * __popc(s)) >> 32), m = s;
      for (; idx > 0; idx--) m &= m - 1u;
      ((uint8_t *)row)[col] = (uint8_t)(__ffs(m) - 1);
    }
    __syncthreads();
    if (c < L) {
      const uint32_t st = row[tid];
      store4(A + (int64_t)v * L, c, L, st);
      if (nsub) {
        if (v > 0) count(hist[0], pa, st, c);
        if (dl <= 0) count(hist[1], st, xl, c);
        if (dr <= 0) count(hist[2], st, xr, c);
      }
    }
  }
  if (!nsub) return;
  __syncthreads();
  int *ns = nsub + r * 2 * (N - 1) * 25;
  for (int k = tid; k < 75; k += NT) {
    const int h = k / 25, e = k % 25;
    if (h == 0) { if (v > 0) ns[en.w * 25 + e] = hist[0][e]; }
    else if ((h == 1 ? dl : dr) <= 0) ns[(2 * v + h - 1) * 25 + e] = hist[h][e];
  }
}
template <int NT>
__global__ void __launch_bounds__(NT) k_fitch_down(const int4 *__restrict__ ent, int64_t N, int64_t L,
                                                   const uint8_t *__restrict__ ax,
                                                   const uint64_t *__restrict__ seeds, const int *__restrict__ flag,
                                                   const uint8_t *__restrict__ mask, uint8_t *__restrict__ all, int64_t rs,
                                                   int *__restrict__ nsub)
{
  down_block<NT>(ent[blockIdx.x], N, L, ax, seeds, flag, mask, all, rs, nsub);
}

// the shuffled root of rows too long for k_shuffle_root: column c takes column perm[c] of the root's
// ancestral states
__global__ void k_gather_root(const uint8_t *__restrict__ all, const int *__restrict__ perm, int64_t L,
                              uint8_t *__restrict__ inner, int64_t rs)
{
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= L) return;
  inner[blockIdx.y * rs + c] = all[blockIdx.y * rs + perm[blockIdx.y * L + c]];
}

// Replay of the branches below the internal nodes of one depth, one work group per branch (x) and
// replicate (y).  For each old symbol the reference takes the parent's positions holding it
// (ascending, P[0..n)), does a partial Fisher-Yates -- step t swaps P[n - 1 - t] with P[k_t], k_t
// uniform in [0, n - t) -- and substitutes at P[n - 1 - t], t < take.  All steps of all symbols run
// at once: what ends at index n - 1 - t is what index k_t held before step t, and index j
// before step t holds what the latest step s < t with k_s = j moved there (index n - 1 - s before
// step s), or its own position if there is none: a walk of a link or two.  The steps that
// drew an index hang off it as a list.
// A row of bytes, the positions by symbol (low half: the position, high half: head of the
// index's list) and the lists' links are in LDS (7 L bytes; the draws stay in registers).
// Bound by latency (one depth after another) for the small depths, by LDS traffic and the draws for
// the wide ones.  One wave per branch applying the swaps one by one took 3075 us for 20 replicates
// of N = 5000 x L = 1500; this takes 600 us.
#define FITCH_LDS_L 9000
// (the symbols' ranges come as scalars by value: selecting among the elements of an array, or of a
// lambda's captures, puts them in scratch)
// index drawn by step g, uniform in [0, m) of its symbol's m = n - t positions
__device__ __forceinline__ int replay_draw(uint64_t seed, uint32_t node, int g, int n0, int n1, int n2, int n3, int n4, int b1,
                                           int b2, int b3, int b4)
{
  int o = 0, no = n0, oo = 0, bo = 0;
  if (g >= b1) { o = 1; no = n1; oo = n0; bo = b1; }
  if (g >= b2) { o = 2; no = n2; oo = n0 + n1; bo = b2; }
  if (g >= b3) { o = 3; no = n3; oo = n0 + n1 + n2; bo = b3; }
  if (g >= b4) { o = 4; no = n4; oo = n0 + n1 + n2 + n3; bo = b4; }
  const int m = no - (g - bo);
  int k = 0;
  if (m >= 2) k = (int)(((uint64_t)rsg_philox(seed, 4u, node + (uint32_t)o, (uint32_t)m, 4u) * (uint64_t)m) >> 32);
  return oo + k;
}
// step g onto the list of the index i it drew
__device__ __forceinline__ void replay_hang(uint32_t *P, uint16_t *nxt, int g, int i)
{
  const uint32_t pos = P[i] & 0xFFFFu;
  nxt[g] = (uint16_t)(atomicExch(&P[i], ((uint32_t)g << 16) | pos) >> 16);
}
// the position step g substitutes at (off5 = L: end of the last symbol's range), and its new symbol
__device__ __forceinline__ void replay_resolve(const uint32_t *P, const uint16_t *nxt, const int4 *cum, uint8_t *row, int g, int idx,
                                               int off1, int off2, int off3, int off4, int off5, int b1, int b2, int b3, int b4)
{
  int o = 0, top = off1 - 1, bo = 0;
  if (g >= b1) { o = 1; top = off2 - 1; bo = b1; }
  if (g >= b2) { o = 2; top = off3 - 1; bo = b2; }
  if (g >= b3) { o = 3; top = off4 - 1; bo = b3; }
  if (g >= b4) { o = 4; top = off5 - 1; bo = b4; }
  const int4 cm = cum[o];
  const int tt = g - bo;
  int tm = g;
  uint32_t p = P[idx];
  for (;;) {                                               // tm falls with every round
    int s = -1;
    for (int e = (int)(p >> 16); e != 0xFFFF; e = nxt[e]) if (e < tm && e > s) s = e;
    if (s < 0) break;
    tm = s; idx = top - (s - bo);
    p = P[idx];
  }
  row[p & 0xFFFFu] = (uint8_t)((tt >= cm.x) + (tt >= cm.y) + (tt >= cm.z) + (tt >= cm.w));
}

// The shuffled root of every replicate (one work group each): the column permutation of
// rsg_fitch_perm, a Fisher-Yates whose step t swaps the positions L - 1 - t and k_t, all steps at once
// as in the replay (one symbol, L positions, L steps), and column L - 1 - t of the root takes the
// ancestral state of the position found there.  Bound by latency: 12 us for 1500 columns, where the host's
// permutations of 20 replicates took 145 us and their upload came on top.  Rows to FITCH_LDS_L columns.
__global__ void __launch_bounds__(512) k_shuffle_root(const uint8_t *__restrict__ all, const uint64_t *__restrict__ seeds, int L,
                                                      uint8_t *__restrict__ inner, int64_t rs)
{
  extern __shared__ uint32_t lds[];
  uint32_t *P = lds;
  uint16_t *nxt = (uint16_t *)(P + L);
  const uint64_t seed = seeds[blockIdx.x];
  const uint8_t *a = all + blockIdx.x * rs;
  uint8_t *o = inner + blockIdx.x * rs;
  auto draw = [&](int t) {
    const uint32_t n = (uint32_t)(L - t);
    return n >= 2u ? (int)(((uint64_t)rsg_philox(seed, 3u, 0u, n, 3u) * (uint64_t)n) >> 32) : 0;
  };
  for (int i = threadIdx.x; i < L; i += 512) P[i] = 0xFFFF0000u | (uint32_t)i;
  __syncthreads();
  for (int t = threadIdx.x; t < L; t += 512) replay_hang(P, nxt, t, draw(t));
  __syncthreads();
  for (int t = threadIdx.x; t < L; t += 512) {
    int idx = draw(t), tm = t;
    uint32_t p = P[idx];
    for (;;) {                                             // tm falls with every round
      int s = -1;
      for (int e = (int)(p >> 16); e != 0xFFFF; e = nxt[e]) if (e < tm && e > s) s = e;
      if (s < 0) break;
      tm = s; idx = L - 1 - s;
      p = P[idx];
    }
    o[L - 1 - t] = a[p & 0xFFFFu];
  }
}

template <int NT>
__device__ __forceinline__ void replay_block(int bx, const int4 *__restrict__ ent, int64_t N, int L,
                                             const uint64_t *__restrict__ seeds, const int *__restrict__ nsub,
                                             uint8_t *__restrict__ leaves, uint8_t *__restrict__ inner, int64_t rs)
{
  extern __shared__ uint32_t lds[];
  constexpr int NW = NT / 64;
  const int L4 = (L + 3) / 4;
  uint32_t *P = lds;                                     // [L] list head << 16 | position
  uint16_t *nxt = (uint16_t *)(P + L);                   // [L] list links
  uint32_t *row = (uint32_t *)(nxt + ((L + 1) & ~1));    // [L4]
  __shared__ int4 cum[5];                                // per old symbol: running counts of new symbols 0..3
  __shared__ uint2 wsum[NW];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t r = blockIdx.y;
  const int4 en = ent[bx >> 1];
  const int v = en.x, side = bx & 1, d = side ? en.z : en.y;
  const uint32_t node = (uint32_t)row_of(d, N) * 5u;
  const uint64_t seed = seeds[r];
  const uint8_t *pa = inner + r * rs + (int64_t)v * L;
  uint8_t *ch = (d > 0) ? inner + r * rs + (int64_t)d * L : leaves + r * N * (int64_t)L + (int64_t)(-d) * L;
  const int *cnt = nsub + (r * 2 * (N - 1) + 2 * v + side) * 25;
  if (tid < 5) {
    const int *q = cnt + 5 * tid;
    const int a = q[0], b = a + q[1], c = b + q[2];
    cum[tid] = make_int4(a, b, c, c + q[3]);
  }
  // the parent's row: thread t takes the dwords t q .. t q + q - 1, so positions ascend with threads;
  // counts of symbols 0..3 in 16-bit halves
  const int q = (L4 + NT - 1) / NT, w0 = tid * q, w1 = min(w0 + q, L4);
  uint32_t c01 = 0u, c23 = 0u;
  for (int w = w0; w < w1; w++) {
    const uint32_t x = load4(pa, 4 * (int64_t)w, L);
    row[w] = x;
    uint32_t h = bits4(x);
    if (4 * w + 4 > L) h &= (1u << (8 * (L - 4 * w))) - 1u;
    c01 += __popc(h & 0x01010101u) + (__popc(h & 0x02020202u) << 16);
    c23 += __popc(h & 0x04040404u) + (__popc(h & 0x08080808u) << 16);
  }
  uint32_t s01 = wave_scan(c01), s23 = wave_scan(c23);   // inclusive
  if (lane == 63) wsum[wv] = make_uint2(s01, s23);
  __syncthreads();
  uint32_t t01 = 0u, t23 = 0u;
#pragma unroll
  for (int k = 0; k < NW; k++) {
    const uint2 ws = wsum[k];
    if (k < wv) { s01 += ws.x; s23 += ws.y; }
    t01 += ws.x; t23 += ws.y;
  }
  t01 = __builtin_amdgcn_readfirstlane(t01); t23 = __builtin_amdgcn_readfirstlane(t23);
  // symbol o: n_o positions from off_o, steps b_o .. b_(o + 1) - 1 (uniform)
  const int n0 = (int)(t01 & 0xFFFFu), n1 = (int)(t01 >> 16), n2 = (int)(t23 & 0xFFFFu), n3 = (int)(t23 >> 16),
            n4 = L - n0 - n1 - n2 - n3;
  const int off1 = n0, off2 = off1 + n1, off3 = off2 + n2, off4 = off3 + n3;
  auto subs = [=](int o) { const int *z = cnt + 5 * o; return z[0] + z[1] + z[2] + z[3] + z[4]; };
  const int b1 = min(subs(0), n0), b2 = b1 + min(subs(1), n1), b3 = b2 + min(subs(2), n2), b4 = b3 + min(subs(3), n3);
  const int total = b4 + min(subs(4), n4);
  if (total > 0) {
    int nx[5];
    nx[0] = (int)((s01 - c01) & 0xFFFFu); nx[1] = (int)((s01 - c01) >> 16);
    nx[2] = (int)((s23 - c23) & 0xFFFFu); nx[3] = (int)((s23 - c23) >> 16);
    nx[4] = 4 * w0 - nx[0] - nx[1] - nx[2] - nx[3];      // (unused where w0 >= L4)
    nx[1] += off1; nx[2] += off2; nx[3] += off3; nx[4] += off4;
    for (int w = w0; w < w1; w++) {
      const uint32_t x = row[w];
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const unsigned s = (x >> (8 * b)) & 0xFFu;
        if (4 * w + b < L) {
          int at = nx[4];
#pragma unroll
          for (int o = 0; o < 4; o++) at = (s == (unsigned)o) ? nx[o] : at;
#pragma unroll
          for (int o = 0; o < 5; o++) nx[o] += (s == (unsigned)o);
          P[at] = 0xFFFF0000u | (uint32_t)(4 * w + b);
        }
      }
    }
    __syncthreads();
    int ki[4];                                             // the first rounds' indices; later ones are drawn again
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int g = tid + u * NT;
      if (g < total) { ki[u] = replay_draw(seed, node, g, n0, n1, n2, n3, n4, b1, b2, b3, b4); replay_hang(P, nxt, g, ki[u]); }
    }
    for (int g = tid + 4 * NT; g < total; g += NT)
      replay_hang(P, nxt, g, replay_draw(seed, node, g, n0, n1, n2, n3, n4, b1, b2, b3, b4));
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int g = tid + u * NT;
      if (g < total) replay_resolve(P, nxt, cum, (uint8_t *)row, g, ki[u], off1, off2, off3, off4, L, b1, b2, b3, b4);
    }
    for (int g = tid + 4 * NT; g < total; g += NT)
      replay_resolve(P, nxt, cum, (uint8_t *)row, g, replay_draw(seed, node, g, n0, n1, n2, n3, n4, b1, b2, b3, b4), off1, off2,
                     off3, off4, L, b1, b2, b3, b4);
  }
  __syncthreads();
  for (int w = tid; w < L4; w += NT) store4(ch, 4 * (int64_t)w, L, row[w]);
}
template <int NT>
__global__ void __launch_bounds__(NT) k_fitch_replay(const int4 *__restrict__ ent, int64_t N, int L,
                                                     const uint64_t *__restrict__ seeds, const int *__restrict__ nsub,
                                                     uint8_t *__restrict__ leaves, uint8_t *__restrict__ inner, int64_t rs)
{
  replay_block<NT>((int)blockIdx.x, ent, N, L, seeds, nsub, leaves, inner, rs);
}

// The replay of one depth (the first nrep work groups) beside the downward pass two depths below it,
// which counts the substitutions of the next depths' branches: narrow depths are bound by
// the latency of a launch, so two share one.
template <int NT>
__global__ void __launch_bounds__(NT) k_fitch_down_replay(const int4 *__restrict__ rent, int nrep, const int4 *__restrict__ dent,
                                                          int64_t N, int64_t L, const uint8_t *__restrict__ ax,
                                                          const uint64_t *__restrict__ seeds, const int *__restrict__ flag,
                                                          const uint8_t *__restrict__ mask, uint8_t *__restrict__ all, int64_t rs,
                                                          int *__restrict__ nsub, uint8_t *__restrict__ leaves,
                                                          uint8_t *__restrict__ inner)
{
  if ((int)blockIdx.x < nrep) replay_block<NT>((int)blockIdx.x, rent, N, (int)L, seeds, nsub, leaves, inner, rs);
  else                        down_block<NT>(dent[blockIdx.x - nrep], N, L, ax, seeds, flag, mask, all, rs, nsub);
}

// The replay for rows too long for LDS (L > FITCH_LDS_L): one wave per branch.  For each
// old symbol: the parent's positions holding it (ascending, ballot compaction) in cols_all (L ints
// per wave slot, 2 maxw slots per replicate), the swaps, whose indices the 64 lanes draw ahead,
// applied in order by lane 0, then the positions that receive substitutions written in parallel.
__global__ void __launch_bounds__(256) k_fitch_replay_long(const int4 *__restrict__ ent, int nn, int64_t N, int64_t L,
                                                           const uint64_t *__restrict__ seeds, const int *__restrict__ nsub,
                                                           uint8_t *__restrict__ leaves, uint8_t *__restrict__ inner,
                                                           int *__restrict__ cols_all, int maxw)
{
  __shared__ int kbuf[4][64];                                 // drawn swap indices, per wave
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int slot = blockIdx.x * 4 + wv;                       // branch slot in this level
  if (slot >= 2 * nn) return;
  const int64_t r = blockIdx.y;
  const uint64_t seed = seeds[r];
  nsub += r * 2 * (N - 1) * 25;
  leaves += r * N * L;
  inner += r * (N - 1) * L;
  const int4 en = ent[slot >> 1];
  const int v = en.x, side = slot & 1;
  const int d = side ? en.z : en.y;
  const int chrow = row_of(d, N);
  const int b = 2 * v + side;
  const uint8_t *pa = inner + (int64_t)v * L;
  uint8_t *ch = (d > 0) ? inner + (int64_t)d * L : leaves + (int64_t)(-d) * L;
  int *cols = cols_all + (r * 2 * maxw + slot) * L;
  for (int64_t c = lane; c < L; c += 64) ch[c] = pa[c];
  wave_sync();
  for (int oldc = 0; oldc < 5; oldc++) {
    int cnt[5], nst = 0;
    for (int nw = 0; nw < 5; nw++) { cnt[nw] = nsub[b * 25 + oldc * 5 + nw]; nst += cnt[nw]; }
    if (!nst) continue;
    // positions of the parent holding oldc, ascending (ballot compaction)
    int ncol = 0;
    for (int64_t c0 = 0; c0 < L; c0 += 64) {
      const int64_t c = c0 + lane;
      const bool hit = c < L && pa[c] == oldc;
      const unsigned long long bal = __ballot(hit);
      if (hit) cols[ncol + __popcll(bal & ((1ull << lane) - 1ull))] = (int)c;
      ncol += __popcll(bal);
    }
    wave_sync();                                              // cols visible to lane 0
    if (ncol == 0) continue;
    // partial Fisher-Yates: step n (ncol down to nlow) swaps positions n - 1 and k_n; only the
    // last take = min(nst, ncol) positions receive substitutions
    const int take = nst < ncol ? nst : ncol;
    const int nlow = (ncol - take + 1 > 2) ? ncol - take + 1 : 2;
    for (int n0 = ncol; n0 >= nlow; n0 -= 64) {
      const int n = n0 - lane;
      if (n >= nlow) {
        const uint32_t u = rsg_philox(seed, 4u, (uint32_t)(chrow * 5 + oldc), (uint32_t)n, 4u);
        kbuf[wv][lane] = (int)(((uint64_t)u * (uint64_t)n) >> 32);
      }
      wave_sync();
      if (lane == 0) {
        const int steps = (n0 - nlow + 1 < 64) ? n0 - nlow + 1 : 64;
        for (int t = 0; t < steps; t++) {
          const int nn1 = n0 - t - 1, k = kbuf[wv][t];
          const int x = cols[nn1]; cols[nn1] = cols[k]; cols[k] = x;
        }
      }
      wave_sync();
    }
    // position ncol - 1 - t (t < take) gets the new symbol whose cumulative count first exceeds t
    for (int t = lane; t < take; t += 64) {
      int acc = 0, sym = 4;
      for (int nw = 0; nw < 5; nw++) { if (t < acc + cnt[nw]) { sym = nw; break; } acc += cnt[nw]; }
      ch[cols[ncol - 1 - t]] = (uint8_t)sym;
    }
    wave_sync();
  }
}

struct Buf {
  std::vector<void *> p;
  ~Buf() { for (void *q : p) hipFree(q); }
  template <typename T> bool get(T **o, size_t n)
  {
    void *q = nullptr;
    if (rsg_dev_malloc(&q, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) return false;
    p.push_back(q); *o = (T *)q;
    return true;
  }
};

} // namespace

int rsg_fitch_plan(int64_t N, int64_t L, const int *left, const int *right, FitchPlan &P, char *errbuf)
{
  if (!left || !right || N < 2 || L < 1) return rsg_fail(errbuf, "Fitch null: bad arguments");
  if (N > (1 << 28) || L > (1 << 30)) return rsg_fail(errbuf, "Fitch null: alignment too large");
  const int m = (int)(N - 1);
  // depths of the internal nodes (walk from the root; malformed trees rejected), parents
  std::vector<int> depth((size_t)m, -1), stack(1, 0);
  std::vector<int> parent((size_t)m, 0);                     // 2 * parent + side
  depth[0] = 0;
  int seen = 1, maxd = 0;
  while (!stack.empty()) {
    const int v = stack.back(); stack.pop_back();
    for (int side = 0; side < 2; side++) {
      const int d = side ? right[v] : left[v];
      if (d > 0) {
        if (d >= m || depth[(size_t)d] >= 0) return rsg_fail(errbuf, "Fitch null: malformed tree at node %d", v);
        depth[(size_t)d] = depth[(size_t)v] + 1; parent[(size_t)d] = 2 * v + side; maxd = std::max(maxd, depth[(size_t)d]);
        stack.push_back(d); seen++;
      } else if (-d >= N) return rsg_fail(errbuf, "Fitch null: leaf index %d out of range", -d);
    }
  }
  if (seen != m) return rsg_fail(errbuf, "Fitch null: %d internal nodes unreachable from the root", m - seen);
  P.lev0.assign((size_t)maxd + 2, 0);
  for (int v = 0; v < m; v++) P.lev0[(size_t)depth[(size_t)v] + 1]++;
  for (int k = 0; k <= maxd; k++) P.lev0[(size_t)k + 1] += P.lev0[(size_t)k];
  P.ent.resize((size_t)m);
  {
    std::vector<int> fill(P.lev0.begin(), P.lev0.end() - 1);
    for (int v = 0; v < m; v++)
      P.ent[(size_t)fill[(size_t)depth[(size_t)v]]++] = make_int4(v, left[v], right[v], parent[(size_t)v]);
  }
  P.maxw = 0;
  for (int k = 0; k <= maxd; k++) P.maxw = std::max(P.maxw, P.lev0[(size_t)k + 1] - P.lev0[(size_t)k]);
  P.N = N; P.L = L; P.m = m; P.maxd = maxd;
  return RSG_OK;
}

// one permutation of all columns (Fisher-Yates as esl_vec_IShuffle), for rows of more than FITCH_LDS_L
void rsg_fitch_perm(uint64_t seed, int64_t L, int *perm)
{
  for (int64_t k = 0; k < L; k++) perm[k] = (int)k;
  for (int64_t n = L; n > 1; n--) {
    const uint32_t u = rsg_philox(seed, 3u, 0u, (uint32_t)n, 3u);
    const int64_t k = (int64_t)(((uint64_t)u * (uint64_t)n) >> 32);
    std::swap(perm[n - 1], perm[k]);
  }
}

// Fitch ancestral states (Tree_FitchAlgorithmAncenstral) of R replicates: D.all receives every
// internal node's state, D.nsub (unless null) the branches' substitution counts.  D.flag is 0 on
// entry, or what an earlier run on the same alignment left.
template <int NT>
static void fitch_up(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R)
{
  const int64_t N = P.N, L = P.L, rs = (N - 1) * L;
  hipLaunchKernelGGL(k_fitch_scan, dim3((unsigned)std::min<int64_t>(1024, N * L / 4096 + 1)), dim3(256), 0, c->stream, D.ax, N * L,
                     D.flag);
  for (int k = P.maxd; k >= 0; k--) {
    const int nn = P.lev0[(size_t)k + 1] - P.lev0[(size_t)k];
    // runs of narrow depths in one launch
    UpRun U;
    int k0 = k + 1;
    while (k0 > 0 && k - k0 + 1 < FITCH_RUN_D && P.lev0[(size_t)k0] - P.lev0[(size_t)k0 - 1] <= FITCH_RUN_W) k0--;
    U.n = k - k0 + 1;
    if (U.n > 1) {
      for (int d = 0; d <= U.n; d++) U.lev[d] = P.lev0[(size_t)(k0 + d)];
      const int64_t nx = (L + 63) / 64;
      const unsigned ru = (unsigned)std::min<int64_t>(R, std::max<int64_t>(5, 4096 / nx));
      hipLaunchKernelGGL(k_fitch_up_run, dim3((unsigned)nx, ru), dim3(16 * FITCH_RUN_W), 0, c->stream, D.ent, U, L, D.ax, D.seeds,
                         D.flag, R, D.mask, rs);
      k = k0;
      continue;
    }
    // where the sets are shared all work groups of a node but the first end at once: no more than
    // 4096 of them per launch (five per node at least, so that a launch still fills the device
    // when every replicate has its own sets)
    const unsigned ry = (unsigned)std::min(R, std::max(5, 4096 / nn));
    hipLaunchKernelGGL(k_fitch_up<NT>, dim3((unsigned)nn, ry), dim3(NT), 0, c->stream, D.ent + P.lev0[(size_t)k], L, D.ax, D.seeds, D.flag, R, D.mask, rs);
  }
}
template <int NT>
static void fitch_down(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R, int k)
{
  const int nn = P.lev0[(size_t)k + 1] - P.lev0[(size_t)k];
  // wide depths: two waves per row, whose rounds are filled (1500 columns, 20 replicates, the widest
  // depth: 34 us; one wave 39, four 39, six 48)
  if (NT > 128 && (int64_t)nn * R > 1024)
    hipLaunchKernelGGL(k_fitch_down<128>, dim3((unsigned)nn, (unsigned)R), dim3(128), 0, c->stream, D.ent + P.lev0[(size_t)k], P.N,
                       P.L, D.ax, D.seeds, D.flag, D.mask, D.all, (P.N - 1) * P.L, D.nsub);
  else
    hipLaunchKernelGGL(k_fitch_down<NT>, dim3((unsigned)nn, (unsigned)R), dim3(NT), 0, c->stream, D.ent + P.lev0[(size_t)k], P.N, P.L,
                       D.ax, D.seeds, D.flag, D.mask, D.all, (P.N - 1) * P.L, D.nsub);
}

// Threads of a work group of the passes: enough for a dword (four columns) each, so that a row takes one
// round of a pass's barriers, 512 at most.  1500 columns: 256 threads take a second round for 119 dwords
// (upward pass 4.3 us a depth), 384 take one (3.5).  Past 2048 columns the rounds go on at 512: a null of
// 1000 sequences of 2049, 4096 and 9000 columns takes 366, 618 and 1956 us, with 256 threads 422, 727 and
// 2208, with 384 389, 682 and 2067; ten of them at once, where a depth has work groups enough, 1227 and
// 3231 us at 2049 and 4096 columns, with 256 threads 1225 and 3395.
template <class F>
static int fitch_width(int64_t L, F f)
{
  if (L <= 256)  return f(std::integral_constant<int, 64>());
  if (L <= 512)  return f(std::integral_constant<int, 128>());
  if (L <= 1024) return f(std::integral_constant<int, 256>());
  if (L <= 1536) return f(std::integral_constant<int, 384>());
  return f(std::integral_constant<int, 512>());
}

template <int NT>
static int fitch_ancestral(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R)
{
  fitch_up<NT>(c, P, D, R);
  for (int k = 0; k <= P.maxd; k++) fitch_down<NT>(c, P, D, R, k);
  return hipGetLastError() == hipSuccess ? RSG_OK : RSG_FAIL;
}
int rsg_fitch_ancestral(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R)
{
  return fitch_width(P.L, [&](auto nt) { return fitch_ancestral<decltype(nt)::value>(c, P, D, R); });
}

// The whole null: up, down, and the replay of each depth two depths behind the downward pass (it
// needs the counts of the branches below, which the next depth's pass forms).
template <int NT>
static int fitch_null(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R)
{
  const int64_t N = P.N, L = P.L, rs = (N - 1) * L;
  const unsigned ry = (unsigned)R;
  const size_t lds = 4 * (size_t)L + 2 * (size_t)((L + 1) & ~1) + 4 * (size_t)((L + 3) / 4);
  fitch_up<NT>(c, P, D, R);
  for (int t = 0; t <= P.maxd + 2; t++) {
    const int k = t - 2;                                     // the depth to replay
    const bool down = t <= P.maxd;
    if (k < 0) {
      if (down) fitch_down<NT>(c, P, D, R, t);
      if (t == 0 && L <= FITCH_LDS_L)
        hipLaunchKernelGGL(k_shuffle_root, dim3(ry), dim3(512), 4 * (size_t)L + 2 * (size_t)((L + 1) & ~1), c->stream, D.all,
                           D.seeds, (int)L, D.inner, rs);
      else if (t == 0)
        hipLaunchKernelGGL(k_gather_root, dim3((unsigned)((L + 255) / 256), ry), dim3(256), 0, c->stream, D.all, D.perm, L, D.inner, rs);
      continue;
    }
    if (k > P.maxd) break;
    const int nn = P.lev0[(size_t)k + 1] - P.lev0[(size_t)k];
    const int4 *ent = D.ent + P.lev0[(size_t)k];
    // wide depths are bound by instructions: two waves per branch spend fewer on sums and partly
    // filled rounds of steps than four, which shorten the latency of the narrow ones
    const bool wide = NT != 64 && (int64_t)2 * nn * R > 2048;
    if (L <= FITCH_LDS_L && !wide && down) {
      const int nd = P.lev0[(size_t)t + 1] - P.lev0[(size_t)t];
      hipLaunchKernelGGL(k_fitch_down_replay<NT>, dim3((unsigned)(2 * nn + nd), ry), dim3(NT), lds, c->stream, ent, 2 * nn,
                         D.ent + P.lev0[(size_t)t], N, L, D.ax, D.seeds, D.flag, D.mask, D.all, rs, D.nsub, D.leaves, D.inner);
      continue;
    }
    if (down) fitch_down<NT>(c, P, D, R, t);
    if (L > FITCH_LDS_L)
      hipLaunchKernelGGL(k_fitch_replay_long, dim3((unsigned)((2 * nn + 3) / 4), ry), dim3(256), 0, c->stream, ent, nn, N, L,
                         D.seeds, D.nsub, D.leaves, D.inner, D.cols, P.maxw);
    else if (wide)
      hipLaunchKernelGGL(k_fitch_replay<128>, dim3((unsigned)(2 * nn), ry), dim3(128), lds, c->stream, ent, N, (int)L,
                         D.seeds, D.nsub, D.leaves, D.inner, rs);
    else
      hipLaunchKernelGGL(k_fitch_replay<NT>, dim3((unsigned)(2 * nn), ry), dim3(NT), lds, c->stream, ent, N, (int)L,
                         D.seeds, D.nsub, D.leaves, D.inner, rs);
  }
  return hipGetLastError() == hipSuccess ? RSG_OK : RSG_FAIL;
}

int rsg_fitch_launch(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R)
{
  return fitch_width(P.L, [&](auto nt) { return fitch_null<decltype(nt)::value>(c, P, D, R); });
}

bool rsg_fitch_host_perm(const FitchPlan &P) { return P.L > FITCH_LDS_L; }
size_t rsg_fitch_cols(const FitchPlan &P) { return P.L > FITCH_LDS_L ? 2 * (size_t)P.maxw * (size_t)P.L : 1; }

extern "C" int rsg_null_fitch(rsg_ctx *c, const uint8_t *ax, int64_t N, int64_t L, const int *left, const int *right,
                              uint64_t seed, uint8_t *leaves, char *errbuf)
{
  if (!c || !ax || !left || !right || !leaves) return rsg_fail(errbuf, "rsg_null_fitch: bad arguments");
  HIPCHK(hipSetDevice(c->device));
  FitchPlan P;
  if (rsg_fitch_plan(N, L, left, right, P, errbuf) != RSG_OK) return RSG_FAIL;
  std::vector<int> perm;
  if (rsg_fitch_host_perm(P)) { perm.resize((size_t)L); rsg_fitch_perm(seed, L, perm.data()); }
  const int64_t m = P.m;
  Buf B;
  uint8_t *d_ax, *d_mask, *d_all, *d_inner, *d_leaves; int4 *d_ent; int *d_perm, *d_nsub, *d_cols;
  uint64_t *d_seed;
  const uint64_t seed2[2] = {seed, 0u};                     // the seed, then the flag
  if (!B.get(&d_ax, (size_t)(N * L)) || !B.get(&d_mask, (size_t)(m * L)) || !B.get(&d_all, (size_t)(m * L)) ||
      !B.get(&d_inner, (size_t)(m * L)) || !B.get(&d_leaves, (size_t)(N * L)) || !B.get(&d_ent, (size_t)m) ||
      !B.get(&d_perm, perm.size()) || !B.get(&d_nsub, (size_t)(2 * m) * 25) || !B.get(&d_cols, rsg_fitch_cols(P)) ||
      !B.get(&d_seed, 2))
    return rsg_fail(errbuf, "rsg_null_fitch: out of device memory");
  HIPCHK(hipMemcpyAsync(d_ax, ax, (size_t)(N * L), hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(d_ent, P.ent.data(), sizeof(int4) * m, hipMemcpyHostToDevice, c->stream));
  if (!perm.empty()) HIPCHK(hipMemcpyAsync(d_perm, perm.data(), sizeof(int) * L, hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(d_seed, seed2, sizeof(seed2), hipMemcpyHostToDevice, c->stream));
  FitchDev D{d_ax, d_ent, d_perm, d_seed, (int *)(d_seed + 1), d_mask, d_all, d_inner, d_leaves,
             d_nsub, d_cols};
  int t; rsg_tstart(c, "fitch_null", &t);
  const int st = rsg_fitch_launch(c, P, D, 1);
  rsg_tstop(c, t);
  if (st != RSG_OK) return rsg_fail(errbuf, "rsg_null_fitch: launch failed");
  HIPCHK(hipMemcpyAsync(leaves, d_leaves, (size_t)(N * L), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  return RSG_OK;
}
