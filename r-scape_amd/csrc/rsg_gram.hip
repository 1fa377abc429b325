// rsg_gram.hip -- pair-count tables as one-hot Gram contractions on CDNA4 MFMA.
//
// Replaces the O(L^2 N) gather loop of mutual_naive_ppij (src/correlators.c:1695-1780,
// driven by corr_NaivePP :1300-1317).  With GAPASCHAR == 0 (src/rscape_config.h:48) the
// table of a column pair is 4 x 4: c[x][y] = sum_s w_s [a_si == x][a_sj == y] over
// canonical symbols.  Writing X for the N x 4L one-hot matrix, all tables at once are the
// Gram C = X^T diag(w) X; only upper-triangular column blocks are formed.
//
// Staging: a one-hot nibble (unit weights) or byte (weights) per (column, sequence), 1 << symbol,
// 0 for gap / N, stored K-chunked ("x4": [Npad / 32][Lpad][16 bytes], "xt": [Npad / 16][Lpad][16
// bytes]: the 32 or 16 sequences of a chunk for every column, chunk after chunk), so the rows of a
// stage are contiguous in HBM and in LDS and the Grams move them with LDS-direct loads.  A wave
// owns 32 i-columns x 32 j-columns and keeps the symbol cells as MFMA accumulators
// ("symbol-major" tiles): each lane reads the 16 staged bytes of its column once per chunk and
// derives the symbol operands in registers.
//
// Unit weights: FP4 MFMA (v_mfma_f32_32x32x64_f8f6f4, E2M1 operands, FP32 accumulation), exact.
//   The operand of symbols A, C, G is the staged nibble masked with 1, 2, 4: the FP4 numbers 0.5,
//   1, 2 or 0; U's nibble (8 would be -0) is shifted right first, giving 2 or 0.  A product is
//   one of 1/4 .. 4 exactly, the cell's unit; an accumulator starts at 2^23 units, where one
//   FP32 ulp is one unit, so every sum is exact and the low mantissa bits are the count (up to
//   65535 sequences; above, from 0, in K segments past FP4_EXACT sequences, and the count is the
//   accumulator over the unit).  The FP4 matrix rate is twice the int8 one (9.8 against
//   4.95 PFLOP/s measured from registers) and a panel holds half the bytes: the same Gram on int8
//   operands took 67 us at N = 5000 x L = 1500 (44 us here, of which 18 at the full matrix rate;
//   the rest is each tile's epilogue, the masks that share the issue slots with the matrix
//   instructions, and the last, partial wave of tiles), 49 us at 4096 x 768 (20.7 us,
//   k_gram_fp4_deep), 3.76 ms at 24576 x 6144 (2.1 ms, 7.0 PFLOP/s).
// Weights: int8 limbs (v_mfma_i32_32x32x32_i8), or split-BF16 (w = hi + lo [+ lo2]) MFMA
//   (v_mfma_f32_32x32x16_bf16); the i-side operand is 1.0 where the symbol matches, the j-side
//   operand the split weight part; all parts accumulate into one FP32 accumulator.
//
// MFMA 32x32 operand / result lane layout (CDNA3/4): A row m and B column n belong to
// lanes with lane % 32 == m (resp. n); the K values split across lane / 32; result
// register r of lane l holds D[8*(r/4) + 4*(l/32) + r%4][l % 32].  A rows are j columns,
// B columns are i columns.  A Gram uses the same K assignment on both sides, so the
// order in which the hardware pairs K values need not be known.
//
// Output: a 16-cell record per column pair i < j at record rsg_rec(i, j) = j*L + i,
// cell x*4+y (the layout of pp[i][j][IDX(x,y,4)] in the reference); unit-weight records hold
// uint16 counts (N <= 65535), weighted ones FP32.
#include "rsg_device.h"
#include <dlfcn.h>
#include <map>
#include <mutex>
#include <tuple>
#include <algorithm>

typedef int   v4i  __attribute__((ext_vector_type(4)));
typedef int   v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef int   v8i  __attribute__((ext_vector_type(8)));
typedef unsigned v16u __attribute__((ext_vector_type(16)));

#define NPAD_Q 512            // sequence padding quantum (covers every K-tile size below)

int64_t rsg_npad(int64_t N) { return ((N + NPAD_Q - 1) / NPAD_Q) * NPAD_Q; }

// ------------------------------------------------------------------------------------
// What rides on a packing launch, in the grid rows from y = gy on: the logarithms of counts 0 .. N
// (lgc; k_logtab's values) and the list of 32 x 32-column tiles of the pair triangle in the Gram's
// order (bi ascending, then bj = bi .. nb - 1; the last diagonal tile is left out when its block
// holds one column).  As kernels of their own in the chain of a small alignment they took 2 us
// each and their share of the launches (200 x 120 scored in 54 us with them and whole tiles in the
// statistic, in 41 us without).
struct PackAux { int gy; int64_t N; double *lgc; int2 *tiles; int nb, ntiles; };
__device__ __forceinline__ void pack_aux(const PackAux &X)
{
  const int64_t e = ((int64_t)(blockIdx.y - X.gy) * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
  if (X.lgc && e <= X.N) log_entry(X.N, e, X.lgc);
  if (e < X.ntiles) {
    const int t = (int)e;
    int bi = 0;
    while ((bi + 1) * X.nb - ((bi + 1) * bi) / 2 <= t) bi++;    // first entry of row bi + 1 > t
    const int off = bi * X.nb - (bi * (bi - 1)) / 2;
    X.tiles[t] = make_int2(bi, bi + (t - off));
  }
}

// The packed forms of a resident alignment (pack_block).
template <int WHAT>
__global__ void __launch_bounds__(256) k_pack(const uint8_t *__restrict__ ax, int64_t N, int64_t L, int64_t Npad, int64_t Lpad,
                                              uint8_t *__restrict__ axT, uint8_t *__restrict__ xt, uint8_t *__restrict__ x4,
                                              PackAux X)
{
  if ((int)blockIdx.y >= X.gy) { pack_aux(X); return; }
  pack_block<WHAT>(ax, N, L, Npad, Lpad, (int64_t)blockIdx.y * 128, (int64_t)blockIdx.x * 128, axT, xt, x4);
}

template <int WHAT>
static void launch_pack(rsg_ctx *c, rsg_msa *m, PackAux X)
{
  const int64_t gx = (m->Lpad + 127) / 128, extra = std::max<int64_t>(X.lgc ? m->N + 1 : 0, X.ntiles);
  X.gy = (int)(m->Npad / 128);
  hipLaunchKernelGGL((k_pack<WHAT>), dim3((unsigned)gx, (unsigned)(X.gy + (extra + 256 * gx - 1) / (256 * gx))), dim3(256), 0,
                     c->stream, m->d_ax, m->N, m->L, m->Npad, m->Lpad, m->d_axT, m->d_xt, m->d_x4, X);
}

int rsg_need(rsg_ctx *c, rsg_msa *m, int what, char *errbuf, int2 *tiles, int nb, int ntiles)
{
  PackAux X{0, m->N, nullptr, tiles, nb, ntiles};
  const bool lgc = (what & PACK_LGC) && m->lgc_n != m->N && m->N <= 65535;   // (few grid rows)
  what &= ~(m->packed | PACK_LGC);
  if (!what) return RSG_OK;              // (a table still missing is made with the probabilities)
  if (lgc) {
    if (!m->d_lgc) HIPCHK(rsg_msa_get(m, &m->d_lgc, sizeof(double) * 3 * (size_t)(m->N + 1)));
    X.lgc = m->d_lgc;
  }
  const size_t tp = (size_t)m->Lpad * (size_t)m->Npad;
  if ((what & PACK_AXT) && !m->d_axT) HIPCHK(rsg_msa_get(m, &m->d_axT, tp));
  if ((what & PACK_XT) && !m->d_xt) HIPCHK(rsg_msa_get(m, &m->d_xt, tp));
  if ((what & PACK_X4) && !m->d_x4) HIPCHK(rsg_msa_get(m, &m->d_x4, tp / 2));
  int t; rsg_tstart(c, "pack", &t);
  switch (what) {
  case PACK_AXT: launch_pack<PACK_AXT>(c, m, X); break;
  case PACK_XT:  launch_pack<PACK_XT>(c, m, X); break;
  case PACK_X4:  launch_pack<PACK_X4>(c, m, X); break;
  case PACK_AXT | PACK_XT: launch_pack<PACK_AXT | PACK_XT>(c, m, X); break;
  case PACK_AXT | PACK_X4: launch_pack<PACK_AXT | PACK_X4>(c, m, X); break;
  default: launch_pack<PACK_AXT | PACK_XT | PACK_X4>(c, m, X); what = PACK_AXT | PACK_XT | PACK_X4;
  }
  rsg_tstop(c, t);
  HIPCHK(hipGetLastError());
  m->packed |= what;
  if (lgc) m->lgc_n = m->N;
  return RSG_OK;
}

// ------------------------------------------------------------------------------------
// Staging of codes for one K-tile in LDS: the j side [chunk (SPC seqs)][BJ columns][16 B]
// (CSA bytes per chunk row), then the i side [chunk][BI columns][16 B]; no padding (a
// ds_read_b128 pass of 16 lanes reads 16 consecutive columns: conflict-free).  SPC sequences per
// chunk: 32 (x4) or 16 (xt).
template <int BI, int BJ, int KT, int NT, int SPC>
struct CodeStage {
  static constexpr int NKC = KT / SPC;
  static constexpr int CSA = BJ * 16, CSB = BI * 16;
  static constexpr int BYTES = NKC * (CSA + CSB);
  static constexpr int NCH = (BI + BJ) * NKC;
  static constexpr int NR = (NCH + NT - 1) / NT;
  static constexpr int NINST = NCH / 64;                    // 64-chunk LDS-direct loads per stage
  // LDS of the FP4 Gram: three stage images; with fused marginals at least the epilogue's
  // exchange (8 uint4 per lane and wave, NT * 128 bytes) and row sums (4 doubles per lane of
  // half the waves, NT * 16 bytes)
  static constexpr int lds_bytes(bool pm) { return (pm && NT * 144 > 3 * BYTES) ? NT * 144 : 3 * BYTES; }
};

// VGPR staging (the BF16 Gram): every thread moves exactly NR chunks (NCH is a multiple of
// the thread count for all shapes); consecutive threads take consecutive columns of a chunk
// row, so loads and LDS stores are contiguous.
#define STAGE_GLOAD(St, pre, xt, Lpad, i0, j0, k0, tid)                                        \
  static_assert(St::NCH % NT == 0, "stage chunks must divide evenly among threads");         \
  _Pragma("unroll") for (int r_ = 0; r_ < St::NR; r_++) {                                      \
    const int ch_ = (tid) + r_ * NT;                                                           \
    const int kc_ = ch_ / (BI + BJ), cc_ = ch_ % (BI + BJ);                                    \
    const int64_t col_ = (cc_ < BJ) ? ((j0) + cc_) : ((i0) + cc_ - BJ);                        \
    pre[r_] = *(const uint4 *)((xt) + (((k0) / 16 + kc_) * (Lpad) + col_) * 16);               \
  }
#define STAGE_SSTORE(St, pre, base, tid)                                                        \
  _Pragma("unroll") for (int r_ = 0; r_ < St::NR; r_++) {                                      \
    const int ch_ = (tid) + r_ * NT;                                                           \
    const int kc_ = ch_ / (BI + BJ), cc_ = ch_ % (BI + BJ);                                    \
    uint8_t *p_ = (cc_ < BJ) ? ((base) + kc_ * St::CSA + cc_ * 16)                             \
                             : ((base) + St::NKC * St::CSA + kc_ * St::CSB + (cc_ - BJ) * 16); \
    *(uint4 *)p_ = pre[r_];                                                                    \
  }

// LDS-direct staging (the FP4 and int8-limb Grams): global_load_lds_dwordx4 moves 16 bytes per lane from
// the lane's own global address to LDS at M0 + 16 * lane, without VGPRs.  The compiler does
// not model the LDS write of the instruction, so it is issued through inline asm and every
// wait for it is an explicit vmcnt wait.
__device__ __forceinline__ void lds_direct16(const uint8_t *g, uint8_t *l)
{
  const uint32_t la = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)l);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(la), "v"(g) : "memory", "m0");
}

// One stage (K-tile `kt`) into LDS image `base`: the stage's NCH chunks are the j-side chunk
// rows then the i-side chunk rows, 64 consecutive chunks per wave instruction (a j-side
// image of NKC * BJ chunks is a multiple of 64, so no instruction straddles the sides).
// Every wave issues exactly NINST / NW instructions.
template <class St, int BI, int BJ, int NW>
__device__ __forceinline__ void stage_lds_direct(const uint8_t *__restrict__ xt, int64_t Lpad, int64_t i0, int64_t j0,
                                                 int64_t kt, uint8_t *base, int wave, int lane)
{
  static_assert(St::NINST % NW == 0 && (St::NKC * BJ) % 64 == 0, "LDS-direct stage shape");
#pragma unroll
  for (int q = 0; q < St::NINST / NW; q++) {
    const int c0 = (wave + NW * q) * 64, c = c0 + lane;
    const bool aside = c < St::NKC * BJ;
    const int cs = aside ? c : c - St::NKC * BJ, w = aside ? BJ : BI;
    const int kc = cs / w, cc = cs % w;
    const int64_t colg = (aside ? j0 : i0) + cc;
    lds_direct16(xt + ((kt * St::NKC + kc) * Lpad + colg) * 16, base + c0 * 16);
  }
}

// D += A B for 64 sequences: FP4 (E2M1) operands in the first four of the instruction's eight
// operand dwords, FP32 accumulators, scales 1.
__device__ __forceinline__ v16f mfma_fp4(v4i a, v4i b, v16f c)
{
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4((v8i){a[0], a[1], a[2], a[3], 0, 0, 0, 0},
                                                         (v8i){b[0], b[1], b[2], b[3], 0, 0, 0, 0}, c, 4, 4, 0, 0, 0, 0);
}
__device__ __forceinline__ v4i and4(uint4 v, unsigned mk, int sh)
{
  return (v4i){(int)((v.x >> sh) & mk), (int)((v.y >> sh) & mk), (int)((v.z >> sh) & mk), (int)((v.w >> sh) & mk)};
}
// Sequences an accumulator that starts at 0 takes (uint32 records): FP32 sums are exact to 2^24 units, a
// unit per sequence at most.  More (the branches of a tree of millions of leaves) go in K segments of this
// many, whose counts k_gram_fix adds as integers.
#define FP4_EXACT (1 << 22)
// FP4 value of symbol s's operand
__host__ __device__ constexpr float fp4_unit(int s) { return s == 0 ? 0.5f : s == 1 ? 1.f : 2.f; }

// Counts in the low 16 bits of two accumulators (started at 2^23 units) as one word.
__device__ __forceinline__ unsigned pack_cells(float a, float b)
{
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x05040100u);
}

// c + the two 16-bit halves of w
__device__ __forceinline__ int sum16(unsigned w, unsigned c)
{
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  const unsigned one = 0x00010001u;
  return (int)__builtin_amdgcn_udot2(*(const u16x2 *)&w, *(const u16x2 *)&one, c, false);
}

// FP4 Gram: 2 x WI x WJ waves; wave w owns the 32 i-columns x 32 j-columns block w % (WI WJ)
// and the symbol rows x of its half (w / (WI WJ)): x in {0, 1} or {2, 3}, 8 accumulators of
// 16 floats per lane.  Two waves share every SIMD (at most 256 registers each), so one wave's
// LDS and barrier waits are covered by the other's MFMAs.  KT sequences per stage.  The
// epilogue writes uint16 (OK = CNT_U16) or uint32 (CNT_U32) records; each half writes the cells
// of its own symbol rows.
// One work-group tile (i0, j0) of one alignment over K-tiles [kt0, kt1); `lds` holds
// St::lds_bytes(pm_i != nullptr).  Without PART the records go to `out`; with it the tile's partial
// counts go, unconditionally and in the record format, to partial record jj * BI + ii (ii, jj:
// column offsets in the tile) for a later reduction.
// With pm_i != nullptr (uint16 records over the whole K range only) the epilogue also leaves the
// marginal partials of the tile's 32 x 32 blocks (pm_i / pm_j, layout and order in rsg_device.h).
template <int WI, int WJ, int KT, int OK, bool PART = false>
__device__ __forceinline__ void gram_tile_fp4(const uint8_t *__restrict__ x4, int64_t Lpad, int64_t L,
                                              void *__restrict__ out, int64_t i0, int64_t j0, uint8_t *lds,
                                              int64_t kt0, int64_t kt1, void *__restrict__ part,
                                              double *__restrict__ pm_i = nullptr, double *__restrict__ pm_j = nullptr,
                                              int64_t nb32 = 0, int64_t tailc = -1)
{
#pragma clang fp contract(off)
  constexpr int BI = 32 * WI, BJ = 32 * WJ, NT = 128 * WI * WJ, KS = KT / 64;
  typedef CodeStage<BI, BJ, KT, NT, 32> St;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int blk = wave % (WI * WJ), half = __builtin_amdgcn_readfirstlane(wave / (WI * WJ)), x0 = 2 * half;
  const int wi = blk % WI, wj = blk / WI;
  const int col = lane & 31, khalf = lane >> 5;
  const int offA = (wj * 32 + col) * 16 + khalf * St::CSA;
  const int offB = St::NKC * St::CSA + (wi * 32 + col) * 16 + khalf * St::CSB;
  // i-side operands: symbols 0, 1 (masks 1, 2) or 2, 3 (mask 4, then shift 1 and mask 4)
  const unsigned mb0 = half ? 0x44444444u : 0x11111111u, mb1 = half ? 0x44444444u : 0x22222222u;
  const float ux[2] = {half ? 2.f : 0.5f, half ? 2.f : 1.f};

  v16f acc[2][4];                                  // [x - x0][y]
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const float z = (OK == CNT_U16) ? 8388608.f * ux[x] * fp4_unit(y) : 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[x][y][r] = z;
    }
  auto kstep = [&](const uint4 ra, const uint4 rb) {
    const v4i a[4] = {and4(ra, 0x11111111u, 0), and4(ra, 0x22222222u, 0), and4(ra, 0x44444444u, 0), and4(ra, 0x44444444u, 1)};
    const v4i b[2] = {and4(rb, mb0, 0), and4(rb, mb1, half)};
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 4; y++) acc[x][y] = mfma_fp4(a[y], b[x], acc[x][y]);
  };
  // tailc >= 0: the sequences past the last whole K-tile fill one 64-sequence k-step (chunks
  // tailc, tailc + 1; zero codes past N), loaded here straight into the lane's fragments and
  // multiplied after the loop, so the loop runs whole K-tiles only
  uint4 ta = make_uint4(0, 0, 0, 0), tb = make_uint4(0, 0, 0, 0);
  if (tailc >= 0) {
    ta = *(const uint4 *)(x4 + ((tailc + khalf) * Lpad + j0 + wj * 32 + col) * 16);
    tb = *(const uint4 *)(x4 + ((tailc + khalf) * Lpad + i0 + wi * 32 + col) * 16);
  }

  // three LDS images, loads two stages ahead: stage kt0 + it is read from image it % 3 while
  // stage kt0 + it + 2 lands in image (it + 2) % 3, which was last read in iteration it - 1
  // (ended by a barrier).  Stages past kt1 - 1 reload kt1 - 1 into an image nobody reads.
  constexpr int NW = 2 * WI * WJ, QW = St::NINST / NW; // LDS-direct loads per wave per stage
  static_assert(QW >= 1 && QW <= 15, "vmcnt range");
  const int nit = (int)(kt1 - kt0);
  auto stage_of = [&](int it) -> int64_t { return kt0 + ((it < nit) ? it : nit - 1); };
  stage_lds_direct<St, BI, BJ, NW>(x4, Lpad, i0, j0, stage_of(0), lds, wave, lane);
  stage_lds_direct<St, BI, BJ, NW>(x4, Lpad, i0, j0, stage_of(1), lds + St::BYTES, wave, lane);
  __builtin_amdgcn_s_waitcnt(0x0F70 | QW);     // vmcnt(QW): this wave's loads of stage 0 landed
  __syncthreads();                             // ... and every wave's
  // The wait for stage it + 1 and the barrier sit before the last k-step of stage it: every read
  // of image it % 3 has completed there (the barrier waits for LDS reads), so the loads issued at
  // the next iteration's start may overwrite it, and the first fragments of stage it + 1 are read
  // right after the barrier while the last MFMAs of stage it run.
  static_assert(KS >= 2, "the barrier precedes the last k-step");
  uint4 ra = *(const uint4 *)(lds + offA);
  uint4 rb = *(const uint4 *)(lds + offB);
  for (int it = 0; it < nit; it++) {
    stage_lds_direct<St, BI, BJ, NW>(x4, Lpad, i0, j0, stage_of(it + 2), lds + ((it + 2) % 3) * St::BYTES, wave, lane);
    const uint8_t *base = lds + (it % 3) * St::BYTES;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      uint4 na = ra, nb = rb;
      if (ks + 1 < KS) {
        na = *(const uint4 *)(base + offA + (ks + 1) * 2 * St::CSA);
        nb = *(const uint4 *)(base + offB + (ks + 1) * 2 * St::CSB);
      } else {
        __builtin_amdgcn_s_waitcnt(0x0F70 | QW); // vmcnt(QW): stage it + 1 landed
        __syncthreads();
        const uint8_t *nbase = lds + ((it + 1) % 3) * St::BYTES;
        na = *(const uint4 *)(nbase + offA);
        nb = *(const uint4 *)(nbase + offB);
      }
      kstep(ra, rb);
      ra = na; rb = nb;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);          // no LDS-direct load outlives the loop
  if (tailc >= 0) kstep(ta, tb);

  // epilogue: lane owns i column `col`; register r holds j = 8*(r/4) + 4*khalf + r%4.  A tile with
  // every pair i < j < L (all but those on the diagonal and at the right edge) stores without
  // conditions.
  const int ii = wi * 32 + col, jj0 = wj * 32 + 4 * khalf;
  const int64_t i = i0 + ii;
  constexpr int NQ = (OK == CNT_U16) ? 2 : 4;               // uint4 per record
  uint4 *dst = PART ? (uint4 *)part + ((int64_t)jj0 * BI + ii) * NQ : (uint4 *)out + rsg_rec(i, j0 + jj0, L) * NQ;
  const int64_t js = (PART ? BI : L) * NQ;                   // one j column further
  const bool full = PART || (i0 + BI <= j0 && j0 + BJ <= L);
  if constexpr (OK != CNT_U16) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int jo = 8 * (r >> 2) + (r & 3);
      if (!full && !(i < j0 + jj0 + jo && j0 + jj0 + jo < L)) continue;
#pragma unroll
      for (int x = 0; x < 2; x++) {
        const float q = 1.f / ux[x];              // a power of two, as every unit
        dst[jo * js + x0 + x] = make_uint4((unsigned)(acc[x][0][r] * (q * 2.f)), (unsigned)(acc[x][1][r] * q),
                                           (unsigned)(acc[x][2][r] * (q * 0.5f)), (unsigned)(acc[x][3][r] * (q * 0.5f)));
      }
    }
    return;
  }
  // cells 8 half .. 8 half + 7, the 16 bytes of this half, word by word (vectors: rows are selected by
  // half below, which would put an array in scratch)
  v16u pk[4];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    pk[0][r] = pack_cells(acc[0][0][r], acc[0][1][r]); pk[1][r] = pack_cells(acc[0][2][r], acc[0][3][r]);
    pk[2][r] = pack_cells(acc[1][0][r], acc[1][1][r]); pk[3][r] = pack_cells(acc[1][2][r], acc[1][3][r]);
  }
#define PK(r) make_uint4(pk[0][r], pk[1][r], pk[2][r], pk[3][r])
  if (full) {
#pragma unroll
    for (int r = 0; r < 16; r++) dst[(8 * (r >> 2) + (r & 3)) * js + half] = PK(r);
  } else {
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int64_t j = j0 + jj0 + 8 * (r >> 2) + (r & 3);
      if (i < j && j < L) dst[(8 * (r >> 2) + (r & 3)) * js + half] = PK(r);
    }
  }
  if (PART || pm_i == nullptr) return;

  // marginal partials.  The two halves of a block split its 16 r rows: half h takes
  // r = 8 h .. 8 h + 7 and receives the sibling's cells of those rows (8 x uint16 per pair, 64 KiB
  // for 8 waves) through the LDS images, which every wave has finished with.  No FMA contraction
  // anywhere in this function, so every producer rounds alike.  Sums of cells are exact in 16 bits
  // (none exceeds the sequence count): rows by two-term dot products of the packed words,
  // columns by adding the words.  Instructions bound this part (with unpacked cells and shuffles
  // through LDS 2200 per wave and tile, as long as a third of the K loop at N = 5000).
  __syncthreads();
  uint4 *xch = (uint4 *)lds;
  if (half) {
#pragma unroll
    for (int rl = 0; rl < 8; rl++) xch[(wave * 8 + rl) * 64 + lane] = PK(rl);
  } else {
#pragma unroll
    for (int rl = 0; rl < 8; rl++) xch[(wave * 8 + rl) * 64 + lane] = PK(8 + rl);
  }
  __syncthreads();
  const int sib = blk + (1 - half) * (WI * WJ);
  const int bi32 = (int)(i0 / 32) + wi, bj32 = (int)(j0 / 32) + wj, Li = (int)L, ic = bi32 * 32 + col;
  const bool blkok = bi32 <= bj32 && bj32 < (int)nb32;      // blocks of the pm32 layout only
  double ao[2] = {0., 0.}, as[2] = {0., 0.}, cv[32];        // row terms of own and of the sibling's symbols
#pragma unroll
  for (int rl = 0; rl < 8; rl++) {
    const int r = 8 * half + rl, j = bj32 * 32 + 8 * (r >> 2) + 4 * khalf + (r & 3);
    const uint4 sv = xch[(sib * 8 + rl) * 64 + lane];
    const uint4 ov = make_uint4(half ? pk[0][8 + rl] : pk[0][rl], half ? pk[1][8 + rl] : pk[1][rl],
                                half ? pk[2][8 + rl] : pk[2][rl], half ? pk[3][8 + rl] : pk[3][rl]);
    const int ro[2] = {sum16(ov.x, sum16(ov.y, 0u)), sum16(ov.z, sum16(ov.w, 0u))};
    const int rsb[2] = {sum16(sv.x, sum16(sv.y, 0u)), sum16(sv.z, sum16(sv.w, 0u))};
    const unsigned c01 = (ov.x + ov.z) + (sv.x + sv.z), c23 = (ov.y + ov.w) + (sv.y + sv.w);
    const double inv = pm_inv(full || (blkok && ic < j && j < Li), (ro[0] + ro[1]) + (rsb[0] + rsb[1]));
#pragma unroll
    for (int x = 0; x < 2; x++) { ao[x] += pm_term(ro[x], inv); as[x] += pm_term(rsb[x], inv); }
    cv[4 * rl] = pm_term((int)(c01 & 0xFFFFu), inv); cv[4 * rl + 1] = pm_term((int)(c01 >> 16), inv);
    cv[4 * rl + 2] = pm_term((int)(c23 & 0xFFFFu), inv); cv[4 * rl + 3] = pm_term((int)(c23 >> 16), inv);
  }
  const double ai[4] = {half ? as[0] : ao[0], half ? as[1] : ao[1], half ? ao[0] : as[0], half ? ao[1] : as[1]};
  const double sj = pm_rscatter32(cv, col);                  // index col: r = 8 half + col / 4, y = col % 4
  const int64_t bq = blkok ? pm_tri(bi32, bj32, nb32) : 0;
  const int rj = 8 * half + (col >> 2), jbo = 8 * (rj >> 2) + 4 * khalf + (rj & 3);
  if (blkok) pm_j[(bq * 32 + jbo) * 4 + (col & 3)] = sj;
  // i side: half 1 hands its sums over r = 8..15 to half 0, which adds them to its own (r = 0..7)
  double *aix = (double *)(lds + NT * 128);
  if (half == 1)
#pragma unroll
    for (int x = 0; x < 4; x++) aix[(blk * 4 + x) * 64 + lane] = ai[x];
  __syncthreads();
  if (half == 0)
#pragma unroll
    for (int x = 0; x < 4; x++) {
      const double si = pm_khalf_sum(ai[x] + aix[(blk * 4 + x) * 64 + lane]);
      if (blkok && khalf == 0) pm_i[(bq * 32 + col) * 4 + x] = si;
    }
#undef PK
}

// K segments of the split tiles: nsu units over the nrem = ntiles - ndp last tiles, tile t
// taking sbase + 1 segments if t < sextra, else sbase (so nsu = nrem * sbase + sextra can match
// the CU count); tile t's units are split_first(t) .. split_first(t) + segments - 1.
__host__ __device__ __forceinline__ int split_first(int t, int sbase, int sextra)
{
  return t * sbase + (t < sextra ? t : sextra);
}
__device__ __forceinline__ void split_unit(int u, int sbase, int sextra, int &t, int &sg, int &ns)
{
  const int big = sextra * (sbase + 1);
  if (u < big) { t = u / (sbase + 1); sg = u % (sbase + 1); ns = sbase + 1; }
  else { t = sextra + (u - big) / sbase; sg = (u - big) % sbase; ns = sbase; }
}

// Grid: first 8 * per_xcd work groups for the first ndp tiles (whole K range), then the nsu
// split units, each over one K segment of one of the last tiles, writing partial records for
// k_gram_fix.  The split keeps the last, partial wave of tiles from leaving most CUs idle; the
// units go to the work-group slots as the full tiles free them, so the spread of the full
// tiles' end times is filled rather than added to the kernel's length.
template <int WI, int WJ, int KT, int OK>
__global__ void __launch_bounds__(128 * WI * WJ) __attribute__((amdgpu_waves_per_eu(2)))
k_gram_fp4(const uint8_t *__restrict__ x4, int64_t nkt, int64_t tailc, int64_t Lpad, int64_t L, void *__restrict__ out,
          const int2 *__restrict__ tiles, int ndp, int per_xcd, int ntiles, int sbase, int sextra,
          uint8_t *__restrict__ part, double *__restrict__ pm_part, int *__restrict__ pmflag)
{
  typedef CodeStage<32 * WI, 32 * WJ, KT, 128 * WI * WJ, 32> St;
  __shared__ __attribute__((aligned(16))) uint8_t lds[St::lds_bytes(OK == CNT_U16)];
  const int nsu = (ntiles - ndp) * sbase + sextra;
  int t;
  int64_t k0 = 0, k1 = nkt;
  uint8_t *p = nullptr;
  if ((int)blockIdx.x < 8 * per_xcd) {
    // XCD-aware mapping (work group g runs on XCD g & 7): consecutive tiles of the
    // (bi, bj)-sorted list run on one XCD (one L2)
    const int g = blockIdx.x;
    t = (g & 7) * per_xcd + (g >> 3);
    if (t >= ndp) return;
  } else {
    const int u = blockIdx.x - 8 * per_xcd;
    if (u >= nsu) return;
    int tr, sg, ns;
    split_unit(u, sbase, sextra, tr, sg, ns);
    t = ndp + tr;
    k0 = nkt * sg / ns; k1 = nkt * (sg + 1) / ns;
    p = part + (int64_t)u * (32 * WI) * (32 * WJ) * (OK == CNT_U16 ? 32 : 64);
  }
  if (pmflag && blockIdx.x == 0 && threadIdx.x == 0) *pmflag = 0;    // set by the marginal reduction
  const int2 tl = tiles[t];
  const int64_t nb32 = (L + 31) / 32, i0 = (int64_t)tl.x * 32 * WI, j0 = (int64_t)tl.y * 32 * WJ, tc = k1 == nkt ? tailc : -1;
  if (p) gram_tile_fp4<WI, WJ, KT, OK, true>(x4, Lpad, L, out, i0, j0, lds, k0, k1, p, nullptr, nullptr, nb32, tc);
  else   gram_tile_fp4<WI, WJ, KT, OK>(x4, Lpad, L, out, i0, j0, lds, k0, k1, nullptr, pm_part,        // split: in k_gram_fix
                                       pm_part ? pm_part + pm32_n(nb32) : nullptr, nb32, tc);
}

// The marginal terms of one row r of a 32 x 32 block, every cell of the lane's uint16 record in s, to
// LDS (row terms [16][4][64], then column terms), and the block's partials from them with the
// arithmetic and order of the Gram epilogue: wave 0 adds the row terms over r = 0..7 and
// r = 8..15 and then the two sums, waves 2 and 3 reduce-scatter the column terms of r = 0..7 and
// r = 8..15 (index 4 (r % 8) + y).
typedef double PmTerms[2][16][4][64];
__device__ __forceinline__ void block_terms(const uint4 s0, const uint4 s1, bool on, int r, int lane, PmTerms &T)
{
#pragma clang fp contract(off)
  const int rs[4] = {sum16(s0.x, sum16(s0.y, 0u)), sum16(s0.z, sum16(s0.w, 0u)), sum16(s1.x, sum16(s1.y, 0u)),
                     sum16(s1.z, sum16(s1.w, 0u))};
  const unsigned c01 = (s0.x + s0.z) + (s1.x + s1.z), c23 = (s0.y + s0.w) + (s1.y + s1.w);   // no half exceeds 65535
  const int cs[4] = {(int)(c01 & 0xFFFFu), (int)(c01 >> 16), (int)(c23 & 0xFFFFu), (int)(c23 >> 16)};
  const double inv = pm_inv(on, (rs[0] + rs[1]) + (rs[2] + rs[3]));
#pragma unroll
  for (int x = 0; x < 4; x++) { T[0][r][x][lane] = pm_term(rs[x], inv); T[1][r][x][lane] = pm_term(cs[x], inv); }
}
// The same terms of FP32 cells (weighted records): t = the row terms, then the column terms.
__device__ __forceinline__ void block_terms_w(const float4 (&c)[4], bool on, double (&t)[8])
{
#pragma clang fp contract(off)
  double rs[4], cs[4];
#pragma unroll
  for (int x = 0; x < 4; x++) rs[x] = (((double)c[x].x + (double)c[x].y) + (double)c[x].z) + (double)c[x].w;
  cs[0] = (((double)c[0].x + (double)c[1].x) + (double)c[2].x) + (double)c[3].x;
  cs[1] = (((double)c[0].y + (double)c[1].y) + (double)c[2].y) + (double)c[3].y;
  cs[2] = (((double)c[0].z + (double)c[1].z) + (double)c[2].z) + (double)c[3].z;
  cs[3] = (((double)c[0].w + (double)c[1].w) + (double)c[2].w) + (double)c[3].w;
  const double ns = (rs[0] + rs[1]) + (rs[2] + rs[3]), inv = (on && ns > 0.) ? 1. / (ns + 16e-10) : 0.;
#pragma unroll
  for (int x = 0; x < 4; x++) { t[x] = (rs[x] + 4e-10) * inv; t[4 + x] = (cs[x] + 4e-10) * inv; }
}
__device__ __forceinline__ void block_partials(const PmTerms &T, int bi32, int bj32, int nb32, int wave, int lane,
                                               double *__restrict__ pm_part)
{
  if (!(bi32 <= bj32 && bj32 < nb32) || wave == 1 || wave > 3) return;
  const int col = lane & 31, khalf = lane >> 5;
  double *pm_i = pm_part, *pm_j = pm_part + pm32_n(nb32);
  const int64_t bq = pm_tri(bi32, bj32, nb32);
  if (wave == 0) {
#pragma unroll
    for (int x = 0; x < 4; x++) {
      double a0 = 0., a1 = 0.;
#pragma unroll
      for (int rl = 0; rl < 8; rl++) { a0 += T[0][rl][x][lane]; a1 += T[0][8 + rl][x][lane]; }
      const double si = pm_khalf_sum(a0 + a1);
      if (khalf == 0) pm_i[(bq * 32 + col) * 4 + x] = si;
    }
  } else {
    const int h = wave - 2;
    double cv[32];
#pragma unroll
    for (int rl = 0; rl < 8; rl++)
#pragma unroll
      for (int y = 0; y < 4; y++) cv[4 * rl + y] = T[1][8 * h + rl][y][lane];
    const double sj = pm_rscatter32(cv, col);
    const int rj = 8 * h + (col >> 2), jbo = 8 * (rj >> 2) + 4 * khalf + (rj & 3);
    pm_j[(bq * 32 + jbo) * 4 + (col & 3)] = sj;
  }
}

// Split tiles: one work group (16 waves) per 32 x 32 block sums the block's partial records over
// the tile's K segments (integer sums: exact; uint16 records add as words, no half exceeding
// 65535) and writes the records; wave w takes row r = w of the MFMA result layout, all its
// segments' loads in flight together.  For uint16 records with pm_part the block's marginal
// partials follow.
#define FIX_WAVES 16
template <int BI, int BJ, int OK>
__global__ void __launch_bounds__(64 * FIX_WAVES)
k_gram_fix(const uint8_t *__restrict__ part, const int2 *__restrict__ tiles, int ndp, int sbase, int sextra, int64_t L,
           void *__restrict__ out, double *__restrict__ pm_part)
{
  constexpr int NQ = (OK == CNT_U16) ? 2 : 4;                       // uint4 per record
  constexpr int NBI = BI / 32, NB = NBI * (BJ / 32);
  __shared__ PmTerms T;
  const int tr = blockIdx.x / NB, sb = blockIdx.x % NB, wi = sb % NBI, wj = sb / NBI;
  const int r = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 31, khalf = lane >> 5;
  const int2 tl = tiles[ndp + tr];
  const int bi32 = tl.x * NBI + wi, bj32 = tl.y * (BJ / 32) + wj, Li = (int)L, ic = bi32 * 32 + col;
  const int ns = sbase + (tr < sextra ? 1 : 0);
  const uint4 *p0 = (const uint4 *)part + (int64_t)split_first(tr, sbase, sextra) * BI * BJ * NQ;
  uint4 s[NQ];
#pragma unroll
  for (int h = 0; h < NQ; h++) s[h] = make_uint4(0, 0, 0, 0);
  const int jb = 8 * (r >> 2) + 4 * khalf + (r & 3);
  const int64_t pr = (int64_t)(wj * 32 + jb) * BI + wi * 32 + col;   // partial record in the tile
#pragma unroll 4
  for (int k = 0; k < ns; k++)
#pragma unroll
    for (int h = 0; h < NQ; h++) {
      const uint4 v = p0[((int64_t)k * BI * BJ + pr) * NQ + h];
      s[h].x += v.x; s[h].y += v.y; s[h].z += v.z; s[h].w += v.w;
    }
  const int nb32 = (Li + 31) / 32, j = bj32 * 32 + jb;
  const bool valid = ic < j && j < Li;
  if (valid)
#pragma unroll
    for (int h = 0; h < NQ; h++) ((uint4 *)out)[rsg_rec(ic, j, L) * NQ + h] = s[h];
  if (OK != CNT_U16 || pm_part == nullptr) return;
  block_terms(s[0], s[1], bi32 <= bj32 && bj32 < nb32 && valid, r, lane, T);
  __syncthreads();
  block_partials(T, bi32, bj32, nb32, r, lane, pm_part);
}

// FP4 Gram of few tiles: a 32 x 32-column tile per work group, its 64-sequence k-steps dealt to KG
// groups of two waves (as the halves of gram_tile_fp4); then the groups' counts meet in LDS as
// packed words (no half exceeds 65535), and every wave takes 8 / KG rows of the tile through records
// and marginal terms.  Where the tiles do not fill the device a tile's own chain bounds the
// kernel.  The K loop has no barriers: every lane loads its fragments itself, DEEP k-steps
// ahead (the second wave of a group finds them in the L1; staged through LDS images with a barrier
// per two k-steps the loop took 205 ns per k-step and SIMD, 160 this way).  Two waves per tile took
// 30 us at 4096 x 768, 10.2 at 1013 x 407, 6.6 at 200 x 120; this takes 20.7, 7.9 and 5.9 us.
#define DEEP 4
template <int KG>
__global__ void __launch_bounds__(128 * KG) __attribute__((amdgpu_waves_per_eu(2)))
k_gram_fp4_deep(const uint8_t *__restrict__ x4, int nk, int64_t Lpad, int64_t L, uint4 *__restrict__ out,
                const int2 *__restrict__ tiles, int ntiles, int per_xcd, double *__restrict__ pm_part, int *__restrict__ pmflag)
{
  constexpr int RPW = 8 / KG;
  constexpr int LDS = KG * 32768 > (int)sizeof(PmTerms) ? KG * 32768 : (int)sizeof(PmTerms);
  __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];
  if (pmflag && blockIdx.x == 0 && threadIdx.x == 0) *pmflag = 0;    // set by the marginal reduction
  const int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (t >= ntiles) return;
  const int2 tl = tiles[t];
  const int64_t i0 = (int64_t)tl.x * 32, j0 = (int64_t)tl.y * 32;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = wave >> 1, half = wave & 1;
  const int col = lane & 31, khalf = lane >> 5;
  const unsigned mb0 = half ? 0x44444444u : 0x11111111u, mb1 = half ? 0x44444444u : 0x22222222u;
  const float ux[2] = {half ? 2.f : 0.5f, half ? 2.f : 1.f};

  const int n = (nk - g + KG - 1) / KG, last = n > 0 ? n - 1 : 0;   // this group's k-steps g, g + KG, ..
  const uint8_t *pa = x4 + ((int64_t)(2 * (n > 0 ? g : 0) + khalf) * Lpad + j0 + col) * 16, *pb = pa + (i0 - j0) * 16;
  const int64_t ks = 2 * KG * Lpad * 16;
  uint4 fa[DEEP], fb[DEEP];
#pragma unroll
  for (int u = 0; u < DEEP; u++) {
    const int64_t o = (int64_t)min(u, last) * ks;
    fa[u] = *(const uint4 *)(pa + o); fb[u] = *(const uint4 *)(pb + o);
  }
  v16f acc[2][4];
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const float z = 8388608.f * ux[x] * fp4_unit(y);
#pragma unroll
      for (int r = 0; r < 16; r++) acc[x][y][r] = z;
    }
  auto kstep = [&](const uint4 ra, const uint4 rb) {
    const v4i a[4] = {and4(ra, 0x11111111u, 0), and4(ra, 0x22222222u, 0), and4(ra, 0x44444444u, 0), and4(ra, 0x44444444u, 1)};
    const v4i b[2] = {and4(rb, mb0, 0), and4(rb, mb1, half)};
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 4; y++) acc[x][y] = mfma_fp4(a[y], b[x], acc[x][y]);
  };
  int st = 0;
  for (; st + DEEP <= n; st += DEEP)
#pragma unroll
    for (int u = 0; u < DEEP; u++) {
      const uint4 ra = fa[u], rb = fb[u];
      const int64_t o = (int64_t)min(st + u + DEEP, last) * ks;
      fa[u] = *(const uint4 *)(pa + o); fb[u] = *(const uint4 *)(pb + o);
      kstep(ra, rb);
    }
#pragma unroll
  for (int u = 0; u < DEEP - 1; u++)
    if (st + u < n) kstep(fa[u], fb[u]);

  // every wave's words: [g][half][r][lane]
  uint4 *xw = (uint4 *)lds;
#pragma unroll
  for (int r = 0; r < 16; r++)
    xw[(wave * 16 + r) * 64 + lane] = make_uint4(pack_cells(acc[0][0][r], acc[0][1][r]), pack_cells(acc[0][2][r], acc[0][3][r]),
                                                 pack_cells(acc[1][0][r], acc[1][1][r]), pack_cells(acc[1][2][r], acc[1][3][r]));
  __syncthreads();
  const int bi32 = tl.x, bj32 = tl.y, nb32 = (int)((L + 31) / 32), ic = bi32 * 32 + col, Li = (int)L;
  uint4 s[RPW][2];
#pragma unroll
  for (int q = 0; q < RPW; q++) {
    const int r = RPW * wave + q, j = bj32 * 32 + 8 * (r >> 2) + 4 * khalf + (r & 3);
#pragma unroll
    for (int h = 0; h < 2; h++) {
      uint4 v = xw[(h * 16 + r) * 64 + lane];
#pragma unroll
      for (int k = 1; k < KG; k++) {
        const uint4 u = xw[((2 * k + h) * 16 + r) * 64 + lane];
        v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
      }
      s[q][h] = v;
    }
    if (ic < j && j < Li) {
      uint4 *o = out + rsg_rec(ic, j, L) * 2;
      o[0] = s[q][0]; o[1] = s[q][1];
    }
  }
  if (pm_part == nullptr) return;
  __syncthreads();                                         // every wave has its rows
  PmTerms &T = *(PmTerms *)lds;
#pragma unroll
  for (int q = 0; q < RPW; q++) {
    const int r = RPW * wave + q, j = bj32 * 32 + 8 * (r >> 2) + 4 * khalf + (r & 3);
    block_terms(s[q][0], s[q][1], bi32 <= bj32 && bj32 < nb32 && ic < j && j < Li, r, lane, T);
  }
  __syncthreads();
  block_partials(T, bi32, bj32, nb32, wave, lane, pm_part);
}

// Batched FP4 Gram over many alignments: one work group per (item, tile); tiles are
// pre-sorted by decreasing sequence count (cost).  Large alignments: 64 x 32 columns, two
// waves per half, 512-sequence K tiles; small ones: 32 x 32 columns, one wave per half,
// 128-sequence K tiles.
template <int WI, int WJ, int KT>
__global__ void __launch_bounds__(128 * WI * WJ) __attribute__((amdgpu_waves_per_eu(2)))
k_gram_fp4_batch(const int4 *__restrict__ tiles, const int64_t *__restrict__ desc, const uint8_t *__restrict__ x4,
                 uint16_t *__restrict__ cnt, double *__restrict__ pm_part, int pm_field)
{
  typedef CodeStage<32 * WI, 32 * WJ, KT, 128 * WI * WJ, 32> St;
  __shared__ __attribute__((aligned(16))) uint8_t lds[St::lds_bytes(true)];
  const int4 tl = tiles[blockIdx.x];                    // (item, bi, bj, -)
  const int64_t *d = desc + (int64_t)tl.x * RSG_BDESC;  // item descriptor (see rsg_batch.hip)
  const int64_t nb32 = (d[1] + 31) / 32;
  double *pmi = pm_part + d[pm_field];
  gram_tile_fp4<WI, WJ, KT, CNT_U16>(x4 + d[4], d[3], d[1], cnt + d[5], (int64_t)tl.y * 32 * WI, (int64_t)tl.z * 32 * WJ,
                                     lds, 0, (d[0] + KT - 1) / KT, nullptr, pmi, pmi + pm32_n(nb32), nb32);
}

// The same tiles in a persistent grid (as many work groups as fit the device at once) fed by
// per-XCD queues: work groups are dispatched to the 8 XCDs round-robin, so group g serves queue
// x = g % 8, which holds the tiles t = x, x + 8, x + 16, ... of the list (each XCD gets the same
// mix of long and short tiles); a pop takes the next index of its queue from an atomic counter.
// The list is sorted by decreasing K length, so this is longest-first greedy scheduling of
// uneven items; eight counters instead of one keep the pops from serialising on one address.
// The counters are cleared by a fill kernel ahead of the launch (graph-safe).
template <int WI, int WJ, int KT>
__global__ void __launch_bounds__(128 * WI * WJ) __attribute__((amdgpu_waves_per_eu(2)))
k_gram_fp4_queue(const int4 *__restrict__ tiles, int ntiles, int *__restrict__ queue, const int64_t *__restrict__ desc,
                const uint8_t *__restrict__ x4, uint16_t *__restrict__ cnt, double *__restrict__ pm_part, int pm_field)
{
  typedef CodeStage<32 * WI, 32 * WJ, KT, 128 * WI * WJ, 32> St;
  __shared__ __attribute__((aligned(16))) uint8_t lds[St::lds_bytes(true)];
  __shared__ int next;
  const int x = blockIdx.x & 7;
  int *q = queue + 16 * x;                              // one counter per 64-byte line
  if (threadIdx.x == 0) next = 8 * atomicAdd(q, 1) + x;
  __syncthreads();
  int t = next;
  while (t < ntiles) {
    int nxt = 0;                                        // the next pop overlaps this tile's first loads
    if (threadIdx.x == 0) nxt = 8 * atomicAdd(q, 1) + x;
    const int4 tl = tiles[t];
    const int64_t *d = desc + (int64_t)tl.x * RSG_BDESC;
    const int64_t nb32 = (d[1] + 31) / 32;
    double *pmi = pm_part + d[pm_field];
    gram_tile_fp4<WI, WJ, KT, CNT_U16>(x4 + d[4], d[3], d[1], cnt + d[5], (int64_t)tl.y * 32 * WI, (int64_t)tl.z * 32 * WJ,
                                       lds, 0, (d[0] + KT - 1) / KT, nullptr, pmi, pmi + pm32_n(nb32), nb32);
    __syncthreads();                                    // every wave is done with lds and has read next
    if (threadIdx.x == 0) next = nxt;
    __syncthreads();
    t = next;
  }
}

// the 8 queue counters (16 ints apart)
__global__ void k_clear_queues(int *__restrict__ q) { if (threadIdx.x < 128) q[threadIdx.x] = 0; }

int rsg_gram_batch_launch(rsg_ctx *c, const int4 *d_big, int nbig, const int4 *d_small, int nsmall,
                          const int64_t *d_desc, const uint8_t *d_x4, uint16_t *d_cnt, double *d_pm_part, int pm_field,
                          int *d_queue)
{
  const int ncu = c->ncu > 0 ? c->ncu : 256;
  if (c->batch_persistent && d_queue) {
    // Large tiles (64 x 32 columns, tens of microseconds each) keep one work group per tile:
    // the hardware dispatcher is already a longest-first queue over the sorted list, and the
    // queue loop's extra live registers make that tile body spill (measured 30% slower).  The
    // many short 32 x 32 tiles run persistent, saving a dispatch per tile.
    if (nbig > 0)
      hipLaunchKernelGGL((k_gram_fp4_batch<2, 1, 512>), dim3((unsigned)nbig), dim3(256), 0, c->stream, d_big, d_desc, d_x4,
                         d_cnt, d_pm_part, pm_field);
    if (nsmall > 0) {                   // 2 waves per group, four groups per CU
      hipLaunchKernelGGL(k_clear_queues, dim3(1), dim3(256), 0, c->stream, d_queue);
      hipLaunchKernelGGL((k_gram_fp4_queue<1, 1, 128>), dim3((unsigned)(std::min(nsmall, 4 * ncu) + 7) & ~7u), dim3(128), 0,
                         c->stream, d_small, nsmall, d_queue, d_desc, d_x4, d_cnt, d_pm_part, pm_field);
    }
    return hipGetLastError() == hipSuccess ? RSG_OK : RSG_FAIL;
  }
  if (nbig > 0)
    hipLaunchKernelGGL((k_gram_fp4_batch<2, 1, 512>), dim3((unsigned)nbig), dim3(256), 0, c->stream, d_big, d_desc, d_x4, d_cnt,
                       d_pm_part, pm_field);
  if (nsmall > 0)
    hipLaunchKernelGGL((k_gram_fp4_batch<1, 1, 128>), dim3((unsigned)nsmall), dim3(128), 0, c->stream, d_small, d_desc, d_x4, d_cnt,
                       d_pm_part, pm_field);
  return hipGetLastError() == hipSuccess ? RSG_OK : RSG_FAIL;
}

// ------------------------------------------------------------------------------------
// Weighted Gram, split-BF16.  Staged from the byte codes plus the split weight parts of
// the K-tile's sequences (bf16 bits, [part][KT]).
//
// Operand expansion for symbol s from 4 staged bytes (one dword d): t = (d >> s) & 0x01010101
// holds 0/1 per byte; v_perm spreads bytes 0,1 (or 2,3) into the two 16-bit halves and a
// 24-bit multiply turns each 0/1 half into 0x0000/0xFFFF (mask) or 0x0000/0x3F80 (1.0).
__device__ __forceinline__ void spread(unsigned d, int s, unsigned &lo, unsigned &hi)
{
  unsigned t = (d >> s) & 0x01010101u;
  lo = __builtin_amdgcn_perm(t, t, 0x0C010C00u);
  hi = __builtin_amdgcn_perm(t, t, 0x0C030C02u);
}

template <int WI, int WJ, int KT, int NS>
__global__ void __launch_bounds__(64 * WI * WJ)
k_gram_bf16(const uint8_t *__restrict__ xt, const uint16_t *__restrict__ wsplit, int64_t nkt, int64_t Npad, int64_t Lpad, int64_t L,
            float *__restrict__ out, const int2 *__restrict__ tiles, int ntiles, int per_xcd)
{
  constexpr int BI = 32 * WI, BJ = 32 * WJ, NT = 64 * WI * WJ, KS = KT / 32;
  typedef CodeStage<BI, BJ, KT, NT, 16> St;
  constexpr int WBYTES = NS * KT * 2;
  constexpr int SB = St::BYTES + WBYTES;
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * SB];

  const int g = blockIdx.x;
  const int t = (g & 7) * per_xcd + (g >> 3);
  if (t >= ntiles) return;
  const int2 tl = tiles[t];
  const int64_t i0 = (int64_t)tl.x * BI, j0 = (int64_t)tl.y * BJ;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wi = wave % WI, wj = wave / WI;
  const int col = lane & 31, khalf = lane >> 5;
  const int offA = (wj * 32 + col) * 16 + khalf * St::CSA;
  const int offB = St::NKC * St::CSA + (wi * 32 + col) * 16 + khalf * St::CSB;

  v16f acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; x++)
#pragma unroll
    for (int y = 0; y < 4; y++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[x][y][r] = 0.f;

  uint4 pre[St::NR];
  uint4 wpre = make_uint4(0, 0, 0, 0);            // weight chunk of this thread (if any)
  constexpr int NWCH = WBYTES / 16;               // 16-byte weight chunks per stage
  auto wload = [&](int64_t k0) {
    if (tid < NWCH) {
      int p = tid / (KT / 8), kc = tid % (KT / 8);
      wpre = *(const uint4 *)(wsplit + p * Npad + k0 + kc * 8);
    }
  };
  auto wstore = [&](uint8_t *base) {
    if (tid < NWCH) *(uint4 *)(base + St::BYTES + tid * 16) = wpre;
  };
  STAGE_GLOAD(St, pre, xt, Lpad, i0, j0, 0, tid);
  wload(0);
  STAGE_SSTORE(St, pre, lds, tid);
  wstore(lds);
  __syncthreads();
  for (int64_t kt = 0; kt < nkt; kt++) {
    const int buf = (int)(kt & 1);
    const int64_t knext = ((kt + 1 < nkt) ? kt + 1 : kt) * KT;
    STAGE_GLOAD(St, pre, xt, Lpad, i0, j0, knext, tid);
    wload(knext);
    const uint8_t *base = lds + buf * SB;
    const uint16_t *wl = (const uint16_t *)(base + St::BYTES);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const uint4 ra = *(const uint4 *)(base + offA + ks * 2 * St::CSA);
      const uint4 rb = *(const uint4 *)(base + offB + ks * 2 * St::CSB);
#pragma unroll
      for (int h = 0; h < 2; h++) {               // two 16-sequence MFMA steps per 32-sequence chunk
        const unsigned da0 = h ? ra.z : ra.x, da1 = h ? ra.w : ra.y;
        const unsigned db0 = h ? rb.z : rb.x, db1 = h ? rb.w : rb.y;
        uint4 wv[NS];
#pragma unroll
        for (int p = 0; p < NS; p++)
          wv[p] = *(const uint4 *)(wl + p * KT + ks * 32 + khalf * 16 + h * 8);
        v8bf bo[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
          unsigned l0, h0, l1, h1;
          spread(db0, s, l0, h0); spread(db1, s, l1, h1);
          uint4 v = make_uint4(__umul24(l0, 0x3F80u), __umul24(h0, 0x3F80u),
                               __umul24(l1, 0x3F80u), __umul24(h1, 0x3F80u));
          bo[s] = *(v8bf *)&v;
        }
#pragma unroll
        for (int y = 0; y < 4; y++) {
          unsigned l0, h0, l1, h1;
          spread(da0, y, l0, h0); spread(da1, y, l1, h1);
          const unsigned m0 = __umul24(l0, 0xFFFFu), m1 = __umul24(h0, 0xFFFFu);
          const unsigned m2 = __umul24(l1, 0xFFFFu), m3 = __umul24(h1, 0xFFFFu);
#pragma unroll
          for (int p = 0; p < NS; p++) {
            uint4 v = make_uint4(wv[p].x & m0, wv[p].y & m1, wv[p].z & m2, wv[p].w & m3);
            const v8bf ao = *(v8bf *)&v;
#pragma unroll
            for (int x = 0; x < 4; x++)
              acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ao, bo[x], acc[x][y], 0, 0, 0);
          }
        }
      }
    }
    STAGE_SSTORE(St, pre, lds + (buf ^ 1) * SB, tid);
    wstore(lds + (buf ^ 1) * SB);
    __syncthreads();
  }

  const int64_t i = i0 + wi * 32 + col;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int64_t j = j0 + wj * 32 + 8 * (r >> 2) + 4 * khalf + (r & 3);
    if (i < j && j < L) {
      float4 *p = (float4 *)(out + rsg_rec(i, j, L) * 16);
#pragma unroll
      for (int x = 0; x < 4; x++) p[x] = make_float4(acc[x][0][r], acc[x][1][r], acc[x][2][r], acc[x][3][r]);
    }
  }
}

// ------------------------------------------------------------------------------------
// Tile shapes (the autotuner sweeps these): waves per work group and K-tile.
struct GramShape { int WI, WJ, KT; const char *name; };
static const GramShape kShapes[] = {
  {2, 2, 256, "64x64c/8w/kt256"},
  {2, 2, 128, "64x64c/8w/kt128"},
  {2, 2, 512, "64x64c/8w/kt512"},
  {1, 1, 256, "32x32c/2w/kt256"},
  {2, 1, 256, "64x32c/4w/kt256"},
  {1, 2, 256, "32x64c/4w/kt256"},
  {2, 1, 512, "64x32c/4w/kt512"},
  {1, 2, 512, "32x64c/4w/kt512"},
  {1, 1, 512, "32x32c/2w/kt512"},
};
static const int kNShapes = (int)(sizeof(kShapes) / sizeof(kShapes[0]));

extern "C" int rsg_gram_nshapes(void) { return kNShapes; }
extern "C" const char *rsg_gram_shape_name(int s) { return (s >= 1 && s <= kNShapes) ? kShapes[s - 1].name : "auto"; }

// Upper-triangular tile list for (L, BI, BJ), cached per process and device.
static const int2 *tile_list(int device, int64_t L, int BI, int BJ, int *ntiles, char *errbuf)
{
  static std::map<std::tuple<int, int64_t, int, int>, std::pair<int2 *, int>> cache;
  static std::mutex mu;                                 // contexts of several threads
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_tuple(device, L, BI, BJ);
  auto it = cache.find(key);
  if (it != cache.end()) { *ntiles = it->second.second; return it->second.first; }
  std::vector<int2> v;
  int64_t nbi = (L + BI - 1) / BI, nbj = (L + BJ - 1) / BJ;
  for (int64_t bi = 0; bi < nbi; bi++)
    for (int64_t bj = 0; bj < nbj; bj++) {
      int64_t jmax = std::min((bj + 1) * BJ, L) - 1;
      if (bi * BI < jmax) v.push_back(make_int2((int)bi, (int)bj));
    }
  int2 *d = nullptr;
  if (rsg_dev_malloc(&d, sizeof(int2) * std::max<size_t>(v.size(), 1)) != hipSuccess) { rsg_fail(errbuf, "tile list: out of device memory"); return nullptr; }
  if (!v.empty() && hipMemcpy(d, v.data(), sizeof(int2) * v.size(), hipMemcpyHostToDevice) != hipSuccess) { rsg_fail(errbuf, "tile list copy"); return nullptr; }
  cache[key] = std::make_pair(d, (int)v.size());
  *ntiles = (int)v.size();
  return d;
}

// 32 x 32-column tiles that fit the device at once: up to one per compute unit on eight waves each,
// up to two on four (with their last, second round on eight waves 300 tiles of 4096 sequences
// take 27.6 us, on four 20.7).  Against the best of the other shapes, with their segments along K and
// the fix-up launch: 8.2 and 10.0 us at 384 x 384, 11.3 and 17.5 at 3072 x 384, 17.3 and 22.7 at
// 3072 x 768, 39 and 44 at 12288 x 768; past 16384 sequences those win (24.8 and 25.8 us at
// 16384 x 320, 66 and 35 at 49152).
static int launch_fp4_deep(rsg_ctx *c, rsg_msa *m, void *out, const int2 *tiles, int ntiles, double *pm_part, int *pmflag,
                           char *errbuf)
{
  const int per = (ntiles + 7) / 8, nk = (int)((m->N + 63) / 64);
  int t; rsg_tstart(c, "gram_fp4", &t);
  if (ntiles <= (c->ncu > 0 ? c->ncu : 256))
    hipLaunchKernelGGL(k_gram_fp4_deep<4>, dim3((unsigned)(8 * per)), dim3(512), 0, c->stream, m->d_x4, nk, m->Lpad, m->L,
                       (uint4 *)out, tiles, ntiles, per, pm_part, pmflag);
  else
    hipLaunchKernelGGL(k_gram_fp4_deep<2>, dim3((unsigned)(8 * per)), dim3(256), 0, c->stream, m->d_x4, nk, m->Lpad, m->L,
                       (uint4 *)out, tiles, ntiles, per, pm_part, pmflag);
  rsg_tstop(c, t);
  HIPCHK(hipGetLastError());
  return RSG_OK;
}

template <int WI, int WJ, int KT, int OK>
static int launch_fp4(rsg_ctx *c, rsg_msa *m, void *out, double *pm_part, int *pmflag, char *errbuf)
{
  constexpr int BI = 32 * WI, BJ = 32 * WJ;
  if (m->Lpad % BI || m->Lpad % BJ || m->Npad % KT) return rsg_fail(errbuf, "gram: padding does not fit the tile");
  int ntiles = 0;
  const int2 *tiles;
  if (c->tiles_fixed) {                      // an allocation-free call brings its own tile list
    if (BI != 32 || BJ != 32) return rsg_fail(errbuf, "gram: a fixed tile list needs 32 x 32-column tiles");
    tiles = c->tiles_fixed; ntiles = c->ntiles_fixed;
  } else tiles = tile_list(c->device, m->L, BI, BJ, &ntiles, errbuf);
  if (!tiles) return RSG_FAIL;
  if (ntiles == 0) return RSG_OK;
  if (OK == CNT_U16 && m->N > RSG_U16_MAXN) return rsg_fail(errbuf, "gram: uint16 records hold up to %d sequences", RSG_U16_MAXN);
  if constexpr (WI == 1 && WJ == 1 && KT == 256 && OK == CNT_U16)
    if (ntiles <= 2 * (c->ncu > 0 ? c->ncu : 256)) return launch_fp4_deep(c, m, out, tiles, ntiles, pm_part, pmflag, errbuf);
  // whole waves of tiles run over the full K range; when there are few waves (under four
  // tiles per work-group slot) and the last wave is at most half full, its tiles are split along
  // K into one segment per CU, which run after the full tiles in the slots the first of them
  // free (the two work groups that share a CU finish far apart), then reduced (with many waves
  // the tail is small and the partial traffic costs more).  A CU holds 8 waves of this kernel
  // (two per SIMD): 4 / (WI WJ) work groups.  Of more tiles than CUs (half a wave of the smallest ones)
  // some would be left without a segment.
  const int ncu = c->ncu > 0 ? c->ncu : 256;
  const int slots = std::max(ncu * 4 / (WI * WJ), 1);
  // whole K-tiles; when the sequences past the last whole one fit one 64-sequence k-step, that
  // step runs from registers after the loop instead of as a K-tile of mostly padding
  int64_t nkt = (m->N + KT - 1) / KT, tailc = -1;
  {
    const int64_t nfull = m->N / KT, r = m->N - nfull * KT;
    if (nfull >= 1 && r > 0 && r <= 64) { nkt = nfull; tailc = nfull * (KT / 32); }
  }
  int ndp = ntiles, sbase = 1, sextra = 0;
  const int rem = ntiles % slots;
  if (OK == CNT_U32 && m->N > FP4_EXACT) {        // every tile in segments whose FP32 sums are exact
    ndp = 0;
    sbase = (int)(m->N / FP4_EXACT) + 1;
  } else if (c->gram_split && ntiles < 4 * slots && rem > 0 && rem <= std::min(slots / 2, ncu) && nkt >= 2) {
    ndp = ntiles - rem;
    const int nsu = (int)std::min<int64_t>((int64_t)ncu, (int64_t)rem * nkt);
    sbase = nsu / rem; sextra = nsu % rem;
  }
  const int nrem = ntiles - ndp, nsu = nrem * sbase + sextra;
  uint8_t *part = nullptr;
  if (nrem > 0) {
    const size_t need = (size_t)nsu * BI * BJ * rsg_rec_bytes(OK);
    if (c->gscr_cap < need && c->no_alloc) return rsg_fail(errbuf, "gram: split-K partials need an allocation");
    if (c->gscr_cap < need) {
      if (c->d_gscr) hipFree(c->d_gscr);
      c->d_gscr = nullptr; c->gscr_cap = 0;
      HIPCHK(rsg_dev_malloc(&c->d_gscr, need));
      c->gscr_cap = need;
    }
    part = (uint8_t *)c->d_gscr;
  }
  const int per = (ndp + 7) / 8;
  dim3 grid((unsigned)(8 * per + nsu)), block(128 * WI * WJ);
  // one timer over the Gram and its split-K fix-up
  int t; rsg_tstart(c, "gram_fp4", &t);
  hipLaunchKernelGGL((k_gram_fp4<WI, WJ, KT, OK>), grid, block, 0, c->stream, m->d_x4, nkt, tailc, m->Lpad, m->L, out,
                     tiles, ndp, per, ntiles, sbase, sextra, part, pm_part, pmflag);
  if (nrem > 0)
    hipLaunchKernelGGL((k_gram_fix<BI, BJ, OK>), dim3((unsigned)(nrem * (BI / 32) * (BJ / 32))), dim3(64 * FIX_WAVES), 0, c->stream,
                       part, tiles, ndp, sbase, sextra, m->L, out, pm_part);
  rsg_tstop(c, t);
  HIPCHK(hipGetLastError());
  return RSG_OK;
}

// The autotuner's table: the fastest shape per size bucket (ceil(log2 N), ceil(log2 L)), one
// "logN logL shape" line each ('#' starts a comment).  Loaded once per process from
// gram_tiles.tsv next to the library (or rsg_gram_tiles_load); sizes without an entry use
// the built-in rule below.
static std::mutex g_tiles_mu;
static std::map<std::pair<int, int>, int> g_tiles;
static bool g_tiles_tried = false;

static int ceil_log2(int64_t v)
{
  int k = 0;
  while (((int64_t)1 << k) < v) k++;
  return k;
}

static int parse_tiles(const char *path, std::map<std::pair<int, int>, int> &t, char *errbuf)
{
  FILE *f = path ? fopen(path, "r") : nullptr;
  if (!f) return rsg_fail(errbuf, "rsg_gram_tiles_load: cannot open %s", path ? path : "(null)");
  char line[256];
  int ln = 0;
  while (fgets(line, sizeof line, f)) {
    ln++;
    char *h = strchr(line, '#');
    if (h) *h = 0;
    int a, b, sh;
    char extra;
    const int n = sscanf(line, "%d %d %d %c", &a, &b, &sh, &extra);
    if (n <= 0) continue;                               // blank or comment
    if (n != 3 || a < 0 || a > 40 || b < 0 || b > 40 || sh < 1 || sh > kNShapes) {
      fclose(f);
      return rsg_fail(errbuf, "rsg_gram_tiles_load: %s line %d: expected \"logN logL shape\" with shape 1..%d", path, ln,
                      kNShapes);
    }
    t[std::make_pair(a, b)] = sh;
  }
  fclose(f);
  return RSG_OK;
}

extern "C" int rsg_gram_tiles_load(const char *path, char *errbuf)
{
  std::map<std::pair<int, int>, int> t;
  if (parse_tiles(path, t, errbuf) != RSG_OK) return RSG_FAIL;
  std::lock_guard<std::mutex> g(g_tiles_mu);
  g_tiles.swap(t);
  g_tiles_tried = true;
  return RSG_OK;
}

static int table_shape(int64_t N, int64_t L)
{
  std::lock_guard<std::mutex> g(g_tiles_mu);
  if (!g_tiles_tried) {
    g_tiles_tried = true;
    Dl_info info;
    if (dladdr((void *)&rsg_gram_tiles_load, &info) && info.dli_fname) {
      std::string p(info.dli_fname);
      const size_t k = p.rfind('/');
      p = (k == std::string::npos ? std::string(".") : p.substr(0, k)) + "/gram_tiles.tsv";
      std::map<std::pair<int, int>, int> t;
      char eb[256];
      if (FILE *f = fopen(p.c_str(), "r")) {
        fclose(f);
        if (parse_tiles(p.c_str(), t, eb) == RSG_OK) g_tiles.swap(t);   // a malformed table is ignored
      }
    }
  }
  auto it = g_tiles.find(std::make_pair(ceil_log2(N), ceil_log2(L)));
  return it == g_tiles.end() ? 0 : it->second;
}

// The shape of a unit-weight Gram: the caller's, else the table's, else by rule.  (A line of the table
// counts for its whole bucket: 32 x 32-column tiles, measured at 768 columns on launch_fp4_deep, also
// past its 992 columns, where they cost at most a few per cent: 26.7 and 27.8 us, 71.3 and 68.1 against
// 64 x 32 at 3072 and 12288 x 1008.)
static int pick_shape(const rsg_ctx *c, int64_t N, int64_t L)
{
  int s = c ? c->gram_shape : 0;
  if (s >= 1 && s <= kNShapes) return s;
  s = table_shape(N, L);
  if (s >= 1 && s <= kNShapes) return s;
  // sizes outside the table: 64 x 32-column tiles of four waves with 512-sequence K tiles win or tie
  // at N >= 1536 (two work groups per CU, so one's epilogue runs under the other's K loop); below
  // ~1000 sequences (a few K tiles) 32 x 32 tiles of two waves are as fast; where those fit the device at
  // once launch_fp4_deep takes them
  const int64_t nb = (L + 31) / 32;
  const bool deep = nb * (nb + 1) / 2 <= 2 * (c && c->ncu > 0 ? c->ncu : 256);
  return (N < 1024 || (deep && N <= 16384)) ? 4 : 7;
}

extern "C" int rsg_gram_shape_for(const rsg_ctx *c, int64_t N, int64_t L) { return pick_shape(c, N, L); }

int rsg_gram_counts_fp4(rsg_ctx *c, rsg_msa *m, void *out, int kind, double *pm_part, int *pmflag, char *errbuf)
{
  if (rsg_need(c, m, PACK_X4, errbuf) != RSG_OK) return RSG_FAIL;
  if (kind == CNT_U32)            // more than 65535 sequences: the two default shapes only, no fused marginals
    return (m->L >= 768) ? launch_fp4<2, 2, 512, CNT_U32>(c, m, out, nullptr, nullptr, errbuf)
                         : launch_fp4<1, 1, 256, CNT_U32>(c, m, out, nullptr, nullptr, errbuf);
  if (kind != CNT_U16) return rsg_fail(errbuf, "gram: bad record kind %d", kind);
  switch (pick_shape(c, m->N, m->L)) {
  case 1: return launch_fp4<2, 2, 256, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 2: return launch_fp4<2, 2, 128, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 3: return launch_fp4<2, 2, 512, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 4: return launch_fp4<1, 1, 256, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 5: return launch_fp4<2, 1, 256, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 6: return launch_fp4<1, 2, 256, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 7: return launch_fp4<2, 1, 512, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 8: return launch_fp4<1, 2, 512, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  case 9: return launch_fp4<1, 1, 512, CNT_U16>(c, m, out, pm_part, pmflag, errbuf);
  }
  return rsg_fail(errbuf, "bad gram shape");
}

// split weights: part p of w_s as bf16 bits, [NS][Npad]; hi = bf16(w), lo = bf16(w - hi), ...
__global__ void k_split_weights(const double *__restrict__ w, int64_t N, int64_t Npad, int nsplit,
                                uint16_t *__restrict__ out)
{
  int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= Npad) return;
  double r = (s < N) ? w[s] : 0.;
  for (int p = 0; p < nsplit; p++) {
    __hip_bfloat16 b = __float2bfloat16((float)r);
    r -= (double)__bfloat162float(b);
    out[p * Npad + s] = __bfloat16_as_ushort(b);
  }
}

int rsg_upload_weights_bf16(rsg_ctx *c, rsg_msa *m, int nsplit, char *errbuf)
{
  if (m->nsplit_ready == nsplit) return RSG_OK;
  if (!m->d_wsplit) HIPCHK(rsg_msa_get(m, &m->d_wsplit, sizeof(uint16_t) * 3 * (size_t)m->Npad));
  hipLaunchKernelGGL(k_split_weights, dim3((unsigned)((m->Npad + 255) / 256)), dim3(256), 0, c->stream,
                     m->d_w, m->N, m->Npad, nsplit, m->d_wsplit);
  HIPCHK(hipGetLastError());
  m->nsplit_ready = nsplit;
  return RSG_OK;
}

template <int WI, int WJ, int KT, int NS>
static int launch_bf16(rsg_ctx *c, rsg_msa *m, float *out, char *errbuf)
{
  constexpr int BI = 32 * WI, BJ = 32 * WJ;
  if (m->Lpad % BI || m->Lpad % BJ || m->Npad % KT) return rsg_fail(errbuf, "gram: padding does not fit the tile");
  int ntiles = 0;
  const int2 *tiles;
  if (c->tiles_fixed) {                      // an allocation-free call brings its own tile list
    if (BI != 32 || BJ != 32) return rsg_fail(errbuf, "gram: a fixed tile list needs 32 x 32-column tiles");
    tiles = c->tiles_fixed; ntiles = c->ntiles_fixed;
  } else tiles = tile_list(c->device, m->L, BI, BJ, &ntiles, errbuf);
  if (!tiles) return RSG_FAIL;
  if (ntiles == 0) return RSG_OK;
  int per = (ntiles + 7) / 8;
  int t; rsg_tstart(c, "gram_bf16", &t);
  hipLaunchKernelGGL((k_gram_bf16<WI, WJ, KT, NS>), dim3((unsigned)(8 * per)), dim3(64 * WI * WJ), 0, c->stream,
                     m->d_xt, m->d_wsplit, (m->N + KT - 1) / KT, m->Npad, m->Lpad, m->L, out, tiles, ntiles, per);
  rsg_tstop(c, t);
  HIPCHK(hipGetLastError());
  return RSG_OK;
}

int rsg_gram_counts_bf16(rsg_ctx *c, rsg_msa *m, int nsplit, float *out, char *errbuf)
{
  if (rsg_need(c, m, PACK_XT, errbuf) != RSG_OK || rsg_upload_weights_bf16(c, m, nsplit, errbuf) != RSG_OK) return RSG_FAIL;
  const bool big = m->L >= 768;
  if (nsplit > 2) return big ? launch_bf16<2, 2, 64, 3>(c, m, out, errbuf) : launch_bf16<1, 1, 64, 3>(c, m, out, errbuf);
  return big ? launch_bf16<2, 2, 64, 2>(c, m, out, errbuf) : launch_bf16<1, 1, 64, 2>(c, m, out, errbuf);
}

// ------------------------------------------------------------------------------------
// Weighted Gram from int8 weight limbs (exact integer accumulation).  Each sequence weight is
// rounded to 21-bit fixed point relative to the largest weight, q_s = round(w_s / W) with
// W = max_s w_s / (2^21 - 1), and split into three 7-bit limbs q = q0 + 2^7 q1 + 2^14 q2.  The
// int8 MFMA then forms, per limb k, G_k[x][y] = sum_s q_{s,k} [a_si = x][a_sj = y] exactly in
// int32 (the j-side operand is the one-hot code masked for symbol y, scaled by 2^y; the i-side
// operand is the limb byte where the code is symbol x, else 0), and the epilogue combines
// W (G_0 + 2^7 G_1 + 2^14 G_2) in FP64 (exact) before the FP32 record store.  The only error
// is the weight rounding: |w_s - W q_s| <= W / 2 = 2^-22 max_s w_s.
//
// Layout of the limb panel: [Npad / 16][4][16] bytes, limbs 0..2 of the 16 sequences of a
// K-chunk (slot 3 zero), so one stage's limbs are NKC * 64 contiguous bytes, staged into LDS
// behind the stage's codes by wave 0 (one more LDS-direct instruction for that wave).
#define W8_BITS 21
__global__ void __launch_bounds__(1024) k_quant_weights(const double *__restrict__ w, int64_t N, int64_t Npad,
                                                         uint8_t *__restrict__ wq, double *__restrict__ scale)
{
  __shared__ double red[1024];
  const int tid = threadIdx.x;
  double mx = 0.;
  for (int64_t s = tid; s < N; s += 1024) mx = fmax(mx, w[s]);
  red[tid] = mx;
  __syncthreads();
  for (int st = 512; st > 0; st >>= 1) {
    if (tid < st) red[tid] = fmax(red[tid], red[tid + st]);
    __syncthreads();
  }
  const double wmax = red[0];
  const double qmax = (double)((1 << W8_BITS) - 1);
  const double W = (wmax > 0.) ? wmax / qmax : 1.;
  if (tid == 0) *scale = W;
  for (int64_t s = tid; s < Npad; s += 1024) {
    double qd = (s < N && wmax > 0.) ? rint(w[s] / W) : 0.;
    qd = fmin(fmax(qd, 0.), qmax);
    const uint32_t q = (uint32_t)qd;
    uint8_t *p = wq + (s / 16) * 64 + (s % 16);
    p[0] = (uint8_t)(q & 127u); p[16] = (uint8_t)((q >> 7) & 127u); p[32] = (uint8_t)((q >> 14) & 127u); p[48] = 0;
  }
}

// One 32 x 32-column tile, four waves: wave x owns the i-side symbol x and all four j-side
// symbols for the three limbs (12 accumulators of 16 int32 per lane).  Staging as in the FP4
// Gram (three LDS images, LDS-direct loads two stages ahead), each image followed by the
// stage's limb bytes.
// K-tiles [kt0, kt1).  With SPLIT (a split-K segment) the combined limb sums
// g = G_0 + 2^7 G_1 + 2^14 G_2 of every cell of every pair of the tile go, unconditionally, to
// the partial record jj * 32 + ii of eight planes of two int64 cells (a lane's cells side by side
// instead took k_gram_w8_fix twice as long) for k_gram_w8_fix, and no record or nseff is written.
// (SPLIT: the partial-sum epilogue, a template argument so that each variant of the loop gets its
// own register allocation -- with both epilogues after one loop the kernel spilled.)
template <int KT, bool SPLIT>
__device__ __forceinline__ void gram_tile_w8(const uint8_t *__restrict__ xt, const uint8_t *__restrict__ wq, double W,
                                             int64_t Lpad, int64_t L, float *__restrict__ out, double *__restrict__ nsx,
                                             int64_t i0, int64_t j0, uint8_t *lds, int64_t kt0, int64_t kt1,
                                             int64_t *__restrict__ part, double *__restrict__ pm_part)
{
#pragma clang fp contract(off)
  constexpr int NT = 256, KS = KT / 32, NW = 4;
  typedef CodeStage<32, 32, KT, NT, 16> St;
  constexpr int IS = St::BYTES + St::NKC * 64;     // one image: codes, then limbs
  constexpr int WCH = St::NKC * 4;                 // 16-byte limb chunks per stage
  constexpr int QW = St::NINST / NW;               // code loads per wave per stage (+1 for wave 0)
  static_assert(QW >= 1 && QW + 1 <= 15 && WCH <= 64, "stage shape");
  static_assert(KS >= 2, "the barrier precedes the last k-step");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, x = wave;
  const int col = lane & 31, khalf = lane >> 5;
  const int offA = col * 16 + khalf * St::CSA;                           // j side
  const int offB = St::NKC * St::CSA + col * 16 + khalf * St::CSB;       // i side
  const int offW = St::BYTES + khalf * 64;                               // limbs of the lane's chunk

  v16i acc[3][4];                                  // [limb][y]
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int y = 0; y < 4; y++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[k][y][r] = 0;

  auto stage = [&](int64_t kt, uint8_t *base) {
    stage_lds_direct<St, 32, 32, NW>(xt, Lpad, i0, j0, kt, base, wave, lane);
    if (wave == 0 && lane < WCH) lds_direct16(wq + (kt * WCH + lane) * 16, base + St::BYTES);
  };
  auto wait_stage = [&]() {                        // this wave's loads of the older stage landed
    if (wave == 0) __builtin_amdgcn_s_waitcnt(0x0F70 | (QW + 1));
    else           __builtin_amdgcn_s_waitcnt(0x0F70 | QW);
  };
  const int nit = (int)(kt1 - kt0);
  auto stage_of = [&](int it) -> int64_t { return kt0 + ((it < nit) ? it : nit - 1); };
  stage(stage_of(0), lds);
  stage(stage_of(1), lds + IS);
  wait_stage();
  __syncthreads();
  uint4 ra = *(const uint4 *)(lds + offA);
  uint4 rb = *(const uint4 *)(lds + offB);
  for (int it = 0; it < nit; it++) {
    stage(stage_of(it + 2), lds + ((it + 2) % 3) * IS);
    const uint8_t *base = lds + (it % 3) * IS;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      // this k-step's limbs: read before the last k-step's barrier, after which the image may
      // be overwritten by the next iteration's loads
      const uint4 *wp = (const uint4 *)(base + offW + ks * 128);
      const uint4 w0 = wp[0], w1 = wp[1], w2 = wp[2];
      uint4 na = ra, nb = rb;
      if (ks + 1 < KS) {
        na = *(const uint4 *)(base + offA + (ks + 1) * 2 * St::CSA);
        nb = *(const uint4 *)(base + offB + (ks + 1) * 2 * St::CSB);
      } else {
        wait_stage();
        __syncthreads();
        const uint8_t *nbase = lds + ((it + 1) % 3) * IS;
        na = *(const uint4 *)(nbase + offA);
        nb = *(const uint4 *)(nbase + offB);
      }
      // i side: byte 0xFF where the code is symbol x, else 0
      const unsigned t0 = (rb.x >> x) & 0x01010101u, t1 = (rb.y >> x) & 0x01010101u,
                     t2 = (rb.z >> x) & 0x01010101u, t3 = (rb.w >> x) & 0x01010101u;
      const unsigned m0 = (t0 << 8) - t0, m1 = (t1 << 8) - t1, m2 = (t2 << 8) - t2, m3 = (t3 << 8) - t3;
      v4i a[4];
#pragma unroll
      for (int y = 0; y < 4; y++) {
        const unsigned mk = 0x01010101u << y;
        a[y] = (v4i){(int)(ra.x & mk), (int)(ra.y & mk), (int)(ra.z & mk), (int)(ra.w & mk)};
      }
      const v4i b0 = (v4i){(int)(m0 & w0.x), (int)(m1 & w0.y), (int)(m2 & w0.z), (int)(m3 & w0.w)};
#pragma unroll
      for (int y = 0; y < 4; y++) acc[0][y] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[y], b0, acc[0][y], 0, 0, 0);
      const v4i b1 = (v4i){(int)(m0 & w1.x), (int)(m1 & w1.y), (int)(m2 & w1.z), (int)(m3 & w1.w)};
#pragma unroll
      for (int y = 0; y < 4; y++) acc[1][y] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[y], b1, acc[1][y], 0, 0, 0);
      const v4i b2 = (v4i){(int)(m0 & w2.x), (int)(m1 & w2.y), (int)(m2 & w2.z), (int)(m3 & w2.w)};
#pragma unroll
      for (int y = 0; y < 4; y++) acc[2][y] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[y], b2, acc[2][y], 0, 0, 0);
      ra = na; rb = nb;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);             // no LDS-direct load outlives the loop

  if constexpr (SPLIT) {                           // a split-K segment: the exact partial sums
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int jj = 8 * (r >> 2) + 4 * khalf + (r & 3);
      int64_t g[4];
#pragma unroll
      for (int y = 0; y < 4; y++)
        g[y] = (int64_t)((unsigned)acc[0][y][r] >> y) + 128 * (int64_t)((unsigned)acc[1][y][r] >> y) +
               16384 * (int64_t)((unsigned)acc[2][y][r] >> y);
      longlong2 *p = (longlong2 *)part + 2 * x * 1024 + jj * 32 + col;
      p[0] = make_longlong2(g[0], g[1]);
      p[1024] = make_longlong2(g[2], g[3]);
    }
    return;
  }

  // epilogue: lane owns i column `col`; register r holds j = 8*(r/4) + 4*khalf + r%4; cells
  // x*4 .. x*4+3 of each record are this wave's.  They meet in LDS (which every wave has finished
  // with after the barrier), eight rows at a time, and each wave takes whole records: the 64 bytes
  // to memory, nseff, the marginal terms.  nseff of every pair comes from the exact integer sums (the
  // FP32 cells each carry a rounding, and ngap = total - nseff cancels most of nseff): one rounding
  // W * sum goes to nsx.  The marginal partials of the 32 x 32 block follow as in the FP4 Gram, from the
  // FP32 cells (a pass of its own over the records took 17 us at 5000 x 1500, 191 us at
  // 20000 x 5000).
  float4 *xc = (float4 *)lds;                      // [x][8 rows][lane]
  int64_t *xs = (int64_t *)(lds + 32768);          // their sums
  const int64_t i = i0 + col;
  double tm[4][8];
#pragma unroll
  for (int hh = 0; hh < 2; hh++) {
    __syncthreads();
#pragma unroll
    for (int rl = 0; rl < 8; rl++) {
      const int r = 8 * hh + rl;
      int64_t g[4], sx = 0;
#pragma unroll
      for (int y = 0; y < 4; y++) {
        g[y] = (int64_t)((unsigned)acc[0][y][r] >> y) + 128 * (int64_t)((unsigned)acc[1][y][r] >> y) +
               16384 * (int64_t)((unsigned)acc[2][y][r] >> y);
        sx += g[y];
      }
      xs[(x * 8 + rl) * 64 + lane] = sx;
      xc[(x * 8 + rl) * 64 + lane] =
        make_float4((float)((double)g[0] * W), (float)((double)g[1] * W), (float)((double)g[2] * W), (float)((double)g[3] * W));
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int rl = 2 * wave + q, r = 8 * hh + rl;
      const int64_t j = j0 + 8 * (r >> 2) + 4 * khalf + (r & 3);
      const bool valid = i < j && j < L;
      float4 c[4];
#pragma unroll
      for (int k = 0; k < 4; k++) c[k] = xc[(k * 8 + rl) * 64 + lane];
      if (valid) {
        float4 *o = (float4 *)(out + rsg_rec(i, j, L) * 16);
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = c[k];
        const int64_t tot = xs[rl * 64 + lane] + xs[(8 + rl) * 64 + lane] + xs[(16 + rl) * 64 + lane] + xs[(24 + rl) * 64 + lane];
        nsx[rsg_rec(i, j, L)] = (double)tot * W;
      }
      block_terms_w(c, valid, tm[2 * hh + q]);
    }
  }
  if (pm_part == nullptr) return;
  __syncthreads();
  PmTerms &T = *(PmTerms *)lds;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int r = 8 * (k >> 1) + 2 * wave + (k & 1);
#pragma unroll
    for (int y = 0; y < 4; y++) { T[0][r][y][lane] = tm[k][y]; T[1][r][y][lane] = tm[k][4 + y]; }
  }
  __syncthreads();
  block_partials(T, (int)(i0 / 32), (int)(j0 / 32), (int)((L + 31) / 32), wave, lane, pm_part);
}

// Grid: 8 * per_xcd work groups for the first ndp tiles (whole K range, neighbouring tiles on one
// XCD), then the split units of the last tiles (K segments as in k_gram_fp4: tile ndp + t takes
// sbase + 1 segments if t < sextra, else sbase), which run in the slots the full tiles free.
template <int KT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
k_gram_w8(const uint8_t *__restrict__ xt, const uint8_t *__restrict__ wq, const double *__restrict__ wscale, int64_t nkt,
          int64_t Lpad, int64_t L, float *__restrict__ out, double *__restrict__ nsx, const int2 *__restrict__ tiles,
          int ndp, int per_xcd, int ntiles, int sbase, int sextra, int64_t *__restrict__ part, double *__restrict__ pm_part,
          int *__restrict__ pmflag)
{
  typedef CodeStage<32, 32, KT, 256, 16> St;
  constexpr int STAGES = 3 * (St::BYTES + St::NKC * 64);
  __shared__ __attribute__((aligned(16))) uint8_t lds[STAGES > (int)sizeof(PmTerms) ? STAGES : (int)sizeof(PmTerms)];
  if (pmflag && blockIdx.x == 0 && threadIdx.x == 0) *pmflag = 0;    // set by the marginal reduction
  const int g = blockIdx.x;
  int t;
  int64_t k0 = 0, k1 = nkt;
  int64_t *p = nullptr;
  if (g < 8 * per_xcd) {
    t = (g & 7) * per_xcd + (g >> 3);
    if (t >= ndp) return;
  } else {
    const int u = g - 8 * per_xcd, nsu = (ntiles - ndp) * sbase + sextra;
    if (u >= nsu) return;
    int tr, sg, ns;
    split_unit(u, sbase, sextra, tr, sg, ns);
    t = ndp + tr;
    k0 = nkt * sg / ns; k1 = nkt * (sg + 1) / ns;
    p = part + (int64_t)u * 1024 * 16;
  }
  const int2 tl = tiles[t];
  if (p) gram_tile_w8<KT, true>(xt, wq, *wscale, Lpad, L, out, nsx, (int64_t)tl.x * 32, (int64_t)tl.y * 32, lds, k0, k1, p, nullptr);
  else   gram_tile_w8<KT, false>(xt, wq, *wscale, Lpad, L, out, nsx, (int64_t)tl.x * 32, (int64_t)tl.y * 32, lds, k0, k1, p, pm_part);
}

// Split tiles: one work group (16 waves) per tile adds the tile's int64 partial sums over its K
// segments (exact) and writes the records, nseff and the marginal partials with the arithmetic
// of the gram_tile_w8 epilogue, so they equal the unsplit kernel's bit for bit.  Wave r takes row
// r of the MFMA layout.
__global__ void __launch_bounds__(1024)
k_gram_w8_fix(const int64_t *__restrict__ part, const int2 *__restrict__ tiles, int ndp, int sbase, int sextra,
              const double *__restrict__ wscale, int64_t L, float *__restrict__ out, double *__restrict__ nsx,
              double *__restrict__ pm_part)
{
#pragma clang fp contract(off)
  __shared__ PmTerms T;
  const int tr = blockIdx.x, r = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 31, khalf = lane >> 5;
  const int2 tl = tiles[ndp + tr];
  const int ns = sbase + (tr < sextra ? 1 : 0);
  const double W = *wscale;
  const int jj = 8 * (r >> 2) + 4 * khalf + (r & 3);
  const int64_t i = (int64_t)tl.x * 32 + col, j = (int64_t)tl.y * 32 + jj;
  const longlong2 *p0 = (const longlong2 *)part + (int64_t)split_first(tr, sbase, sextra) * 8 * 1024 + jj * 32 + col;
  int64_t g[16];
#pragma unroll
  for (int c = 0; c < 16; c++) g[c] = 0;
#pragma unroll 2
  for (int k = 0; k < ns; k++) {
    const longlong2 *q = p0 + (int64_t)k * 8 * 1024;
#pragma unroll
    for (int h = 0; h < 8; h++) { const longlong2 v = q[h * 1024]; g[2 * h] += v.x; g[2 * h + 1] += v.y; }
  }
  const bool valid = i < j && j < L;
  int64_t tot = 0;
  float4 c[4];
#pragma unroll
  for (int x = 0; x < 4; x++) {
    tot += (g[x * 4] + g[x * 4 + 1]) + (g[x * 4 + 2] + g[x * 4 + 3]);
    c[x] = make_float4((float)((double)g[x * 4] * W), (float)((double)g[x * 4 + 1] * W), (float)((double)g[x * 4 + 2] * W),
                       (float)((double)g[x * 4 + 3] * W));
  }
  if (valid) {
    float4 *o = (float4 *)(out + rsg_rec(i, j, L) * 16);
#pragma unroll
    for (int x = 0; x < 4; x++) o[x] = c[x];
    nsx[rsg_rec(i, j, L)] = (double)tot * W;
  }
  if (pm_part == nullptr) return;
  double t[8];
  block_terms_w(c, valid, t);
#pragma unroll
  for (int y = 0; y < 4; y++) { T[0][r][y][lane] = t[y]; T[1][r][y][lane] = t[4 + y]; }
  __syncthreads();
  block_partials(T, tl.x, tl.y, (int)((L + 31) / 32), r, lane, pm_part);
}

int rsg_gram_counts_w8(rsg_ctx *c, rsg_msa *m, float *out, double *pm_part, int *pmflag, char *errbuf)
{
  constexpr int KT = 256;
  if (m->Npad % KT || m->Lpad % 32) return rsg_fail(errbuf, "gram: padding does not fit the tile");
  if (m->N > (1 << 21)) return rsg_fail(errbuf, "weighted int8 counts: at most %d sequences", 1 << 21);
  if (rsg_need(c, m, PACK_XT, errbuf) != RSG_OK) return RSG_FAIL;
  if (!m->d_wq) {
    HIPCHK(rsg_msa_get(m, &m->d_wq, (size_t)m->Npad * 4 + 64));
  }
  double *d_scale = (double *)(m->d_wq + (size_t)m->Npad * 4);
  if (!m->wq_ready) {
    hipLaunchKernelGGL(k_quant_weights, dim3(1), dim3(1024), 0, c->stream, m->d_w, m->N, m->Npad, m->d_wq, d_scale);
    HIPCHK(hipGetLastError());
    m->wq_ready = 1;
  }
  if (!m->d_nsx) HIPCHK(rsg_msa_get(m, &m->d_nsx, sizeof(double) * (size_t)m->L * (size_t)m->L));
  int ntiles = 0;
  const int2 *tiles;
  if (c->tiles_fixed) { tiles = c->tiles_fixed; ntiles = c->ntiles_fixed; }
  else tiles = tile_list(c->device, m->L, 32, 32, &ntiles, errbuf);
  if (!tiles) return RSG_FAIL;
  if (ntiles == 0) return RSG_OK;
  // the tail as in launch_fp4: a CU holds two of these 4-wave work groups; when the last wave of
  // tiles is at most half full its tiles are split along K, one segment per CU, after the full
  // tiles, and k_gram_w8_fix adds the exact partial sums.  From twelve K-tiles on: below, the
  // segments are too short for the partials and the second launch (300 columns: 26 us split and 17
  // whole at 600 sequences, 36 and 29 at 2000, 43 and 58 at 5000)
  const int ncu = c->ncu > 0 ? c->ncu : 256, slots = 2 * ncu;
  const int64_t nkt = (m->N + KT - 1) / KT;
  int ndp = ntiles, sbase = 1, sextra = 0;
  const int rem = ntiles % slots;
  if (c->gram_split && ntiles < 4 * slots && rem > 0 && rem <= slots / 2 && nkt >= 12) {
    ndp = ntiles - rem;
    const int nsu = (int)std::min<int64_t>((int64_t)ncu, (int64_t)rem * nkt);
    sbase = nsu / rem; sextra = nsu % rem;
  }
  const int nrem = ntiles - ndp, nsu = nrem * sbase + sextra;
  int64_t *part = nullptr;
  if (nrem > 0) {
    const size_t need = (size_t)nsu * 1024 * 16 * sizeof(int64_t);
    if (c->gscr_cap < need && c->no_alloc) return rsg_fail(errbuf, "gram: split-K partials need an allocation");
    if (c->gscr_cap < need) {
      if (c->d_gscr) hipFree(c->d_gscr);
      c->d_gscr = nullptr; c->gscr_cap = 0;
      HIPCHK(rsg_dev_malloc(&c->d_gscr, need));
      c->gscr_cap = need;
    }
    part = (int64_t *)c->d_gscr;
  }
  const int per = (ndp + 7) / 8;
  int t; rsg_tstart(c, "gram_w8", &t);
  hipLaunchKernelGGL((k_gram_w8<KT>), dim3((unsigned)(8 * per + nsu)), dim3(256), 0, c->stream, m->d_xt, m->d_wq, d_scale,
                     nkt, m->Lpad, m->L, out, m->d_nsx, tiles, ndp, per, ntiles, sbase, sextra, part, pm_part, pmflag);
  if (nrem > 0)
    hipLaunchKernelGGL(k_gram_w8_fix, dim3((unsigned)nrem), dim3(1024), 0, c->stream, part, tiles, ndp, sbase, sextra, d_scale,
                       m->L, out, m->d_nsx, pm_part);
  rsg_tstop(c, t);
  HIPCHK(hipGetLastError());
  return RSG_OK;
}
