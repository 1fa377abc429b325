// rsg_internal.h -- internal state and helpers of librscape_hip (not part of the C-ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <cstdint>
#include <cstdio>
#include <cstdarg>
#include <cstring>
#include <string>
#include <vector>
#include <thread>
#include <memory>
#include <mutex>
#include <algorithm>
#include "../../include/rscape_hip.h"
#include "rsg_pool.h"

#define RSG_MAX_TIMERS 64

// Pair record of columns i < j (16 cells c[x*4+y]) lives at record index j*L + i, so
// consecutive i (the MFMA result lanes) store to consecutive records.
__host__ __device__ static inline int64_t rsg_rec(int64_t i, int64_t j, int64_t L) { return j * L + i; }

// a ^ b ^ c: one instruction on the device (the compiler makes two of the operators)
__host__ __device__ static inline uint32_t rsg_xor3(uint32_t a, uint32_t b, uint32_t c)
{
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
#else
  return a ^ b ^ c;
#endif
}

// Philox4x32-10 counter-based generator (Salmon, Moraes, Dror & Shaw, SC'11).  A draw is a
// pure function of (seed, stream, node, position, tag), so simulation is order-free.  One block
// gives four 32-bit words; rsg_philox returns the first.
__host__ __device__ static inline void rsg_philox4(uint64_t seed, uint32_t stream, uint32_t node, uint32_t pos,
                                                   uint32_t tag, uint32_t out[4])
{
  uint32_t c0 = pos, c1 = node, c2 = stream, c3 = tag;
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
  for (int r = 0; r < 10; r++) {
    uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0, hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    uint32_t n0 = rsg_xor3(hi1, c1, k0), n2 = rsg_xor3(hi0, c3, k1);
    c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
    k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
  }
  out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}
__host__ __device__ static inline uint32_t rsg_philox(uint64_t seed, uint32_t stream, uint32_t node,
                                                     uint32_t pos, uint32_t tag)
{
  uint32_t w[4];
  rsg_philox4(seed, stream, node, pos, tag, w);
  return w[0];
}
// Tag of the per-node draws of the GTR evolution: the block keyed (internal node v, column)
// gives the left child's symbol draw, the right child's, and the two leaf-gap draws.
#define RSG_TAG_CHILDREN 5u

// Kinds of stored pair counts.
//   CNT_U16: unit-weight Gram records, 16 uint16 counts (cell x*4+y), 32 bytes per record; for
//            N <= RSG_U16_MAXN sequences.
//   CNT_U32: unit-weight Gram records for larger N, 16 uint32 counts, 64 bytes per record.
//   CNT_F32: split-BF16 weighted records, FP32 cells, 64 bytes per record.
enum { CNT_U16 = 1, CNT_F32 = 2, CNT_U32 = 3 };
#define RSG_U16_MAXN 65535
static inline int rsg_int_kind(int64_t N) { return N <= RSG_U16_MAXN ? CNT_U16 : CNT_U32; }
__host__ __device__ static inline int rsg_rec_bytes(int kind) { return kind == CNT_U16 ? 32 : 64; }

// The packed forms of an alignment (N x L codes, row-major), built on demand (rsg_need):
//   axT: [Lpad][Npad] raw codes, pad = 4 (a gap);
//   x4:  one-hot FP4 Gram operand, K-chunked [Npad / 32][Lpad][16 bytes]: nibble e of a chunk is
//        1 << symbol of the chunk's sequence e for canonical residues, 0 otherwise;
//   xt:  one-hot byte Gram operand (weighted Grams), [Npad / 16][Lpad][16 bytes], byte 1 << symbol.
enum { PACK_AXT = 1, PACK_XT = 2, PACK_X4 = 4, PACK_LGC = 8 };   // PACK_LGC: with them, the logarithm table

#ifdef __HIPCC__
// One-hot bytes (1 << c for c < 4, else 0) of four codes: byte permute from a table, the selector
// of any code past 3 pointing at a zero byte.
__device__ __forceinline__ unsigned onehot4(unsigned codes)
{
  const unsigned big = (((codes >> 2) & 0x3F3F3F3Fu) + 0x7F7F7F7Fu) & 0x80808080u;   // code > 3
  return __builtin_amdgcn_perm(0u, 0x08040201u, (codes & 0x03030303u) | (big >> 5));
}

// Orders what the lanes of a wave exchange through memory (LDS or global): stores before it are seen by
// every lane's loads after it.  For waves that share data with no other wave of their work group.
__device__ __forceinline__ void wave_sync()
{
  __threadfence_block();
  __builtin_amdgcn_wave_barrier();
}

// Packs the 128-sequence x 128-column block at (s0, c0) with 256 threads: the codes come in as
// dwords of four columns (unaligned: L is any number; 16 loads in flight per thread), cross an
// LDS tile, and leave as 16-byte stores, two columns per thread: consecutive threads take
// consecutive column pairs (x4, xt) or consecutive 16-sequence runs of a column pair (axT).
// Bound by HBM: 20 alignments of 5000 x 1500 pack to x4 in 60 us (3.8 TB/s); with a byte per load
// and LDS access the same took 177 us.
template <int WHAT>
__device__ __forceinline__ void pack_block(const uint8_t *__restrict__ ax, int64_t N, int64_t L, int64_t Npad, int64_t Lpad,
                                           int64_t s0, int64_t c0, uint8_t *__restrict__ axT, uint8_t *__restrict__ xt,
                                           uint8_t *__restrict__ x4)
{
  typedef uint32_t u32u __attribute__((aligned(1)));
  __shared__ uint32_t tile[128][33];
  const int tid = threadIdx.x;
  {
    const int cw = tid & 31, r0 = tid >> 5;
    const int64_t c = c0 + 4 * cw;
    uint32_t v[16];
    if (L >= 4) {
      // every load in range and none behind a branch, so all 16 are in flight at once: rows past N
      // read row N - 1, the columns' last dword is read at L - 4 and shifted; what is past N or
      // L becomes a gap afterwards
      const int64_t cc = min(c, L - 4), sc = min((int64_t)3, c - cc);
#pragma unroll
      for (int k = 0; k < 16; k++) v[k] = *(const u32u *)(ax + min(s0 + r0 + 8 * k, N - 1) * L + cc);
      const uint32_t in = (c >= L) ? 0u : (c + 4 <= L) ? 0xFFFFFFFFu : (1u << (8 * (int)(L - c))) - 1u;
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const uint32_t m = (s0 + r0 + 8 * k < N) ? in : 0u;
        v[k] = ((v[k] >> (8 * (int)sc)) & m) | (0x04040404u & ~m);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const int64_t s = s0 + r0 + 8 * k;
        v[k] = 0x04040404u;
        if (s < N)
          for (int b = 0; b < 3; b++)
            if (c + b < L) v[k] = (v[k] & ~(0xFFu << (8 * b))) | ((uint32_t)ax[s * L + c + b] << (8 * b));
      }
    }
#pragma unroll
    for (int k = 0; k < 16; k++) tile[r0 + 8 * k][cw] = v[k];
  }
  __syncthreads();
  const uint16_t *t16 = (const uint16_t *)tile;           // [128][66]: column pairs
  if (WHAT & PACK_X4) {
    const int cp = tid & 63, q = tid >> 6;                // 32-sequence chunk q
    if (c0 + 2 * cp < Lpad) {
      unsigned w0[4], w1[4];
#pragma unroll
      for (int d = 0; d < 4; d++) {
        w0[d] = w1[d] = 0u;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const int s = q * 32 + d * 8 + e;
          const unsigned h = onehot4((unsigned)t16[s * 66 + cp] | ((unsigned)t16[(s + 1) * 66 + cp] << 16));
          w0[d] |= ((h & 0xFu) | ((h >> 12) & 0xF0u)) << (4 * e);
          w1[d] |= (((h >> 8) & 0xFu) | ((h >> 20) & 0xF0u)) << (4 * e);
        }
      }
      uint4 *o = (uint4 *)(x4 + ((s0 / 32 + q) * Lpad + c0 + 2 * cp) * 16);
      o[0] = make_uint4(w0[0], w0[1], w0[2], w0[3]);
      o[1] = make_uint4(w1[0], w1[1], w1[2], w1[3]);
    }
  }
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int u = tid + 256 * k;
    if (WHAT & PACK_AXT) {
      const int g = u & 7, cp = u >> 3;
      if (c0 + 2 * cp < Lpad) {
        unsigned w0[4], w1[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
          w0[d] = w1[d] = 0u;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const unsigned h = t16[(g * 16 + d * 4 + e) * 66 + cp];
            w0[d] |= (h & 0xFFu) << (8 * e);
            w1[d] |= (h >> 8) << (8 * e);
          }
        }
        uint8_t *o = axT + (c0 + 2 * cp) * Npad + s0 + 16 * g;
        *(uint4 *)o = make_uint4(w0[0], w0[1], w0[2], w0[3]);
        *(uint4 *)(o + Npad) = make_uint4(w1[0], w1[1], w1[2], w1[3]);
      }
    }
    if (WHAT & PACK_XT) {
      const int cp = u & 63, g = u >> 6;
      if (c0 + 2 * cp < Lpad) {
        unsigned w0[4], w1[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
          w0[d] = w1[d] = 0u;
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            const int s = g * 16 + d * 4 + e;
            const unsigned h = onehot4((unsigned)t16[s * 66 + cp] | ((unsigned)t16[(s + 1) * 66 + cp] << 16));
            w0[d] |= ((h & 0xFFu) | ((h >> 8) & 0xFF00u)) << (8 * e);
            w1[d] |= (((h >> 8) & 0xFFu) | ((h >> 16) & 0xFF00u)) << (8 * e);
          }
        }
        uint4 *o = (uint4 *)(xt + ((s0 / 16 + g) * Lpad + c0 + 2 * cp) * 16);
        o[0] = make_uint4(w0[0], w0[1], w0[2], w0[3]);
        o[1] = make_uint4(w1[0], w1[1], w1[2], w1[3]);
      }
    }
  }
}
#endif

struct rsg_timer { const char *name; hipEvent_t a, b; double host_ms; };   // host_ms >= 0: a host phase

struct rsg_ctx {
  int          device = 0;
  hipStream_t  stream = nullptr;
  int          timing = 0;
  int          ntimers = 0;
  rsg_timer    timers[RSG_MAX_TIMERS];
  int          gram_shape = 0;          // 0 = automatic
  int          gram_split = 1;          // split the last partial wave of Gram tiles along K
  int          batch_persistent = 1;    // batched kernels: persistent grids (1) or one group per work unit (0)
  int          defer = 0;               // queue status/min/max copies; the caller synchronises once
  int          skip_minmax = 0;         // a correction follows: the statistic's min / max are not needed
  int          ncu = 0;                 // compute units of the device
  void        *d_gscr = nullptr;  size_t gscr_cap = 0;   // Gram split partials
  void        *d_arena = nullptr; size_t arena_cap = 0;  // batched-null buffers (grow-only)
  // the last batched-null graph: instantiated once per launch geometry (sizes, tiles, tree
  // levels, scalar arguments, arena address: the bytes in bexec_sig), replayed by later calls
  // of the same geometry with new inputs
  hipGraphExec_t bexec = nullptr;
  std::vector<uint8_t> bexec_sig;
  int          bexec_hits = 0;          // replays that reused the cached graph (for tests)
  void        *d_hits = nullptr;  size_t hits_cap = 0;   // hit-list compaction (grow-only, entries)
  void        *h_hits = nullptr;                          // its pinned host mirror, same capacity
  void        *d_rank = nullptr, *h_rank = nullptr;       // rank histogram: slices, list, counters, pinned results
  int          rank_dirty = 0;                            // its dense counters to clear before the next call
  // small reusable device scratch (reductions)
  double      *d_red = nullptr;  size_t red_cap = 0;
  int         *d_flag = nullptr;
  // results of one scoring call, in the layout of h_pinned[0..4]: min, max, correction NaN flag
  // (int), COVavg, marginal validation flag (int); one copy brings them to the host, or the
  // chain's last kernel (the min / max reduction) writes them there itself (res_on_host).
  double      *d_res = nullptr;
  double      *h_pinned = nullptr;      // 64 doubles of pinned host staging
  double      *d_hres = nullptr;        // h_pinned as the device addresses it
  int          res_on_host = 0;
  // completion stamp: the min / max reduction writes hstamp to h_pinned[63] after the result
  // block (system-scope release)
  unsigned long long hstamp = 0;
  int          stamp_wait_us = 0;       // spin on the stamp this long before the stream is synchronised
  void        *d_small = nullptr;       // 64 KB of device scratch for small per-call tables
  // set for the duration of an allocation-free call (rsg_noalloc.hip): the Gram takes this
  // 32 x 32-column tile list instead of its cached one, and d_red is not grown past red_cap
  const int2  *tiles_fixed = nullptr;
  int          ntiles_fixed = 0;
  int          no_alloc = 0;
  RsgPool      tmp;                     // scratch of single calls, used on `stream` only
  std::shared_ptr<RsgPool> pool = std::make_shared<RsgPool>();   // buffers of the alignments made here
};

// Scratch of one call, used by work on the context's stream only.
struct RsgTmp {
  rsg_ctx *c;
  std::vector<void *> p;
  explicit RsgTmp(rsg_ctx *ctx) : c(ctx) {}
  RsgTmp(const RsgTmp &) = delete;
  RsgTmp &operator=(const RsgTmp &) = delete;
  ~RsgTmp() { for (void *q : p) c->tmp.put(q); }
  template <typename T> hipError_t get(T **out, size_t bytes)
  {
    void *q = nullptr;
    try { p.reserve(p.size() + 1); } catch (const std::bad_alloc &) { return hipErrorOutOfMemory; }
    const hipError_t e = c->tmp.get(&q, bytes);
    if (e == hipSuccess) { p.push_back(q); *out = (T *)q; }
    return e;
  }
};

struct rsg_msa {
  std::shared_ptr<RsgPool> pool;  // where its buffers come from
  int      device = 0;
  int64_t  N = 0, L = 0;        // sequences, columns
  int64_t  Npad = 0, Lpad = 0;  // padded to the Gram K-tile / column tile
  uint8_t *d_ax  = nullptr;     // N x L raw codes (row-major, as uploaded)
  uint8_t *d_axT = nullptr;     // packed forms (above), those of `packed` current
  uint8_t *d_xt  = nullptr;
  uint8_t *d_x4  = nullptr;
  int      packed = 0;
  double  *d_w   = nullptr;     // N weights (FP64); all 1 when unweighted
  int      weighted = 0;
  int      weights_ok = 1;    // every weight finite and >= 0 (else pp cannot validate)
  double   wsum = 0.;
  // split-BF16 weight parts of the weighted Gram: [3][Npad] bf16 bits
  uint16_t *d_wsplit = nullptr;
  int      nsplit_ready = 0;
  uint8_t *d_wq = nullptr;      // int8 weight limbs [Npad/16][4][16] and (after them) the FP64 scale
  int      wq_ready = 0;
  int      wq_counts = 0;       // the current counts come from the rounded weights (RSG_COUNTS_W8)
  double  *d_nsx = nullptr;     // with wq_counts: nseff of every pair (record index) in FP64
  double   wsum_q = 0.;         // sum of the rounded weights W * q_s
  // pair tables
  void    *d_cnt = nullptr;     // L x L x 16 (i<j records), kind below
  int      cnt_kind = -1;
  int      pm_fused = 0;          // the last FP4 Gram left the marginal partials in d_red
  size_t   cnt_bytes = 0;
  void    *d_cnt_u = nullptr;   // unit-weight counts kept for RAF when the main counts are weighted
  int      cnt_u_kind = -1;
  double  *d_pm = nullptr;      // L x 4
  double  *d_ps = nullptr;      // L x 5
  double  *d_lgc = nullptr;     // log table for integer counts, N+2 entries
  int64_t  lgc_n = -1;          // the N the log table holds (rebuilt when it differs)
  double  *d_cov = nullptr;     // L x L (FP64)
  double  *d_tmp = nullptr;     // L x L scratch (RAFS source)
  double  *d_rowx = nullptr;    // 2 L + 2: row means, row sums, COVavg
  double  *d_eval = nullptr;    // L x L E-values (kept on the device for the hit list)
  int      have_eval = 0;
  double   minCOV = 0., maxCOV = 0.;
  int      have_probs = 0, have_cov = 0;
};
template <typename T> static inline hipError_t rsg_msa_get(rsg_msa *m, T **p, size_t bytes) { return m->pool->get((void **)p, bytes); }

// Total weight the counts were formed with (ngap = total - nseff): the rounded weights' sum for
// counts from int8 weight limbs, so ngap is the gapped sequences' rounded weight
static inline double rsg_count_wsum(const rsg_msa *m) { return m->wq_counts ? m->wsum_q : m->wsum; }


// Host threads for planning work: the hardware's, at most 16 (one GPU's share of a node).
static inline int rsg_host_threads()
{
  const unsigned h = std::thread::hardware_concurrency();
  return (int)std::min(16u, std::max(1u, h));
}

// fn(k0, k1) over contiguous ranges of [0, n) of about equal total weight w(k) (total: their
// sum), one range per host thread (fewer when the total is under min_work per thread); the
// calling thread takes the first range.
template <class W, class F>
static void rsg_parallel_ranges(int n, int64_t total, W w, F fn, int64_t min_work = 1 << 16)
{
  const int nt = (int)std::max<int64_t>(1, std::min<int64_t>({(int64_t)rsg_host_threads(), (int64_t)n, total / min_work + 1}));
  std::vector<int> rb((size_t)nt + 1, n);
  rb[0] = 0;
  int64_t acc = 0;
  for (int k = 0, t = 1; k < n && t < nt; k++) {
    acc += w(k);
    while (t < nt && acc * nt >= total * t) rb[(size_t)t++] = k + 1;
  }
  std::vector<std::thread> th;
  for (int t = 1; t < nt; t++) th.emplace_back(fn, rb[(size_t)t], rb[(size_t)t + 1]);
  fn(rb[0], rb[1]);
  for (auto &x : th) x.join();
}

// ---- error helpers ----
static inline int rsg_fail(char *errbuf, const char *fmt, ...)
{
  if (errbuf) {
    va_list ap; va_start(ap, fmt);
    vsnprintf(errbuf, RSG_ERRBUFSIZE, fmt, ap);
    va_end(ap);
  }
  return RSG_FAIL;
}

#define HIPCHK(call) do { hipError_t e_ = (call); if (e_ != hipSuccess) \
  return rsg_fail(errbuf, "%s: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); } while (0)

// ---- timers ----
static inline void rsg_tstart(rsg_ctx *c, const char *name, int *slot)
{
  *slot = -1;
  if (!c->timing || c->ntimers >= RSG_MAX_TIMERS) return;
  if (c->timing == 2 && strncmp(name, "gram", 4) != 0) return;     // Gram launches only
  rsg_timer &t = c->timers[c->ntimers];
  if (!t.a) { hipEventCreate(&t.a); hipEventCreate(&t.b); }
  t.name = name; t.host_ms = -1.;
  hipEventRecord(t.a, c->stream);
  *slot = c->ntimers++;
}
static inline void rsg_tstop(rsg_ctx *c, int slot)
{
  if (slot >= 0) hipEventRecord(c->timers[slot].b, c->stream);
}
// a host-side phase measured by the caller (wall clock, ms), reported with the device timers
static inline void rsg_thost(rsg_ctx *c, const char *name, double ms)
{
  if (c->timing != 1 || c->ntimers >= RSG_MAX_TIMERS) return;
  rsg_timer &t = c->timers[c->ntimers++];
  t.name = name; t.host_ms = ms;
}

// ---- kernel launchers implemented in the .hip files ----
int rsg_noalloc_init(int device, char *errbuf);   // rsg_noalloc.hip: the scratch array's address
// packed forms, allocated and built if missing (and, on the same launch, a list of ntiles Gram tiles)
int rsg_need(rsg_ctx *c, rsg_msa *m, int what, char *errbuf, int2 *tiles = nullptr, int nb = 0, int ntiles = 0);
int rsg_msa_alloc(rsg_ctx *c, int64_t nseq, int64_t alen, rsg_msa **ret, char *errbuf);   // rsg_capi.hip
// pm_part (uint16 records only; nullptr = none): marginal partials of every 32 x 32 block
// (pm32 layout, rsg_device.h); pmflag: cleared for the marginal reduction that follows
int rsg_gram_counts_fp4(rsg_ctx *c, rsg_msa *m, void *d_out, int kind, double *pm_part, int *pmflag, char *errbuf);
int rsg_gram_counts_bf16(rsg_ctx *c, rsg_msa *m, int nsplit, float *d_out, char *errbuf);
int rsg_gram_counts_w8(rsg_ctx *c, rsg_msa *m, float *d_out, double *pm_part, int *pmflag, char *errbuf);
int rsg_probs_from_counts(rsg_ctx *c, rsg_msa *m, double tol, char *errbuf);
double *rsg_pm32_scratch(rsg_ctx *c, int64_t L, char *errbuf);
int rsg_stat(rsg_ctx *c, rsg_msa *m, int base, int cls, const double *allow16, int prec, char *errbuf);
int rsg_raf(rsg_ctx *c, rsg_msa *m, int rafs, const double *allow16, char *errbuf);
int rsg_correct(rsg_ctx *c, rsg_msa *m, int actype, int shiftnonneg, char *errbuf);
int rsg_reserve_scratch(rsg_ctx *c, int64_t L, bool pm_pass, char *errbuf);
int rsg_minmax(rsg_ctx *c, rsg_msa *m, char *errbuf);
int rsg_upload_weights_bf16(rsg_ctx *c, rsg_msa *m, int nsplit, char *errbuf);
int64_t rsg_npad(int64_t N);

// One simulated alignment: tree + output rows (rsg_sim.hip).
struct SimItem {
  int64_t N, L;           // leaves, columns
  int64_t tree_off;       // first internal node of this item in the concatenated tree arrays
  int64_t seq_off;        // offset of its (N-1) x L internal-node symbol rows
  int64_t leaf_off;       // offset of its N x L leaf output
  uint64_t seed; uint32_t stream; uint32_t gapthr;   // a leaf symbol is gapped if its tag-1 draw < gapthr
  int64_t col_blk0;       // first 64-column block of this item in the launch
  int64_t model_off;      // offset (doubles) of its 40-double GTR model
};
// Tree levels of a set of items: entries {item, internal node, left child, right child}
// grouped by depth.
// Host staging array without value-initialisation (every element is written before it is read).
template <class T> struct HostArr {
  std::unique_ptr<T[]> p;
  size_t n = 0;
  void alloc(size_t k) { p.reset(new T[k]); n = k; }
  T *data() { return p.get(); }
  const T *data() const { return p.get(); }
  size_t size() const { return n; }
  T &operator[](size_t i) { return p[i]; }
  const T &operator[](size_t i) const { return p[i]; }
};

struct SimLevels {
  HostArr<int4> ent;
  std::vector<int64_t> lev_ent0;     // entry offset of each level (size nlev + 1)
  std::vector<int64_t> lev_blocks;   // 64-column blocks of each level
  std::vector<int64_t> lev_maxl;     // longest alignment among each level's entries
};
int rsg_sim_levels(const SimItem *items, int nitems, const int *const *left, const int *const *right, SimLevels &lv, char *errbuf);
int rsg_sim_launch(rsg_ctx *c, const SimItem *d_items, int nitems, int64_t nodes, int64_t blocks,
                   const SimLevels &lv, const int4 *d_ent,
                   const double *d_ld, const double *d_rd, const double *d_models, uint32_t *d_cdf,
                   uint8_t *d_seqs, uint8_t *d_leaves, const uint8_t *root0, int64_t root_len);
int rsg_simulate_device(rsg_ctx *c, int nitems, const int64_t *N, const int64_t *L,
                        const int *left, const int *right, const double *ld, const double *rd,
                        const double *models, const uint64_t *seed, const uint32_t *stream, const double *gapfrac,
                        uint8_t *d_leaves, const int64_t *leaf_off, char *errbuf, const uint8_t *root0 = nullptr);
// one alignment's leaves to the host, the root drawn from pi (root == nullptr) or given (L codes)
int rsg_sim_one(rsg_ctx *c, const rsg_null_job *job, const uint8_t *root, uint8_t *leaves, char *errbuf);
int rsg_sim_pairs(rsg_ctx *c, const rsg_null_job *job, const int *ct, const double *model16, const uint8_t *root,
                  uint8_t *leaves, char *errbuf);

// R-scape's null of one alignment for R replicates at once (rsg_fitch.hip): the tree's levels
// (internal nodes grouped by depth, ent[lev0[k] .. lev0[k+1]) at depth k: {node, left child, right
// child, 2 * parent + side}) and the widest level, then one launch per kernel and depth covering
// every replicate.
struct FitchPlan {
  int64_t N = 0, L = 0;
  int m = 0, maxd = 0, maxw = 0;
  std::vector<int4> ent;
  std::vector<int> lev0;
};
// Device buffers of R replicates: ax (N x L codes), the tree's levels (ent: m), perm
// (R x L, read where rsg_fitch_host_perm), seeds (R), flag (1 where ax holds a code past 4; 0 before the first run),
// mask, all and inner (R x m x L: the internal nodes' state sets, states and shuffled rows), leaves
// (R x N x L: the null alignments), nsub (R x 2m x 25; null: not counted), cols (R x
// rsg_fitch_cols ints).
struct FitchDev {
  const uint8_t *ax;
  const int4 *ent;
  const int *perm;
  const uint64_t *seeds;
  int *flag;
  uint8_t *mask, *all, *inner, *leaves;
  int *nsub, *cols;
};
size_t rsg_fitch_cols(const FitchPlan &P);
int rsg_fitch_plan(int64_t N, int64_t L, const int *left, const int *right, FitchPlan &P, char *errbuf);
bool rsg_fitch_host_perm(const FitchPlan &P);              // whether the launch reads D.perm
void rsg_fitch_perm(uint64_t seed, int64_t L, int *perm);
int rsg_fitch_launch(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R);
int rsg_fitch_ancestral(rsg_ctx *c, const FitchPlan &P, const FitchDev &D, int R);

// Batched pipeline: per-item descriptor of RSG_BDESC int64 fields
// {N, L, Npad, Lpad, off_x4, off_cnt, off_cov, off_pm, off_rows, (unused), off_leaf, blk0_pack,
//  blk0_stat, blk0_el, nb32, group, blk0_hist, off_pm32 (marginal partials), blk0_col16
//  (16-column blocks), blk0_row}
#define RSG_BDESC 20
// Surrogate features (rsg_features.hip): column statistics of items {x4 panel offset, N,
// Npad, L, first 4-column block, Lpad} into 36 uint64 counters per item; the host turns them into
// RSG_NULL_NFEAT floats.
int rsg_feat_launch(rsg_ctx *c, const int64_t *d_items, int nitems, int64_t nblocks, const uint8_t *d_base,
                    unsigned long long *d_out);
void rsg_feat_finish(const unsigned long long *cnt, int64_t N, int64_t L, const int *left, const int *right,
                     const double *ld, const double *rd, float *f);
// Large alignments of a batch use 64 x 32-column tiles (4 waves, 512-sequence K tiles), the
// others 32 x 32-column tiles (2 waves, 128-sequence K tiles).
static inline bool rsg_batch_big_tiles(int64_t N, int64_t L) { return L >= 256 && N >= 256; }
// d_queue: 128 ints of device memory for the persistent kernel's per-XCD tile counters (unused
// by the one-work-group-per-tile launch, rsg_ctx::batch_persistent = 0).
int rsg_gram_batch_launch(rsg_ctx *c, const int4 *d_big, int nbig, const int4 *d_small, int nsmall,
                          const int64_t *d_desc, const uint8_t *d_x4, uint16_t *d_cnt, double *d_pm_part, int pm_field,
                          int *d_queue);
