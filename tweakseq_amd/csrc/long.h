// Long pairs (tens of thousands of residues per side), global alignment, int32.
//
// Forward pass (long_fwd_kernel): the strips of all long pairs, 512 query rows
// each (64 lanes x 8 rows, strip.h without direction bits: five operations a
// cell), form one device work queue, pair-major; a wave takes the next strip,
// which trails the one above on whichever CU it landed, through bottom rows in
// device memory whose entries are their own flags (strips.h).  Every strip a
// wave waits on was dequeued before its own, by a wave that is running, so
// the pipeline cannot deadlock.  Two waves per SIMD (LONG_WAVES per CU): they
// fill its issue slots, and need 204 registers each; with 128, for four, the
// sweep spills and 48 pairs take 54 ms, with one wave 30 ms, with two 19 ms.
//
// The forward pass is score only.  The bottom rows stay, which makes every
// 512th row a checkpoint, and when a traceback follows the column (G, E of
// every row) at every CKX-th column is kept too.
//
// Traceback (long_tb_kernel, one workgroup of 4 waves per pair) walks the
// matrix from (m, n) in regions.  A region is the rows of one forward strip up
// to the walk's row and a band of columns ending at the walk's column and
// starting at a column checkpoint far enough left for a path near the diagonal
// to leave through the strip's top.  The region is recomputed with direction
// codes (strip.h, 4 strips of 128 rows, one per wave, pipelined through LDS)
// and one wave walks it a CIGAR run at a time (walk.h) until the path leaves
// through the top or the left; the next region starts there.  The recomputed
// cells are the forward pass's cells, so the walk is the full-matrix walk of
// the specification (oracle/gotoh.c), bit for bit.  Small regions: their time
// is columns + 64 strips of dependent steps, and the columns beyond the
// diagonal (LMARGIN, half a CKX) are what a region computes for nothing.
//
// One after the other, the regions of the longest pair (120 us each) would set
// the time of a batch of few pairs.  So where the path will pass is guessed
// first: at every strip's bottom row, the column of the largest H near the
// diagonal (long_cross_kernel) -- for related sequences on the path, or next
// to it.  A region around every guess is recomputed by a workgroup of its own
// (long_regions_kernel), all over the GPU at once, and the walk uses such a
// region wherever it contains the walk's cell (a region's codes are exact
// whatever made it), else recomputes one itself as above.  Batches whose
// pairs fill the GPU by themselves do without.
//
// 48 DNA pairs of 10,000 to 60,000 with CIGARs: forward 36 -> 19 ms, traceback
// 63 -> 17 ms with small regions and run walks, -> 2.8 ms with regions ahead;
// 256 of 10,000 to 100,000: 449 -> 277 -> 242 ms a run.  (Before: plain recurrence,
// progress counters every 64 columns, regions of 4,096 rows on 8 waves, a walk
// of one thread.)
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"
#include "longplan.h"
#include "strips.h"
#include "traceback.h"
#include "walk.h"

namespace ta {

constexpr int LONG_WAVES = 8;             // forward waves per CU
constexpr int LAHEAD = 128;               // columns of a region ahead on either side of its guesses
constexpr int LGUESS = 8192;              // columns on either side of the diagonal a guess is looked for in
static_assert(LST == GWAVE * LR && strip_spd(2) == 4, "shapes of longplan.h");

struct LongPair {
  uint64_t a_off, b_off;  // residue codes (16-byte aligned, 32 bytes readable past the end)
  uint64_t ring;          // (G, F) entries: S - 1 rows of T + 8
  uint64_t colck;         // (G, E) entries: (n - 1) / CKX columns x S * LST rows
  int32_t pid, m, n, S, T;
  int32_t item0;          // its first queue item
};

struct LongItem {
  int32_t lp, s;  // long pair, strip
};

struct LongArgs {
  const LongPair *lp;
  int32_t nlp;
  const LongItem *items;
  int32_t nitems;
  int32_t *ctr;         // [0] forward items taken, [1] traceback pairs taken
  const int8_t *table;  // Kp x Kp
  int32_t Kp;
  const uint8_t *codes;
  int2 *ring, *colck;
  uint32_t *wpl;        // traceback workgroups: direction codes, LPLANES dwords each
  uint32_t *ahead;      // codes of the regions ahead, an item's at LPLANES (item - ahead0); null: none
  int32_t *cross;       // per item: the column (1-based) its strip's bottom row is guessed to be left at
  int32_t ahead0;
  const PairDev *pd;
  FillOut *fo;
  ResultDev *res;
  char *cig;
  int32_t open, ext;
  int32_t ckpt_on;      // keep column checkpoints (a traceback follows)
  int32_t spin_limit;   // looks before a wait gives up
  int32_t *err;         // set when a wait gave up (results are then invalid)
};

// LDS of a forward wave, after what strips.h lays out: the score slot, then a
// ring of column codes (1,024 columns, the first 8 repeated after the last).
template <int NC, bool BYTES>
constexpr int SL_CODES = SL_SLOT + strip_slot_bytes(LR, NC, BYTES);
template <int NC, bool BYTES>
constexpr int long_fwd_lds = SL_CODES<NC, BYTES> + 1024 + 16;

template <int NC_, bool BYTES_>
struct LongIO : StripRingIO {
  static constexpr bool TB = false, KEEP = true, BYTES = BYTES_;
  static constexpr int NC = NC_;
  uint32_t slot_add;
  const uint8_t *cb;        // the pair's column codes
  int n, K;
  uint32_t next = 0;        // this lane's 4 codes of the next 256 columns
  int2 *ck;                 // this lane's rows in column checkpoint 0; null: none are kept
  uint64_t ck_step;         // entries per checkpoint

  __device__ __forceinline__ void ahead_codes(int col) {
    const int c = col + 4 * (int)(threadIdx.x & 63), left = n - c;
    const uint32_t keep = left >= 4 ? 0xffffffffu : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
    next = ((left > 0 ? *(const uint32_t *)(cb + c) : 0u) & keep) | ((0x01010101u * (uint32_t)K) & ~keep);
  }
  __device__ __forceinline__ uint64_t codes(int b) {
    uint8_t *w = lds + SL_CODES<NC, BYTES>;
    const int lane = threadIdx.x & 63;
    if ((b & 31) == 0) {  // 256 more columns
      const int at = (8 * b + 4 * lane) & 1023;
      *(uint32_t *)(w + at) = next;
      if (at < 8) *(uint32_t *)(w + 1024 + at) = next;
      ahead_codes(8 * b + 256);
    }
    uint64_t v;
    __builtin_memcpy(&v, w + ((8 * b - lane) & 1023), 8);
    return v;
  }
  __device__ __forceinline__ void planes(uint32_t) const {}
  __device__ __forceinline__ bool keeps(int b) const {
    const int hi = (8 * b + 8) / CKX * CKX;  // the last checkpoint column a lane may be at
    return ck && hi >= CKX && hi >= 8 * b - 62;
  }
  template <int PR>
  __device__ __forceinline__ void column(int c, const int (&G)[PR], const int (&E)[PR]) const {
    if (ck && c >= 0 && ((c + 1) & (CKX - 1)) == 0 && c + 1 < n) {
      int4 *d = (int4 *)(ck + (uint64_t)((c + 1) / CKX - 1) * ck_step);
#pragma unroll
      for (int k = 0; k < PR; k += 2) d[k / 2] = make_int4(G[k], E[k], G[k + 1], E[k + 1]);
    }
  }
};

// Before a forward pass: every bottom-row entry empty, the queue heads at 0.
template <int = 0>
__global__ void long_init_kernel(uint4 *ring, uint64_t n16, int32_t *ctr) {
  const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
  const uint32_t e = (uint32_t)STRIP_EMPTY;
  for (uint64_t k = tid; k < n16; k += stride) ring[k] = make_uint4(e, e, e, e);
  if (tid < 2) ctr[tid] = 0;
}

// Forward pass: one wave per workgroup, strips off the device queue.
// BYTES: scores plus |open| + |ext| fit in int8.
template <int NC, bool BYTES>
__global__ __launch_bounds__(64, 2) void long_fwd_kernel(LongArgs A) {
  extern __shared__ __align__(256) uint8_t lds[];
  const int lane = threadIdx.x & 63, K = A.Kp - 1;
  for (int x = lane; x < 1024; x += 64) {
    const int r = x >> 5, c = x & 31;
    lds[SL_TAB + x] = r < K && c < K ? (uint8_t)A.table[r * A.Kp + c] : (uint8_t)PAD_SCORE;
  }
  ((int *)(lds + SL_CONST))[lane & 31] = (lane & 31) < 16 ? 0 : 2 * (A.open - A.ext);
  bool lost = false;
  for (;;) {
    int it = 0;
    if (lane == 0) it = atomicAdd(&A.ctr[0], 1);
    it = __builtin_amdgcn_readfirstlane(it);
    if (it >= A.nitems) break;
    const LongItem w = A.items[it];
    const LongPair P = A.lp[w.lp];
    const int s = w.s, r0 = (s * 64 + lane) * LR;
    const uint8_t *line[LR];
#pragma unroll
    for (int k = 0; k < LR; ++k) line[k] = lds + SL_TAB + 32 * (r0 + k < P.m ? A.codes[P.a_off + r0 + k] : 31);
    strip_slot<LR, NC, BYTES>(lds + SL_SLOT, line, K, -A.open - A.ext, A.ext - A.open);
    ((uint32_t *)(lds + SL_CODES<NC, BYTES>))[240 + (lane & 15)] = 0x01010101u * (uint32_t)K;  // columns -64 .. -1: pads
    LongIO<NC, BYTES> io;
    io.lds = lds;
    io.slot_add = 0x01010101u * (((uint32_t)(uintptr_t)(lds_u8 *)lds + SL_SLOT) >> 8);
    io.rin = s ? A.ring + P.ring + (uint64_t)(s - 1) * (P.T + 8) : nullptr;
    io.rout = A.ring + P.ring + (uint64_t)s * (P.T + 8);
    io.cols = P.T - 63;
    io.spin_limit = A.spin_limit;
    io.err = A.err;
    io.lost = lost;
    io.cb = A.codes + P.b_off;
    io.n = P.n;
    io.K = K;
    io.ck = A.ckpt_on && P.n > CKX ? A.colck + P.colck + r0 : nullptr;
    io.ck_step = (uint64_t)P.S * LST;
    io.ahead_codes(0);
    asm volatile("" ::: "memory");  // staged by all lanes (a wave's LDS accesses keep their order)
    if (io.rin) io.look();
    StripEnd end;
    strip_sweep<LR, false>(io, s, s + 1 == P.S, P.m, P.n, P.T, A.open, A.ext, end);
    lost = io.lost;
    if (end.has) {
      FillOut o;
      o.score = end.h; o.end_i = P.m; o.end_j = P.n; o.flags = 1 | 4;  // int32, long path
      A.fo[P.pid] = o;
    }
  }
}

// LDS of a traceback workgroup.  Its strips share one ring: each stores its
// bottom row over the one it read, 63 columns behind.
enum { LT_TAB = 0, LT_SYNC = 1024, LT_SLOTS = 1280, LT_CODES = LT_SLOTS + LTW * strip_slot_bytes(2),
       LT_RING = LT_CODES + ((64 + LREG_T + 32 + 15) & ~15), LT_WIN = LT_RING + (LREG_T + 80) * 8,
       LONG_TB_LDS = LT_WIN + StripWindow<2>::WL * StripWindow<2>::WD * 4 };
// Its sync words.
enum { LS_PAIR = 0, LS_I = 1, LS_J = 2, LS_PROG = 4, LS_READY = 25, LS_ZERO = 32, LS_EDGE = 48 };

// What a traceback workgroup's regions share.
__device__ __forceinline__ void long_tb_setup(const LongArgs &A, uint8_t *lds, int32_t *sy) {
  static_assert(LT_SLOTS % STRIP_ROW == 0 && LT_SLOTS + LTW * strip_slot_bytes(2) <= 256 * STRIP_ROW, "slot rows");
  const int tid = threadIdx.x, K = A.Kp - 1;
  for (int x = tid; x < 1024; x += 64 * LTW) {
    const int r = x >> 5, c = x & 31;
    lds[LT_TAB + x] = r < K && c < K ? (uint8_t)A.table[r * A.Kp + c] : (uint8_t)PAD_SCORE;
  }
  if (tid < 64) sy[tid] = tid == LS_READY ? 0x7fffffff : tid >= LS_EDGE ? 2 * (A.open - A.ext) : 0;
  if (tid < 64) lds[LT_CODES + tid] = (uint8_t)K;
}

// A region's codes: rows of strip beta up to row i (1-based), columns
// c_left + 1 .. c_left + ncols (c_left: 0 or a checkpoint), by the workgroup.
__device__ __forceinline__ void long_region(const LongArgs &A, const LongPair &P, uint8_t *lds, int32_t *sy, int beta,
                                            int i, int c_left, int ncols, uint32_t *pl, bool &lost) {
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), K = A.Kp - 1;
  const int top = beta * LST, T = (ncols + 63 + 7) & ~7, S = (i - top + 127) / 128;
  uint8_t *bcode = lds + LT_CODES;
  int2 *ring = (int2 *)(lds + LT_RING);
  const uint8_t *cb = A.codes + P.b_off + c_left;
  for (int x = 4 * tid; x < T + 16; x += 256 * LTW) {
    const int left = ncols - x;
    const uint32_t keep = left >= 4 ? 0xffffffffu : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
    *(uint32_t *)(bcode + 64 + x) =
        ((left > 0 ? *(const uint32_t *)(cb + x) : 0u) & keep) | ((0x01010101u * (uint32_t)K) & ~keep);
  }
  if (beta) {  // the row above: the forward strip's bottom row
    const int2 *row = A.ring + P.ring + (uint64_t)(beta - 1) * (P.T + 8) + c_left;
    for (int x = tid; x < ncols; x += 64 * LTW) ring[64 + x] = row[x];
  }
  if (tid < LTW) sy[LS_PROG + tid] = 0;
  __syncthreads();
  if (wv < S) {
    const int sa = top / 128 + wv, r0 = (sa * 64 + lane) * 2;  // strips of 128 rows, counted over the pair
    const uint8_t *line[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) line[k] = lds + LT_TAB + 32 * (r0 + k < P.m ? A.codes[P.a_off + r0 + k] : 31);
    const int slot = LT_SLOTS + wv * strip_slot_bytes(2);
    strip_slot<2>(lds + slot, line, K, -A.open - A.ext, A.ext - A.open);
    struct IO : StripGroupIO {
      const int2 *left;
    } io;
    io.left = c_left ? A.colck + P.colck + (uint64_t)(c_left / CKX - 1) * P.S * LST + r0 : nullptr;
    io.bcode = bcode + 64 - lane;
    io.slot_add = 0x01010101u * ((uint32_t)((uint32_t)(uintptr_t)(lds_u8 *)lds + slot) >> 8);
    io.status = A.err;
    io.gave_up = 1;
    io.spin_limit = 1 << 22;
    io.lost = lost;
    io.pin = sy + (wv ? LS_PROG + wv - 1 : LS_READY);
    io.pout = sy + LS_PROG + wv;
    io.rin = lane ? (int2 *)(sy + LS_ZERO) : wv || beta ? ring + 64 : (int2 *)(sy + LS_EDGE);
    io.rin_step = lane == 0 && (wv || beta) ? 8 : 0;
    io.rout = ring;
    io.need0 = wv << 20;
    io.s = wv;
    io.cols = T - 63;
    io.pl = pl + (uint64_t)wv * (T / strip_spd(2)) * 64 + lane;
    io.pl_step = 64;
    asm volatile("" ::: "memory");  // staged by all lanes (a wave's LDS accesses keep their order)
    StripEnd end;
    strip_sweep<2, false>(io, sa, wv + 1 == S, i, ncols, T, A.open, A.ext, end);
    lost = io.lost;
  }
  __syncthreads();  // the codes are in place
}

// The columns of the region ahead of strip beta (item x): from a checkpoint
// left of where the strip above is guessed to be left, to right of this one's
// guess, at most LREG of them.
__device__ __forceinline__ void long_ahead_cols(const LongArgs &A, const LongPair &P, int beta, int &c_left, int &right) {
  const int32_t *cross = A.cross + P.item0 + beta;
  const int here = cross[0], up = beta ? cross[-1] : 0;
  right = here + LAHEAD < P.n ? here + LAHEAD : P.n;
  const int from = (up < here ? up : here) - LAHEAD;
  c_left = from <= 0 ? 0 : from / CKX * CKX;
  if (right - c_left > LREG) c_left = (right - LREG + CKX - 1) / CKX * CKX;
}

// Guesses: per queue item, the column of the largest H of its strip's bottom
// row near the diagonal (the last strip's: n).  Also clears the pair counter
// of the traceback that follows.
template <int = 0>
__global__ __launch_bounds__(256) void long_cross_kernel(LongArgs A) {
  __shared__ int2 part[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const LongItem it = A.items[blockIdx.x];
  const LongPair P = A.lp[it.lp];
  if (blockIdx.x == 0 && tid == 0) A.ctr[1] = 0;
  if (it.s == P.S - 1) {
    if (tid == 0) A.cross[P.item0 + it.s] = P.n;
    return;
  }
  const int2 *row = A.ring + P.ring + (uint64_t)it.s * (P.T + 8);
  const int mid = (int)((int64_t)P.n * (it.s + 1) * LST / P.m);
  const int lo = mid > LGUESS ? mid - LGUESS : 0, hi = mid + LGUESS < P.n ? mid + LGUESS : P.n;
  int best = INT32_MIN, col = lo;
  for (int x = lo + tid; x < hi; x += 256) {
    const int h = row[x].x + A.ext * x;
    if (h > best) { best = h; col = x; }
  }
  auto join = [&](int h, int c) {
    if (h > best || (h == best && c < col)) { best = h; col = c; }
  };
#pragma unroll
  for (int w = 32; w >= 1; w >>= 1) {
    const int h = __shfl_xor(best, w, 64), c = __shfl_xor(col, w, 64);
    join(h, c);
  }
  if (lane == 0) part[tid >> 6] = make_int2(best, col);
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) join(part[w].x, part[w].y);
    A.cross[P.item0 + it.s] = col + 1;
  }
}

// The regions ahead, a workgroup per queue item.
template <int = 0>
__global__ __launch_bounds__(64 * LTW, 4) void long_regions_kernel(LongArgs A) {
  extern __shared__ __align__(256) uint8_t lds[];
  int32_t *sy = (int32_t *)(lds + LT_SYNC);
  const LongItem it = A.items[blockIdx.x];
  const LongPair P = A.lp[it.lp];
  long_tb_setup(A, lds, sy);
  __syncthreads();
  int c_left, right;
  long_ahead_cols(A, P, it.s, c_left, right);
  const int i = (it.s + 1) * LST < P.m ? (it.s + 1) * LST : P.m;
  bool lost = false;
  long_region(A, P, lds, sy, it.s, i, c_left, right - c_left, A.ahead + (uint64_t)(P.item0 + it.s - A.ahead0) * LPLANES,
              lost);
}

// Traceback: one workgroup of LTW waves per pair (pairs off a counter).
template <int = 0>
__global__ __launch_bounds__(64 * LTW) void long_tb_kernel(LongArgs A) {
  extern __shared__ __align__(256) uint8_t lds[];
  int32_t *sy = (int32_t *)(lds + LT_SYNC);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t *const own = A.wpl + (uint64_t)blockIdx.x * LPLANES;
  long_tb_setup(A, lds, sy);
  bool lost = false;
  for (;;) {
    __syncthreads();
    if (tid == 0) sy[LS_PAIR] = atomicAdd(&A.ctr[1], 1);
    __syncthreads();
    const int q = __builtin_amdgcn_readfirstlane(sy[LS_PAIR]);
    if (q >= A.nlp) break;
    const LongPair P = A.lp[q];
    const PairDev pd = A.pd[P.pid];
    WaveRuns rw;  // wave 0's
    rw.end = (uint32_t *)(A.cig + pd.cig_off + pd.cig_cap);
    rw.cap = pd.cig_cap / 4;
    int i = P.m, j = P.n, state = 0;
    bool failed = false;
    while (i > 0 && j > 0) {
      // Region: rows of the strip holding row i, columns c_left + 1 .. j (or more).
      const int beta = (i - 1) / LST, top = beta * LST;
      int c_left = 0, right = 0;
      const uint32_t *pl = own;
      if (A.ahead) {
        long_ahead_cols(A, P, beta, c_left, right);
        pl = A.ahead + (uint64_t)(P.item0 + beta - A.ahead0) * LPLANES;
      }
      if (j <= c_left || j > right) {  // no region ahead, or not this cell in it
        c_left = j - (i - top) - LMARGIN;
        c_left = c_left <= 0 ? 0 : (c_left / CKX) * CKX;
        right = j;
        pl = own;
        long_region(A, P, lds, sy, beta, i, c_left, right - c_left, own, lost);
      }
      const int T = (right - c_left + 63 + 7) & ~7;
      if (wv == 0) {
        StripWindow<2> src{pl, (uint32_t *)(lds + LT_WIN), T, -1, -1};
        int li = i - top, lj = j - c_left, steps = 0;
        src.refill(li, lj);
        if (wave_walk<WALK_GLOBAL>(src, rw, li, lj, state, INT32_MAX, steps) == WALK_GAVE_UP) {
          failed = true;  // cannot happen: end the walk rather than loop
          li = lj = 0;
        }
        if (lane == 0) {
          sy[LS_I] = failed ? 0 : top + li;
          sy[LS_J] = failed ? 0 : c_left + lj;
        }
      }
      __syncthreads();
      i = __builtin_amdgcn_readfirstlane(sy[LS_I]);
      j = __builtin_amdgcn_readfirstlane(sy[LS_J]);
      // Read by every wave before wave 0 stores the next cell: where the next
      // region is one computed ahead, no other barrier lies between the two.
      __syncthreads();
    }
    if (wv == 0) {
      if (i == 0 && j > 0) rw.emit(1, j);
      if (j == 0 && i > 0) rw.emit(2, i);
      failed |= !rw.finish();
      const FillOut f = A.fo[P.pid];
      ResultDev r;
      r.score = f.score;
      r.a_begin = 0; r.a_end = P.m - 1; r.b_begin = 0; r.b_end = P.n - 1;
      const int nr = rw.n < rw.cap ? rw.n : rw.cap;
      r.cigar_off = (int64_t)(pd.cig_off + pd.cig_cap) - 4 * nr;
      r.cigar_len = 4 * nr;
      r.flags = f.flags | (failed ? WALK_FAILED : 0);
      if (lane == 0) A.res[P.pid] = r;
    }
  }
}

}  // namespace ta
