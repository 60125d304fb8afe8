// A batch of few pairs, for latency: every strip of every pair on a wave of
// its own, anywhere on the GPU.
//
// The fill of fill.h gives a task (up to two pairs) one wave, or the four
// fill waves of one workgroup, whose time on a long pair is then the run's:
// 16 pairs of up to 5,000 residues kept 16 of 256 CUs busy.  Here a pair's
// strips (64 lanes x 2 rows, strip.h) are items of one queue, pair by
// pair, and trail each other by about 100 columns whichever CUs they run on.
//
// A strip's bottom row goes to device memory, a row of (G, F) entries per
// strip, each entry one 8-byte device-coherent store and never stored twice;
// before the run every entry holds a value no strip stores (STRIP_EMPTY), so
// an entry is its own flag: the strip below reads 64 entries ahead at once,
// takes the leading ones that are there into its LDS and looks again two
// blocks later.  No counter, and no wait for a store, sits between the two.
// Every strip a wave waits on was taken from the queue before its own by a
// running wave, so the pipeline cannot deadlock; waits are bounded.
//
// What it takes (from run to results in place, one wave or workgroup per task
// against this): 16 pairs of 50 to 5,000 residues, global, 10.6 -> 1.13 ms a
// call; one 1,500 x 1,571 pair 2.88 -> 0.43 ms; 1,024 local pairs of 300 to
// 600 890 -> 423 us.
//
// Direction codes go to device memory, and a second kernel walks each pair
// back with a wave of its own, a CIGAR run at a time (walk.h), over windows
// of the codes staged in LDS.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"
#include "strip.h"
#include "traceback.h"
#include "walk.h"

namespace ta {

constexpr int STRIPS_MAXN = 32768;    // columns a pair may have (its codes are staged in LDS)
constexpr int STRIPS_PR = 2;          // rows per lane (4: as fast where SIMDs are short, slower where they are not)
constexpr int STRIPS_PER_SIMD = 8;    // most strips per SIMD a batch takes this form with (plan_strips)
constexpr int STRIP_EMPTY = INT32_MIN;

struct StripPair {
  uint64_t a_off, b_off;  // residue codes (16-byte aligned, 32 bytes readable past the end)
  uint64_t ring;          // (G, F) entries: S - 1 rows of T + 8
  uint64_t planes;        // direction codes, dwords: S x T / SPD x 64
  int32_t pid, m, n, S, T;
  int32_t i16;            // the pair is one the packed int16 lanes would take (its flags say so)
};

struct StripItem {
  int32_t sp, s;
};

struct StripsArgs {
  const StripPair *sp;
  const StripItem *items;
  int32_t nitems, npairs;
  int32_t *ctr;
  const int8_t *table;    // Kp x Kp
  int32_t Kp;
  const uint8_t *codes;
  int2 *ring;
  uint32_t *planes;
  uint64_t *best;         // local, per pair: its best cell, packed (strips_key), 0 none
  int32_t *score;         // global, per pair
  int32_t open, ext, sat_limit, spin_limit;
  int32_t *err;           // | 8: a wait gave up
  TbArgs tb;              // results
  int32_t bcode_bytes;    // LDS for column codes
};

// Best cells compare by h, then the smaller i, then the smaller j (each < 2^20).
__device__ __forceinline__ uint64_t strips_key(int h, int i, int j) {
  return ((uint64_t)h << 40) | ((uint64_t)(0xFFFFF - i) << 20) | (uint64_t)(0xFFFFF - j);
}

// LDS: 32-byte table lines, the ring window (128 entries), 16 words of zeros
// and borders, the score slot, the column codes.
enum { SL_TAB = 0, SL_RING = 1024, SL_CONST = 2048, SL_SLOT = 2304 };
__host__ __device__ constexpr int strips_lds(int bcode_bytes) {
  return SL_SLOT + strip_slot_bytes(STRIPS_PR) + bcode_bytes;
}

// A strip whose neighbours are anywhere on the GPU: bottom rows in device
// memory, entries that are their own flags, and a window of the row above in LDS.
struct StripRingIO : StripIODefaults {
  uint8_t *lds;
  const int2 *rin;          // the strip above's entries, column 0 on; null above the first strip
  int2 *rout;               // this strip's
  int cols, spin_limit;     // cols: columns the strip above stores
  int32_t *err;
  int avail = 0;            // columns in the LDS window
  int2 ahead;               // the 64 entries from `avail` on, as of the last look
  int age = 0;
  bool lost = false;

  __device__ __forceinline__ void look() {
    const int col = avail + (int)(threadIdx.x & 63);
    ahead = make_int2(0, 0);  // past the last stored column: zeros
    if (col < cols) {
      const uint64_t v = __hip_atomic_load((const uint64_t *)(rin + col), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      ahead = make_int2((int)(uint32_t)v, (int)(uint32_t)(v >> 32));
    }
  }
  // The leading entries of the last look that are there, into the window.
  __device__ __forceinline__ void take() {
    const uint64_t none = __ballot(ahead.x == STRIP_EMPTY);
    const int k = none ? __builtin_ctzll(none) : 64, lane = threadIdx.x & 63;
    if (lane < k) ((int2 *)(lds + SL_RING))[(avail + lane) & 127] = ahead;
    avail += k;
  }
  __device__ __forceinline__ void peek() {}
  __device__ __forceinline__ void await(int b) {
    if (!rin || lost) return;
    const int want = 8 * b + 8;
    // every second block, and whenever columns are missing; the window holds
    // at most 128 columns, from this block's on
    if (b > 0 && avail >= want && (++age & 1)) return;
    if (avail + 64 <= 8 * b + 120) {
      take();
      int spins = 0;
      while (avail < want) {
        look();
        take();
        if (++spins > spin_limit) {
          if ((threadIdx.x & 63) == 0) atomicOr(err, 8);
          lost = true;
          break;
        }
        // a strip that has not begun may wait for long, beside hundreds like it
        if (avail < want && b == 0) __builtin_amdgcn_s_sleep(32);
      }
      look();
    }
  }
  __device__ __forceinline__ void tops(int b, int half, int (&g)[8], int (&f)[8]) const {
    const int lane = threadIdx.x & 63, q = 4 * half;
    const int4 *r = (const int4 *)(lds + (lane ? SL_CONST : rin ? SL_RING + ((8 * b + q) & 127) * 8 : SL_CONST + 64));
    const int4 v = r[0], w = r[1];
    g[q] = v.x; f[q] = v.y; g[q + 1] = v.z; f[q + 1] = v.w;
    g[q + 2] = w.x; f[q + 2] = w.y; g[q + 3] = w.z; f[q + 3] = w.w;
  }
  __device__ __forceinline__ void bottom(int b, const int (&g)[8], const int (&f)[8]) const {
    if ((threadIdx.x & 63) == 63) {
      int2 *r = rout + 8 * b - 63;
      auto put = [&](int q) {
        __hip_atomic_store((uint64_t *)(r + q), (uint64_t)(uint32_t)g[q] | ((uint64_t)(uint32_t)f[q] << 32),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      if (b >= 8) {
#pragma unroll
        for (int q = 0; q < 8; ++q) put(q);
      } else if (b == 7) {  // column 0; the ones before are left of the border
        put(7);
      }
    }
  }
};

struct StripsIO : StripRingIO {
  const uint8_t *bcode;
  uint32_t slot_add;
  __amdgpu_buffer_rsrc_t pl;
  uint32_t pl_at = 0;

  __device__ __forceinline__ uint64_t codes(int b) const {
    uint64_t w;
    __builtin_memcpy(&w, bcode + 8 * b, 8);
    return w;
  }
  __device__ __forceinline__ void planes(uint32_t dw) {
    __builtin_amdgcn_raw_buffer_store_b32(dw, pl, 4u * (threadIdx.x & 63), pl_at, 0);
    pl_at += 256;
  }
};

template <bool LOCAL>
__global__ __launch_bounds__(64) void strips_kernel(StripsArgs A) {
  constexpr int PR = STRIPS_PR;
  extern __shared__ __align__(256) uint8_t lds[];
  constexpr int SPD = strip_spd(PR);
  const int lane = threadIdx.x & 63, K = A.Kp - 1;
  for (int x = lane; x < 1024; x += 64) {
    const int r = x >> 5, c = x & 31;
    lds[SL_TAB + x] = r < K && c < K ? (uint8_t)A.table[r * A.Kp + c] : (uint8_t)PAD_SCORE;
  }
  ((int *)(lds + SL_CONST))[lane & 31] = (lane & 31) < 16 || LOCAL ? 0 : 2 * (A.open - A.ext);
  uint8_t *bcode = lds + SL_SLOT + strip_slot_bytes(PR);
  bool lost = false;
  for (;;) {
    int it = 0;
    if (lane == 0) it = atomicAdd(A.ctr, 1);
    it = __builtin_amdgcn_readfirstlane(it);
    if (it >= A.nitems) break;
    const StripItem w = A.items[it];
    const StripPair P = A.sp[w.sp];
    const int s = w.s, m = P.m, n = P.n, T = P.T;
    // column codes: 64 pads, the columns, pads
    lds[SL_SLOT + strip_slot_bytes(PR) + lane] = (uint8_t)K;
    const uint8_t *cb = A.codes + P.b_off;
    for (int x = 16 * lane; x < T + 16; x += 1024) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (x < n) v = *(const uint4 *)(cb + x);
      uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int left = n - x - 4 * q;  // codes of this dword inside the sequence
        const uint32_t keep = left >= 4 ? 0xffffffffu : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
        u[q] = (u[q] & keep) | ((0x01010101u * (uint32_t)K) & ~keep);
      }
      *(uint4 *)(bcode + 64 + x) = make_uint4(u[0], u[1], u[2], u[3]);
    }
    const int r0 = (s * 64 + lane) * PR;
    const uint8_t *line[PR];
#pragma unroll
    for (int k = 0; k < PR; ++k) line[k] = lds + SL_TAB + 32 * (r0 + k < m ? A.codes[P.a_off + r0 + k] : 31);
    strip_slot<PR>(lds + SL_SLOT, line, K, LOCAL ? 0 : -A.open - A.ext, LOCAL ? PAD_SCORE : A.ext - A.open);
    asm volatile("" ::: "memory");  // staged by all lanes (a wave's LDS accesses keep their order)
    StripsIO io;
    io.bcode = bcode + 64 - lane;
    io.slot_add = 0x01010101u * (((uint32_t)(uintptr_t)(lds_u8 *)lds + SL_SLOT) >> 8);
    io.lds = lds;
    io.rin = s ? A.ring + P.ring + (uint64_t)(s - 1) * (T + 8) : nullptr;
    io.rout = A.ring + P.ring + (uint64_t)s * (T + 8);
    io.pl = __builtin_amdgcn_make_buffer_rsrc(A.planes + P.planes + (uint64_t)s * (T / SPD) * 64, 0, (T / SPD) * 256,
                                              0x00020000);
    io.cols = T - 63;
    io.spin_limit = A.spin_limit;
    io.err = A.err;
    io.lost = lost;
    if (io.rin) io.look();
    StripEnd end;
    strip_sweep<PR, LOCAL>(io, s, s + 1 == P.S, m, n, T, A.open, A.ext, end);
    lost = io.lost;
    if (LOCAL) {
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) {
        const int oh = __shfl_xor(end.h, d, 64), oi = __shfl_xor(end.i, d, 64), oj = __shfl_xor(end.j, d, 64);
        if (strip_better(oh, oi, oj, end.h, end.i, end.j)) { end.h = oh; end.i = oi; end.j = oj; }
      }
      if (lane == 0 && end.h > 0)
        atomicMax((unsigned long long *)(A.best + w.sp), (unsigned long long)strips_key(end.h, end.i, end.j));
    } else if (end.has) {
      A.score[w.sp] = end.h;
    }
  }
}

// A walk over codes in device memory, local scores not needed (the stop is marked).
template <bool LOCAL>
__global__ __launch_bounds__(64) void strips_walk_kernel(StripsArgs A) {
  using Win = StripWindow<STRIPS_PR>;
  __shared__ uint32_t win[Win::WL * Win::WD];
  const StripPair P = A.sp[blockIdx.x];
  const PairDev pd = A.tb.pairs[P.pid];
  const int lane = threadIdx.x & 63;
  ResultDev r;
  int i = P.m, j = P.n;
  r.cigar_off = (int64_t)(pd.cig_off + pd.cig_cap);
  r.cigar_len = 0;
  if (LOCAL) {
    const uint64_t k = A.best[blockIdx.x];
    r.score = (int)(k >> 40);
    i = k ? 0xFFFFF - (int)((k >> 20) & 0xFFFFF) : 0;
    j = k ? 0xFFFFF - (int)(k & 0xFFFFF) : 0;
    // as the packed lanes report it: beyond their range a rerun in int32
    r.flags = !P.i16 ? 1 : r.score > A.sat_limit ? 3 : 0;
    if (!k) r.flags |= 8;
    r.a_begin = r.b_begin = -1;
    r.a_end = i - 1;
    r.b_end = j - 1;
  } else {
    r.score = A.score[blockIdx.x];
    r.flags = P.i16 ? 0 : 1;
    r.a_begin = 0; r.a_end = P.m - 1; r.b_begin = 0; r.b_end = P.n - 1;
  }
  i = __builtin_amdgcn_readfirstlane(i);
  j = __builtin_amdgcn_readfirstlane(j);
  if (LOCAL ? i > 0 : A.tb.do_cigar != 0) {
    WaveRuns rw;
    rw.on = A.tb.do_cigar != 0;
    rw.end = (uint32_t *)(A.tb.cig + pd.cig_off + pd.cig_cap);
    rw.cap = pd.cig_cap / 4;
    Win src{A.planes + P.planes, win, P.T, -1, -1};
    src.refill(i, j);
    int state = 0, steps = 0;
    // a walk may take fewer than `cap` steps, or end on that step (local)
    const int full = 2 * (pd.la + pd.lb) + 2, cap = (full < A.tb.guard_cap ? full : A.tb.guard_cap) - (LOCAL ? 0 : 1);
    const int how = wave_walk<LOCAL ? WALK_MARKED : WALK_GLOBAL>(src, rw, i, j, state, cap, steps);
    if (how == WALK_GAVE_UP) r.flags |= WALK_FAILED;
    if (!LOCAL && how != WALK_GAVE_UP) {
      if (i == 0 && j > 0) rw.emit(1, j);
      if (j == 0 && i > 0) rw.emit(2, i);
    }
    if (!rw.finish() && rw.on) r.flags |= WALK_FAILED;
    if (LOCAL) { r.a_begin = i; r.b_begin = j; }
    if (rw.on) {
      const int nr = rw.n < rw.cap ? rw.n : rw.cap;
      r.cigar_off -= 4 * nr;
      r.cigar_len = 4 * nr;
    }
  }
  if (lane == 0) put_result(A.tb, P.pid, r);
}

// Before a run: every ring entry empty, no best cell.
__global__ void strips_init_kernel(uint4 *ring, uint64_t n16, uint64_t *best, int npairs) {
  const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
  const uint32_t e = (uint32_t)STRIP_EMPTY;
  for (uint64_t k = tid; k < n16; k += stride) ring[k] = make_uint4(e, e, e, e);
  for (uint64_t k = tid; k < (uint64_t)npairs; k += stride) best[k] = 0;
}

}  // namespace ta
