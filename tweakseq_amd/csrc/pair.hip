// One pair at low latency: the editor's "realign selection" path.
//
// In the reference, realigning two selected rows runs the external aligner
// on them (tweakseq/UI/SeqEditMainWin.cpp:1616-1663) and splices the result
// back at the selection (tweakseq/Core/Project.cpp:964-1026).  Here it is
// one launch of one workgroup that takes the letters and returns the CIGAR
// runs, with nothing else on the device:
//  * the letters are read straight from host staging (mapped, pinned
//    memory) and encoded in LDS, beside a substitution table compiled in;
//  * the fill is strip.h's int32 sweep: strips of 64 lanes x 1, 2 or 4 rows,
//    strip s on wave s % 4, trailing strip s-1 through a ring of bottom rows
//    in LDS (progress counters, workgroup scope, bounded waits);
//  * direction codes (4 bits per cell) stay in LDS (in device memory where
//    they do not fit beside the tables), and wave 0 walks them back a CIGAR
//    run at a time (walk.h);
//  * the result and the runs go straight back to host staging.
// Pairs larger than that take the batch path (the caller's entry point
// decides).  Recurrence, boundaries and tie-breaks are those of the
// specification the CPU oracle implements (oracle/gotoh.c); the local
// stop cell (H = 0) is marked in its code as d = 0, x = 1 (a combination
// the H-source never takes), since no walk reads another bit of such a cell.
//
// Bound by dependent steps: n + 80 (strips) of the fill, each as long as one
// wave takes to issue it, and a lookup per CIGAR run of the walk.  Call to
// CIGAR, with two rows per lane, 322 cycles a step and a walk of 430 cycles a
// cell, and now: 24 x 28 global protein 36 / 19 us, 300 x 320 155 / 71 us (of
// 2.4 GHz cycles: fill 117,000, walk 28,000, tables and letters 7,500),
// 400 x 420 local DNA 217 / 100 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "../../include/tweakalign.h"
#include "blosum62.h"
#include "common.h"
#include "pair.h"
#include "runtime_internal.h"
#include "strip.h"
#include "walk.h"

namespace ta {

namespace {

// Substitution lines (32 bytes a residue, pads at PAD_SCORE) and letter maps,
// compiled in and loaded as they are.
struct alignas(16) PairTables {
  int8_t prot[32 * 32];
  int8_t map[2][256];  // TA_PROTEIN, TA_DNA: letter -> code, -1 outside the alphabet
};
constexpr PairTables pair_tables() {
  constexpr int8_t lower[] = {TA_BLOSUM62_LOWER};
  constexpr char order[] = TA_PROT_ORDER;
  PairTables t{};
  for (int x = 0; x < 32 * 32; ++x) t.prot[x] = PAD_SCORE;
  for (int r = 0; r < TA_PROT_K; ++r)
    for (int c = 0; c < TA_PROT_K; ++c) {
      const int hi = r > c ? r : c, lo = r > c ? c : r;
      t.prot[32 * r + c] = lower[hi * (hi + 1) / 2 + lo];
    }
  for (int x = 0; x < 256; ++x) {
    const int u = (x >= 'a' && x <= 'z') ? x - 32 : x;
    int p = -1;
    for (int r = 0; r < TA_PROT_K; ++r)
      if (order[r] == u) p = r;
    if (u == 'J' || u == 'O' || u == 'U') p = TA_PROT_K - 1;  // scored as X
    t.map[0][x] = (int8_t)p;
    t.map[1][x] = (int8_t)(u == 'A' ? 0 : u == 'C' ? 1 : u == 'G' ? 2 : u == 'T' ? 3 : -1);
  }
  return t;
}
static_assert(TA_PROTEIN == 0 && TA_DNA == 1 && TA_PROT_K + 1 <= STRIP_NC, "alphabet codes");
__device__ const PairTables kPairTables = pair_tables();

// LDS words of the sync area.
enum { SY_STATUS = 0, SY_SCORE = 1, SY_PROG = 4, SY_BEST = 8, SY_DUMP = 24, SY_READY = 25, SY_ZERO = 32, SY_EDGE = 48,
       SY_WORDS = 64 };

// 16 letters of a sequence (positions x .. x + 15, those past len ignored) as
// codes, `pad` past its end; bad: a letter outside the alphabet.
__device__ __forceinline__ uint4 encode16(const int8_t *lmap, uint4 v, int x, int len, int pad, int &bad) {
  uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t o = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const bool in = x + 4 * q + b < len;
      const int c = lmap[(w[q] >> (8 * b)) & 0xff];
      bad |= in && c < 0;
      o |= (uint32_t)(in && c >= 0 ? c : pad) << (8 * b);
    }
    w[q] = o;
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// Direction codes in LDS, all at hand: dwords [strip][t / SPD][lane], the
// last strip as wide as it has lanes.
template <int PR>
struct PairCodes {
  const uint32_t *pl;
  uint32_t strip_dw;         // dwords of a full strip
  uint32_t last, last_lanes; // the last strip, and its width
  __device__ __forceinline__ int code(int i, int j) const {
    constexpr uint32_t SPD = strip_spd(PR);
    const uint32_t r = (uint32_t)i - 1, L = r / PR, s = L >> 6, l = L & 63, t = (uint32_t)j - 1 + l;
    const uint32_t dw = pl[__umul24(s, strip_dw) + __umul24(t / SPD, s == last ? last_lanes : 64u) + l];
    return strip_code<PR>(dw, t % SPD, r % PR);
  }
  __device__ __forceinline__ int direct(int i, int j) const { return code(i, j); }
  __device__ __forceinline__ bool refill(int, int) { return false; }
};

template <int PR, bool LOCAL, bool GP>
__global__ __launch_bounds__(64 * PAIR_WAVES) __attribute__((amdgpu_waves_per_eu(1, 1))) void pair_kernel(PairArgs A) {
  extern __shared__ __align__(256) uint8_t lds[];
  const PairLayout &Y = A.lay;
  uint8_t *tab = lds;                            // 32-byte line per residue code
  int8_t *lmap = (int8_t *)(lds + 1024);         // letter -> code, -1 outside the alphabet
  uint8_t *acode = lds + Y.acode;
  uint8_t *bcode = lds + Y.bcode;                // 64 pads, the columns, pads
  int32_t *sy = (int32_t *)(lds + Y.sync);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = A.m, n = A.n, T = Y.T, S = Y.S, nthr = blockDim.x;
  const bool prot = A.alphabet == TA_PROTEIN;
  const int K = prot ? TA_PROT_K : 4, pad = K;

  // Tables and letters: every load before the first use (the letters come
  // over the host link).  Each thread takes 16 letters of either sequence.
  const uint4 *ga = (const uint4 *)A.a, *gb = (const uint4 *)A.b;
  uint4 va = make_uint4(0, 0, 0, 0), vb = va;
  if (16 * tid < m) va = ga[tid];
  if (16 * tid < n) vb = gb[tid];
  for (int x = tid; x < 256; x += nthr) {
    uint32_t v = ((const uint32_t *)kPairTables.prot)[x];
    if (!prot) {
      v = 0;
      for (int b = 0; b < 4; ++b) {
        const int r = x >> 3, c = ((x & 7) << 2) + b;
        v |= (uint32_t)(uint8_t)(r < 4 && c < 4 ? (r == c ? A.match : A.mismatch) : PAD_SCORE) << (8 * b);
      }
    }
    ((uint32_t *)tab)[x] = v;
    if (x < 64) ((uint32_t *)lmap)[x] = ((const uint32_t *)kPairTables.map[prot ? 0 : 1])[x];
  }
  if (tid < SY_WORDS) sy[tid] = tid == SY_READY ? 0x7fffffff : tid >= SY_EDGE && !LOCAL ? 2 * (A.open - A.ext) : 0;
  if (LOCAL && S > 1) {  // ring columns no strip stores (from T - 63 on): 0
    int2 *tail = (int2 *)(lds + Y.ring) + T + 1;
    const int rings = S - 1 < PAIR_WAVES ? S - 1 : PAIR_WAVES, w = Y.ring_len - T - 1;
    for (int x = tid; x < rings * w; x += nthr) tail[(x / w) * Y.ring_len + x % w] = make_int2(0, 0);
  }
  if (tid < 16) ((uint32_t *)bcode)[tid] = 0x01010101u * (uint32_t)pad;
  __syncthreads();
  int bad = 0;
  for (int x = 16 * tid; x < m || x < T + 16; x += 16 * nthr) {
    if (x != 16 * tid) {
      if (x < m) va = ga[x / 16];
      if (x < n) vb = gb[x / 16];
    }
    if (x < m) *(uint4 *)(acode + x) = encode16(lmap, va, x, m, pad, bad);
    if (x < T + 16) *(uint4 *)(bcode + 64 + x) = encode16(lmap, vb, x, n, pad, bad);
  }
  if (bad) atomicOr(&sy[SY_STATUS], PAIR_BAD_LETTER);
  __syncthreads();
  if (sy[SY_STATUS] & PAIR_BAD_LETTER) {
    if (tid == 0) {
      A.out->status = sy[SY_STATUS];
      if (A.polled) __hip_atomic_store(&A.out->done, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return;
  }

  // ---- fill
  constexpr int SPD = strip_spd(PR);
  const int slot = Y.slots + wv * Y.slot_bytes;
  int2 *const ring = (int2 *)(lds + Y.ring);
  const int last_lanes = (m - (S - 1) * 64 * PR + PR - 1) / PR;
  StripEnd end;
  for (int s = wv; s < S; s += PAIR_WAVES) {
    const int r0 = (s * 64 + lane) * PR;
    const uint8_t *line[PR];
#pragma unroll
    for (int k = 0; k < PR; ++k) line[k] = tab + 32 * (r0 + k < m ? acode[r0 + k] : PAIR_PAD_LINE);
    strip_slot<PR>(lds + slot, line, K, LOCAL ? 0 : -A.open - A.ext, LOCAL ? PAD_SCORE : A.ext - A.open);
    StripGroupIO io;
    io.bcode = bcode + 64 - lane;
    io.slot_add = 0x01010101u * ((uint32_t)((uint32_t)(uintptr_t)(lds_u8 *)lds + slot) >> 8);
    io.status = sy + SY_STATUS;
    io.pin = sy + (s ? SY_PROG + (s + PAIR_WAVES - 1) % PAIR_WAVES : SY_READY);
    io.pout = sy + SY_PROG + s % PAIR_WAVES;
    io.rin = lane ? (int2 *)(sy + SY_ZERO)
                  : s ? ring + ((s + PAIR_WAVES - 1) % PAIR_WAVES) * Y.ring_len + 64 : (int2 *)(sy + SY_EDGE);
    io.rin_step = lane == 0 && s ? 8 : 0;
    io.rout = ring + (s % PAIR_WAVES) * Y.ring_len;
    io.need0 = s << 20;
    io.cols = T - 63;
    io.s = s;
    io.spin_limit = A.spin_limit;
    io.gave_up = PAIR_GAVE_UP;
    if constexpr (GP) {
      io.pl = (uint32_t *)A.planes + (size_t)s * (T / SPD) * 64 + lane;
      io.pl_step = 64;
    } else {
      const bool own = s + 1 < S || lane < last_lanes;
      io.pl = own ? (uint32_t *)(lds + Y.planes) + s * (T / SPD) * 64 + lane : (uint32_t *)sy + SY_DUMP;
      io.pl_step = !own ? 0 : s + 1 < S ? 64 : last_lanes;
    }
    strip_sweep<PR, LOCAL>(io, s, s + 1 == S, m, n, T, A.open, A.ext, end);
  }
  if (LOCAL) {
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) {
      const int oh = __shfl_xor(end.h, w, 64), oi = __shfl_xor(end.i, w, 64), oj = __shfl_xor(end.j, w, 64);
      if (strip_better(oh, oi, oj, end.h, end.i, end.j)) { end.h = oh; end.i = oi; end.j = oj; }
    }
    if (lane == 0) {
      sy[SY_BEST + 3 * wv] = end.h; sy[SY_BEST + 3 * wv + 1] = end.i; sy[SY_BEST + 3 * wv + 2] = end.j;
    }
  } else if (end.has) {
    sy[SY_SCORE] = end.h;
  }
  __syncthreads();  // (GP: and every plane store of the workgroup is visible to it)
  if (wv != 0) return;

  // ---- end cell and walk (wave 0)
  ResultDev r;
  r.flags = TA_F_I32;
  int i = m, j = n;
  if (LOCAL) {
    int bh = 0, bi = 0x7fffffff, bj = 0x7fffffff;
    for (int w = 0; w < PAIR_WAVES && w < S; ++w) {
      const int oh = sy[SY_BEST + 3 * w], oi = sy[SY_BEST + 3 * w + 1], oj = sy[SY_BEST + 3 * w + 2];
      if (oh > 0 && strip_better(oh, oi, oj, bh, bi, bj)) { bh = oh; bi = oi; bj = oj; }
    }
    r.score = bh;
    if (bh <= 0) {
      r.score = 0;
      r.a_begin = r.a_end = r.b_begin = r.b_end = -1;
      r.flags |= TA_F_EMPTY;
      i = j = 0;
    } else {
      i = __builtin_amdgcn_readfirstlane(bi);
      j = __builtin_amdgcn_readfirstlane(bj);
      r.a_end = i - 1; r.b_end = j - 1;
    }
  } else {
    r.score = sy[SY_SCORE];
    r.a_begin = 0; r.a_end = m - 1; r.b_begin = 0; r.b_end = n - 1;
  }
  const bool walk = LOCAL ? r.score > 0 : A.traceback != 0;
  uint32_t *runs = (uint32_t *)(lds + Y.runs);  // over the slots, which only the fill read
  const int cap = Y.runs_cap;
  WaveRuns rw;
  rw.end = runs + cap;
  rw.cap = cap;
  if (walk) {
    constexpr int KIND = LOCAL ? WALK_MARKED : WALK_GLOBAL;
    int state = 0, steps = 0, how;
    if constexpr (GP) {
      StripWindow<PR> src{(const uint32_t *)A.planes, (uint32_t *)(lds + Y.window), T, -1, -1};
      src.refill(i, j);
      how = wave_walk<KIND>(src, rw, i, j, state, A.walk_cap, steps);
    } else {
      PairCodes<PR> src{(const uint32_t *)(lds + Y.planes), (uint32_t)(T / SPD) * 64, (uint32_t)S - 1,
                        (uint32_t)last_lanes};
      how = wave_walk<KIND>(src, rw, i, j, state, A.walk_cap, steps);
    }
    if (how == WALK_GAVE_UP) {
      r.flags |= TA_F_WALK_FAILED;
    } else if (!LOCAL) {
      if (i == 0 && j > 0) rw.emit(1, j);
      if (j == 0 && i > 0) rw.emit(2, i);
      i = j = 0;
    }
    if (!rw.finish()) r.flags |= TA_F_WALK_FAILED;
  }
  if (LOCAL && r.score > 0) { r.a_begin = i; r.b_begin = j; }
  const int nr = rw.n < cap ? rw.n : cap, wp = cap - nr;
  uint32_t *dst = (uint32_t *)(A.out + 1);
  if (A.traceback)
    for (int q = lane; q < nr; q += 64) dst[q] = runs[wp + q];
  if (lane == 0) {
    r.cigar_off = 0;
    r.cigar_len = A.traceback ? 4 * nr : 0;
    A.out->r = r;
    A.out->nruns = A.traceback ? nr : 0;
    A.out->status = sy[SY_STATUS];
  }
  // (the wave's own stores: one release covers the runs of all its lanes)
  if (A.polled && lane == 0) __hip_atomic_store(&A.out->done, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int PR>
void launch_rows(const PairArgs &A, hipStream_t st) {
  void (*k)(PairArgs) = A.local ? (A.lay.plane_bytes ? pair_kernel<PR, true, true> : pair_kernel<PR, true, false>)
                                : (A.lay.plane_bytes ? pair_kernel<PR, false, true> : pair_kernel<PR, false, false>);
  hipLaunchKernelGGL(k, dim3(1), dim3(64 * std::min(PAIR_WAVES, A.lay.S)), A.lay.bytes, st, A);
}

}  // namespace

PairLayout pair_layout(int m, int n, int K, int lds_max) {
  PairLayout L{};
  auto up = [](long x, int to) { return (x + to - 1) / to * to; };
  // Rows per lane.  A strip's step takes about 16 instructions and 13 more
  // per row, and every wave is one SIMD's: the fewest rows that give each of
  // the four waves at most one strip.
  L.R = m <= 64 * PAIR_WAVES ? 1 : m <= 128 * PAIR_WAVES ? 2 : 4;
  L.T = (n + 63 + 7) & ~7;
  L.S = (m + 64 * L.R - 1) / (64 * L.R);
  const int waves = std::min(PAIR_WAVES, L.S);
  L.ring_len = L.T + 80;
  L.runs_cap = m + n + 2;
  long off = 1280;
  L.sync = (int)off; off += 4 * SY_WORDS;
  L.slots = (int)off;  // in the first 64 KB (strip.h addresses a slot's rows in one byte)
  static_assert((1280 + 4 * SY_WORDS) % STRIP_ROW == 0 &&
                1280 + 4 * SY_WORDS + PAIR_WAVES * strip_slot_bytes(4) <= 256 * STRIP_ROW, "slot rows");
  const int rows = (int)up(K + 1, 4);
  L.slot_bytes = (L.R == 4 ? STRIP_NC + rows : rows) * STRIP_ROW;
  off += (long)waves * L.slot_bytes;
  L.acode = (int)off; off += up(m, 16);
  L.bcode = (int)off; off += up(64 + L.T + 32, 16);
  L.ring = (int)off; off += (long)std::min(PAIR_WAVES, L.S - 1) * L.ring_len * 8;
  // after the fill: the CIGAR runs and, with the codes in device memory, the walk's window
  L.runs = L.slots;
  L.window = (int)(L.slots + up(4L * L.runs_cap, 16));
  const long spd = strip_spd(L.R), after = L.window + 64 * (32 / spd + 1) * 4, strips = (long)L.T / spd * 4;
  const long last = (m - (long)(L.S - 1) * 64 * L.R + L.R - 1) / L.R;
  L.planes = (int)std::max(off, (long)L.window);
  const long with = L.planes + strips * ((L.S - 1) * 64L + last);
  if (with <= lds_max) {
    L.bytes = (int)with;
  } else {
    L.bytes = (int)std::min(std::max(off, after), 1L << 30);
    L.plane_bytes = (int)std::min(strips * 64 * L.S, 1L << 30);
  }
  return L;
}

int pair_launch(const PairArgs &A, hipStream_t st) {
  (void)hipGetLastError();
  if (A.lay.R == 1) launch_rows<1>(A, st);
  else if (A.lay.R == 2) launch_rows<2>(A, st);
  else launch_rows<4>(A, st);
  return hipGetLastError() == hipSuccess ? TA_OK : TA_E_DEVICE;
}

}  // namespace ta

// ---------------------------------------------------------------------------
// Host side.
namespace {

using namespace ta;

// Result, CIGAR text and status of a finished pair kernel (record readable
// on the host).
int pair_finish(const PairOut &o, const uint32_t *runs, const ta_params *p, ta_result *out, char *cigar_buf,
                int64_t cap, int64_t *used) {
  if (o.status & PAIR_BAD_LETTER) return TA_E_ALPHABET;
  if (o.status & PAIR_GAVE_UP) return TA_E_DEVICE;
  const ResultDev &r = o.r;
  out->score = r.score;
  out->a_begin = r.a_begin; out->a_end = r.a_end;
  out->b_begin = r.b_begin; out->b_end = r.b_end;
  out->flags = r.flags;
  out->cigar_off = 0;
  out->cigar_len = 0;
  if (p->traceback && o.nruns > 0) {
    const int64_t len = cigar_text(runs, o.nruns, nullptr);
    out->cigar_len = (int32_t)len;
    if (used) *used = len;
    if (!cigar_buf || len > cap) return TA_E_SPACE;
    cigar_text(runs, o.nruns, cigar_buf);
  } else if (used) {
    *used = 0;
  }
  return (r.flags & TA_F_WALK_FAILED) ? TA_E_WALK : TA_OK;
}

// The pair path takes pairs whose codes take about a CU's LDS at most (codes
// that do not fit beside the fill's tables go to device memory); others (and
// empty sides, and forced long-pair lanes) go through the batch path.  Which
// pairs these are shows in their results (TA_F_I32), so the bound is a fixed
// function of the lengths.
bool pair_fits(int32_t m, int32_t n, int64_t lds_max) {
  const int64_t T = (n + 63 + 7) & ~7, S = ((int64_t)m + 127) / 128;
  auto up16 = [](int64_t x) { return (x + 15) & ~15ll; };
  return 1536 + up16(m) + up16(T + 8) + 32 * ((int64_t)n + 8) + S * T * 64 + 4 * ((int64_t)m + n + 2) <= lds_max;
}

bool pair_path(const ta_ctx *ctx, const ta_params *p, int32_t la, int32_t lb) {
  if (la <= 0 || lb <= 0 || p->lanes == TA_LANES_LONG) return false;
  if (p->mode == TA_GLOBAL && (int64_t)(la + lb + 2) * -p->gap_extend + 2 * (int64_t)-p->gap_open >= (1ll << 28))
    return false;  // scores near the int32 -infinity: the batch path reports it
  if (p->mode == TA_LOCAL) {  // the kernel's end-cell keys hold H in 16 bits
    const int maxS = p->alphabet == TA_PROTEIN ? 11 : std::max(0, std::max(p->match, p->mismatch));
    if ((int64_t)std::min(la, lb) * maxS >= 65535) return false;
  }
  return pair_fits(la, lb, ctx->lds_max);
}

PairArgs pair_args(const ta_ctx *ctx, const ta_params *p, int32_t la, int32_t lb) {
  PairArgs A{};
  A.m = la; A.n = lb;
  A.alphabet = p->alphabet; A.match = p->match; A.mismatch = p->mismatch;
  A.open = p->gap_open; A.ext = p->gap_extend;
  A.local = p->mode == TA_LOCAL; A.traceback = p->traceback != 0;
  A.spin_limit = 1 << 22;
  A.walk_cap = la + lb;  // a walk takes at most la + lb steps
  if (const char *e = getenv("TWEAKALIGN_WALK_GUARD")) A.walk_cap = std::min(A.walk_cap, std::max(0, atoi(e)));
  A.lay = pair_layout(la, lb, p->alphabet == TA_PROTEIN ? TA_PROT_K : 4, ctx->lds_max);
  return A;
}

// Device memory for the codes of a pair that fits: at most the codes' 4 bits
// a cell over whole strips and steps, some 200 KB.
constexpr size_t kPairPlanes = 256 << 10;

}  // namespace

int ta_align_pair(ta_ctx *ctx, const ta_params *p, const char *a, int32_t la, const char *b, int32_t lb,
                  ta_result *out, char *cigar_buf, int64_t cap, int64_t *used) {
  if (!ctx || !p || !out || la < 0 || lb < 0 || (la && !a) || (lb && !b)) return TA_E_INVALID;
  if (params_check(p)) return TA_E_INVALID;
  if (!pair_path(ctx, p, la, lb)) {
    const ta_pair q{a, la, b, lb};
    return ta_align_batch(ctx, p, &q, 1, out, cigar_buf, cap, used);
  }
  if (hipSetDevice(ctx->device) != hipSuccess) return TA_E_DEVICE;
  PairArgs A = pair_args(ctx, p, la, lb);
  if (A.lay.plane_bytes) {
    if (!ctx->pair_planes && !(ctx->pair_planes = device_alloc(kPairPlanes))) return TA_E_NOMEM;
    A.planes = (uint8_t *)ctx->pair_planes;
  }
  // staging: [PairOut][runs][a][b]
  const size_t o_runs = sizeof(PairOut), o_a = (o_runs + 4 * (size_t)A.lay.runs_cap + 15) & ~(size_t)15;
  const size_t o_b = (o_a + (size_t)la + 15) & ~(size_t)15, need = o_b + (size_t)lb + 16;
  if (ctx->pair_stage_cap < need) {
    if (ctx->pair_stage) (void)hipHostFree(ctx->pair_stage);
    ctx->pair_stage = nullptr;
    ctx->pair_stage_cap = 0;
    const size_t want = std::max(need, (size_t)64 << 10);
    if (hipHostMalloc(&ctx->pair_stage, want, hipHostMallocCoherent) != hipSuccess) {
      (void)hipGetLastError();
      ctx->pair_stage = nullptr;
      return TA_E_NOMEM;
    }
    ctx->pair_stage_cap = want;
  }
  uint8_t *st = (uint8_t *)ctx->pair_stage;
  memcpy(st + o_a, a, (size_t)la);
  memcpy(st + o_b, b, (size_t)lb);
  PairOut *o = (PairOut *)st;
  o->status = 0;
  o->done = 0;
  A.polled = 1;
  A.a = (const char *)(st + o_a);
  A.b = (const char *)(st + o_b);
  A.out = o;
  int rc = pair_launch(A, ctx->stream);
  if (rc) return rc;
  // The kernel's last store says that the result is there, a few microseconds
  // before the stream is seen idle; a wait longer than any pair takes is the
  // stream's (which reports errors).
  const auto t0 = std::chrono::steady_clock::now();
  while (!__atomic_load_n(&o->done, __ATOMIC_ACQUIRE)) {
    if (std::chrono::steady_clock::now() - t0 < std::chrono::microseconds(500)) continue;
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return TA_E_DEVICE;
    break;
  }
  return pair_finish(*o, (const uint32_t *)(st + o_runs), p, out, cigar_buf, cap, used);
}

// ---------------------------------------------------------------------------
// The allocation-free variant.  `scratch` is the only device memory it uses:
// [PairOut][runs][letters of a][letters of b].  In host code its name is a
// host-side stand-in, never a device address: every use goes through the
// address hipGetSymbolAddress gives for the device (pair_scratch_setup).
namespace {

static __device__ __align__(256) uint8_t scratch[TA_PAIR_STATIC_SCRATCH];
static __device__ __align__(256) uint8_t scratch_planes[kPairPlanes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint8_t *g_scratch[kMaxDevices] = {}, *g_planes[kMaxDevices] = {};
bool g_scratch_done[kMaxDevices] = {};

uint8_t *scratch_of(int device, uint8_t **planes) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> g(g_scratch_mu);
  *planes = g_planes[device];
  return g_scratch[device];
}

// Offsets inside the scratch for an la x lb pair (within its size whenever
// la + lb <= TA_PAIR_STATIC_MAX).
struct StaticLayout {
  size_t runs, a, b, end;
};
StaticLayout static_layout(int32_t la, int32_t lb) {
  StaticLayout L;
  L.runs = sizeof(PairOut);
  L.a = (L.runs + 4 * ((size_t)la + lb + 2) + 15) & ~(size_t)15;
  L.b = (L.a + (size_t)la + 15) & ~(size_t)15;
  L.end = L.b + (size_t)lb;
  return L;
}
static_assert(sizeof(PairOut) + 4 * (TA_PAIR_STATIC_MAX + 2) + 15 + TA_PAIR_STATIC_MAX + 15 <= TA_PAIR_STATIC_SCRATCH,
              "scratch too small for the largest pair it admits");

// Result of a pair with an empty side, as the batch path gives it.
int empty_side(const ta_params *p, int32_t la, int32_t lb, ta_result *out, char *cigar_buf, int64_t cap,
               int64_t *used) {
  *out = ta_result{};
  out->cigar_off = 0;
  if (p->mode == TA_LOCAL) {
    out->a_begin = out->a_end = out->b_begin = out->b_end = -1;
    out->flags = TA_F_EMPTY;
    if (used) *used = 0;
    return TA_OK;
  }
  const int32_t len = la + lb;
  out->score = len ? p->gap_open + (len - 1) * p->gap_extend : 0;
  out->a_begin = 0; out->a_end = la - 1; out->b_begin = 0; out->b_end = lb - 1;
  uint32_t run = len ? ((uint32_t)len << 2) | (la ? 2u : 1u) : 0u;  // la I's or lb D's
  const int64_t need = (p->traceback && len) ? cigar_text(&run, 1, nullptr) : 0;
  out->cigar_len = (int32_t)need;
  if (used) *used = need;
  if (need > 0) {
    if (!cigar_buf || need > cap) return TA_E_SPACE;
    cigar_text(&run, 1, cigar_buf);
  }
  return TA_OK;
}

}  // namespace

void pair_scratch_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return;
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (g_scratch_done[device]) return;
  g_scratch_done[device] = true;
  void *ptr = nullptr, *pl = nullptr;
  hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e == hipSuccess) e = hipGetSymbolAddress(&pl, HIP_SYMBOL(scratch_planes));
  if (e != hipSuccess) {
    (void)hipGetLastError();
    fprintf(stderr, "tweakalign: no address for the pair scratch on device %d: %s\n", device, hipGetErrorString(e));
    return;
  }
  g_scratch[device] = (uint8_t *)ptr;
  g_planes[device] = (uint8_t *)pl;
}

int ta_align_pair_static(ta_ctx *ctx, const ta_params *p, const char *a, int32_t la, const char *b, int32_t lb,
                         ta_result *out, char *cigar_buf, int64_t cap, int64_t *used) {
  if (!ctx || !p || !out || la < 0 || lb < 0 || (la && !a) || (lb && !b)) return TA_E_INVALID;
  if (params_check(p)) return TA_E_INVALID;
  if ((int64_t)la + lb > TA_PAIR_STATIC_MAX) return TA_E_LIMIT;
  if (la == 0 || lb == 0) return empty_side(p, la, lb, out, cigar_buf, cap, used);
  if (!pair_path(ctx, p, la, lb)) return TA_E_LIMIT;
  uint8_t *planes = nullptr, *scr = scratch_of(ctx->device, &planes);
  if (!scr) return TA_E_DEVICE;
  if (hipSetDevice(ctx->device) != hipSuccess) return TA_E_DEVICE;
  const StaticLayout L = static_layout(la, lb);
  hipStream_t st = ctx->stream;
  if (hipMemcpyAsync(scr + L.a, a, (size_t)la, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemcpyAsync(scr + L.b, b, (size_t)lb, hipMemcpyHostToDevice, st) != hipSuccess)
    return TA_E_DEVICE;
  PairArgs A = pair_args(ctx, p, la, lb);
  A.a = (const char *)(scr + L.a);
  A.b = (const char *)(scr + L.b);
  A.planes = planes;
  A.out = (PairOut *)scr;  // the kernel writes every field the host reads (status included)
  int rc = pair_launch(A, st);
  if (rc) return rc;
  // result and runs to the calling thread's stack
  struct {
    PairOut o;
    uint32_t runs[TA_PAIR_STATIC_MAX + 2];
  } back;
  static_assert(sizeof(PairOut) % 4 == 0, "runs follow the record");
  if (hipMemcpyAsync(&back, scr, sizeof(PairOut) + 4 * ((size_t)la + lb + 2), hipMemcpyDeviceToHost, st) !=
          hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return TA_E_DEVICE;
  return pair_finish(back.o, back.runs, p, out, cigar_buf, cap, used);
}
