// Progressive multiple alignment on the GPU (ta_msa).
//
// tweakseq aligns N > 2 sequences by handing them to an external MSA program
// (tweakseq/UI/SeqEditMainWin.cpp:1647-1659) and reading the aligned FASTA
// back (tweakseq/Core/Project.cpp:908-1032).  This builds the alignment in
// process, to the specification the CPU oracle restates (oracle/msa.c):
//
//  1. global Gotoh scores of all pairs -- one batch of the pairwise engine
//     (n(n-1)/2 pairs, score only: 130,816 pairs for 512 sequences);
//  2. similarities s_ij * 1e6 / max(1, min(self_i, self_j)) (integer), and
//     UPGMA joins on the host with exact integer comparisons (ties to the
//     smallest pair of cluster ids);
//  3. the joins, tree level by tree level: every join of a level is one
//     workgroup of msa_join_kernel, which aligns the columns of the lower
//     cluster's profile (DP rows) with the higher one's (DP columns) by
//     global Gotoh -- match score M(i,j) = cntA[i] . PB[j] with
//     PB[j][x] = sum_y S(x,y) cntB[j][y], gap costs times nA * nB, the
//     pairwise ties (diag > E > F, E / F prefer opening) -- and walks the
//     direction codes back from (la, lb) to runs.
//
// Profiles stay on the device: a cluster's column is a row of 24 residue
// counts and 24 PB entries.  Both are sums over its sequences, so a join's
// workgroup makes the merged columns by adding the rows its runs bring
// together, and records for each column of either side the merged column it
// went to; in the end a thread per residue follows those maps to the root.
// The host sees each join's length only, which sizes the next level.  (A
// sequence's own columns are rows of a table of K, picked by its codes.)
//
// Each level first scores every column pair of every join over the whole GPU
// (msa_scores_kernel; int32: nA * nB is bounded so that 24 codes x 11 x
// nA * nB fits), in the order the sweeps read them, pads included.  A join's
// workgroup then sweeps strips of 128 rows (strip.h, 2 rows a lane), a wave
// each, up to 16 waves; each trails the one above through a ring of bottom
// rows in LDS.  Its values G = H - ext (i + j) + (open - ext) stay between
// 3 (open - ext) nA nB and min(la, lb) (max S + 2 |ext|) nA nB; joins where
// that could leave int32 take the plain recurrence in int64.
//
// Bound by the dependent steps of the largest join of a level: lb + 63 + 72
// a strip of 128 rows, each as long as a wave takes to issue it.  512
// sequences of 100 to 600 (17 levels): with a plain recurrence that passed
// direction bytes to a walk by one thread, and counts made by the host from
// row-by-row profiles, a level took 420 us of join kernel and 800 us in all;
// now 157 us and 240 us; the call 32.6 -> 20.0 ms (14.6 with the score batch's
// creation and fill shortened too).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>
#include <vector>

#include "runtime_internal.h"
#include "strip.h"
#include "walk.h"

namespace {

using namespace ta;

constexpr int JWMAX = 16;                // waves per join at most
constexpr int JR = 2;                    // DP rows per lane
constexpr int JRS = 64 * JR;             // DP rows per strip
constexpr int KS = 24;                   // codes of a column, padded with zeros
constexpr int CI = 2 * KS / 4;           // int4s of a column: its KS counts, then its KS PB entries
constexpr int64_t WMAX = 8000000;        // nA * nB bound: 24 codes x 11 x nA * nB fits int32

// One side of a join: len columns, of a sequence (codes) or of a joined cluster (rows).
struct JoinSide {
  const uint8_t *code;  // a sequence: its residue codes
  const int4 *rows;     // a cluster: CI int4s per column
  int32_t *map;         // the merged column of each of its columns
  int32_t len;
};

struct JoinJob {
  JoinSide a, b;
  int64_t w;        // nA * nB: gap costs scale
  int64_t m_off;    // match scores in the sweep's order: [strip][step][lane][row]
  int64_t tb_off;   // direction codes, dwords of 4 steps x 2 rows: [strip][step / 4][lane]
  int64_t run_off;  // la + lb + 2 runs
  int64_t src_off;  // la + lb merged columns: (A's column or -1, B's column or -1)
  int4 *out;        // the merged columns' rows (null: not needed)
};

struct JoinArgs {
  const JoinJob *jobs;
  const int4 *leaf;   // rows of the K single residues
  int32_t *mbuf;
  uint32_t *tb, *runs;
  int2 *src;
  int32_t *nops;
  int32_t *err;       // | 1: a wait on another wave's progress gave up; | 2: a walk did
  int32_t open, ext, spin_limit;
};

// Steps of a strip of a join with lb columns (lane 63 trails lane 0), in whole blocks of 8.
__host__ __device__ inline int join_steps(int lb) { return (lb + 63 + 7) & ~7; }
__host__ __device__ inline int join_strips(int la) { return (la + JRS - 1) / JRS; }
// LDS of the int32 ring: a column's bottom row at entry column + 64.
__host__ __device__ inline int join_ring(int lb) { return join_steps(lb) + 80; }
// Bytes of the ring of a join with lb columns (int64: H and F of every column).
inline int64_t join_ring_bytes(int lb, bool wide) {
  return wide ? 2 * (int64_t)sizeof(int64_t) * (lb + 2) : (int64_t)sizeof(int2) * join_ring(lb);
}

__device__ __forceinline__ const int4 *join_row(const JoinSide &s, const int4 *leaf, int c) {
  return s.code ? leaf + s.code[c] * CI : s.rows + (int64_t)c * CI;
}

// Every join's match scores M(i, j) = cntA[i] . PB[j] + bias w, over the
// whole GPU.  A tile is a strip of 128 rows and 64 of its steps: its 127
// columns' PB rows in LDS (28 dwords apart: lanes read consecutive columns
// without bank conflicts), a lane's two rows of counts in registers; a
// sequence's row picks one entry.  Columns outside the pair score `pad` w.
// M24: every count and PB entry fits 24 bits (one multiply-add a code).
// blockIdx.x is the join, its tiles dealt over blockIdx.y.
template <bool M24>
__global__ __launch_bounds__(256) void msa_scores_kernel(JoinArgs A, int bias, int pad) {
  constexpr int PS = 28;
  __shared__ __align__(16) int32_t pbs[127 * PS];
  const JoinJob &J = A.jobs[blockIdx.x];
  const int la = J.a.len, lb = J.b.len, T = join_steps(lb), NC = (T + 63) / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wbias = (int)(bias * J.w), wpad = (int)(pad * J.w);
  for (int tile = blockIdx.y; tile < join_strips(la) * NC; tile += gridDim.y) {
    const int s = tile / NC, t0 = (tile % NC) * 64;
    for (int x = threadIdx.x; x < 127 * 6; x += 256) {
      const int c = t0 - 63 + x / 6;
      if (c >= 0 && c < lb) *(int4 *)(pbs + x / 6 * PS + x % 6 * 4) = join_row(J.b, A.leaf, c)[6 + x % 6];
    }
    const int i0 = s * JRS + lane * JR;
    int a[JR][KS], ac[JR];
#pragma unroll
    for (int k = 0; k < JR; ++k) {
      const bool in = i0 + k < la;
      if (J.a.code) {
        ac[k] = in ? J.a.code[i0 + k] : 0;
      } else {
#pragma unroll
        for (int x = 0; x < KS / 4; ++x) {
          const int4 v = in ? J.a.rows[(int64_t)(i0 + k) * CI + x] : make_int4(0, 0, 0, 0);
          a[k][4 * x] = v.x; a[k][4 * x + 1] = v.y; a[k][4 * x + 2] = v.z; a[k][4 * x + 3] = v.w;
        }
      }
    }
    __syncthreads();
    int2 *mm = (int2 *)(A.mbuf + J.m_off) + ((int64_t)s * T + t0) * 64 + lane;
    for (int q = wave; q < 64 && t0 + q < T; q += 4) {
      const int c = t0 + q - lane;
      const int32_t *pb = pbs + (q - lane + 63) * PS;
      int2 m = make_int2(wpad, wpad);
      if (c >= 0 && c < lb) {
        m = make_int2(wbias, wbias);
        if (J.a.code) {
          m.x += pb[ac[0]];
          m.y += pb[ac[1]];
        } else {
#pragma unroll
          for (int x = 0; x < KS; x += 4) {
            const int4 v = *(const int4 *)(pb + x);
            const int p[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int y = 0; y < 4; ++y) {
              m.x += M24 ? __mul24(a[0][x + y], p[y]) : a[0][x + y] * p[y];
              m.y += M24 ? __mul24(a[1][x + y], p[y]) : a[1][x + y] * p[y];
            }
          }
        }
      }
      mm[(int64_t)q * 64] = m;
    }
    __syncthreads();
  }
}

// wave_shr:1 (lane l takes lane l - 1's value, lane 0 keeps `old`).
__device__ __forceinline__ int64_t shr_lane(int64_t old, int64_t v) {
  const int32_t lo = __builtin_amdgcn_update_dpp((int32_t)old, (int32_t)v, 0x138, 0xf, 0xf, false);
  const int32_t hi = __builtin_amdgcn_update_dpp((int32_t)(old >> 32), (int32_t)(v >> 32), 0x138, 0xf, 0xf, false);
  return ((int64_t)hi << 32) | (uint32_t)lo;
}

// A strip of a join: scores from memory, read a block ahead.
struct JoinIO : StripGroupIO {
  static constexpr bool SLOTS = false;
  const int2 *ms;   // this lane's, 64 a step
  int blocks;
  int2 pre[2][4];   // the next block's halves

  __device__ __forceinline__ void load(int b, int half) {
    const int2 *p = ms + (int64_t)(8 * (b < blocks ? b : blocks - 1) + 4 * half) * 64;
#pragma unroll
    for (int q = 0; q < 4; ++q) pre[half][q] = p[q * 64];
  }
  __device__ __forceinline__ void scores(int b, int half, int (&v)[4][JR]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q][0] = pre[half][q].x;
      v[q][1] = pre[half][q].y;
    }
    load(b + 1, half);
  }
};

// LDS words of the sync area: a progress counter per wave, then as in StripGroupIO.
enum { JS_PROG = 0, JS_STATUS = 16, JS_READY = 17, JS_RUNS = 18, JS_ZERO = 32, JS_EDGE = 48, JS_WORDS = 64 };
// A join's LDS beside the ring: the sync area and the walk's window.
constexpr int64_t JOIN_LDS = 4 * (JS_WORDS + StripWindow<JR>::WL * StripWindow<JR>::WD);

// The strips of a join in int64, plain recurrence: H, E, F with a column test
// a step; direction codes as strip.h's.
__device__ __forceinline__ void join_sweep_wide(const JoinArgs &A, const JoinJob &J, int64_t *ringH, int32_t *sy,
                                                int W) {
  constexpr int64_t NEG = INT64_MIN / 4;
  const int la = J.a.len, lb = J.b.len, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t go = A.open * J.w, ge = A.ext * J.w;
  const int S = join_strips(la), NST = join_steps(lb);
  int64_t *ringF = ringH + (lb + 2);
  for (int s = wave; s < S; s += W) {
    const int i0 = s * JRS + lane * JR + 1;  // this lane's first row
    int64_t Hl[JR], El[JR];                  // H(i, j - 1), E(i, j - 1)
#pragma unroll
    for (int k = 0; k < JR; ++k) {
      Hl[k] = go + (i0 + k - 1) * ge;  // H(i, 0)
      El[k] = NEG;
    }
    int64_t hd0 = i0 == 1 ? 0 : go + (i0 - 2) * ge;  // H(i0 - 1, j - 1) for the next column: H(i0 - 1, 0)
    int64_t Hbot = 0, Fbot = NEG;                    // this lane's last row at its last column
    const bool writer = lane == 63 && s + 1 < S;     // stores the strip's last row for strip s + 1
    const int2 *ms = (const int2 *)(A.mbuf + J.m_off) + (int64_t)s * NST * 64 + lane;
    uint32_t *tb = A.tb + J.tb_off + (int64_t)s * (NST / 4) * 64 + lane;
    for (int b = 0; b < NST / 8; ++b) {
      if (s > 0) {  // strip s - 1 must have stored the ring up to this block's last column
        const int need = ((s - 1) / W + 1) << 20 | min(8 * b + 8, lb);
        int spins = 0;
        while (__hip_atomic_load(&sy[JS_PROG + (s - 1) % W], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < need) {
          if (++spins > A.spin_limit) {
            if (lane == 0) atomicOr(&sy[JS_STATUS], 1);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      uint32_t acc = 0;
      for (int q = 0; q < 8; ++q) {
        const int t = 8 * b + q, j = t - lane + 1, c = t + 1;  // c: lane 0's column
        int64_t top = go + (c - 1) * ge, topf = NEG;           // row 0, or the ring
        if (s > 0) {
          top = c <= lb ? ringH[c] : 0;
          topf = c <= lb ? ringF[c] : NEG;
        }
        const int64_t Hup0 = shr_lane(top, Hbot), Fup0 = shr_lane(topf, Fbot);
        const int2 m2 = ms[(int64_t)t * 64];
        uint32_t nib = 0;
        if (j >= 1 && j <= lb) {
          int64_t hup = Hup0, fup = Fup0, hd = hd0;
#pragma unroll
          for (int k = 0; k < JR; ++k) {
            const int64_t eo = Hl[k] + go, ee = El[k] + ge, fo = hup + go, fe = fup + ge;
            const int64_t E = ee > eo ? ee : eo, F = fe > fo ? fe : fo, d = hd + (k ? m2.y : m2.x);
            const int64_t h = max(d, max(E, F));
            nib = nib << 4 | (uint32_t)((ee > eo) | (fe > fo) << 1 | (d < h) << 2 | (E < F) << 3);
            hd = Hl[k];
            Hl[k] = h;
            El[k] = E;
            hup = h;
            fup = F;
          }
          Hbot = hup;
          Fbot = fup;
          hd0 = Hup0;
          if (writer) {
            ringH[j] = hup;
            ringF[j] = fup;
          }
        }
        acc = acc << 8 | nib;
        if ((q & 3) == 3) tb[(int64_t)(t / 4) * 64] = acc;
      }
      // publish the ring columns stored so far (the writer lane's column)
      if (s + 1 < S) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        const int done = min(max(8 * b + 8 - 63, 0), lb);
        if (lane == 63) __hip_atomic_store(&sy[JS_PROG + wave], (s / W + 1) << 20 | done, __ATOMIC_RELEASE,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  }
}

// A join: the DP, the walk back, the merged columns.  WIDE: values in int64.
template <bool WIDE>
__global__ __launch_bounds__(64 * JWMAX) void msa_join_kernel(JoinArgs A) {
  extern __shared__ __align__(16) uint8_t jlds[];  // the strips' ring of bottom rows
  __shared__ __align__(16) int32_t sy[JS_WORDS];
  __shared__ uint32_t win[StripWindow<JR>::WL * StripWindow<JR>::WD];
  const JoinJob &J = A.jobs[blockIdx.x];
  const int la = J.a.len, lb = J.b.len, tid = threadIdx.x, lane = tid & 63, nthr = blockDim.x, W = nthr >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = join_strips(la), T = join_steps(lb);
  const int go = (int)(A.open * J.w), ge = (int)(A.ext * J.w);  // (not WIDE: they fit)
  uint32_t *tb = A.tb + J.tb_off;
  if (tid < JS_WORDS) sy[tid] = tid == JS_READY ? 0x7fffffff : tid >= JS_EDGE ? 2 * (go - ge) : 0;
  __syncthreads();

  // ---- the DP: strip s on wave s % W; every strip stores its bottom row over
  // the one it read, 63 columns behind
  if constexpr (WIDE) {
    join_sweep_wide(A, J, (int64_t *)jlds, sy, W);
  } else {
    int2 *const ring = (int2 *)jlds;
    for (int s = wave; s < S; s += W) {
      JoinIO io;
      io.ms = (const int2 *)(A.mbuf + J.m_off) + (int64_t)s * T * 64 + lane;
      io.blocks = T / 8;
      io.load(0, 0);
      io.load(0, 1);
      io.status = sy + JS_STATUS;
      io.pin = sy + (s ? JS_PROG + (s - 1) % W : JS_READY);
      io.pout = sy + JS_PROG + wave;
      io.rin = lane ? (int2 *)(sy + JS_ZERO) : s ? ring + 64 : (int2 *)(sy + JS_EDGE);
      io.rin_step = lane == 0 && s ? 8 : 0;
      io.rout = ring;
      io.need0 = s ? ((s - 1) / W + 1) << 20 : 0;
      io.s = s / W;
      io.cols = T - 63;
      io.spin_limit = A.spin_limit;
      io.gave_up = 1;
      io.pl = tb + (int64_t)s * (T / 4) * 64 + lane;
      io.pl_step = 64;
      StripEnd end;
      strip_sweep<JR, false>(io, s, s + 1 == S, la, lb, T, go, ge, end);
    }
  }
  __syncthreads();  // every code of the workgroup is visible to it

  // ---- walk back from (la, lb), a run at a time (wave 0)
  const int cap = la + lb + 2;
  uint32_t *const rend = A.runs + J.run_off + cap;
  if (wave == 0) {
    WaveRuns rw;
    rw.end = rend;
    rw.cap = cap;
    StripWindow<JR> src{tb, win, T, -1, -1};
    int i = la, j = lb, state = 0, steps = 0;
    src.refill(i, j);
    const int how = wave_walk<WALK_GLOBAL>(src, rw, i, j, state, la + lb, steps);
    if (how != WALK_GAVE_UP) {
      if (i == 0 && j > 0) rw.emit(1, j);
      if (j == 0 && i > 0) rw.emit(2, i);
    }
    const bool ok = rw.finish() && how != WALK_GAVE_UP;
    if (lane == 0) {
      sy[JS_RUNS] = ok ? rw.n : 0;
      if (!ok) atomicOr(&sy[JS_STATUS], 2);
    }
  }
  __syncthreads();

  // ---- the merged columns' sources and both sides' maps, a run to a wave
  const int nr = sy[JS_RUNS];
  const uint32_t *runs = rend - nr;
  int2 *const src = A.src + J.src_off;
  int x0 = 0, a0 = 0, b0 = 0;  // columns before run `base`
  for (int base = 0; base < nr; base += 64) {
    const uint32_t v = base + lane < nr ? runs[base + lane] : 0;
    const int op = v & 3, len = (int)(v >> 2);
    int na = op == 1 ? 0 : len, nb = op == 2 ? 0 : len, nx = len;  // inclusive sums over the lanes
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int oa = __shfl_up(na, d, 64), ob = __shfl_up(nb, d, 64), ox = __shfl_up(nx, d, 64);
      if (lane >= d) { na += oa; nb += ob; nx += ox; }
    }
    for (int k = wave; k < min(64, nr - base); k += W) {
      const int o = __builtin_amdgcn_readlane(op, k), l = __builtin_amdgcn_readlane(len, k);
      const int x = x0 + __builtin_amdgcn_readlane(nx, k) - l;
      const int ia = a0 + __builtin_amdgcn_readlane(na, k) - (o == 1 ? 0 : l);
      const int ib = b0 + __builtin_amdgcn_readlane(nb, k) - (o == 2 ? 0 : l);
      for (int e = lane; e < l; e += 64) {
        src[x + e] = make_int2(o == 1 ? -1 : ia + e, o == 2 ? -1 : ib + e);
        if (o != 1) J.a.map[ia + e] = x + e;
        if (o != 2) J.b.map[ib + e] = x + e;
      }
    }
    x0 += __builtin_amdgcn_readlane(nx, 63);
    a0 += __builtin_amdgcn_readlane(na, 63);
    b0 += __builtin_amdgcn_readlane(nb, 63);
  }
  if (tid == 0) {
    A.nops[blockIdx.x] = x0;
    if (sy[JS_STATUS]) atomicOr(A.err, sy[JS_STATUS]);
  }
  if (!J.out) return;
  __syncthreads();
  for (int64_t e = tid; e < (int64_t)x0 * CI; e += nthr) {
    const int x = (int)(e / CI), y = (int)(e % CI);
    const int2 s = src[x];
    int4 v = make_int4(0, 0, 0, 0);
    if (s.x >= 0) v = join_row(J.a, A.leaf, s.x)[y];
    if (s.y >= 0) {
      const int4 u = join_row(J.b, A.leaf, s.y)[y];
      v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
    }
    J.out[e] = v;
  }
}

// Every residue's column in the root: up the tree through the joins' maps.
struct MsaNode {
  const int32_t *map;  // the node's columns in its parent's
  int32_t parent;      // -1: the root
};
__global__ __launch_bounds__(256) void msa_columns_kernel(const MsaNode *nodes, const int64_t *off, int32_t *cols,
                                                          int chunks) {
  const int s = blockIdx.x / chunks;
  const int64_t k = (int64_t)(blockIdx.x % chunks) * 256 + threadIdx.x;
  if (k >= off[s + 1] - off[s]) return;
  int c = (int)k;
  for (int v = s; nodes[v].parent >= 0; v = nodes[v].parent) c = nodes[v].map[c];
  cols[off[s] + k] = c;
}

}  // namespace

int ta_msa(ta_ctx *ctx, const ta_params *p, const char *const *seqs, const int32_t *lens, int32_t nseq,
           int32_t *alen, int32_t *cols, int32_t *joins) {
  if (!ctx || !p || !seqs || !lens || nseq <= 0 || !alen || !cols) return TA_E_INVALID;
  if (p->mode != TA_GLOBAL || p->gap_open > 0 || p->gap_extend > 0) return TA_E_INVALID;
  std::vector<int64_t> off(nseq + 1, 0);
  for (int32_t s = 0; s < nseq; ++s) {
    if (lens[s] <= 0 || !seqs[s]) return TA_E_INVALID;
    off[s + 1] = off[s] + lens[s];
  }
  PhaseTrace tr("msa");  // TWEAKALIGN_TRACE=1: host phase times on stderr
  int8_t S[32 * 32];
  int32_t K = 0;
  int rc = ta_matrix(p->alphabet, p->match, p->mismatch, S, &K);
  if (rc) return rc;
  if (K > KS) return TA_E_INVALID;
  int64_t max_abs_s = 1;
  for (int32_t x = 0; x < K * K; ++x) max_abs_s = std::max<int64_t>(max_abs_s, S[x] < 0 ? -S[x] : S[x]);
  std::vector<uint8_t> codes((size_t)off[nseq]);
  for (int32_t s = 0; s < nseq; ++s)
    if ((rc = ta_encode(p->alphabet, seqs[s], lens[s], codes.data() + off[s]))) return rc;
  if (hipSetDevice(ctx->device) != hipSuccess) return TA_E_DEVICE;
  tr.mark("encode");

  // 1. pair scores on the GPU
  const int32_t nc = 2 * nseq - 1;
  std::vector<int64_t> sum((size_t)nc * nc, 0);
  std::vector<int64_t> self(nseq, 0);
  for (int32_t s = 0; s < nseq; ++s)
    for (int64_t q = off[s]; q < off[s + 1]; ++q) self[s] += S[codes[q] * K + codes[q]];
  if (nseq > 1) {
    std::vector<ta_pair> pairs;
    pairs.reserve((size_t)nseq * (nseq - 1) / 2);
    for (int32_t a = 0; a < nseq; ++a)
      for (int32_t b = a + 1; b < nseq; ++b) pairs.push_back({seqs[a], lens[a], seqs[b], lens[b]});
    ta_params q = *p;
    q.traceback = 0;
    ta_batch *B = nullptr;
    std::vector<ta_result> res(pairs.size());
    rc = batch_create_on(ctx, &q, pairs.data(), (int32_t)pairs.size(), ctx->stream, &B);
    tr.mark("score create");
    if (!rc) rc = ta_batch_run(ctx, B);
    if (!rc) rc = ta_batch_wait(ctx, B);
    tr.mark("score run");
    if (!rc) rc = ta_batch_results(ctx, B, res.data(), nullptr, 0, nullptr);
    if (B) ta_batch_destroy(B);
    if (rc) return rc;
    tr.mark("score results");
    size_t k = 0;
    for (int32_t a = 0; a < nseq; ++a)
      for (int32_t b = a + 1; b < nseq; ++b, ++k) {
        const int64_t d = std::max<int64_t>(1, std::min(self[a], self[b]));
        sum[(size_t)a * nc + b] = sum[(size_t)b * nc + a] = (int64_t)res[k].score * 1000000 / d;
      }
  }

  tr.mark("score sums");
  // 2. UPGMA joins (exact), and each join's tree level.  Row a keeps its
  // best partner b > a (largest mean, ties to the smaller b); the join is the
  // best row's (ties to the smaller a) -- the lexicographically first pair of
  // largest mean.  After a join only rows whose partner died are rescanned;
  // every other row compares its partner with the new cluster.
  std::vector<int32_t> size(nc, 0), level(nc, 0), ja(nseq > 1 ? nseq - 1 : 0), jb(ja.size());
  std::vector<char> live(nc, 0);
  std::vector<int32_t> best(nc, -1);
  for (int32_t s = 0; s < nseq; ++s) { size[s] = 1; live[s] = 1; }
  // mean(a, b) > mean(x, y), exactly
  auto above = [&](int32_t a, int32_t b, int32_t x, int32_t y) {
    return (__int128)sum[(size_t)a * nc + b] * size[x] * size[y] > (__int128)sum[(size_t)x * nc + y] * size[a] * size[b];
  };
  auto rescan = [&](int32_t a, int32_t end) {
    best[a] = -1;
    for (int32_t b = a + 1; b < end; ++b)
      if (live[b] && (best[a] < 0 || above(a, b, a, best[a]))) best[a] = b;
  };
  for (int32_t a = 0; a < nseq; ++a) rescan(a, nseq);
  int32_t top = 0;
  for (int32_t t = 0; t + 1 < nseq; ++t) {
    int32_t ba = -1;
    for (int32_t a = 0; a < nseq + t; ++a)
      if (live[a] && best[a] >= 0 && (ba < 0 || above(a, best[a], ba, best[ba]))) ba = a;
    const int32_t bb = best[ba], c = nseq + t;
    ja[t] = ba; jb[t] = bb;
    if (joins) { joins[2 * t] = ba; joins[2 * t + 1] = bb; }
    size[c] = size[ba] + size[bb];
    level[c] = 1 + std::max(level[ba], level[bb]);
    top = std::max(top, level[c]);
    live[ba] = live[bb] = 0;
    live[c] = 1;
    for (int32_t x = 0; x < c; ++x)
      if (live[x]) sum[(size_t)c * nc + x] = sum[(size_t)x * nc + c] = sum[(size_t)ba * nc + x] + sum[(size_t)bb * nc + x];
    for (int32_t a = 0; a < c; ++a) {
      if (!live[a]) continue;
      if (best[a] == ba || best[a] == bb || best[a] < 0) rescan(a, c + 1);
      else if (above(a, c, a, best[a])) best[a] = c;
    }
  }

  tr.mark("upgma");
  // 3. joins level by level
  hipStream_t st = ctx->stream;
  std::vector<void *> held;  // device blocks of the whole call
  auto hold = [&](size_t bytes) {
    void *d = device_alloc(std::max<size_t>(1, bytes));
    if (d) held.push_back(d);
    return d;
  };
  // A level's merged columns, given back once every cluster in it is joined.
  struct Level {
    void *p;
    int32_t live;
  };
  std::vector<Level> levels;
  struct Free {
    std::vector<void *> &held;
    std::vector<Level> &levels;
    ~Free() {
      for (void *d : held) device_free(d);
      for (const Level &l : levels) device_free(l.p);
    }
  } free_all{held, levels};
  // Rows of single residues, and the sequences' codes.
  std::vector<int32_t> hleaf((size_t)K * 2 * KS, 0);
  for (int32_t x = 0; x < K; ++x) {
    hleaf[(size_t)x * 2 * KS + x] = 1;
    for (int32_t y = 0; y < K; ++y) hleaf[(size_t)x * 2 * KS + KS + y] = S[y * K + x];
  }
  int4 *d_leaf = (int4 *)hold(hleaf.size() * sizeof(int32_t));
  uint8_t *d_codes = (uint8_t *)hold((size_t)off[nseq]);
  int32_t *d_err = (int32_t *)hold(sizeof(int32_t));
  if (!d_leaf || !d_codes || !d_err) return TA_E_NOMEM;
  if (hipMemsetAsync(d_err, 0, sizeof(int32_t), st) ||
      hipMemcpyAsync(d_leaf, hleaf.data(), hleaf.size() * sizeof(int32_t), hipMemcpyHostToDevice, st) ||
      hipMemcpyAsync(d_codes, codes.data(), (size_t)off[nseq], hipMemcpyHostToDevice, st) || hipStreamSynchronize(st))
    return TA_E_DEVICE;
  struct Cluster {
    int32_t len = 0, rows = 1, level = -1;  // level: index into `levels`, -1 a sequence
    const int4 *tab = nullptr;
  };
  std::vector<Cluster> cl(nc);
  std::vector<MsaNode> nodes(nc, MsaNode{nullptr, -1});
  for (int32_t s = 0; s < nseq; ++s) cl[s].len = lens[s];
  const int64_t gap_w = -((int64_t)p->gap_open + p->gap_extend);
  for (int32_t L = 1; L <= top; ++L) {
    std::vector<int32_t> ts;
    for (int32_t t = 0; t + 1 < nseq; ++t)
      if (level[nseq + t] == L) ts.push_back(t);
    const int32_t nj = (int32_t)ts.size();
    std::vector<JoinJob> jobs(nj);
    int64_t tb_total = 0, run_total = 0, col_total = 0, m_total = 0;
    int32_t max_lb = 0, strips = 0, tiles = 0;
    bool wide = false;  // some join's DP values need int64
    bool m24 = true;    // every count and PB entry fits 24 bits
    for (int32_t q = 0; q < nj; ++q) {
      const Cluster &ca = cl[ja[ts[q]]], &cb = cl[jb[ts[q]]];
      JoinJob &J = jobs[q];
      J.a = {ca.tab ? nullptr : d_codes + off[ja[ts[q]]], ca.tab, nullptr, ca.len};
      J.b = {cb.tab ? nullptr : d_codes + off[jb[ts[q]]], cb.tab, nullptr, cb.len};
      J.w = (int64_t)ca.rows * cb.rows;
      // joins whose column scores could leave int32
      if (J.w > WMAX || (int64_t)ca.len * cb.len > INT32_MAX) return TA_E_INVALID;
      const int64_t c = (int64_t)p->gap_open - p->gap_extend;
      const int64_t reach = std::min(ca.len, cb.len) * (max_abs_s - 2ll * p->gap_extend) +
                            (ca.len + cb.len + 2) * std::max<int64_t>(0, c) + 4 * (gap_w + max_abs_s);
      if (reach >= (1ll << 30) / J.w) wide = true;
      if (std::max(ca.rows, cb.rows) * max_abs_s >= (1 << 23)) m24 = false;
      const int64_t S = join_strips(ca.len), T = join_steps(cb.len);
      J.m_off = m_total;
      m_total += S * T * 64 * JR;
      J.tb_off = tb_total;
      tb_total += S * (T / 4) * 64;
      J.run_off = run_total;
      run_total += ca.len + cb.len + 2;
      J.src_off = col_total;
      col_total += ca.len + cb.len;
      max_lb = std::max(max_lb, cb.len);
      strips = (int32_t)std::max<int64_t>(strips, S);
      tiles = (int32_t)std::max<int64_t>(tiles, S * ((T + 63) / 64));
    }
    // The ring holds a bottom row of every column: 20,017 of them fit a CU's
    // LDS (10,078 in int64).  A larger launch would take the whole queue down.
    if (join_ring_bytes(max_lb, wide) + JOIN_LDS > ctx->lds_max) return TA_E_INVALID;
    const bool root = L == top;
    int32_t *d_map = (int32_t *)hold(sizeof(int32_t) * (size_t)col_total);
    int4 *d_out = root ? nullptr : (int4 *)device_alloc(sizeof(int4) * CI * (size_t)col_total);
    if (d_out) levels.push_back({d_out, nj});
    for (int32_t q = 0; q < nj && d_map; ++q) {
      JoinJob &J = jobs[q];
      J.a.map = d_map + J.src_off;
      J.b.map = J.a.map + J.a.len;
      J.out = d_out ? d_out + J.src_off * CI : nullptr;
      nodes[ja[ts[q]]] = {J.a.map, nseq + ts[q]};
      nodes[jb[ts[q]]] = {J.b.map, nseq + ts[q]};
    }
    tr.mark("level sizes");
    std::vector<int32_t> hnops(nj);
    int32_t herr = 0;
    JoinArgs a{};
    JoinJob *d_jobs = (JoinJob *)device_alloc(sizeof(JoinJob) * nj);
    a.jobs = d_jobs;
    a.leaf = d_leaf;
    a.mbuf = (int32_t *)device_alloc(sizeof(int32_t) * (size_t)m_total);
    a.tb = (uint32_t *)device_alloc(sizeof(uint32_t) * (size_t)tb_total);
    a.runs = (uint32_t *)device_alloc(sizeof(uint32_t) * (size_t)run_total);
    a.src = (int2 *)device_alloc(sizeof(int2) * (size_t)col_total);
    a.nops = (int32_t *)device_alloc(sizeof(int32_t) * nj);
    a.err = d_err;
    a.open = p->gap_open; a.ext = p->gap_extend;
    a.spin_limit = 1 << 22;
    rc = (d_map && (root || d_out) && d_jobs && a.mbuf && a.tb && a.runs && a.src && a.nops) ? TA_OK : TA_E_NOMEM;
    if (!rc) {
      (void)hipGetLastError();
      if (hipMemcpyAsync(d_jobs, jobs.data(), sizeof(JoinJob) * nj, hipMemcpyHostToDevice, st)) rc = TA_E_DEVICE;
      // the match scores over the whole GPU, then the joins
      const dim3 grid((unsigned)nj, (unsigned)std::min(tiles, 65535));
      if (!rc) hipLaunchKernelGGL(m24 ? msa_scores_kernel<true> : msa_scores_kernel<false>, grid, dim3(256), 0, st, a,
                                  wide ? 0 : -p->gap_open - p->gap_extend, wide ? 0 : p->gap_extend - p->gap_open);
      const size_t lds = (size_t)join_ring_bytes(max_lb, wide);
      if (!rc) hipLaunchKernelGGL(wide ? msa_join_kernel<true> : msa_join_kernel<false>, dim3((unsigned)nj),
                                  dim3(64 * std::min(strips, JWMAX)), lds, st, a);
      if (rc || hipGetLastError() != hipSuccess ||
          hipMemcpyAsync(hnops.data(), a.nops, sizeof(int32_t) * nj, hipMemcpyDeviceToHost, st) ||
          hipMemcpyAsync(&herr, d_err, sizeof(int32_t), hipMemcpyDeviceToHost, st) || hipStreamSynchronize(st))
        rc = TA_E_DEVICE;
      if (rc) (void)hipStreamSynchronize(st);
      if (!rc && herr) {
        fprintf(stderr, "tweakalign: %s gave up (msa join)\n", herr & 1 ? "a wait on another wave's progress" : "a walk");
        rc = TA_E_DEVICE;
      }
    }
    device_free(d_jobs); device_free(a.mbuf); device_free(a.tb); device_free(a.runs); device_free(a.src);
    device_free(a.nops);
    if (rc) return rc;
    for (int32_t q = 0; q < nj; ++q) {
      const int32_t t = ts[q];
      for (const int32_t child : {ja[t], jb[t]})
        if (cl[child].level >= 0 && --levels[cl[child].level].live == 0) {
          device_free(levels[cl[child].level].p);
          levels[cl[child].level].p = nullptr;
        }
      cl[nseq + t] = {hnops[q], cl[ja[t]].rows + cl[jb[t]].rows, root ? -1 : (int32_t)levels.size() - 1, jobs[q].out};
    }
    tr.mark("level gpu");
  }

  // 4. every residue's column
  *alen = cl[nc - 1].len;
  int32_t *d_cols = (int32_t *)hold(sizeof(int32_t) * (size_t)off[nseq]);
  int64_t *d_off = (int64_t *)hold(sizeof(int64_t) * (nseq + 1));
  MsaNode *d_nodes = (MsaNode *)hold(sizeof(MsaNode) * nc);
  if (!d_cols || !d_off || !d_nodes) return TA_E_NOMEM;
  const int32_t chunks = (*std::max_element(lens, lens + nseq) + 255) / 256;
  (void)hipGetLastError();
  rc = hipMemcpyAsync(d_off, off.data(), sizeof(int64_t) * (nseq + 1), hipMemcpyHostToDevice, st) ||
               hipMemcpyAsync(d_nodes, nodes.data(), sizeof(MsaNode) * nc, hipMemcpyHostToDevice, st)
           ? TA_E_DEVICE
           : TA_OK;
  if (!rc)
    hipLaunchKernelGGL(msa_columns_kernel, dim3((unsigned)nseq * (unsigned)chunks), dim3(256), 0, st, d_nodes, d_off,
                       d_cols, chunks);
  if (rc || hipGetLastError() != hipSuccess ||
      hipMemcpyAsync(cols, d_cols, sizeof(int32_t) * (size_t)off[nseq], hipMemcpyDeviceToHost, st))
    rc = TA_E_DEVICE;
  if (hipStreamSynchronize(st) != hipSuccess || rc) return TA_E_DEVICE;  // (nothing queued reads the blocks after)
  tr.mark("columns");
  return TA_OK;
}
