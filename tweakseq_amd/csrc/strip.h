// One strip of a pair's DP in int32, swept by a wave for latency.
//
// A strip is 64 lanes x PR query rows; lane l works on column t - l at step
// t, its bottom row going to the next lane one step later.  What a single
// wave takes per step is its instruction count (it issues about one every 5.3
// cycles), so the step is kept short: 210 cycles for 2 rows (322 with the
// plain recurrence, a column test, codes passed from lane to lane and
// branches inside the block).
//  * Global values are held as G = H - ext (i + j) + (open - ext).  In these
//    terms extending a gap costs nothing, a gap opens at G, and the diagonal
//    adds S + |open| + |ext|:
//        E = max(E, G_left)   F = max(F, G_up)   H = max(G_diag + S', E, F)
//        G = H + (open - ext)
//    five operations a cell instead of eight, one value (G) kept for all
//    three neighbours.  Every comparison is between values of one cell, which
//    shift alike, so the direction bits are those of the plain recurrence.
//  * Local values are H, and X = max(H - |open|, 0); E and F are floored at 0
//    (unsigned saturating subtractions), which needs no floor for H.
//  * The row above reaches a lane as `v_add_u32_dpp`: the lane above's value,
//    or 0 in lane 0, plus a register that holds lane 0's top input and 0 in
//    the other lanes.  F is handed down as the next row's finished maximum.
//  * A lane's PR scores of a column come from its own slot, [code][lane]
//    (conflict-free); the address is one v_perm of the packed column codes
//    and the lane's base, the codes of 8 columns one unaligned read.
//  * Direction bits are sign bits of differences, shifted into a dword by
//    v_alignbit; a dword holds 8 / PR steps.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"

namespace ta {

typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) const uint32_t lds_cu32;

// Steps a dword of direction codes holds.
__host__ __device__ constexpr int strip_spd(int PR) { return 8 / PR; }
// A dword's code of step offset q (t mod SPD), row k of the lane: e f d x in bits 0..3.
template <int PR>
__device__ __forceinline__ int strip_code(uint32_t dw, int q, int k) { return (int)(dw >> (28 - 4 * (q * PR + k))) & 15; }

// Score slots: a row of 64 entries per code; an entry holds a lane's rows, int32 for
// one row, int16 pairs for two, PR / 2 tables of such pairs for more (NC rows apart),
// or int8 quadruples in PR / 4 tables (BYTES; where every score fits).
constexpr int STRIP_NC = 24;                  // codes (23 residues and a pad)
constexpr int STRIP_NC_DNA = 8;               // 4 and a pad
constexpr int STRIP_ROW = 256;                // bytes per code
__host__ __device__ constexpr int strip_slot_tables(int PR, bool BYTES) { return PR <= 2 ? 1 : PR / (BYTES ? 4 : 2); }
__host__ __device__ constexpr int strip_slot_bytes(int PR, int NC = STRIP_NC, bool BYTES = false) {
  return strip_slot_tables(PR, BYTES) * NC * STRIP_ROW;
}

// Fills the calling lane's slot entries at LDS byte `slot` + 4 lane: row k's score
// against code c < nc is line[k][c] + bias (line: 32-byte table lines in LDS); code
// nc, the pad outside the columns, scores `pad`.
template <int PR, int NC = STRIP_NC, bool BYTES = false>
__device__ __forceinline__ void strip_slot(uint8_t *slot, const uint8_t *const (&line)[PR], int nc, int bias, int pad) {
  const int lane = threadIdx.x & 63;
  for (int c4 = 0; c4 <= nc; c4 += 4) {
    uint32_t w[PR];
#pragma unroll
    for (int k = 0; k < PR; ++k) w[k] = *(const uint32_t *)(line[k] + c4);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      uint32_t *d = (uint32_t *)(slot + (c4 + b) * STRIP_ROW) + lane;
      int v[PR];
#pragma unroll
      for (int k = 0; k < PR; ++k) v[k] = c4 + b == nc ? pad : (int)(int8_t)(w[k] >> (8 * b)) + bias;
      if constexpr (PR == 1) {
        d[0] = (uint32_t)v[0];
      } else if constexpr (BYTES) {
#pragma unroll
        for (int k = 0; k < PR; k += 4)
          d[(k / 4) * NC * STRIP_ROW / 4] = ((uint32_t)v[k] & 0xffu) | (((uint32_t)v[k + 1] & 0xffu) << 8) |
                                            (((uint32_t)v[k + 2] & 0xffu) << 16) | ((uint32_t)v[k + 3] << 24);
      } else {
#pragma unroll
        for (int k = 0; k < PR; k += 2)
          d[(k / 2) * NC * STRIP_ROW / 4] = ((uint32_t)v[k] & 0xffffu) | ((uint32_t)v[k + 1] << 16);
      }
    }
  }
}

__device__ __forceinline__ int strip_satsub(int x, int g) {
  return (int)__builtin_elementwise_sub_sat((uint32_t)x, (uint32_t)g);
}

// The strip's outcome: global, H(m, n) in the lane that owns row m (has = true);
// local, the lane's best cell (h 0: none), 1-based.
struct StripEnd {
  int h = 0, i = 0x7fffffff, j = 0x7fffffff;
  bool has = false;
};

// (h desc, i asc, j asc): the local end-cell order.
__device__ __forceinline__ bool strip_better(int h, int i, int j, int bh, int bi, int bj) {
  return h > bh || (h == bh && (i < bi || (i == bi && j < bj)));
}

// What most strips' surroundings have in common: direction codes kept, the
// matrix's own left border, no columns kept, scores from slots.
struct StripIODefaults {
  static constexpr bool TB = true, KEEP = false, BYTES = false, SLOTS = true;
  static constexpr int NC = STRIP_NC;
  static constexpr const int2 *left = nullptr;
  __device__ __forceinline__ bool keeps(int) const { return false; }
  template <int PR>
  __device__ __forceinline__ void column(int, const int (&)[PR], const int (&)[PR]) const {}
};

// Strip s (0-based) of an m x n pair over T = n + 63 steps (rounded up to 8).
// IO is the strip's surroundings:
//   SLOTS (scores from this wave's slot):
//   uint64_t codes(b)            the codes of this lane's 8 columns of block b <= T / 8 (pads outside the columns)
//   uint32_t slot_add            added to every 4 packed codes (the slot's first row, in each byte)
//   or scores(b, half, v)        the scores of 4 of this lane's steps, each row's, |open| + |ext| added, and pads
//   void peek(), await(b)        reads the strip above's progress; waits until that strip has stored block
//                                b's columns (b <= T / 8), of the T - 63 it stores
//   void tops(b, half, g, f)     4 of those columns' bottom row, in lane 0, and 0 in the others; above the
//                                first strip every value is the border's (0, or 2 (open - ext)), and local
//                                columns from T - 63 on are 0
//   void bottom(b, g, f)         this strip's bottom row after block b, in lane 63 (columns 8 b - 63 ..)
//   void planes(dw)              the next dword of direction codes (SPD steps; IO::TB only)
//   bool keeps(b)                IO::KEEP: whether block b calls column(c, G, E) after each step, c the lane's column
//   const int2 *left             (G, E) of the lane's rows in the column left of the strip's first, null at the
//                                matrix border; the rows above it precede it
// Local columns and H stay below 2^16 - 128 (the end-cell keys).
//
// Lanes left or right of the columns run along on pads: left of column 0 the
// pad's score reproduces the border (global: H = open - ext in G's terms,
// which needs |open| >= |ext|; else those blocks are masked by column; local:
// 0), right of the last column the values go nowhere.  So no step tests its
// column but the last ones of the strip that holds row m, which keep H(m, n).
// Strips that start inside the matrix (io.left) mask their first blocks too.
template <int PR, bool LOCAL, class IO>
__device__ __forceinline__ void strip_sweep(IO &io, int s, bool last, int m, int n, int T, int open, int ext,
                                            StripEnd &end) {
  constexpr bool TB = IO::TB;
  constexpr int SPD = TB ? strip_spd(PR) : 1, NS = IO::SLOTS ? strip_slot_tables(PR, IO::BYTES) : PR;
  const int lane = threadIdx.x & 63;
  const int r0 = (s * 64 + lane) * PR;  // 0-based first row of the lane
  const int c = open - ext, go = -open, ge = -ext;
  const int edge = LOCAL ? 0 : 2 * c;   // G (local: H) along the left border and above the first row
  int G[PR], E[PR], X[PR], cap[PR];
  uint32_t key[PR];
#pragma unroll
  for (int k = 0; k < PR; ++k) { G[k] = edge; E[k] = edge; X[k] = 0; key[k] = 0; cap[k] = 0; }
  int hd = (!LOCAL && r0 == 0) ? c : edge;  // the row above at the previous column
  const bool inner = !LOCAL && io.left != nullptr;
  if (inner) {
#pragma unroll
    for (int k = 0; k < PR; ++k) {
      const int2 v = io.left[k];
      G[k] = v.x;
      E[k] = v.y;
    }
    hd = r0 == 0 ? edge : io.left[-1].x;
  }
  int Gb = edge, Fb = edge;                 // handed to the lane below
  int tg[8], tf[8];                         // lane 0's top inputs, each half read once its last values are used
  io.peek();
  io.await(0);
  io.tops(0, 0, tg, tf);
  const uint32_t lbase = 4u * (uint32_t)lane;
  // Scores of 4 steps, read half a block ahead: from 4 packed codes, or from the IO.
  struct Sc { std::conditional_t<IO::SLOTS, uint32_t, int> v[4][NS]; } sa, sb;  // of the block's first and second half
  auto fetch = [&](uint32_t w, Sc &sc) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // byte 1 = code q's slot row, byte 0 = 4 lane
      const uint32_t a = __builtin_amdgcn_perm(w, lbase, 0x0c0c0000u | ((uint32_t)(4 + q) << 8));
#pragma unroll
      for (int x = 0; x < NS; ++x) sc.v[q][x] = *(lds_cu32 *)(uintptr_t)(a + x * IO::NC * STRIP_ROW);
    }
  };
  auto score = [](const Sc &sc, int q, int k) {
    if constexpr (!IO::SLOTS) return (int)sc.v[q][k];
    if constexpr (IO::BYTES) return (int)(int8_t)(sc.v[q][k >> 2] >> (8 * (k & 3)));
    const uint32_t w = (uint32_t)sc.v[q][PR > 2 && !IO::BYTES ? k >> 1 : 0];
    return PR == 1 ? (int)w : (k & 1) ? (int)w >> 16 : (int)(int16_t)w;
  };
  uint64_t cw = 0;   // the codes of the next block, then its second half's
  uint32_t w1 = 0;
  if constexpr (IO::SLOTS) {
    cw = io.codes(0);
    w1 = (uint32_t)(cw >> 32) + io.slot_add;
    fetch((uint32_t)cw + io.slot_add, sa);
  } else {
    io.scores(0, 0, sa.v);
  }
  // The row whose direction bits are still to be taken, and the row at hand.
  struct Pending {
    int En, F, D, H, up, oe;
    uint32_t x, dd, f, e, z, kv, kc;
  } pd{};
  int Gu = 0, up = 0, F = 0, En = 0, D = 0, t2 = 0;
  uint32_t acc = 0;
  const int NB = T / 8;
  // One block: masked (first blocks), plain, or keeping H(m, n) (last blocks).
  auto block = [&](int b, auto mode_tag) {
    constexpr int MODE = decltype(mode_tag)::value;
    const int tb = 8 * b;
    int rg[8], rf[8];
    // Four steps, masked on the left by column.
    [[maybe_unused]] auto masked_steps = [&](auto q0_tag) {
      constexpr int Q0 = decltype(q0_tag)::value;
#pragma unroll
      for (int q = Q0; q < Q0 + 4; ++q) {
        const int Gu0 = __builtin_amdgcn_update_dpp(0, Gb, 0x138, 0xf, 0xf, true) + tg[q];
        const int Fu0 = __builtin_amdgcn_update_dpp(0, Fb, 0x138, 0xf, 0xf, true) + tf[q];
        uint32_t nib = 0;
        const int c0 = tb + q - lane;
        if (c0 >= 0) {
          int upk = Gu0, Fk = Fu0, d = hd;
#pragma unroll
          for (int k = 0; k < PR; ++k) {
            const int Dk = d + score(Q0 ? sb : sa, q - Q0, k), Ek = max(E[k], G[k]), H = max(Dk, max(Ek, Fk));
            if constexpr (TB) {
              nib = __builtin_amdgcn_alignbit(nib, (uint32_t)(Ek - Fk), 31);
              nib = __builtin_amdgcn_alignbit(nib, (uint32_t)(Dk - H), 31);
              nib = __builtin_amdgcn_alignbit(nib, (uint32_t)(upk - Fk), 31);
              nib = __builtin_amdgcn_alignbit(nib, (uint32_t)(G[k] - Ek), 31);
            }
            d = G[k];
            E[k] = Ek;
            upk = G[k] = H + c;
            Fk = max(Fk, upk);
          }
          Gb = G[PR - 1];
          Fb = Fk;
          hd = Gu0;
        }
        if constexpr (TB) {
          acc = ((PR == 8 ? 0u : acc << (4 * (PR & 7))) | nib);
          if ((q + 1) % SPD == 0) io.planes(acc);
        }
        rg[q] = Gb;
        rf[q] = Fb;
#pragma unroll
        for (int k = 0; k < PR; ++k) cap[k] = c0 == n - 1 ? G[k] : cap[k];
        if constexpr (IO::KEEP) io.column(c0, G, E);
      }
    };
    // Four steps.  The order is pinned: each operation of a row's recurrence
    // (one dependent chain) is followed by one of the previous row's
    // direction bits, and the reads of the next half's scores stay ahead.
#define STRIP_PIN __builtin_amdgcn_sched_barrier(0)
    auto pend = [&](auto i_tag, int row) {  // the i-th operation of the pending row's bits
      constexpr int I = decltype(i_tag)::value;
      if constexpr (LOCAL) {  // H = 0 (H >= 0 always): d = 0, x = 1; x = 0 on diagonal cells
        if constexpr (I == 0) pd.x = (uint32_t)(pd.En - pd.F);
        if constexpr (I == 1) pd.dd = (uint32_t)(pd.D - pd.H);
        if constexpr (I == 2) pd.z = (uint32_t)(pd.H - 1);
        if constexpr (I == 3) pd.f = (uint32_t)(pd.up - pd.F);
        if constexpr (I == 4) pd.x = (pd.x & pd.dd) | pd.z;
        if constexpr (I == 5) pd.dd &= ~pd.z;
        if constexpr (I == 6) pd.e = (uint32_t)(pd.oe - pd.En);
        if constexpr (I == 7) acc = __builtin_amdgcn_alignbit(acc, pd.x, 31);
        if constexpr (I == 8) pd.kv = ((uint32_t)pd.H << 16) | pd.kc;
        if constexpr (I == 9) acc = __builtin_amdgcn_alignbit(acc, pd.dd, 31);
        if constexpr (I == 10) key[row] = max(key[row], pd.kv);
        if constexpr (I == 11) acc = __builtin_amdgcn_alignbit(acc, pd.f, 31);
        if constexpr (I == 12) acc = __builtin_amdgcn_alignbit(acc, pd.e, 31);
      } else {
        if constexpr (I == 0) pd.x = (uint32_t)(pd.En - pd.F);
        if constexpr (I == 1) pd.dd = (uint32_t)(pd.D - pd.H);
        if constexpr (I == 2) acc = __builtin_amdgcn_alignbit(acc, pd.x, 31);
        if constexpr (I == 3) pd.f = (uint32_t)(pd.up - pd.F);
        if constexpr (I == 4) acc = __builtin_amdgcn_alignbit(acc, pd.dd, 31);
        if constexpr (I == 5) pd.e = (uint32_t)(pd.oe - pd.En);
        if constexpr (I == 6) acc = __builtin_amdgcn_alignbit(acc, pd.f, 31);
        if constexpr (I == 7) acc = __builtin_amdgcn_alignbit(acc, pd.e, 31);
      }
      STRIP_PIN;
    };
#define STRIP_PEND(i) \
  if (have) pend(std::integral_constant<int, i>{}, row)
    auto steps = [&](auto cap_tag, auto keep_tag, auto q0_tag) {
      constexpr bool CAP = decltype(cap_tag)::value, KEEP = decltype(keep_tag)::value;
      constexpr int Q0 = decltype(q0_tag)::value;
#pragma unroll
      for (int q = Q0; q < Q0 + 4; ++q) {
#pragma unroll
        for (int k = 0; k < PR; ++k) {
          const bool have = TB && (q > 0 || k > 0);  // a row is pending (a block starts without)
          const bool lastrow = k == PR - 1;
          int row = (k + PR - 1) % PR;       // its row of the lane
          if (k == 0 && q == 0) {  // the block's first row: nothing to pair with
            Gu = __builtin_amdgcn_update_dpp(0, Gb, 0x138, 0xf, 0xf, true) + tg[0];
            F = __builtin_amdgcn_update_dpp(0, Fb, 0x138, 0xf, 0xf, true) + tf[0];
            up = LOCAL ? strip_satsub(Gu, go) : Gu;
            En = max(LOCAL ? strip_satsub(E[0], ge) : E[0], LOCAL ? X[0] : G[0]);
            D = hd + score(sa, 0, 0);
            if constexpr (LOCAL) t2 = strip_satsub(F, ge);
            STRIP_PIN;
          }
          const int H = max(D, max(En, F));
          STRIP_PIN;
          STRIP_PEND(0);
          const int Gn = LOCAL ? strip_satsub(H, go) : H + c;
          STRIP_PIN;
          STRIP_PEND(1);
          const int Fn = max(LOCAL ? t2 : F, Gn);
          STRIP_PIN;
          STRIP_PEND(2);
          const int oe = LOCAL ? X[k] : G[k], oldG = G[k];
          E[k] = En;
          G[k] = LOCAL ? H : Gn;
          if constexpr (LOCAL) X[k] = Gn;
          // the next row (of this step, or row 0 of the next): its E, its diagonal, the row above it
          const int nk = lastrow ? 0 : k + 1;
          int En1 = 0, D1 = 0, Gu1 = 0, Fu1 = 0, up1 = 0, t1 = 0;
          const bool next = !(lastrow && q == 7);
          if constexpr (LOCAL) {
            if (next) {
              t1 = strip_satsub(E[nk], ge);
              STRIP_PIN;
            }
            STRIP_PEND(3);
          }
          if (next) {
            En1 = LOCAL ? max(t1, X[nk]) : max(E[nk], G[nk]);
            STRIP_PIN;
          }
          if constexpr (LOCAL) {
            STRIP_PEND(4);
            STRIP_PEND(5);
          } else {
            STRIP_PEND(3);
            STRIP_PEND(4);
          }
          if (next && lastrow) {
            Fu1 = __builtin_amdgcn_update_dpp(0, Fn, 0x138, 0xf, 0xf, true) + tf[(q + 1) & 7];
            STRIP_PIN;
          }
          STRIP_PEND(LOCAL ? 6 : 5);
          if (next && lastrow) {
            Gu1 = __builtin_amdgcn_update_dpp(0, G[PR - 1], 0x138, 0xf, 0xf, true) + tg[(q + 1) & 7];
            STRIP_PIN;
          }
          STRIP_PEND(LOCAL ? 7 : 6);
          if (next) {
            const int qs = lastrow ? q + 1 : q;
            D1 = (lastrow ? Gu : oldG) + score(qs < 4 ? sa : sb, qs & 3, nk);
            STRIP_PIN;
          }
          if constexpr (LOCAL) {
            STRIP_PEND(8);
            if (next) {
              t1 = strip_satsub(lastrow ? Fu1 : Fn, ge);
              STRIP_PIN;
            }
            STRIP_PEND(9);
            if (next && lastrow) {
              up1 = strip_satsub(Gu1, go);
              STRIP_PIN;
            }
            STRIP_PEND(10);
            STRIP_PEND(11);
            STRIP_PEND(12);
          } else {
            STRIP_PEND(7);
          }
          if (TB && k == 0 && q % SPD == 0 && q > 0) io.planes(acc);  // the step before is complete
          pd.En = En; pd.F = F; pd.D = D; pd.H = H; pd.up = up; pd.oe = oe;
          pd.kc = (uint32_t)(0xFFBF - (tb + q - lane));
          if (lastrow) {
            Gb = G[PR - 1];
            Fb = Fn;
            rg[q] = Gb;
            rf[q] = Fb;
            hd = Gu;
            if constexpr (CAP) {
              const bool here = tb + q == n - 1 + lane;
#pragma unroll
              for (int x = 0; x < PR; ++x) cap[x] = here ? G[x] : cap[x];
            }
            if constexpr (KEEP) io.column(tb + q - lane, G, E);
          }
          if (next) {
            En = En1; D = D1;
            if constexpr (LOCAL) t2 = t1;
            if (lastrow) {
              up = LOCAL ? up1 : Gu1;
              F = Fu1;
              Gu = Gu1;
            } else {
              up = Gn;
              F = Fn;
            }
          } else if constexpr (TB) {  // the block's last row: its bits, and its dword
            const bool have = true;
            row = PR - 1;
            STRIP_PEND(0); STRIP_PEND(1); STRIP_PEND(2); STRIP_PEND(3);
            STRIP_PEND(4); STRIP_PEND(5); STRIP_PEND(6); STRIP_PEND(7);
            if constexpr (LOCAL) {
              STRIP_PEND(8); STRIP_PEND(9); STRIP_PEND(10); STRIP_PEND(11); STRIP_PEND(12);
            }
            io.planes(acc);
          }
        }
      }
    };
    auto half = [&](auto q0_tag) {
      if constexpr (MODE == 0) masked_steps(q0_tag);
      else steps(std::integral_constant<bool, MODE == 2>{}, std::integral_constant<bool, IO::KEEP && MODE >= 2>{}, q0_tag);
    };
    if constexpr (IO::SLOTS) cw = io.codes(b + 1);
    io.tops(b, 1, tg, tf);
    io.peek();
    if constexpr (IO::SLOTS) fetch(w1, sb);
    else io.scores(b, 1, sb.v);
    __builtin_amdgcn_sched_barrier(0);
    half(std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (IO::SLOTS) {
      w1 = (uint32_t)(cw >> 32) + io.slot_add;
      fetch((uint32_t)cw + io.slot_add, sa);
    } else {
      io.scores(b + 1, 0, sa.v);
    }
    io.await(b + 1);
    io.tops(b + 1, 0, tg, tf);
    __builtin_amdgcn_sched_barrier(0);
    half(std::integral_constant<int, 4>{});
    if (!last) io.bottom(b, rg, rf);
  };
  int b = 0;
  if constexpr (!LOCAL) {
    if (c > 0 || inner)
      for (; b < 8 && b < NB; ++b) block(b, std::integral_constant<int, 0>{});
    for (const int kb = last && n > 0 ? (n - 1) / 8 : NB; b < kb; ++b) {
      if constexpr (IO::KEEP) {
        if (io.keeps(b)) {
          block(b, std::integral_constant<int, 3>{});
          continue;
        }
      }
      block(b, std::integral_constant<int, 1>{});
    }
    for (; b < NB; ++b) block(b, std::integral_constant<int, 2>{});
  } else {
    for (; b < NB; ++b) block(b, std::integral_constant<int, 1>{});
  }
  if constexpr (LOCAL) {
#pragma unroll
    for (int k = 0; k < PR; ++k) {
      const int h = (int)(key[k] >> 16), j = 0xFFC0 - (int)(key[k] & 0xffff);
      if (r0 + k < m && h > 0 && strip_better(h, r0 + k + 1, j, end.h, end.i, end.j)) {
        end.h = h; end.i = r0 + k + 1; end.j = j;
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < PR; ++k)
      if (r0 + k + 1 == m) { end.h = cap[k] - c + ext * (m + n); end.has = true; }
  }
}

// A strip whose neighbours are in its workgroup: their bottom rows in LDS rings
// (column x at entry x + 64), a progress counter each.
struct StripGroupIO : StripIODefaults {
  const uint8_t *bcode;      // this lane's first column code, at step 0
  uint32_t slot_add;
  int32_t *pin, *pout, *status;
  int2 *rin, *rout;          // rin: lane 0's entries (strip 0: 8 border entries), the others' 8 zero entries
  int rin_step, need0, cols, s, spin_limit, seen = 0;
  uint32_t *pl;              // this lane's next dword, pl_step apart (a lane past the query: one unused dword)
  int pl_step;
  int gave_up;               // OR-ed into *status when a wait gives up
  bool lost = false;         // a wait gave up: no more waits

  __device__ __forceinline__ uint64_t codes(int b) const {
    uint64_t w;
    __builtin_memcpy(&w, bcode + 8 * b, 8);
    return w;
  }
  __device__ __forceinline__ int need(int b) const { return need0 | (8 * b + 8 < cols ? 8 * b + 8 : cols); }
  __device__ __forceinline__ void peek() {
    seen = __hip_atomic_load(pin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ void await(int b) {
    const int want = need(b);
    int spins = 0;
    while (!lost && __builtin_amdgcn_readfirstlane(seen) < want) {
      if (++spins > spin_limit) {
        if ((threadIdx.x & 63) == 0) atomicOr(status, gave_up);
        lost = true;
      }
      __builtin_amdgcn_s_sleep(1);
      peek();
    }
    asm volatile("" ::: "memory");  // the ring's reads stay below (a wave's LDS accesses keep their order)
  }
  __device__ __forceinline__ void tops(int b, int half, int (&g)[8], int (&f)[8]) const {
    const int4 *r = (const int4 *)(rin + b * rin_step) + 2 * half;
    const int4 v = r[0], w = r[1];
    const int q = 4 * half;
    g[q] = v.x; f[q] = v.y; g[q + 1] = v.z; f[q + 1] = v.w;
    g[q + 2] = w.x; f[q + 2] = w.y; g[q + 3] = w.z; f[q + 3] = w.w;
  }
  __device__ __forceinline__ void bottom(int b, const int (&g)[8], const int (&f)[8]) {
    if ((threadIdx.x & 63) == 63) {
      int2 *r = rout + 8 * b + 1;
#pragma unroll
      for (int q = 0; q < 8; ++q) r[q] = make_int2(g[q], f[q]);
      int done = 8 * b + 8 - 63;
      done = done < 0 ? 0 : done;
      asm volatile("" ::: "memory");  // the entries first (a wave's LDS accesses keep their order)
      __hip_atomic_store(pout, ((s + 1) << 20) | done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __device__ __forceinline__ void planes(uint32_t dw) {
    *pl = dw;
    pl += pl_step;
  }
};

// Codes in device memory ([strip][t / SPD][64 lanes]): a window of them in
// LDS, 64 strip lanes' rows up from the walk's cell, for each lane WD dwords
// around the diagonal through it.  A thread brings one strip lane's dwords:
// one address and WD loads.  The window above is on its way while one is
// walked, placed on the same diagonal; a walk that leaves it fetches its own.
// (Windows of 32 lanes fetched when needed, and the shorter lookups of long
// gaps and gaps of one, before / now: 48 DNA pairs 1,662 / 1,068 us, requests
// of 8 pairs of up to 2,500 202 / 137, 16 unrelated pairs of up to 5,000
// 239 / 219, a pair of 1,500 53 / 43.)
template <int PR>
struct StripWindow {
  static constexpr int SPD = strip_spd(PR), WL = 64, WD = 32 / SPD + 1;
  const uint32_t *pl;
  uint32_t *win;  // WL x WD
  int T;
  int L0, u0;     // the window's first (lowest) lane, counted over all strips, and its 0-based column
  uint32_t nx[WD] = {};    // the next window: this thread's lane
  int nL0 = -1, nu0 = 0;   // (nL0 < 0: none)
  // (arithmetic shifts: positions left of the columns are negative)
  static __device__ __forceinline__ int dword(int t) { return t >> (SPD == 8 ? 3 : SPD == 4 ? 2 : 1); }
  // where a window on (l0, c0) holds the dword of lane L's column u; -1: not
  __device__ __forceinline__ int at(int l0, int c0, int L, int u) const {
    const int q = l0 - L, s = L & 63, d = dword(u + s) - dword(c0 - q * PR + s) + WD / 2;
    return (uint32_t)q < (uint32_t)WL && (uint32_t)d < (uint32_t)WD ? q * WD + d : -1;
  }
  __device__ __forceinline__ int code(int i, int j) const {
    const int L = (int)((uint32_t)(i - 1) / PR), x = at(L0, u0, L, j - 1);
    const int c = strip_code<PR>(win[x < 0 ? 0 : x], (uint32_t)(j - 1 + (L & 63)) % SPD, (uint32_t)(i - 1) % PR);
    return x < 0 ? -1 : c;
  }
  __device__ __forceinline__ int direct(int i, int j) const {
    const int L = (int)((uint32_t)(i - 1) / PR), t = j - 1 + (L & 63);
    return strip_code<PR>(pl[((size_t)(L >> 6) * (T / SPD) + dword(t)) * 64 + (L & 63)], (uint32_t)t % SPD,
                          (uint32_t)(i - 1) % PR);
  }
  __device__ __forceinline__ void fetch(int l0, int c0) {
    const int q = min((int)(threadIdx.x & 63), l0), L = l0 - q, s = L & 63;
    const uint32_t *p = pl + (size_t)(L >> 6) * (T / SPD) * 64 + s;
    const int d = dword(c0 - q * PR + s) - WD / 2;
#pragma unroll
    for (int k = 0; k < WD; ++k) nx[k] = p[min(max(d + k, 0), T / SPD - 1) * 64];
  }
  __device__ __forceinline__ bool refill(int i, int j) {
    const int L = (i - 1) / PR, u = j - 1;
    bool moved = true;
    if (nL0 < 0 || at(nL0, nu0, L, u) < 0) {
      moved = L != L0 || u != u0;
      nL0 = L;
      nu0 = u;
      fetch(L, u);
    }
    L0 = nL0;
    u0 = nu0;
    uint32_t *w = win + (threadIdx.x & 63) * WD;
#pragma unroll
    for (int k = 0; k < WD; ++k) w[k] = nx[k];
    nL0 = L0 - WL;
    nu0 = u - (L - nL0) * PR;
    if (nL0 >= 0) fetch(nL0, nu0);
    return moved;
  }
};

}  // namespace ta
