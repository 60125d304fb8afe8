// Memory of long pairs: the shapes of long.h's device arrays, what a request
// is admitted for, and how a batch divides what it may take.  Host code only.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <utility>
#include <vector>

namespace ta {

constexpr int LR = 8;                     // rows per lane of a forward strip
constexpr int LST = 64 * LR;              // rows of a forward strip, and of a region at most
constexpr int CKX = 512;                  // column checkpoint spacing
constexpr int LMARGIN = 256;              // region columns beyond the diagonal through the walk's rows
constexpr int LREG = LST + LMARGIN + CKX; // columns of a region at most
constexpr int LREG_T = (LREG + 63 + 7) & ~7;
constexpr int LTW = LST / 128;            // waves of a traceback workgroup: strips of a region
constexpr size_t LPLANES = (size_t)LTW * LREG_T / 4 * 64;  // dwords of a region's codes (4 steps a dword)
constexpr int64_t LREG_BYTES = 4 * (int64_t)LPLANES;       // 344 KB
constexpr int LONG_AHEAD = 16384;         // regions a traceback computes ahead at most (5.6 GB)

// Strips and steps of an la x lb pair; its bottom rows and, for a traceback,
// its checkpoint columns, in 8-byte entries.
inline int long_strips(int64_t la) { return (int)((la + LST - 1) / LST); }
inline int64_t long_steps(int64_t lb) { return (lb + 63 + 7) & ~7ll; }
inline int64_t long_rows(int64_t la, int64_t lb) { return (int64_t)(long_strips(la) - 1) * (long_steps(lb) + 8); }
inline int64_t long_cols(int64_t la, int64_t lb, bool trace) {
  return trace ? (lb - 1) / CKX * long_strips(la) * LST : 0;
}

// Rows and columns take 1/32 byte a cell.  The pairs of a batch may hold them
// one group of pairs after the other, so a pair counts about a third of that
// (5/512 byte a cell, and 11 MB), and the batch at least its largest pair.
inline int64_t long_share(int64_t la, int64_t lb) {
  const int64_t rl = ((lb + 7) & ~7ll) + 80, S = (la + 511) / 512;
  return (S - 1) / 8 * 8 * rl + (lb - 1) / 1024 * S * 512 * 8 + 8 * 64 * ((std::min<int64_t>(lb, 5376) + 71) / 8) * 32;
}

constexpr int64_t LONG_ROOM = (int64_t)16 << 30;  // rows and columns a batch holds at a time where nothing limits it

// What the long pairs of a request take: `least`, in groups and without
// regions ahead, and `full`, side by side up to LONG_ROOM with them.  A
// batch's least is at most the sum of its requests' (full alike), so requests
// admitted one by one fit together.  (Score only: no region, and nothing
// counts as traceback memory, so least is 0.)
struct LongNeed {
  bool trace = true;
  int64_t n = 0, strips = 0, share = 0, most = 0, all = 0;
  void add(int64_t la, int64_t lb) {
    const int64_t rc = 8 * (long_rows(la, lb) + long_cols(la, lb, trace));
    ++n;
    strips += long_strips(la);
    share += long_share(la, lb);
    most = std::max(most, rc);
    all += rc;
  }
  int64_t least() const { return trace && n ? std::max(share, most + n * LREG_BYTES) : 0; }
  int64_t full() const {
    if (!n) return 0;
    const int64_t rc = std::min(all, std::max(LONG_ROOM, most));
    return trace ? std::max(least(), rc + (n + std::min<int64_t>(strips, LONG_AHEAD)) * LREG_BYTES) : rc;
  }
};

// Pairs whose bottom rows and checkpoints share memory with other groups':
// pairs [lp0, + npairs), queue items [it0, + nitems), ring entries [0, ring_n).
struct LongGroup {
  int lp0, npairs, it0, nitems;
  uint64_t ring_n;
};

struct LongPlan {
  struct At {
    uint64_t ring, col;  // its rows' and columns' first entries in the block that the groups share
    int32_t item0;       // its first queue item
  };
  std::vector<LongGroup> groups;
  std::vector<At> at;                   // per pair
  uint64_t entries = 0, col_n = 0;      // the block, and the columns in it at most
  int wgs = 0;                          // traceback workgroups, a region's codes each
  int ahead = 0;                        // regions ahead (0: none)
  int64_t bytes() const { return 8 * (int64_t)entries + (int64_t)(wgs + ahead) * LREG_BYTES; }
};

// Long pairs (la, lb), in the order given, within `limit` bytes (at least
// their LongNeed::least; a lone pair of a score-only batch may take more); -1:
// no limit, which is LONG_ROOM or the pairs' shares, whichever is more, and the
// regions ahead beside it.
inline LongPlan long_plan(const std::vector<std::pair<int32_t, int32_t>> &shape, bool trace, int cus, int64_t limit) {
  LongPlan P;
  if (shape.empty()) return P;
  LongNeed need;
  need.trace = trace;
  int most = 0;
  for (const auto &s : shape) {
    need.add(s.first, s.second);
    most = std::max(most, long_strips(s.first));
  }
  if (trace) {
    P.wgs = std::max(1, std::min((int)shape.size(), 2 * cus));
    // Regions ahead, where the pairs alone would not keep every CU at a
    // region until the longest ends: 48 pairs (S up to 118, 3,300 in all)
    // 16.7 -> 2.8 ms; beyond, the same regions are computed either way.
    if (need.strips < (int64_t)most * cus) P.ahead = std::max(most, (int)std::min<int64_t>(need.strips, LONG_AHEAD));
  }
  int64_t room = std::max(LONG_ROOM, need.share);
  if (limit >= 0) {
    // Short of the full need, groups come first: regions ahead save a batch
    // milliseconds, groups too small to fill the GPU's waves multiply its time.
    const int64_t spare = limit - need.most - P.wgs * LREG_BYTES;
    if (limit < need.full()) P.ahead = (int)std::min<int64_t>(P.ahead, std::max<int64_t>(0, spare / 4) / LREG_BYTES);
    if (P.ahead < most) P.ahead = 0;
    room = std::min(room, limit - (P.wgs + P.ahead) * LREG_BYTES);
  }
  uint64_t ring = 0, col = 0;
  int items = 0;
  for (size_t k = 0; k < shape.size(); ++k) {
    const int la = shape[k].first, lb = shape[k].second, S = long_strips(la);
    const uint64_t nr = (uint64_t)long_rows(la, lb), nc = (uint64_t)long_cols(la, lb, trace);
    if (P.groups.empty() || (ring + col && 8 * (int64_t)(ring + col + nr + nc) > room)) {
      ring = col = 0;
      P.groups.push_back(LongGroup{(int)k, 0, items, 0, 0});
    }
    P.at.push_back(LongPlan::At{ring, col, items});
    ring += nr;
    col += nc;
    items += S;
    P.entries = std::max(P.entries, ring + col);
    P.col_n = std::max(P.col_n, col);
    LongGroup &g = P.groups.back();
    g.npairs += 1;
    g.nitems += S;
    g.ring_n = ring;
  }
  for (const LongGroup &g : P.groups)  // a group's columns follow its rows
    for (int k = g.lp0; k < g.lp0 + g.npairs; ++k) P.at[k].col += g.ring_n;
  return P;
}

}  // namespace ta
