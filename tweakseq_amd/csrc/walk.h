// Walks back over direction codes, a whole wave per walk.
//
// A walk one cell at a time is a chain of dependent lookups: 180 ns a cell
// from LDS, 300 ns from memory, whatever else the chip does.  Here the 64
// lanes look at the next 64 cells the walk can pass in its state -- up the
// diagonal in state H, along the row in E, up the column in F -- and one
// ballot gives the length of the run, so a step costs one lookup per CIGAR
// run (a few dozen cells) instead of one per cell.
//
// The states and their order are those of the specification (traceback.h):
// H follows the cell's source; a gap source is taken at once with the same
// cell's extend bit; E and F stay while the extend bit is set.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"

namespace ta {

// How a walk ends other than at the matrix border.
enum { WALK_GLOBAL = 0,   // only there
       WALK_MARKED = 1 }; // on a cell whose code is d = 0, x = 1: its H is 0

enum { WALK_AT_BORDER = 0, WALK_STOPPED = 1, WALK_GAVE_UP = 2 };

// CIGAR runs ((len << 2) | op) in walk order, written backwards from `end`:
// 64 at a time from a register, lane k holding the k-th.
struct WaveRuns {
  uint32_t *end;   // the n-th run goes to end[-1 - n]
  int cap;         // slots before end
  int n = 0, op = -1, len = 0;
  uint32_t buf = 0;
  bool on = true;

  __device__ __forceinline__ void store(int base) const {
    const int r = base + (int)(threadIdx.x & 63);
    if (on && r < n && r < cap) end[-1 - r] = buf;
  }
  __device__ __forceinline__ void push() {
    if (!len) return;
    buf = (int)(threadIdx.x & 63) == (n & 63) ? ((uint32_t)len << 2) | (uint32_t)op : buf;
    ++n;
    if ((n & 63) == 0) store(n - 64);
  }
  __device__ __forceinline__ void emit(int o, int k) {
    if (o != op) { push(); op = o; len = 0; }
    len += k;
  }
  // The last runs; false if there were more than slots.
  __device__ __forceinline__ bool finish() {
    push();
    len = 0;
    if (n & 63) store(n & ~63);
    return n <= cap;
  }
};

// Walks from (i, j) (1-based) in `state` (0 H, 1 E, 2 F) until it ends;
// every value is the same in all lanes.  Src gives
//   int code(i, j)        a lane's cell: e f d x in bits 0..3, -1 if not at hand
//   int direct(i, j)      the same from where the codes are, at hand or not
//   bool refill(i, j)     (whole wave) brings cell (i, j) and its surroundings
//                         to hand; false if it cannot
// `steps` counts cells passed, and the walk gives up when they exceed `cap`.
template <int KIND, class Src>
__device__ __forceinline__ int wave_walk(Src &src, WaveRuns &w, int &i, int &j, int &state, int cap,
                                         int &steps) {
  const int lane = threadIdx.x & 63;
  if (i <= 0 || j <= 0) return WALK_AT_BORDER;
  auto look = [&](int ci, int cj, bool far) {  // a lane's cell; -1 beyond the border (no branch: an inner cell stands in)
    const int c = far ? src.direct(max(ci, 1), max(cj, 1)) : src.code(max(ci, 1), max(cj, 1));
    return min(ci, cj) >= 1 ? c : -1;
  };
  bool far = false;  // a gap goes on beyond what is at hand
  for (;;) {
    if (state == 0) {
      const int ci = i - lane, cj = j - lane;
      const int c = look(ci, cj, false);
      const uint64_t stop = __ballot((c & (KIND == WALK_MARKED ? 12 : 4)) != 0);
      const int run = stop ? __builtin_ctzll(stop) : 64;
      if (run) {
        w.emit(0, run);
        i -= run; j -= run; steps += run;
        if (steps > cap) return WALK_GAVE_UP;
        if (run == 64) continue;
      }
      const int at = __builtin_amdgcn_readlane(c, run);  // the cell that ends the run
      if (at < 0) {  // beyond the border, or not at hand
        if (i <= 0 || j <= 0) return WALK_AT_BORDER;
        if (!src.refill(i, j)) return WALK_GAVE_UP;
        continue;
      }
      if (KIND == WALK_MARKED && (at & 12) == 8) return WALK_STOPPED;
      state = (at & 8) ? 2 : 1;
      if (!(at & state)) {  // a gap of one: the same cell opened it
        w.emit(state, 1);
        i -= state == 2;
        j -= state == 1;
        state = 0;
        if (++steps > cap) return WALK_GAVE_UP;
        continue;
      }
    }
    // the gap: cells that extend it, then the one that opened it
    const int ci = i - (state == 2 ? lane : 0), cj = j - (state == 1 ? lane : 0);
    const int c = look(ci, cj, far);
    const uint64_t stop = __ballot(c < 0 || (c & state) == 0);
    const int run = stop ? __builtin_ctzll(stop) : 64;
    const int at = run < 64 ? __builtin_amdgcn_readlane(c, run & 63) : -1;
    const int len = at >= 0 ? run + 1 : run;
    if (len) w.emit(state, len);
    i -= state == 2 ? len : 0;
    j -= state == 1 ? len : 0;
    steps += len;
    if (steps > cap) return WALK_GAVE_UP;
    if (at >= 0) {
      state = 0;
      far = false;
    } else if (run < 64) {
      if (i <= 0 || j <= 0) return WALK_AT_BORDER;
      if (far) return WALK_GAVE_UP;  // cannot happen
      far = true;
    }
  }
}

}  // namespace ta
