// The single-pair (low-latency) kernel's interface to its host code.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"

namespace ta {

constexpr int PAIR_WAVES = 4;                // waves of the workgroup (one per SIMD)
constexpr int PAIR_PAD_LINE = 31;            // table line of a row outside the query
constexpr int PAIR_BAD_LETTER = 1;           // PairOut::status bits
constexpr int PAIR_GAVE_UP = 2;

// Rows per lane, and LDS byte offsets of the kernel's arrays, for an m x n pair.
struct PairLayout {
  int32_t R;                // rows per lane: 1, 2 or 4
  int32_t T, S;             // steps per strip (n + 63, rounded to 8), strips
  int32_t slot_bytes;       // score slot of a wave
  int32_t ring_len;         // int2 entries per ring
  int32_t runs_cap;         // CIGAR run slots
  int32_t acode, bcode, sync, slots, ring, planes, runs, window;
  int32_t bytes;            // total LDS
  int32_t plane_bytes;      // direction codes of all strips in device memory; 0: they are in LDS
};

// Written by the kernel: the result, then nruns CIGAR runs ((len << 2) | op,
// op 0 M / 1 D / 2 I) in alignment order right after this record.
struct PairOut {
  ResultDev r;
  int32_t nruns;
  int32_t status;           // PAIR_BAD_LETTER, PAIR_GAVE_UP
  int32_t done;             // set last, where the caller polls it
  int32_t pad_;
};

struct PairArgs {
  const char *a, *b;        // letters, device-readable (mapped host staging or device scratch)
  int32_t m, n;
  int32_t alphabet, match, mismatch;
  int32_t open, ext, local, traceback;
  int32_t spin_limit;
  int32_t polled;           // set PairOut::done when everything else is stored
  int32_t walk_cap;         // most steps the walk may take before it ends flagged (above any walk normally)
  PairLayout lay;
  uint8_t *planes;          // lay.plane_bytes of device memory, where the codes do not fit in LDS
  PairOut *out;             // device-writable; m + n + 2 run slots follow it
};

// The form for an m x n pair of an alphabet of K letters within lds_max bytes of LDS.
PairLayout pair_layout(int m, int n, int K, int lds_max);
// One workgroup on stream st; TA_E_DEVICE when the launch fails.
int pair_launch(const PairArgs &A, hipStream_t st);

}  // namespace ta
