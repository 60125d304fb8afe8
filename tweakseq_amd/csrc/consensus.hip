// Column consensus of an alignment on the GPU.
//
// Replaces Consensus::calculate (tweakseq/Core/Annotations/Consensus.cpp:80-161),
// which scores, for every column, each sequence's residue against every
// other's (BLOSUM62 for two letters, +1 for two non-letters, -4 for one of
// each) in O(nseq^2) per column, keeps the first sequence with the highest
// score, and takes its character when the number of its positive pairings
// reaches the plurality (else '?').
//
// A sequence's score depends only on the class of its residue (23 BLOSUM62
// rows or "not a letter"), so a column's classes are counted in one pass over
// the rows (coalesced: consecutive lanes read consecutive columns of a row)
// and each class present is scored against the counts,
// O(nseq + 24^2) per column: score(k) = sum_j cnt[j] * S(k, j) - S(k, k),
// the self pairing removed.  The winner is the class of best score whose
// first sequence comes first -- the reference's strict ">" over sequences in
// order.  Scores are integers, as the reference's double sums of integer
// weights are.  HBM-bound: nseq * len bytes read once.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstddef>
#include <cstring>
#include <vector>

#include "runtime_internal.h"

namespace {

constexpr int CK = 24;       // 23 BLOSUM62 rows, then "not a letter"
constexpr int CW = 16;       // waves per workgroup: shares of the rows
constexpr int CU = 8;        // row loads a lane has in flight

struct ConsArgs {
  const uint8_t *msa;        // row s at msa + s * len
  int32_t nseq, len;
  double plurality;
  char *out;
  const int8_t *cls;         // byte -> class (256)
  const int8_t *score;       // CK x CK pairing scores
  const int8_t *match;       // CK x CK: 1 when a pairing counts as a match
};

// A workgroup takes 64 columns (a lane each) and deals its rows to CW waves,
// which count classes into shared LDS tables (a lane's column is its own bank,
// so the atomics never conflict inside a wave).  Bound by the latency of the
// row loads: a thread per column alone, reading its rows one after the other,
// took 233 us for 512 x 2,000 (8 workgroups in all); 16 waves of 8 loads in
// flight take about 14 us.  The scores are dealt by class, one or two a wave.
__global__ __launch_bounds__(64 * CW) void consensus_kernel(ConsArgs A) {
  __shared__ int8_t cls[256];
  __shared__ int32_t sc[CK * CK], mt[CK * CK];
  __shared__ int32_t cnt[CK][64], first[CK][64], sco[CK][64], mat[CK][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 256) cls[tid] = A.cls[tid];
  for (int x = tid; x < CK * CK; x += 64 * CW) {
    sc[x] = A.score[x];
    mt[x] = A.match[x];
  }
  for (int x = tid; x < CK * 64; x += 64 * CW) {
    (&cnt[0][0])[x] = 0;
    (&first[0][0])[x] = INT_MAX;
  }
  __syncthreads();
  const int c = blockIdx.x * 64 + lane;
  const bool in = c < A.len;
  const uint8_t *col = A.msa + (in ? c : 0);
  const int per = (A.nseq + CW - 1) / CW, s0 = wave * per, s1 = s0 + per < A.nseq ? s0 + per : A.nseq;
  for (int s = s0; s < s1; s += CU) {
    uint8_t v[CU];
#pragma unroll
    for (int u = 0; u < CU; ++u) v[u] = col[(size_t)(s + u < s1 ? s + u : s1 - 1) * A.len];
#pragma unroll
    for (int u = 0; u < CU; ++u) {
      if (s + u < s1) {
        const int k = cls[v[u]];
        atomicAdd(&cnt[k][lane], 1);
        atomicMin(&first[k][lane], s + u);
      }
    }
  }
  __syncthreads();
  int32_t cj[CK];
#pragma unroll
  for (int j = 0; j < CK; ++j) cj[j] = cnt[j][lane];
  for (int k = wave; k < CK; k += CW) {
    int s = -sc[k * CK + k], m = -mt[k * CK + k];  // no pairing with itself
#pragma unroll
    for (int j = 0; j < CK; ++j) {
      s += cj[j] * sc[k * CK + j];
      m += cj[j] * mt[k * CK + j];
    }
    sco[k][lane] = s;
    mat[k][lane] = m;
  }
  __syncthreads();
  if (wave != 0 || !in) return;
  int best = INT_MIN, best_first = INT_MAX, best_match = 0;
#pragma unroll
  for (int k = 0; k < CK; ++k) {
    const int f = first[k][lane], s = sco[k][lane];
    if (f != INT_MAX && (s > best || (s == best && f < best_first))) {
      best = s;
      best_first = f;
      best_match = mat[k][lane];
    }
  }
  A.out[c] = (double)best_match >= A.plurality ? (char)col[(size_t)best_first * A.len] : '?';
}

// Class of every byte, pairing scores and match flags (from the engine's own
// BLOSUM62 table and letter map, ta_matrix / ta_encode).
struct ConsTables {
  int8_t cls[256], score[CK * CK], match[CK * CK];
};

ConsTables make_tables() {
  ConsTables t;
  int8_t S[32 * 32];
  int32_t K = 0;
  ta_matrix(TA_PROTEIN, 0, 0, S, &K);
  for (int b = 0; b < 256; ++b) {
    t.cls[b] = CK - 1;
    if (b >= 'A' && b <= 'Z') {  // the reference maps only 'A'..'Z' (latin1 - 65)
      const char ch = (char)b;
      uint8_t code = 0;
      if (ta_encode(TA_PROTEIN, &ch, 1, &code) == TA_OK) t.cls[b] = (int8_t)code;
    }
  }
  for (int a = 0; a < CK; ++a)
    for (int b = 0; b < CK; ++b) {
      int s, m;
      if (a == CK - 1 && b == CK - 1) { s = 1; m = 1; }
      else if (a == CK - 1 || b == CK - 1) { s = -4; m = 0; }
      else { s = S[a * K + b]; m = s > 0; }
      t.score[a * CK + b] = (int8_t)s;
      t.match[a * CK + b] = (int8_t)m;
    }
  return t;
}

}  // namespace

int ta_consensus(ta_ctx *ctx, const char *const *rows, int32_t nseq, int32_t len, double plurality, char *out) {
  if (!ctx || !rows || nseq <= 0 || len < 0 || (len > 0 && !out)) return TA_E_INVALID;
  for (int32_t s = 0; s < nseq; ++s)
    if (!rows[s] && len > 0) return TA_E_INVALID;
  if (len == 0) return TA_OK;
  if (plurality < 0) plurality = nseq / 2.0;  // Consensus::setSequences, weights 1.0
  if (hipSetDevice(ctx->device) != hipSuccess) return TA_E_DEVICE;
  static const ConsTables tables = make_tables();
  const size_t bytes = (size_t)nseq * (size_t)len;
  std::vector<uint8_t> host(bytes);
  for (int32_t s = 0; s < nseq; ++s) memcpy(host.data() + (size_t)s * len, rows[s], (size_t)len);
  uint8_t *d_msa = (uint8_t *)device_alloc(bytes);
  char *d_out = (char *)device_alloc((size_t)len);
  ConsTables *d_tab = (ConsTables *)device_alloc(sizeof(ConsTables));
  int rc = (d_msa && d_out && d_tab) ? TA_OK : TA_E_NOMEM;
  hipStream_t st = ctx->stream;
  if (!rc && (hipMemcpyAsync(d_msa, host.data(), bytes, hipMemcpyHostToDevice, st) != hipSuccess ||
              hipMemcpyAsync(d_tab, &tables, sizeof(ConsTables), hipMemcpyHostToDevice, st) != hipSuccess))
    rc = TA_E_DEVICE;
  if (!rc) {
    ConsArgs a;
    a.msa = d_msa; a.nseq = nseq; a.len = len; a.plurality = plurality; a.out = d_out;
    const int8_t *tb = (const int8_t *)d_tab;
    a.cls = tb + offsetof(ConsTables, cls);
    a.score = tb + offsetof(ConsTables, score);
    a.match = tb + offsetof(ConsTables, match);
    (void)hipGetLastError();
    hipLaunchKernelGGL(consensus_kernel, dim3((len + 63) / 64), dim3(64 * CW), 0, st, a);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(out, d_out, (size_t)len, hipMemcpyDeviceToHost, st) != hipSuccess)
      rc = TA_E_DEVICE;
  }
  if (hipStreamSynchronize(st) != hipSuccess && !rc) rc = TA_E_DEVICE;
  device_free(d_msa);
  device_free(d_out);
  device_free(d_tab);
  return rc;
}
