// Host runtime + C ABI of the alignment engine (include/tweakalign.h).
//
// A batch is encoded once on the host, split into DP tasks (packed int16
// couples where the score range allows, int32 singles otherwise), sorted
// longest-first and uploaded; a run is: persistent fill kernels pulling tasks
// off a device counter, an optional int32 rerun of pairs whose int16 pass
// saturated, and the traceback kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <atomic>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <vector>

#include "../../include/tweakalign.h"
#include "blosum62.h"
#include "common.h"
#include "fill.h"
#include "long.h"
#include "runtime_internal.h"
#include "strips.h"
#include "traceback.h"

using namespace ta;

// ---------------------------------------------------------------------------
// Alphabets.  The protein table is BLOSUM62 in the row order
// A R N D C Q E G H I L K M F P S T W Y V B Z X and the letter map of
// tweakseq/Core/Annotations/Consensus.cpp:34-69 (same numbers, by necessity).
namespace {

const char kProtOrder[] = TA_PROT_ORDER;
const int8_t kBlosumLower[] = {TA_BLOSUM62_LOWER};
constexpr int kProtK = TA_PROT_K;

struct Alphabet {
  int K = 0;
  int8_t S[32 * 32];  // K x K
  int8_t map[256];    // byte -> code, -1 outside the alphabet
  int maxS = 0, minS = 0;
};

Alphabet make_alphabet(int alphabet, int match, int mismatch) {
  Alphabet A;
  memset(A.map, -1, sizeof(A.map));
  if (alphabet == TA_PROTEIN) {
    A.K = kProtK;
    int idx = 0;
    for (int r = 0; r < kProtK; ++r)
      for (int c = 0; c <= r; ++c, ++idx) {
        A.S[r * kProtK + c] = kBlosumLower[idx];
        A.S[c * kProtK + r] = kBlosumLower[idx];
      }
    for (int r = 0; r < kProtK; ++r) {
      A.map[(unsigned char)kProtOrder[r]] = (int8_t)r;
      A.map[(unsigned char)(kProtOrder[r] + 32)] = (int8_t)r;
    }
    for (char c : {'J', 'O', 'U'}) {  // no row of their own: scored as X
      A.map[(unsigned char)c] = 22;
      A.map[(unsigned char)(c + 32)] = 22;
    }
  } else {
    A.K = 4;
    for (int r = 0; r < 4; ++r)
      for (int c = 0; c < 4; ++c) A.S[r * 4 + c] = (int8_t)(r == c ? match : mismatch);
    const char *acgt = "ACGT";
    for (int r = 0; r < 4; ++r) {
      A.map[(unsigned char)acgt[r]] = (int8_t)r;
      A.map[(unsigned char)(acgt[r] + 32)] = (int8_t)r;
    }
  }
  A.maxS = -128;
  A.minS = 127;
  for (int x = 0; x < A.K * A.K; ++x) {
    A.maxS = std::max<int>(A.maxS, A.S[x]);
    A.minS = std::min<int>(A.minS, A.S[x]);
  }
  return A;
}

// Score-only packed couples keep 4-bit scores: the table must span at most
// 16 values, and for local couples the pad code (scored as the minimum) must
// be negative so that leading pad columns hold H at 0.  Other score-only
// tables run in int32.
bool nibble_ok(const Alphabet &A, bool local) { return A.maxS - A.minS <= 15 && (!local || A.minS < 0); }

// (K+1) x (K+1) table of score - minS (0..15), pad row / column at 0.
std::vector<int8_t> nibble_table(const Alphabet &A) {
  const int Kp = A.K + 1;
  std::vector<int8_t> t((size_t)Kp * Kp, 0);
  for (int r = 0; r < A.K; ++r)
    for (int c = 0; c < A.K; ++c) t[(size_t)r * Kp + c] = (int8_t)(A.S[r * A.K + c] - A.minS);
  return t;
}

// (K+1) x (K+1) table with a pad row / column (index K) of PAD_SCORE.
std::vector<int8_t> padded_table(const Alphabet &A) {
  const int Kp = A.K + 1;
  std::vector<int8_t> t((size_t)Kp * Kp, PAD_SCORE);
  for (int r = 0; r < A.K; ++r)
    for (int c = 0; c < A.K; ++c) t[(size_t)r * Kp + c] = A.S[r * A.K + c];
  return t;
}

#define HIPCHK(x)                                                   \
  do {                                                              \
    hipError_t e_ = (x);                                            \
    if (e_ != hipSuccess) {                                         \
      fprintf(stderr, "tweakalign: %s at %s:%d\n", hipGetErrorString(e_), __FILE__, __LINE__); \
      return TA_E_DEVICE;                                           \
    }                                                               \
  } while (0)

// Device memory cache.  Blocks of every size are kept per size class and
// reused: hipFree waits for the whole device, so freeing a batch's planes
// while other batches run would stall them all (the serving loop keeps
// several batches in flight), and hipMalloc per buffer would dominate small
// batches.  Classes are powers of two up to 1 MB, then four per doubling
// (at most 19% rounding).  A request takes a free block of its class or of
// the next classes up to twice its size.  Free blocks stay cached up to half
// the device's memory; past that, and when hipMalloc fails, cached blocks
// are released.
struct MemCache {
  std::mutex mu;
  std::map<std::pair<int, size_t>, std::vector<void *>> free;  // (device, class) -> blocks
  std::unordered_map<void *, std::pair<int, size_t>> live;
  std::map<int, size_t> cached, cap;                              // per device: free bytes, their limit
};
MemCache &memcache() {
  static MemCache *c = new MemCache();  // lives until the process ends
  return *c;
}

size_t size_class(size_t n) {
  size_t c = 256;
  while (c < n && c < (1u << 20)) c <<= 1;
  if (c >= n) return c;
  while (c * 2 < n) c <<= 1;  // c < n <= 2c: classes c * (5, 6, 7, 8) / 4
  for (int q = 5; q <= 8; ++q)
    if (c / 4 * q >= n) return c / 4 * q;
  return 2 * c;
}

// Releases every cached free block of `dev` (lock held).
void cache_release(MemCache &mc, int dev) {
  for (auto it = mc.free.begin(); it != mc.free.end(); ++it) {
    if (it->first.first != dev) continue;
    for (void *p : it->second) (void)hipFree(p);
    it->second.clear();
  }
  mc.cached[dev] = 0;
}

void *cache_alloc(size_t bytes) {
  int dev = 0;
  (void)hipGetDevice(&dev);
  MemCache &mc = memcache();
  const size_t cls = size_class(bytes);
  std::lock_guard<std::mutex> g(mc.mu);
  if (!mc.cap.count(dev)) {
    size_t fr = 0, tot = 0;
    mc.cap[dev] = hipMemGetInfo(&fr, &tot) == hipSuccess ? tot / 2 : (size_t)64 << 30;
  }
  for (auto it = mc.free.lower_bound({dev, cls}); it != mc.free.end() && it->first.first == dev &&
                                                  it->first.second <= 2 * cls;
       ++it) {
    if (it->second.empty()) continue;
    void *p = it->second.back();
    it->second.pop_back();
    mc.cached[dev] -= it->first.second;
    mc.live[p] = it->first;
    return p;
  }
  void *p = nullptr;
  if (hipMalloc(&p, cls) != hipSuccess) {
    (void)hipGetLastError();
    cache_release(mc, dev);
    if (hipMalloc(&p, cls) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
  }
  mc.live[p] = {dev, cls};
  return p;
}

void cache_free(void *p) {
  if (!p) return;
  MemCache &mc = memcache();
  std::lock_guard<std::mutex> g(mc.mu);
  auto it = mc.live.find(p);
  if (it == mc.live.end()) return;
  const auto key = it->second;
  mc.live.erase(it);
  mc.free[key].push_back(p);
  mc.cached[key.first] += key.second;
  if (mc.cached[key.first] > mc.cap[key.first]) cache_release(mc, key.first);
}

template <typename T>
int dalloc(T **p, size_t n) {
  *p = nullptr;
  if (n == 0) return TA_OK;
  *p = (T *)cache_alloc(n * sizeof(T));
  return *p ? TA_OK : TA_E_NOMEM;
}

template <typename T>
int upload(T **dst, const std::vector<T> &src, hipStream_t st) {
  int rc = dalloc(dst, src.size());
  if (rc) return rc;
  if (!src.empty()) HIPCHK(hipMemcpyAsync(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice, st));
  return TA_OK;
}

template <typename T>
void dfree(T *&p) {
  cache_free((void *)p);
  p = nullptr;
}

// Host staging for the residue codes, the results and the CIGAR runs.  A
// copy to or from pageable memory runs at a fraction of the link's rate (the
// runtime copies it through bounce buffers); with pinned memory the DMA
// engine reads or writes the block itself.  Pinning a block takes
// milliseconds, so blocks are kept and reused: batch creation takes one and
// encodes into it, result fetching takes two and reads from them, and each
// goes back once its copy has finished.  At most 16 free blocks and 1 GB stay
// pinned; blocks above 256 MB come from the heap (pinning them would cost
// about what it saves).
struct Staging {
  uint8_t *p = nullptr;
  size_t cap = 0;
  bool pinned = false;
};
struct StagePool {
  std::mutex mu;
  std::vector<Staging> free;
};
StagePool &stage_pool() {
  static StagePool *s = new StagePool();  // lives until the process ends
  return *s;
}

Staging stage_take(size_t bytes) {
  StagePool &sp = stage_pool();
  {
    std::lock_guard<std::mutex> g(sp.mu);
    int best = -1;  // the smallest free block that fits
    for (int i = 0; i < (int)sp.free.size(); ++i)
      if (sp.free[i].cap >= bytes && (best < 0 || sp.free[i].cap < sp.free[best].cap)) best = i;
    if (best >= 0) {
      const Staging s = sp.free[best];
      sp.free.erase(sp.free.begin() + best);
      return s;
    }
  }
  Staging s;
  s.cap = size_class(std::max(bytes, (size_t)1 << 20));
  if (s.cap <= ((size_t)256 << 20)) {
    if (hipHostMalloc((void **)&s.p, s.cap, hipHostMallocPortable) == hipSuccess) {
      s.pinned = true;
      return s;
    }
    (void)hipGetLastError();
    s.p = nullptr;
  }
  s.p = (uint8_t *)malloc(s.cap);
  if (!s.p) s.cap = 0;
  return s;
}

void stage_give(Staging &s) {
  if (!s.p) return;
  if (!s.pinned) {
    free(s.p);
  } else {
    StagePool &sp = stage_pool();
    std::lock_guard<std::mutex> g(sp.mu);
    sp.free.push_back(s);
    auto by_cap = [](const Staging &x, const Staging &y) { return x.cap < y.cap; };
    size_t bytes = 0;
    for (const Staging &f : sp.free) bytes += f.cap;
    while (sp.free.size() > 16 || bytes > ((size_t)1 << 30)) {  // unpin the smallest, or the largest past 1 GB
      auto it = sp.free.size() > 16 ? std::min_element(sp.free.begin(), sp.free.end(), by_cap)
                                    : std::max_element(sp.free.begin(), sp.free.end(), by_cap);
      bytes -= it->cap;
      (void)hipHostFree(it->p);
      sp.free.erase(it);
    }
  }
  s = Staging{};
}

// A staging block held by one batch creation.  Once a copy from it is
// queued on `stream`, the block goes back only after the stream has drained
// (every return path, device errors included).
struct StageHold {
  Staging s;
  hipStream_t stream = nullptr;
  bool queued = false;
  ~StageHold() {
    if (queued) (void)hipStreamSynchronize(stream);
    stage_give(s);
  }
};

// Host vectors of destroyed batches, kept for the next batches so that
// their pages stay mapped (a fresh multi-MB vector pays a page fault per
// 4 KB, milliseconds per batch): up to 4 per element type, none above 64 MB.
template <typename T>
struct VecBin {
  std::mutex mu;
  std::vector<std::vector<T>> v;
  static VecBin &get() {
    static VecBin *b = new VecBin();
    return *b;
  }
};
template <typename T>
void vec_take(std::vector<T> &x) {
  VecBin<T> &b = VecBin<T>::get();
  std::lock_guard<std::mutex> g(b.mu);
  if (!b.v.empty()) {
    x.swap(b.v.back());
    b.v.pop_back();
  }
  x.clear();
}
template <typename T>
void vec_give(std::vector<T> &x) {
  const size_t bytes = x.capacity() * sizeof(T);
  if (bytes < ((size_t)64 << 10) || bytes > ((size_t)64 << 20)) return;
  VecBin<T> &b = VecBin<T>::get();
  std::lock_guard<std::mutex> g(b.mu);
  if (b.v.size() < 4) {
    b.v.emplace_back();
    b.v.back().swap(x);
  }
}

// Host vectors bound for the device, gathered into one pinned staging block
// and sent with one asynchronous copy into one device block (a copy from
// pageable memory is staged by the runtime and waits for the link; a copy
// per vector took a small batch's creation 3.4 us each).  The vectors must
// live until commit(); the staging block until the stream drains.
struct BulkUpload {
  struct Item { void **dst; const void *src; size_t bytes, at; };
  std::vector<Item> items;
  StageHold hold;
  template <typename T>
  void add(T **dst, const std::vector<T> &v) {
    *dst = nullptr;
    if (!v.empty()) items.push_back(Item{(void **)dst, v.data(), v.size() * sizeof(T), 0});
  }
  int commit(void **block, hipStream_t st) {
    *block = nullptr;
    size_t total = 0;
    for (Item &x : items) {
      x.at = total;
      total += (x.bytes + 255) & ~(size_t)255;
    }
    if (!total) return TA_OK;
    hold.s = stage_take(total);
    if (!hold.s.p) return TA_E_NOMEM;
    if (!(*block = cache_alloc(total))) return TA_E_NOMEM;
    for (Item &x : items) {
      memcpy(hold.s.p + x.at, x.src, x.bytes);
      *x.dst = (uint8_t *)*block + x.at;
    }
    hold.stream = st;
    hold.queued = true;
    return hipMemcpyAsync(*block, hold.s.p, total, hipMemcpyHostToDevice, st) == hipSuccess ? TA_OK : TA_E_DEVICE;
  }
};


}  // namespace

// The device-memory cache for the library's other sources (runtime_internal.h).
void *device_alloc(size_t bytes) { return cache_alloc(bytes); }
void device_free(void *p) { cache_free(p); }

// ---------------------------------------------------------------------------
const char *ta_strerror(int code) {
  switch (code) {
    case TA_OK: return "ok";
    case TA_E_INVALID: return "invalid argument";
    case TA_E_ALPHABET: return "residue outside the alphabet";
    case TA_E_SPACE: return "output buffer too small";
    case TA_E_DEVICE: return "HIP runtime error";
    case TA_E_NOMEM: return "out of memory";
    case TA_E_BUDGET: return "request exceeds the traceback-memory budget";
    case TA_E_CANCELLED: return "request cancelled";
    case TA_E_TICKET: return "unknown ticket";
    case TA_E_NODEVICE: return "no usable GPU";
    case TA_E_WALK: return "a traceback walk did not complete";
    case TA_E_LIMIT: return "input exceeds the fixed scratch of the allocation-free entry point";
    case TA_E_PENDING: return "pending";
    default: return "unknown error";
  }
}

int ta_matrix(int32_t alphabet, int32_t match, int32_t mismatch, int8_t *out, int32_t *K) {
  if (alphabet != TA_PROTEIN && alphabet != TA_DNA) return TA_E_INVALID;
  Alphabet A = make_alphabet(alphabet, match, mismatch);
  if (K) *K = A.K;
  if (out) memcpy(out, A.S, (size_t)A.K * A.K);
  return TA_OK;
}

int ta_encode(int32_t alphabet, const char *s, int32_t len, uint8_t *out) {
  if (alphabet != TA_PROTEIN && alphabet != TA_DNA) return TA_E_INVALID;
  if (len < 0 || (len > 0 && (!s || !out))) return TA_E_INVALID;
  Alphabet A = make_alphabet(alphabet, 1, -1);
  for (int32_t i = 0; i < len; ++i) {
    int c = A.map[(unsigned char)s[i]];
    if (c < 0) return TA_E_ALPHABET;
    out[i] = (uint8_t)c;
  }
  return TA_OK;
}

int ta_create(ta_ctx **out, int device) {
  if (!out) return TA_E_INVALID;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return TA_E_NODEVICE;
  if (device < 0 || device >= ndev) return TA_E_INVALID;
  HIPCHK(hipSetDevice(device));
  ta_ctx *c = new ta_ctx();
  c->device = device;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0)
    c->cus = cus;
  int lds = 0;
  if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) == hipSuccess && lds > 0)
    c->lds_max = lds;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return TA_E_DEVICE;
  }
  pair_scratch_setup(device);  // ta_align_pair_static's array on this device (reports its own failure)
  *out = c;
  return TA_OK;
}

void ta_destroy(ta_ctx *c) {
  if (!c) return;
  serve_shutdown(c);
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  if (c->pair_stage) (void)hipHostFree(c->pair_stage);
  device_free(c->pair_planes);
  c->seq_arena.reset();  // freed here unless a batch still holds it (none after serve_shutdown)
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

int params_check(const ta_params *p) {
  if (!p) return TA_E_INVALID;
  if (p->mode != TA_GLOBAL && p->mode != TA_LOCAL) return TA_E_INVALID;
  if (p->alphabet != TA_PROTEIN && p->alphabet != TA_DNA) return TA_E_INVALID;
  if (p->gap_open > 0 || p->gap_extend > 0 || p->gap_open < -1000 || p->gap_extend < -1000) return TA_E_INVALID;
  if (p->alphabet == TA_DNA && (p->match < -100 || p->match > 100 || p->mismatch < -100 || p->mismatch > 100))
    return TA_E_INVALID;
  if (p->lanes != TA_LANES_AUTO && p->lanes != TA_LANES_I16 && p->lanes != TA_LANES_I32 &&
      p->lanes != TA_LANES_LONG)
    return TA_E_INVALID;
  if (p->lanes == TA_LANES_LONG && p->mode != TA_GLOBAL) return TA_E_INVALID;
  return TA_OK;
}

// ---------------------------------------------------------------------------
// Batch construction.
namespace {

struct HostPair {
  uint64_t a_off, b_off;
  int32_t la, lb;
  int path;  // 3 long-pair pipeline, 2 packed int16, 1 int32, 0 no DP (empty side)
  bool maysat = false;  // path 2, local: the int16 fill may saturate (int32 rerun then)
};

// Global pairs of at least this many cells go through the long-pair
// pipeline: one task would otherwise hold a single wave for the whole sweep
// (and 4 bits per cell of direction planes).
constexpr int64_t kLongCells = 1ll << 25;

bool long_pair(const ta_params &p, int la, int lb) {
  if (p.mode != TA_GLOBAL || la == 0 || lb == 0) return false;
  if (p.lanes == TA_LANES_LONG) return true;
  return p.lanes == TA_LANES_AUTO && (int64_t)la * lb >= kLongCells;
}

// Direction-plane bytes a pair of the other paths is admitted for.
int64_t planes_estimate(int la, int lb) {
  return (int64_t)((la + STRIP - 1) / STRIP) * ((lb + G + 7) / 8) * (G * R * 4);
}

// Residue codes one task's strips and columns read (expand_codes_kernel).
struct CodeJob {
  uint64_t row_off, col_off;
  int32_t nrows, ncol, lo, hi, off0, off1;
};

__host__ __device__ inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Where a task's row codes, column codes, ring and direction planes start in
// the plan's arrays, or (task_span) how many entries / bytes it takes there.
struct TaskAt {
  uint64_t row, col, ring, tb;
};

// A couple (or single) that becomes a task.
struct Unit {
  int lo, hi;
  bool single;
  int m, n;  // rows and columns (maxima over the two halves)
};

// Tasks of one shape that a wave takes together: units [u0, u0 + cnt) of n
// columns and S strips, their entries one after the other from `at`.
struct TaskSpan {
  TaskAt at;
  uint32_t u0, cnt;
  int32_t n, S;
};

// Tasks swept by groups of GG lanes, GWAVE / GG to a span (short spans are
// filled with copies of their first task that write nothing).
struct TaskList {
  int P = 2, GG = GWAVE;
  std::vector<Unit> units;
  std::vector<TaskSpan> spans;  // in the order they are taken
  int tasks() const { return (int)spans.size() * (GWAVE / GG); }
};

struct Plan {
  // [0] whole-wave groups, [1] G-lane groups (NGW per wave unit), [2] 8-lane
  // groups (8 per wave unit; packed couples only, list1[2] stays empty)
  TaskList list2[3], list1[3];
  uint64_t rows_n = 0, cols_n = 0;        // rowcodes / colcodes entries planned
  uint64_t ring_elems = 0, tb_bytes = 0;
  // Tasks written on the host (int32 reruns, the plain form)
  std::vector<CodeJob> cjobs;
  std::vector<PairTB> ptb;
  Plan() {
    const int gg[3] = {GWAVE, G, 8};
    for (int g = 0; g < 3; ++g) {
      list2[g].GG = list1[g].GG = gg[g];
      list1[g].P = 1;
    }
  }
};

// Resident one-wave fill workgroups per CU: one per SIMD.  A fill wave keeps
// its SIMD's VALU busy by itself (the recurrence's dependent chain per row is
// a fraction of a step's instructions), and a second wave on the SIMD only
// halves the speed of the long tasks that end the batch (measured on the
// 65,536-pair local batch: 9.1 ms at 4 waves per CU, 9.9 at 8, 10.5 at 12).
// Fill waves per CU: as wanted, within LDS; walking fills have WALK_FW (one
// workgroup per CU).
int fill_waves_per_cu(int P, int Kp, bool nib, int want, bool walk = false) {
  if (walk) return WALK_FW;
  return std::max(1, std::min(want, (160 * 1024) / fill_lds_bytes(P, Kp, nib)));
}

// Raw letters to residue codes in place, 16 bytes per thread step, through a
// 256-entry map (0xff: outside the alphabet, which sets *bad).
struct LetterMap {
  uint32_t w[64];
};
__global__ __launch_bounds__(256) void encode_kernel(uint4 *codes, size_t words, LetterMap map, int32_t *bad) {
  __shared__ uint8_t m[256];
  if (threadIdx.x < 64) ((uint32_t *)m)[threadIdx.x] = map.w[threadIdx.x];
  __syncthreads();
  uint32_t any = 0;
  for (size_t w = (size_t)blockIdx.x * blockDim.x + threadIdx.x; w < words; w += (size_t)gridDim.x * blockDim.x) {
    uint4 v = codes[w];
    uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t b0 = m[x[q] & 0xff], b1 = m[(x[q] >> 8) & 0xff], b2 = m[(x[q] >> 16) & 0xff], b3 = m[x[q] >> 24];
      any |= b0 | b1 | b2 | b3;
      x[q] = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
    }
    codes[w] = make_uint4(x[0], x[1], x[2], x[3]);
  }
  if (__any(any & 0x80) && (threadIdx.x & 63) == 0) atomicOr(bad, 1);
}

// The row and column codes of a task (pairs A, B), expanded by threads
// tid < nthr from the uploaded residues: row r of a half is its pair's query residue r
// (pad past m), column j its reference residue j - off (pad before the
// leading columns and past n).
__device__ __forceinline__ void expand_job(const CodeJob &c, const PairDev &A, const PairDev &B, const uint8_t *codes,
                                           int pad, uint16_t *rowcodes, uint16_t *colcodes, int tid, int nthr) {
  for (int r = tid; r < c.nrows; r += nthr) {
    const int ca = r < A.la ? codes[A.a_off + r] : pad;
    const int cb = r < B.la ? codes[B.a_off + r] : pad;
    rowcodes[c.row_off + r] = (uint16_t)(ca | (cb << 8));
  }
  for (int j = tid; j < c.ncol; j += nthr) {
    const int ja = j - c.off0, jb = j - c.off1;
    const int ca = (ja >= 0 && ja < A.lb) ? codes[A.b_off + ja] : pad;
    const int cb = (jb >= 0 && jb < B.lb) ? codes[B.b_off + jb] : pad;
    colcodes[c.col_off + j] = (uint16_t)(ca | (cb << 8));
  }
}

// The codes of a list of tasks, one workgroup per task.
__global__ void expand_codes_kernel(const CodeJob *jobs, int njobs, const PairDev *pairs, const uint8_t *codes,
                                    int pad, uint16_t *rowcodes, uint16_t *colcodes) {
  for (int q = blockIdx.x; q < njobs; q += gridDim.x) {
    const CodeJob c = jobs[q];
    expand_job(c, pairs[c.lo], pairs[c.hi], codes, pad, rowcodes, colcodes, threadIdx.x, blockDim.x);
  }
}

// Allocates a plan's row and column codes on the device and expands them
// there (the residues and pair descriptors are already uploaded).
int expand_codes(const std::vector<CodeJob> &jobs, uint64_t rows_n, uint64_t cols_n, const PairDev *d_pairs,
                 const uint8_t *d_codes, int Kp, uint16_t **d_rows, uint16_t **d_cols, hipStream_t st) {
  int rc = dalloc(d_rows, (size_t)rows_n);
  rc = rc ? rc : dalloc(d_cols, (size_t)cols_n);
  if (rc || jobs.empty()) return rc;
  CodeJob *d_jobs = nullptr;
  rc = upload(&d_jobs, jobs, st);
  if (rc) return rc;
  (void)hipGetLastError();
  hipLaunchKernelGGL(expand_codes_kernel, dim3((unsigned)std::min<size_t>(jobs.size(), 65536)), dim3(256), 0, st,
                     d_jobs, (int)jobs.size(), d_pairs, d_codes, Kp - 1, *d_rows, *d_cols);
  if (hipGetLastError() != hipSuccess) rc = TA_E_DEVICE;
  // the job list goes back to the cache once the expansion has read it
  if (hipStreamSynchronize(st) != hipSuccess && !rc) rc = TA_E_DEVICE;
  dfree(d_jobs);
  return rc;
}

// Row codes: S * ST entries; column codes: 8 NB + 8 (a multiple of 8, so
// every task's columns start 16-byte aligned); ring: two arrays of
// 8 NB + 2 GG + 16 when there is more than one strip.
__host__ __device__ inline TaskAt task_span(int P, int GG, bool trace, int n, int S) {
  const int NB = ceil_div(n + GG, 8);
  return TaskAt{(uint64_t)S * GG * R, (uint64_t)(8 * NB + 8), S > 1 ? 2ull * (8 * NB + 2 * GG + 16) : 0,
                trace ? (uint64_t)S * tb_strip_bytes(P, NB, GG) : 0};
}

// One task (pair lo / hi; hi == lo for a single; la, lb: their lengths) of n
// columns and S strips at the given offsets.
__host__ __device__ inline Task make_task(const TaskAt &at, int GG, bool trace, int lo, int hi, const int (&la)[2],
                                          const int (&lb)[2], bool single, int n, int S) {
  Task T{};
  T.pair[0] = lo; T.pair[1] = hi;
  T.m[0] = la[0]; T.m[1] = la[1];
  T.n = n;
  T.off[0] = n - lb[0]; T.off[1] = n - lb[1];
  T.S = S;
  T.NB = ceil_div(n + GG, 8);
  T.single = single ? 1 : 0;
  T.row_off = at.row;
  T.col_off = at.col;
  T.ring_len = S > 1 ? 8 * T.NB + 2 * GG + 16 : 0;
  T.ring_off = at.ring;
  T.tb_off = trace ? at.tb : 0;
  return T;
}
// The direction-plane record of a task's half.
__host__ __device__ inline PairTB task_ptb(const Task &T, int P, int GG, int h) {
  PairTB d{};
  d.tb_off = T.tb_off; d.P = P; d.half = h; d.NB = T.NB; d.off = T.off[h]; d.GG = GG;
  return d;
}

// A task on the host at the plan's running offsets, appended to dst with its
// code-expansion job and its pairs' records.
void add_task(Plan &pl, std::vector<Task> &dst, int P, int GG, bool trace, const std::vector<HostPair> &hp,
              int lo, int hi, bool single, int n = 0, int S = 0) {
  const int la[2] = {hp[lo].la, hp[hi].la}, lb[2] = {hp[lo].lb, hp[hi].lb};
  if (!n) n = std::max(lb[0], lb[1]);
  if (!S) S = ceil_div(std::max(la[0], la[1]), GG * R);
  const TaskAt at{pl.rows_n, pl.cols_n, pl.ring_elems, pl.tb_bytes}, sz = task_span(P, GG, trace, n, S);
  dst.push_back(make_task(at, GG, trace, lo, hi, la, lb, single, n, S));
  const Task &T = dst.back();
  pl.cjobs.push_back(CodeJob{T.row_off, T.col_off, T.S * GG * R, 8 * T.NB + 8, lo, hi, T.off[0], T.off[1]});
  for (int h = 0; h < (single ? 1 : 2); ++h) pl.ptb[h ? hi : lo] = task_ptb(T, P, GG, h);
  pl.rows_n += sz.row; pl.cols_n += sz.col; pl.ring_elems += sz.ring; pl.tb_bytes += sz.tb;
}

// Start of a batch on the device: its pairs' fill outputs before a run (an
// empty side: the finished result) and their direction-plane records (pairs
// of at least long_cells cells: the long-pair kernels').
__global__ void pairs_init_kernel(const PairDev *pairs, int n, FillOut *fo, PairTB *ptb, int local, int open, int ext,
                                  int64_t long_cells) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const int la = pairs[k].la, lb = pairs[k].lb;
    FillOut f{0, 0, 0, 0};
    PairTB d{};
    if (la == 0 || lb == 0) {
      if (local) {
        f.flags = 8;
      } else {
        f.score = la + lb ? open + (la + lb - 1) * ext : 0;
        f.end_i = la; f.end_j = lb;
      }
    } else if ((int64_t)la * lb >= long_cells) {
      d.P = 3;
    }
    fo[k] = f;
    ptb[k] = d;
  }
}

// The planned tasks, their pairs' direction-plane records and their row and
// column codes, a wave per task (a workgroup each took 132 us: a chain of
// dependent reads before a few codes a thread).  The host plans spans only (shapes,
// offsets, which units): tasks, code jobs and records written there and
// copied over were 15 of the 20 MB that the creation of a batch of 130,816
// pairs wrote and sent.  With the pairs' table written by the host threads
// and its copy under the planning, and sorts of packed 64-bit keys, that
// creation takes 3.1 ms instead of 6.5.
struct PlanArgs {
  struct List {
    const Unit *units;
    const TaskSpan *spans;
    Task *dst;
    int32_t ntasks, P, GG;
  } list[6];
  int32_t trace, pad;
  const PairDev *pairs;
  const uint8_t *codes;
  PairTB *ptb;
  uint16_t *rowcodes, *colcodes;
};
__global__ __launch_bounds__(256) void plan_tasks_kernel(PlanArgs A, int total) {
  const int lane = threadIdx.x & 63;
  for (int x = blockIdx.x * 4 + (int)(threadIdx.x >> 6); x < total; x += 4 * gridDim.x) {
    int q = __builtin_amdgcn_readfirstlane(x), l = 0;
    while (q >= A.list[l].ntasks) q -= A.list[l++].ntasks;
    const PlanArgs::List &L = A.list[l];
    const int NG = GWAVE / L.GG, i = q % NG;
    const TaskSpan s = L.spans[q / NG];
    const bool filler = i >= (int)s.cnt;
    const int at_i = filler ? 0 : i;
    const Unit u = L.units[s.u0 + at_i];
    const PairDev a = A.pairs[u.lo], b = A.pairs[u.hi];
    const TaskAt sz = task_span(L.P, L.GG, A.trace, s.n, s.S);
    const TaskAt at{s.at.row + at_i * sz.row, s.at.col + at_i * sz.col, s.at.ring + at_i * sz.ring,
                    s.at.tb + at_i * sz.tb};
    const int la[2] = {a.la, b.la}, lb[2] = {a.lb, b.lb};
    Task T = make_task(at, L.GG, A.trace, u.lo, u.hi, la, lb, u.single, s.n, s.S);
    if (filler) T.single = 2;
    if (lane == 0) {
      L.dst[q] = T;
      if (!filler) {
        A.ptb[u.lo] = task_ptb(T, L.P, L.GG, 0);
        if (!u.single) A.ptb[u.hi] = task_ptb(T, L.P, L.GG, 1);
      }
    }
    if (filler) continue;
    const CodeJob c{T.row_off, T.col_off, T.S * L.GG * R, 8 * T.NB + 8, u.lo, u.hi, T.off[0], T.off[1]};
    expand_job(c, a, b, A.codes, A.pad, A.rowcodes, A.colcodes, lane, 64);
  }
}

// Positions 0..n-1 in ascending order of key, equal keys in position order:
// key and position packed in 64 bits, an LSD radix sort over the 11-bit
// digits in which the keys differ.  The planner orders tens of thousands of
// pairs and units per batch, where comparison sorts that read their keys
// through the pair table cost milliseconds.  `key` is used up.
std::vector<int32_t> order_by_key(std::vector<uint64_t> &key) {
  const size_t n = key.size();
  std::vector<int32_t> idx;
  vec_take(idx);
  idx.resize(n);
  if (!n) return idx;
  uint64_t lo = key[0], hi = key[0];
  for (uint64_t k : key) { lo = std::min(lo, k); hi = std::max(hi, k); }
  int nb = 0, kb = 0;  // bits of a position, of a key's range
  while ((uint64_t)(n - 1) >> nb) ++nb;
  while (kb < 64 && (hi - lo) >> kb) ++kb;
  if (nb + kb > 64) {
    for (size_t t = 0; t < n; ++t) idx[t] = (int32_t)t;
    std::stable_sort(idx.begin(), idx.end(), [&](int32_t a, int32_t b) { return key[a] < key[b]; });
    return idx;
  }
  uint64_t any = 0;
  for (size_t t = 0; t < n; ++t) {
    key[t] = nb < 64 ? (key[t] - lo) << nb | t : t;
    any |= key[t] ^ key[0];
  }
  std::vector<uint64_t> tmp;
  vec_take(tmp);
  tmp.resize(n);
  for (int sh = nb; sh < nb + kb; sh += 11) {
    if (!(any >> sh & 2047)) continue;
    size_t at[2049] = {0};
    for (uint64_t k : key) ++at[((k >> sh) & 2047) + 1];
    for (int d = 0; d < 2048; ++d) at[d + 1] += at[d];
    for (uint64_t k : key) tmp[at[(k >> sh) & 2047]++] = k;
    key.swap(tmp);
  }
  const uint64_t mask = (1ull << nb) - 1;
  for (size_t t = 0; t < n; ++t) idx[t] = (int32_t)(key[t] & mask);
  vec_give(tmp);
  return idx;
}

// `v` reordered by ascending key[v's position]; `key` is used up.
template <typename T>
void gather_by_key(std::vector<T> &v, std::vector<uint64_t> &key) {
  std::vector<int32_t> o = order_by_key(key);
  std::vector<T> w;
  vec_take(w);
  w.resize(v.size());
  for (size_t t = 0; t < o.size(); ++t) w[t] = v[o[t]];
  v.swap(w);
  vec_give(w);
  vec_give(o);
}

// Lengths are at most 1,000,000 (< 2^20), strips of STRIP rows at most 2^13.
constexpr uint64_t LEN_TOP = (1u << 20) - 1, STRIPS_TOP = (1u << 13) - 1;
static_assert((1000000 + STRIP - 1) / STRIP <= (int)STRIPS_TOP, "strip count exceeds its key field");

// Wave units: GWAVE / GG tasks of GG lanes and one shape that one wave runs
// in lockstep.  Local couples are ordered by (strips, columns) and take their
// unit's column count as leading pad columns; global couples need equal
// column counts (H(m, n) is read at the last column), so they are grouped by
// columns.  Whole-wave tasks are units of one.  Units go out largest first
// (more 8-step blocks first, S * NB < 2^40, stable), with offsets in that order.
void plan_units(Plan &pl, TaskList &L, bool local, bool trace) {
  const int GG = L.GG, NG = GWAVE / GG;
  std::vector<Unit> &u = L.units;
  auto strips = [GG](int m) { return ceil_div(std::max(m, 1), GG * R); };
  std::vector<uint64_t> key;
  vec_take(key);
  if (NG > 1) {  // local: more strips first, then more columns; global: columns first
    key.resize(u.size());
    for (size_t t = 0; t < u.size(); ++t) {
      const uint64_t sk = STRIPS_TOP - (uint64_t)strips(u[t].m), nk = LEN_TOP - (uint64_t)u[t].n;
      key[t] = local ? (sk << 20 | nk) : (nk << 13 | sk);
    }
    gather_by_key(u, key);
  }
  std::vector<TaskSpan> spans;
  vec_take(spans);
  key.clear();
  for (size_t k = 0; k < u.size();) {
    size_t e = k;
    int nq = 0, mq = 0;
    for (; e < u.size() && e - k < (size_t)NG && (local || u[e].n == u[k].n); ++e) {
      nq = std::max(nq, u[e].n);
      mq = std::max(mq, u[e].m);
    }
    spans.push_back(TaskSpan{TaskAt{0, 0, 0, 0}, (uint32_t)k, (uint32_t)(e - k), nq, strips(mq)});
    key.push_back((1ull << 40) - (uint64_t)strips(mq) * (uint64_t)ceil_div(nq + GG, 8));
    k = e;
  }
  gather_by_key(spans, key);
  vec_give(key);
  for (TaskSpan &s : spans) {
    const TaskAt sz = task_span(L.P, GG, trace, s.n, s.S);
    s.at = TaskAt{pl.rows_n, pl.cols_n, pl.ring_elems, pl.tb_bytes};
    pl.rows_n += s.cnt * sz.row; pl.cols_n += s.cnt * sz.col;
    pl.ring_elems += s.cnt * sz.ring; pl.tb_bytes += s.cnt * sz.tb;
  }
  L.spans.swap(spans);
  vec_give(spans);
}

// The wave units of int32 singles `u`, written on the host.
void add_units(Plan &pl, std::vector<Task> &dst, std::vector<Unit> u, bool local, bool trace,
               const std::vector<HostPair> &hp) {
  TaskList L;
  L.P = 1; L.GG = G;
  L.units.swap(u);
  Plan shapes;
  plan_units(shapes, L, local, trace);
  for (const TaskSpan &s : L.spans) {
    const size_t first = dst.size();
    for (uint32_t i = s.u0; i < s.u0 + s.cnt; ++i)
      add_task(pl, dst, 1, G, trace, hp, L.units[i].lo, L.units[i].hi, L.units[i].single, s.n, s.S);
    for (uint32_t q = s.cnt; q < (uint32_t)NGW; ++q) {  // fillers: copies that write nothing
      Task f = dst[first];
      f.single = 2;
      dst.push_back(f);
    }
  }
}

// Steps a G-lane group needs for a task of these shapes, in 8-step blocks.
double group_cost(int mmax, int n) { return (double)ceil_div(mmax, G * R) * ceil_div(n + G, 8); }

// The same for an 8-lane group (64-row strips, a 7-column skew).
double cost8(int mmax, int n) { return (double)ceil_div(mmax, 8 * R) * ceil_div(n + 8, 8); }

// Packed couples whose 8-lane sweep takes at most this fraction of the mean
// work of a group slot go into 8-lane units (8 tasks per wave; global ones of
// equal column counts): 64-row strips and a 7-column skew compute fewer pad
// cells than 128-row strips and a 15-column skew (65,536-pair log-normal
// local batch: 1.11x the real cells instead of 1.164x; the 130,816-pair
// all-vs-all fill 4.07 -> 3.85 ms), while the 16-lane units keep the tasks
// whose 8-lane units would be long enough to end the run late.  A
// list-scheduling model of the local batch gives the shortest run between
// 0.4x and 0.9x; 8-lane units of every task end it ~50% late.
double eight_lane_limit() {
  const char *e = getenv("TWEAKALIGN_EIGHT_LANE");  // fraction; "0" turns 8-lane units off
  return e ? atof(e) : 0.5;
}


// Whole-wave groups for tasks long enough to set the makespan of a group
// sweep: more than 0.75x the mean work of a group slot (a list-scheduling
// simulation of the 65,536-pair log-normal batch gives 99% slot efficiency
// there, 68% at 1.5x), and tall enough (>= 384 rows) not to waste most of a
// 512-row strip.  With fewer tasks than resident waves (`few`) the run takes
// as long as one task's sweep, so every task taller than one group strip
// gets a whole wave (a lone 300 x 320 pair: 384 steps instead of 1,008 in
// 16-lane strips).
int pick_gg(int mmax, int n, double mean_slot, bool few) {
  if (mmax <= G * R) return G;
  if (few) return GWAVE;
  return (mmax >= 3 * GWAVE * R / 4 && group_cost(mmax, n) > 0.75 * mean_slot) ? GWAVE : G;
}

// Direction-plane records of single pairs, rewritten.
struct PtbPatch {
  PairTB d;
  int32_t pair, pad_;
};
__global__ void patch_ptb_kernel(const PtbPatch *p, int n, PairTB *ptb) {
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) ptb[p[q].pair] = p[q].d;
}

// Start of a run: work-queue counters to 0, fill outputs to their initial
// values (empty pairs keep theirs).  A kernel rather than memset / memcpy
// nodes, so a captured run is all kernels.
__global__ void init_kernel(int32_t *ctr, int nctr, FillOut *fo, const FillOut *fo_init, int n) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  for (int k = tid; k < nctr; k += stride) ctr[k] = 0;
  for (int k = tid; k < n; k += stride) fo[k] = fo_init[k];
}

}  // namespace

struct ta_batch {
  hipStream_t stream = nullptr;  // the context stream, or a serving stream
  ta_params p{};
  int32_t n = 0;
  Alphabet alph;
  int Kp = 0;
  bool trace = false;       // direction planes are stored (local, or CIGAR asked)
  bool may_saturate = false;
  int64_t cells = 0;
  std::vector<HostPair> hp;
  FillOut *d_fo_init = nullptr;
  int32_t *d_order = nullptr;  // traceback walker -> pair, longest first
  // Walks inside the fill kernel (direction planes, no int32 rerun possible):
  // the traceback kernel then takes only the pairs no fill task holds.
  bool walk = false;
  // Walking batches of few tasks: the first ncoop[P-1]... whole-wave tasks of
  // each lane width are swept by a workgroup's fill waves together.
  int32_t ncoop2 = 0, ncoop1 = 0;
  int32_t n_rest = 0;
  int32_t *d_order_rest = nullptr;
  uint64_t cig_bytes = 0;
  Plan plan;
  // device
  uint8_t *d_codes = nullptr;
  std::shared_ptr<uint8_t> codes_owner;  // set when d_codes is a resident-sequence arena (held, not freed)
  void *d_bulk = nullptr;         // the block of the tables that go up in one copy (BulkUpload)
  int8_t *d_table = nullptr;
  int8_t *d_table_nib = nullptr;  // packed couples: 4-bit biased scores
  bool nib = false;
  bool shift = false;             // packed couples, score only: shifted values fit (shift_fits)
  int fill_waves = 0;             // resident fill waves per CU (0: default_waves)
  bool wave_tasks = false;        // whole-wave groups for every multi-strip task
  Task *d_tasks2[3] = {nullptr, nullptr, nullptr}, *d_tasks1[3] = {nullptr, nullptr, nullptr};
  uint16_t *d_rowcodes = nullptr, *d_colcodes = nullptr;
  uint32_t *d_ring = nullptr;
  uint8_t *d_tb = nullptr;
  PairTB *d_ptb = nullptr;
  PairDev *d_pairs = nullptr;
  FillOut *d_fo = nullptr;
  ResultDev *d_res = nullptr;
  char *d_cig = nullptr;
  int32_t *d_ctr = nullptr;
  // int32 rerun of saturated pairs (allocated on demand)
  Task *d_tasks_r = nullptr;
  uint16_t *d_rowcodes_r = nullptr, *d_colcodes_r = nullptr;
  uint32_t *d_ring_r = nullptr;
  uint8_t *d_tb_r = nullptr;
  PtbPatch *d_patch_r = nullptr;
  int32_t n_rerun = 0;
  // long-pair pipeline
  std::vector<LongPair> longs;
  std::vector<LongItem> litems;
  std::vector<LongGroup> lgroups;
  LongPair *d_lp = nullptr;
  LongItem *d_litems = nullptr;
  int2 *d_lring = nullptr;    // bottom rows, then checkpoint columns, of a group
  uint32_t *d_wpl = nullptr;  // region codes of the traceback workgroups
  // Regions computed ahead (0: none), and the guesses they are placed by.
  int32_t lahead = 0;
  uint32_t *d_lahead = nullptr;
  int32_t *d_lcross = nullptr;
  uint64_t lring_n = 0, lcol_n = 0;
  int32_t long_wgs = 0, spin_limit = 1 << 20;  // about a second of polling
  // Most steps a traceback walk may take (TWEAKALIGN_WALK_GUARD lowers it so
  // that walks end flagged; otherwise above every walk's length).
  int32_t guard_cap = INT32_MAX;
  // Batches of few pairs (strips.h).
  bool strips = false;
  int strips_bcode = 0;
  std::vector<StripPair> spairs;
  std::vector<StripItem> sitems;
  StripPair *d_spairs = nullptr;
  StripItem *d_sitems = nullptr;
  int2 *d_sring = nullptr;
  uint32_t *d_splanes = nullptr;
  uint64_t *d_sbest = nullptr;
  int32_t *d_sscore = nullptr;
  uint64_t sring_n = 0, splanes_n = 0;
  // captured run
  bool graph_on = false, phases_timed = false;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  // timing
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  std::vector<hipEvent_t> gev;  // around the tracebacks of all long groups but the last
  bool gev_timed = false;       // by the last run
  double ms[4] = {0, 0, 0, 0};
  // plain (one launch per pair) resources, built on first use
  bool plain_ready = false;
  std::vector<Task> plain_tasks;
  Task *d_plain_tasks = nullptr;
  // int32 reruns of the pairs whose int16 fill may saturate: NGW entries
  // each (index plain_rerun[k]), their planes' PairTB in d_pptb_r
  std::vector<int32_t> plain_rerun;
  Task *d_plain_rtasks = nullptr;
  PairTB *d_pptb_r = nullptr;
  uint16_t *d_prow = nullptr, *d_pcol = nullptr;
  uint32_t *d_pring = nullptr;
  uint8_t *d_ptbuf = nullptr;
  PairTB *d_pptb = nullptr;
};

namespace {

bool global_i16_safe(const ta_params &p, int maxS, int la, int lb) {
  const long lo = 3L * -p.gap_open + (long)(la + lb + 2) * -p.gap_extend + 128;
  const long hi = (long)std::min(la, lb) * maxS + maxS;
  return lo < 16000 && hi < 32000;
}
}  // namespace

bool global_int16_safe(const ta_params *p, int maxS, int la, int lb) { return global_i16_safe(*p, maxS, la, lb); }

namespace {

// Resident fill waves per CU a batch asks for: its tuning, else one per SIMD
// when direction planes are written (those kernels keep a SIMD busy alone and
// more waves slowed the 65,536-pair batch: 8.4 ms at 4 per CU, 9.1 at 8),
// else three per SIMD (the score-only kernels are leaner and latency-exposed:
// packed int16 ops issue at 77% of peak with one wave, 90% with two; the
// all-vs-all batch runs 5.6 ms at 4 per CU, 4.3 at 8, 4.0 at 12).
int waves_wanted(const ta_batch *B) { return B->fill_waves ? B->fill_waves : (B->trace ? 4 : 12); }

void free_rerun(ta_batch *B) {
  dfree(B->d_tasks_r); dfree(B->d_rowcodes_r); dfree(B->d_colcodes_r);
  dfree(B->d_ring_r); dfree(B->d_tb_r); dfree(B->d_patch_r);
  B->n_rerun = 0;
}

}  // namespace

void ta_batch_destroy(ta_batch *B) {
  if (!B) return;
  // The blocks go back to the cache, where a batch on another stream may take
  // them at once: the batch's last run (every run form ends by recording
  // ev[3]) must have finished first.  The event is the batch's own, so this
  // holds even where the run's stream is gone.
  if (B->ev[3]) (void)hipEventSynchronize(B->ev[3]);
  if (B->codes_owner) B->d_codes = nullptr;
  dfree(B->d_codes); dfree(B->d_bulk);
  for (int g = 0; g < 3; ++g) { dfree(B->d_tasks2[g]); dfree(B->d_tasks1[g]); }
  dfree(B->d_rowcodes); dfree(B->d_colcodes); dfree(B->d_ring); dfree(B->d_tb);
  dfree(B->d_ptb); dfree(B->d_pairs); dfree(B->d_fo); dfree(B->d_res); dfree(B->d_cig);
  dfree(B->d_ctr); dfree(B->d_fo_init);
  free_rerun(B);
  dfree(B->d_lring); dfree(B->d_wpl);
  dfree(B->d_lahead); dfree(B->d_lcross);
  dfree(B->d_sring); dfree(B->d_splanes); dfree(B->d_sbest);
  dfree(B->d_sscore);
  dfree(B->d_plain_tasks); dfree(B->d_prow); dfree(B->d_pcol); dfree(B->d_pring);
  dfree(B->d_ptbuf); dfree(B->d_pptb); dfree(B->d_plain_rtasks); dfree(B->d_pptb_r);
  for (auto &e : B->ev)
    if (e) (void)hipEventDestroy(e);
  for (auto &e : B->gev)
    if (e) (void)hipEventDestroy(e);
  if (B->gexec) (void)hipGraphExecDestroy(B->gexec);
  if (B->graph) (void)hipGraphDestroy(B->graph);
  vec_give(B->hp);
  for (int g = 0; g < 3; ++g) {
    vec_give(B->plan.list2[g].units);
    vec_give(B->plan.list2[g].spans);
    vec_give(B->plan.list1[g].units);
    vec_give(B->plan.list1[g].spans);
  }
  delete B;
}

// Origin of a shifted fill's values, which makes the lowest one -32,700.
static int shift_base(const ta_params &p) { return -32700 - 3 * (p.gap_open - p.gap_extend); }

// Whether score-only global couples take the shifted fill: it takes 17% fewer
// instructions (1.75e9 against 2.12e9 for 130,816 pairs, 3.2 ms against 3.9)
// and is the faster one wherever its values fit.  Opening must
// cost at least extending (or gaps raise the values), and the nibbles'
// constant must be a byte's (0..240).  A pair that global_i16_safe admits
// has 3 |open| + (la + lb) |ext| < 16,000 and min(la, lb) max S < 32,000, so
// its largest value is below -32,700 + 48,000.
static bool shift_fits(const ta_params &p, const Alphabet &A) {
  const int k0 = A.minS - p.gap_open - p.gap_extend;
  return p.gap_open <= p.gap_extend && k0 >= 0 && k0 <= 240;
}

// A pair the batch runtime takes: lengths in range, letters present, and
// (global) scores clear of the int32 kernels' -infinity (-2^29).
static bool pair_ok(const ta_params &p, const ta_pair &q) {
  if (q.la < 0 || q.lb < 0 || q.la > 1000000 || q.lb > 1000000 || (q.la && !q.a) || (q.lb && !q.b)) return false;
  return p.mode == TA_LOCAL ||
         (int64_t)(q.la + q.lb + 2) * -p.gap_extend + 2 * (int64_t)-p.gap_open < (1ll << 28);
}

// Whether a batch's pairs all go strip by strip over the whole GPU (strips.h),
// and their items.  Its steps are int32 and single pairs, about twice the
// instructions per cell of the packed fill, and buy a run as long as the
// longest pair's pipeline instead of its sweep by one or four waves.  Both
// sides measured on related protein pairs, lengths up to L (half of it at
// least), from run to results in place, us, task form / strips:
//   strips per SIMD   global                           local
//     0.9 (L 1200)    1,482 / 341                      1,635 / 393
//     3.5 (L 600)       811 / 333                        890 / 423
//     7   (L 1200)    2,552 / 793                      1,899 / 1,095
//     9   (L 400)       862 / 439                        947 / 590
//    19   (L 200)       486 / 570                        521 / 738
// so batches of up to 8 strips per SIMD take it, except very short pairs,
// whose whole run is launches: a pair costs it 18 ns, and three launches and
// a status copy 25 us, which a longest pair of la + lb = 60 + pairs / 24 gains
// back (L 30: 2 pairs 72 / 73, 2,048 95 / 117; L 120: 4,096 218 / 185,
// 8,192 219 / 245).
static void plan_strips(ta_ctx *ctx, ta_batch *B) {
  if (!B->trace || getenv("TWEAKALIGN_COOP") || getenv("TWEAKALIGN_WALK_IN_FILL")) return;
  const bool local = B->p.mode == TA_LOCAL;
  int64_t strips = 0;
  int max_t = 0, longest = 0;
  std::vector<int32_t> ks;
  for (int32_t k = 0; k < B->n; ++k) {
    const HostPair &h = B->hp[k];
    if (h.path != 1 && h.path != 2) continue;
    if (h.lb > STRIPS_MAXN) return;
    // local H and its bound in the end-cell keys
    if (local && (int64_t)std::min(h.la, h.lb) * std::max(0, B->alph.maxS) >= 65400) return;
    ks.push_back(k);
    strips += ceil_div(h.la, 64 * STRIPS_PR);
    max_t = std::max(max_t, (h.lb + 63 + 7) & ~7);
    longest = std::max(longest, h.la + h.lb);
    if (strips > (int64_t)ctx->cus * 4 * STRIPS_PER_SIMD) return;
  }
  if (ks.empty() || longest < 60 + (int)(ks.size() / 24) || strips_lds(max_t + 96) > ctx->lds_max) return;
  B->strips = true;
  B->strips_bcode = max_t + 96;
  B->may_saturate = false;
  // longest pipelines first
  std::vector<uint64_t> key(ks.size());
  for (size_t t = 0; t < ks.size(); ++t) {
    const HostPair &h = B->hp[ks[t]];
    key[t] = (1ull << 32) - (uint64_t)h.lb - 100ull * ceil_div(h.la, 64 * STRIPS_PR);
  }
  gather_by_key(ks, key);
  B->spairs.reserve(ks.size());
  B->sitems.reserve((size_t)strips);
  for (int32_t k : ks) {
    const HostPair &h = B->hp[k];
    StripPair P{};
    P.a_off = h.a_off; P.b_off = h.b_off;
    P.pid = k; P.m = h.la; P.n = h.lb;
    P.S = ceil_div(h.la, 64 * STRIPS_PR);
    P.T = (h.lb + 63 + 7) & ~7;
    P.i16 = h.path == 2;
    P.ring = B->sring_n;
    B->sring_n += (uint64_t)(P.S - 1) * (P.T + 8);
    P.planes = B->splanes_n;
    B->splanes_n += (uint64_t)P.S * (P.T / strip_spd(STRIPS_PR)) * 64;
    for (int s = 0; s < P.S; ++s) B->sitems.push_back(StripItem{(int32_t)B->spairs.size(), s});
    B->spairs.push_back(P);
  }
}

int ta_batch_create(ta_ctx *ctx, const ta_params *p, const ta_pair *pairs, int32_t n, ta_batch **out) {
  return batch_create_on(ctx, p, pairs, n, ctx ? ctx->stream : nullptr, out);
}

int batch_create_on(ta_ctx *ctx, const ta_params *p, const ta_pair *pairs, int32_t n, hipStream_t stream,
                    ta_batch **out, const ta_tuning *force, const ResidentBatch *res, int64_t admitted) {
  if (!ctx || !p || !out || n < 0 || (n > 0 && !pairs && !res)) return TA_E_INVALID;
  *out = nullptr;
  if (params_check(p)) return TA_E_INVALID;
  if (res && ((int64_t)res->la.size() != n || (n > 0 && !res->arena))) return TA_E_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  PhaseTrace tr("create");

  ta_batch *B = new ta_batch();
  B->stream = stream;
  B->p = *p;
  B->n = n;
  B->alph = make_alphabet(p->alphabet, p->match, p->mismatch);
  B->Kp = B->alph.K + 1;
  const bool local = p->mode == TA_LOCAL;
  B->trace = local || p->traceback;
  B->nib = nibble_ok(B->alph, local);
  // Launch shape: the autotuner's candidate, else the context's tuning for
  // this kind of batch, else the defaults.
  ta_tuning tu{0, TA_LANES_AUTO, 0};
  if (force) {
    tu = *force;
  } else {
    std::lock_guard<std::mutex> g(ctx->tune_mu);
    int bucket = 0;
    if (ctx->tune.empty()) {
      // (the defaults)
    } else if (res) {  // the bucket from the resident sequences' lengths
      std::vector<ta_pair> lens((size_t)n);
      for (int32_t k = 0; k < n; ++k) lens[k] = ta_pair{nullptr, res->la[k], nullptr, res->lb[k]};
      bucket = ta_tune_bucket(lens.data(), n);
    } else {
      bucket = ta_tune_bucket(pairs, n);
    }
    auto it = ctx->tune.find(tune_key(p, bucket));
    if (it != ctx->tune.end()) tu = it->second;
  }
  B->fill_waves = tu.waves_per_cu;
  B->wave_tasks = tu.wave_tasks != 0;
  const int lanes = p->lanes != TA_LANES_AUTO ? p->lanes : tu.lanes;

  // Encode (sequences shared between pairs are encoded once).  Each
  // sequence also gets the sum over its residues of the best score the
  // residue can reach against any letter (0 if none is positive): no local
  // alignment of it scores more, which decides whether int16 can saturate.
  int best[32] = {0}, maxbest = 0;
  for (int r = 0; r < B->alph.K; ++r)
    for (int c = 0; c < B->alph.K; ++c) best[r] = std::max<int>(best[r], B->alph.S[r * B->alph.K + c]);
  for (int r = 0; r < B->alph.K; ++r) maxbest = std::max(maxbest, best[r]);
  const int64_t sat_limit = 32767 - 2L * B->alph.maxS;
  // Unique sequences (by pointer and length) and their offsets in the code
  // array.  Pointers are split by hash over the host threads; each thread
  // scans every pair and keeps a table for its share only (a few hundred KB,
  // cache-resident), mapping a pointer to its latest unique entry, so the
  // same pointer always meets the same thread, in pair order.
  struct Uniq { const char *s; int32_t len; uint64_t off; int64_t bound; };
  // A pair as the checks and the planner see it (resident sequences: the
  // lengths; their letters are on the device).
  auto pair_at = [&](int32_t k) -> ta_pair {
    if (!res) return pairs[k];
    const int32_t la = res->la[k], lb = res->lb[k];
    return ta_pair{la ? "" : nullptr, la, lb ? "" : nullptr, lb};
  };
  // The pairs in contiguous shares, one per host thread: sums first, then the
  // tables at the offsets they give.
  struct Share {
    bool ok = true, maysat = false;
    int64_t cells = 0;
    uint64_t cig = 0;
    size_t n16 = 0, n32 = 0;
  };
  const int NS = n >= 4096 ? (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency())) : 1;
  auto share_at = [&](int t) { return (int32_t)((int64_t)n * t / NS); };
  std::vector<Share> shares(NS);
  parallel_tasks(NS, [&](int t) {
    Share s;
    for (int32_t k = share_at(t); k < share_at(t + 1); ++k) {
      const ta_pair q = pair_at(k);
      if (!pair_ok(*p, q)) s.ok = false;
      s.cells += (int64_t)q.la * q.lb;
      s.cig += (uint64_t)(p->traceback ? 4 * (q.la + q.lb + 1) : 0);  // one dword per run at most
    }
    shares[t] = s;
  });
  uint64_t cig = 0;
  for (Share &s : shares) {
    if (!s.ok) {
      delete B;
      return TA_E_INVALID;
    }
    B->cells += s.cells;
    const uint64_t at = cig;
    cig += s.cig;
    s.cig = at;
  }
  B->cig_bytes = cig;
  tr.mark("validate");
  auto mix = [](const char *s) -> uint64_t {
    uint64_t x = (uint64_t)(uintptr_t)s;
    x = (x ^ (x >> 29)) * 0xbf58476d1ce4e5b9ull;
    return x ^ (x >> 32);
  };
  const int T = n >= 8192 ? (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency())) : 1;
  // a pointer's thread: the hash's top 32 bits scaled to [0, T) (no division)
  auto part_of = [T](uint64_t x) { return (int)(((x >> 32) * (uint64_t)T) >> 32); };
  // The calling thread's buffers, kept between calls: their pages stay
  // mapped (first-touch page faults cost more than the work here).
  // (Named through references: the worker threads below must reach the
  // calling thread's copies, not their own.)
  static thread_local std::vector<int32_t> tl_ua, tl_ub;
  static thread_local std::vector<std::vector<Uniq>> tl_part;
  static thread_local std::vector<Uniq> tl_uq;
  std::vector<int32_t> &ua = tl_ua, &ub = tl_ub;
  std::vector<std::vector<Uniq>> &part = tl_part;
  std::vector<Uniq> &uq = tl_uq;
  size_t ctotal = 0;  // bytes of the unique sequences' codes
  std::vector<int32_t> base(T + 1, 0);  // first unique entry of each thread's share
  std::vector<char> sums(T, 0);         // whether a share has a sequence whose bound must be summed
  if (!res) {
    ua.resize((size_t)n);
    ub.resize((size_t)n);
    if ((int)part.size() < T) part.resize(T);
    for (int t = 0; t < T; ++t) part[t].clear();
    parallel_tasks(T, [&](int t) {
      struct Slot { const char *s; int32_t idx; };
      // sized for this thread's expected share at most a quarter full; the
      // thread keeps it between calls (the host pool's threads live on)
      size_t cap = 64;
      while (cap < 8 * (size_t)n / (size_t)T) cap <<= 1;
      static thread_local std::vector<Slot> tl_tab;
      std::vector<Slot> &tab = tl_tab;
      if (tab.size() != cap) tab.assign(cap, Slot{nullptr, -1});
      else std::fill(tab.begin(), tab.end(), Slot{nullptr, -1});
      std::vector<Uniq> &mine = part[t];
      auto grow = [&]() {  // keep the table at most half full
        std::vector<Slot> old(2 * cap, Slot{nullptr, -1});
        old.swap(tab);
        cap *= 2;
        for (const Slot &e : old) {
          if (e.idx < 0) continue;
          size_t h = (size_t)mix(e.s) & (cap - 1);
          while (tab[h].idx >= 0) h = (h + 1) & (cap - 1);
          tab[h] = e;
        }
      };
      auto uniq = [&](const char *s, int32_t len, uint64_t x) -> int32_t {
        size_t h = (size_t)x & (cap - 1);
        while (tab[h].idx >= 0 && tab[h].s != s) h = (h + 1) & (cap - 1);
        if (tab[h].idx >= 0 && mine[tab[h].idx].len == len) return tab[h].idx;
        const bool fresh = tab[h].idx < 0;
        mine.push_back(Uniq{s, len, 0, -1});
        tab[h] = Slot{s, (int32_t)mine.size() - 1};
        if (fresh && 2 * mine.size() > cap) grow();
        return (int32_t)mine.size() - 1;
      };
      for (int32_t k = 0; k < n; ++k) {
        const ta_pair &q = pairs[k];
        const uint64_t xa = mix(q.a), xb = mix(q.b);
        if (part_of(xa) == t) ua[k] = uniq(q.a, q.la, xa);
        if (part_of(xb) == t) ub[k] = uniq(q.b, q.lb, xb);
      }
    });
    tr.mark("dedupe hash");
    // Global order: partition by partition; each sequence starts 16-byte
    // aligned (walker windows).  Offsets, bounds from the lengths alone and the
    // flat array, per partition on the threads, from the partitions' counts and
    // byte totals.
    std::vector<size_t> bbase(T + 1, 0);
    for (int t = 0; t < T; ++t) {
      base[t + 1] = base[t] + (int32_t)part[t].size();
      size_t bytes = 0;
      for (const Uniq &e : part[t]) bytes += ((size_t)e.len + 15) & ~(size_t)15;
      bbase[t + 1] = bbase[t] + bytes;
    }
    uq.resize((size_t)base[T]);
    parallel_tasks(T, [&](int t) {
      size_t at = bbase[t];
      Uniq *dst = uq.data() + base[t];
      for (const Uniq &e : part[t]) {
        *dst = e;
        dst->off = at;
        if (local) {
          dst->bound = (int64_t)e.len * maxbest;
          if (dst->bound > sat_limit) sums[t] = 1;
        }
        at += ((size_t)e.len + 15) & ~(size_t)15;
        ++dst;
      }
    });
    ctotal = bbase[T];
    tr.mark("dedupe offsets");
  }
  // The walker reads 32-byte windows: 32 bytes of slack after the last
  // sequence.  The raw letters go up as they are, each sequence followed by
  // a letter that encodes to 0 up to the next 16-byte start (each host thread
  // copies its sequences, so the pages are first touched in parallel), and
  // the GPU encodes them in place, flagging letters outside the alphabet.
  const size_t cend = ((ctotal + 15) & ~(size_t)15) + 32;
  StageHold codes;  // raw letters of the unique sequences, 16-byte aligned starts
  if (!res) {
    codes.s = stage_take(cend);
    if (!codes.s.p) {
      delete B;
      return TA_E_NOMEM;
    }
  }
  uint8_t map[256], pad_letter = 0;
  for (int b = 255; b >= 0; --b) {
    const int c = B->alph.map[b];
    map[b] = c < 0 ? 0xff : (uint8_t)c;
    if (c == 0) pad_letter = (uint8_t)b;
  }
  if (!res) {
    parallel_for(uq.size(), [&](size_t u) {
      const Uniq &e = uq[u];
      uint8_t *dst = codes.s.p + e.off;
      if (e.len) memcpy(dst, e.s, (size_t)e.len);
      const size_t next = u + 1 < uq.size() ? uq[u + 1].off : cend;
      memset(dst + e.len, pad_letter, next - (e.off + (size_t)e.len));
    });
    if (uq.empty()) memset(codes.s.p, pad_letter, cend);
  }
  tr.mark("letters");
  // The sum over a sequence's residues of the best score each can reach
  // (0 if none is positive) bounds any local alignment of it; it decides
  // whether int16 can saturate, which only a sequence longer than
  // limit / (best of all letters) can reach, so only such sequences are summed.
  // (A pass of the host threads that finds none costs small batches 30-45 us: 256
  // pairs of up to 20 residues 251-271 us a call with it, 207-220 without.)
  if (std::any_of(sums.begin(), sums.end(), [](char x) { return x != 0; }))
    parallel_for(uq.size(), [&](size_t u) {
      Uniq &e = uq[u];
      if (e.bound <= sat_limit) return;
      int64_t sum = 0;
      const unsigned char *src = (const unsigned char *)e.s;
      for (int32_t i = 0; i < e.len; ++i) sum += map[src[i]] < 0x80 ? best[map[src[i]]] : 0;
      e.bound = sum;
    });
  // The letters go up while the host plans: from the pinned block the copy
  // runs on the DMA engine alone; the encoding kernel follows on the stream.
  hipStream_t st = B->stream;
  int rc = TA_OK;
  // the counters, and behind them whether a letter was outside the alphabet
  rc = dalloc(&B->d_ctr, 32);
  if (!rc && hipMemsetAsync(B->d_ctr, 0, 32 * sizeof(int32_t), st) != hipSuccess) rc = TA_E_DEVICE;
  int32_t *d_bad = B->d_ctr + 16;
  if (res) {  // resident sequences: the codes are on the device already
    B->codes_owner = res->arena;
    B->d_codes = res->arena.get();
  } else if (!rc) {
    rc = dalloc(&B->d_codes, cend);
  }
  if (!rc && !res) {
    codes.stream = st;
    codes.queued = true;
    if (hipMemcpyAsync(B->d_codes, codes.s.p, cend, hipMemcpyHostToDevice, st) != hipSuccess) rc = TA_E_DEVICE;
  }
  if (!rc && !res) {
    (void)hipGetLastError();
    LetterMap lm;
    memcpy(lm.w, map, 256);
    const size_t words = cend / 16;
    hipLaunchKernelGGL(encode_kernel, dim3((unsigned)std::min<size_t>((words + 255) / 256, 4096)), dim3(256), 0, st,
                       (uint4 *)B->d_codes, words, lm, d_bad);
    if (hipGetLastError() != hipSuccess) rc = TA_E_DEVICE;
  }
  if (rc) {
    (void)hipStreamSynchronize(st);
    ta_batch_destroy(B);
    return rc;
  }
  tr.mark("upload-encode");
  // The pairs' table goes up while the host plans, too.
  StageHold ptab;
  ptab.s = stage_take(sizeof(PairDev) * (size_t)n + 64);  // (and where the letter check comes back)
  if (!ptab.s.p) rc = TA_E_NOMEM;
  PairDev *pairs_h = (PairDev *)ptab.s.p;
  int32_t *bad_letter = (int32_t *)(pairs_h + n);
  vec_take(B->hp);
  B->hp.resize(n);
  if (!rc) parallel_tasks(NS, [&](int t) {
    Share &s = shares[t];
    uint64_t cig_at = s.cig;
    for (int32_t k = share_at(t); k < share_at(t + 1); ++k) {
      const ta_pair q = pair_at(k);
      HostPair h{};
      int32_t a = 0, b = 0;
      if (!res) {
        a = ua[k] + (T > 1 ? base[part_of(mix(q.a))] : 0);
        b = ub[k] + (T > 1 ? base[part_of(mix(q.b))] : 0);
      }
      h.a_off = res ? res->a_off[k] : uq[a].off;
      h.b_off = res ? res->b_off[k] : uq[b].off;
      h.la = q.la; h.lb = q.lb;
      if (q.la == 0 || q.lb == 0) {
        h.path = 0;
      } else if (long_pair(*p, q.la, q.lb)) {
        h.path = 3;
      } else if (lanes == TA_LANES_I32 || (!B->nib && !B->trace)) {
        h.path = 1;
      } else if (local && q.lb > 32767) {
        h.path = 1;  // packed end-cell keys hold the column in 15 bits
      } else if (local) {
        h.path = 2;
        h.maysat = (res ? std::min(res->a_bound[k], res->b_bound[k]) : std::min(uq[a].bound, uq[b].bound)) > sat_limit;
        if (h.maysat) s.maysat = true;
      } else {
        h.path = global_i16_safe(*p, B->alph.maxS, q.la, q.lb) ? 2 : 1;
      }
      s.n16 += h.path == 2;
      s.n32 += h.path == 1;
      B->hp[k] = h;
      PairDev d{};
      d.a_off = h.a_off; d.b_off = h.b_off; d.la = q.la; d.lb = q.lb;
      d.cig_cap = p->traceback ? 4 * (q.la + q.lb + 1) : 0;
      d.cig_off = cig_at;
      cig_at += (uint64_t)d.cig_cap;
      pairs_h[k] = d;
    }
  });
  for (const Share &s : shares) B->may_saturate = B->may_saturate || s.maysat;
  B->shift = B->nib && !B->trace && shift_fits(*p, B->alph);
  rc = rc ? rc : dalloc(&B->d_pairs, (size_t)std::max(n, 1));
  rc = rc ? rc : dalloc(&B->d_fo_init, (size_t)std::max(n, 1));
  rc = rc ? rc : dalloc(&B->d_ptb, (size_t)std::max(n, 1));
  if (!rc && n) {
    ptab.stream = st;
    ptab.queued = true;
    const int64_t long_cells = local ? INT64_MAX : p->lanes == TA_LANES_LONG ? 1
                                     : p->lanes == TA_LANES_AUTO ? kLongCells : INT64_MAX;
    (void)hipGetLastError();
    if (hipMemcpyAsync(B->d_pairs, pairs_h, sizeof(PairDev) * n, hipMemcpyHostToDevice, st) != hipSuccess)
      rc = TA_E_DEVICE;
    if (!rc) hipLaunchKernelGGL(pairs_init_kernel, dim3((unsigned)std::min(1024, (n + 255) / 256)), dim3(256), 0, st,
                                B->d_pairs, n, B->d_fo_init, B->d_ptb, (int)local, p->gap_open, p->gap_extend, long_cells);
    if (hipGetLastError() != hipSuccess) rc = TA_E_DEVICE;
  }
  if (rc) {
    (void)hipStreamSynchronize(st);
    ta_batch_destroy(B);
    return rc;
  }

  tr.mark("pairs");
  // (a tuning is a shape of the task form, so candidates are timed in it)
  if (!force) plan_strips(ctx, B);
  // Couples: local pairs pad to the longer column count; global couples
  // need equal column counts (so H(m, n) of both sits in the last column).
  Plan &pl = B->plan;
  for (int g = 0; g < 3; ++g) {
    vec_take(pl.list2[g].units);
    vec_take(pl.list1[g].units);
  }
  std::vector<int32_t> i16, i32;
  std::vector<uint64_t> key;
  vec_take(i16);
  vec_take(i32);
  vec_take(key);
  // More strips first, then more columns, then lower pair index (the lists
  // hold ascending pair indices).
  // Local pairs are ranked by 64-row strips (those of 8-lane units), which
  // keeps them in order of 128-row strips too.
  const int rank_rows = local ? 8 * R : STRIP;
  static_assert((1000000 + 8 * R - 1) / (8 * R) < (1 << 15), "strip count exceeds its key field");
  // Global couples: groups of equal columns in ascending order, each ranked so.
  if (!B->strips) {
    size_t n16 = 0, n32 = 0;
    std::vector<size_t> at16(NS), at32(NS);
    for (int t = 0; t < NS; ++t) {
      at16[t] = n16; at32[t] = n32;
      n16 += shares[t].n16; n32 += shares[t].n32;
    }
    i16.resize(n16);
    i32.resize(n32);
    key.resize(n16);
    parallel_tasks(NS, [&](int t) {
      size_t a = at16[t], b = at32[t];
      for (int32_t k = share_at(t); k < share_at(t + 1); ++k) {
        const HostPair &h = B->hp[k];
        if (h.path == 1) i32[b++] = k;
        if (h.path != 2) continue;
        const uint64_t rank = (1ull << 15) - (uint64_t)ceil_div(h.la, rank_rows);
        key[a] = local ? rank << 20 | (LEN_TOP - (uint64_t)h.lb) : (uint64_t)h.lb << 16 | rank;
        i16[a++] = k;
      }
    });
    gather_by_key(i16, key);
  }
  tr.mark("ranks");
  // Neighbours pair off; globally, within a group of equal columns, whose odd
  // one out goes alone.
  // (the lengths gathered on the host threads first: a read of a table that
  // they wrote is a miss in one thread's caches)
  std::vector<std::pair<int32_t, int32_t>> len;
  vec_take(len);
  len.resize(i16.size());
  parallel_for(i16.size(), [&](size_t t) {
    const HostPair &h = B->hp[i16[t]];
    len[t] = {h.la, h.lb};
  });
  std::vector<Unit> couples;
  vec_take(couples);
  couples.reserve(local ? (i16.size() + 1) / 2 : i16.size());
  double work = 0;  // mean group-slot work decides which tasks get whole-wave groups
  for (size_t t = 0; t < i16.size();) {
    const bool two = t + 1 < i16.size() && (local || len[t + 1].second == len[t].second);
    const size_t u = two ? t + 1 : t;
    couples.push_back(Unit{i16[t], i16[u], !two, std::max(len[t].first, len[u].first),
                           std::max(len[t].second, len[u].second)});
    work += group_cost(couples.back().m, couples.back().n);
    t += two ? 2 : 1;
  }
  tr.mark("couples");
  for (int k : i32) work += group_cost(B->hp[k].la, B->hp[k].lb);
  // Walks in the fill kernel: batches with direction planes whose int16 fill
  // cannot saturate (a rerun would replace some pairs' planes after the fill),
  // and more than one fill task: a lone task's walk can only start when its
  // fill ends, and the traceback kernel walks it sooner (a 300 x 320 pair:
  // 0.385 ms from run to results instead of 0.402).
  const char *wenv = getenv("TWEAKALIGN_WALK_IN_FILL");  // "0": walks only after the fill
  B->walk = B->trace && !B->may_saturate && !(wenv && wenv[0] == '0') && couples.size() + i32.size() > 1 &&
            walk_lds_bytes(2, B->Kp) <= ctx->lds_max;
  const int wpc = fill_waves_per_cu(2, B->Kp, !B->trace, waves_wanted(B), B->walk);
  const double slots = (double)ctx->cus * wpc * NGW;
  const double mean_slot = work / slots;
  const bool few = B->wave_tasks || couples.size() + i32.size() <= (size_t)ctx->cus * wpc;
  const double lim8 = !few ? eight_lane_limit() * mean_slot : -1.0;
  for (const Unit &c : couples) {
    const int g = pick_gg(c.m, c.n, mean_slot, few) == GWAVE ? 0
                  : cost8(c.m, c.n) <= lim8 && ceil_div(c.m, 8 * R) <= (int)STRIPS_TOP ? 2  // (fits the unit sort key)
                                                                                       : 1;
    pl.list2[g].units.push_back(c);
  }
  for (int k : i32) {
    const HostPair &h = B->hp[k];
    pl.list1[pick_gg(h.la, h.lb, mean_slot, few) == GWAVE ? 0 : 1].units.push_back(Unit{k, k, true, h.la, h.lb});
  }
  vec_give(couples);
  vec_give(len);
  vec_give(i16);
  vec_give(i32);
  vec_give(key);
  tr.mark("task kinds");
  for (int g = 0; g < 3; ++g) plan_units(pl, pl.list2[g], local, B->trace);
  for (int g = 0; g < 2; ++g) plan_units(pl, pl.list1[g], local, B->trace);
  tr.mark("wave units");
  // With few tasks the run lasts as long as its longest whole-wave task, so
  // tasks of two or more strips get a workgroup's fill waves each (strips
  // pipelined across them), as long as there are at most two per CU.
  const char *cenv = getenv("TWEAKALIGN_COOP");  // "0": never
  if (B->walk && few && !(cenv && cenv[0] == '0')) {
    auto multi = [](const TaskSpan &t) { return t.S >= 2; };
    std::vector<TaskSpan> &s2 = pl.list2[0].spans, &s1 = pl.list1[0].spans;
    const size_t c2 = std::count_if(s2.begin(), s2.end(), multi);
    const size_t c1 = std::count_if(s1.begin(), s1.end(), multi);
    if (c2 + c1 > 0 && c2 + c1 <= (size_t)(2 * ctx->cus)) {
      std::stable_partition(s2.begin(), s2.end(), multi);
      std::stable_partition(s1.begin(), s1.end(), multi);
      B->ncoop2 = (int32_t)c2;
      B->ncoop1 = (int32_t)c1;
    }
  }

  tr.mark("tasks");
  // Long pairs: strips of all pairs form one queue, largest pairs first.
  {
    std::vector<int> lk;
    for (int32_t k = 0; k < n; ++k)
      if (B->hp[k].path == 3) lk.push_back(k);
    std::stable_sort(lk.begin(), lk.end(), [&](int x, int y) {
      return (int64_t)B->hp[x].la * B->hp[x].lb > (int64_t)B->hp[y].la * B->hp[y].lb;
    });
    std::vector<std::pair<int32_t, int32_t>> shape;
    for (int k : lk) shape.push_back({B->hp[k].la, B->hp[k].lb});
    int64_t limit = -1;  // bytes they may take
    if (admitted >= 0 && !lk.empty()) {
      limit = admitted;
      for (const HostPair &h : B->hp)
        if (B->trace && h.path != 0 && h.path != 3) limit -= planes_estimate(h.la, h.lb);
    }
    if (const char *e = getenv("TWEAKALIGN_LONG_BYTES")) limit = std::max(0ll, atoll(e));
    LongPlan lpl = long_plan(shape, p->traceback != 0, ctx->cus, limit);
    for (size_t q = 0; q < lk.size(); ++q) {
      const HostPair &h = B->hp[lk[q]];
      LongPair L{};
      L.pid = lk[q]; L.m = h.la; L.n = h.lb; L.S = long_strips(h.la);
      L.T = (int32_t)long_steps(h.lb);
      L.a_off = h.a_off; L.b_off = h.b_off;
      L.ring = lpl.at[q].ring; L.colck = lpl.at[q].col;
      L.item0 = lpl.at[q].item0;
      for (int s = 0; s < L.S; ++s) B->litems.push_back(LongItem{(int32_t)q, s});
      B->longs.push_back(L);
    }
    B->lgroups.swap(lpl.groups);
    B->lring_n = lpl.entries; B->lcol_n = lpl.col_n;
    B->long_wgs = lpl.wgs; B->lahead = lpl.ahead;
    if (const char *e = getenv("TWEAKALIGN_SPIN_LIMIT")) B->spin_limit = std::max(1, atoi(e));
    if (const char *e = getenv("TWEAKALIGN_WALK_GUARD")) B->guard_cap = std::max(0, atoi(e));
  }

  tr.mark("long pairs");
  // Upload: every host-built table in one pinned block.
  std::vector<int8_t> table = padded_table(B->alph), table_nib;
  BulkUpload up;
  up.add(&B->d_table, table);
  if (B->nib && !B->trace) {
    table_nib = nibble_table(B->alph);
    up.add(&B->d_table_nib, table_nib);
  }
  PlanArgs pa{};
  int32_t total = 0;
  Unit *d_units[6] = {nullptr};
  TaskSpan *d_spans[6] = {nullptr};
  for (int l = 0; l < 6; ++l) {
    TaskList &L = l < 3 ? pl.list2[l] : pl.list1[l - 3];
    pa.list[l].ntasks = L.tasks(); pa.list[l].P = L.P; pa.list[l].GG = L.GG;
    total += L.tasks();
    up.add(&d_units[l], L.units);
    up.add(&d_spans[l], L.spans);
  }
  std::vector<int32_t> order, rest;  // longer pairs first
  auto longest_first = [&](std::vector<int32_t> &v) {
    std::vector<uint64_t> len(v.size());
    for (size_t t = 0; t < v.size(); ++t) len[t] = 2000000 - (uint64_t)(B->hp[v[t]].la + B->hp[v[t]].lb);
    gather_by_key(v, len);
  };
  if (B->walk || B->strips) {  // pairs without a fill task: empty and long pairs
    for (int32_t k = 0; k < n; ++k)
      if (B->hp[k].path == 0 || (B->hp[k].path == 3 && !B->strips)) rest.push_back(k);
    longest_first(rest);
    B->n_rest = (int32_t)rest.size();
    up.add(&B->d_order_rest, rest);
  } else if (B->trace) {
    order.resize(n);
    for (int32_t k = 0; k < n; ++k) order[k] = k;
    longest_first(order);
    up.add(&B->d_order, order);
  }
  up.add(&B->d_lp, B->longs);
  up.add(&B->d_litems, B->litems);
  up.add(&B->d_spairs, B->spairs);
  up.add(&B->d_sitems, B->sitems);
  rc = rc ? rc : up.commit(&B->d_bulk, st);
  rc = rc ? rc : dalloc(&B->d_rowcodes, (size_t)pl.rows_n);
  rc = rc ? rc : dalloc(&B->d_colcodes, (size_t)pl.cols_n);
  for (int l = 0; l < 6; ++l) {
    Task **dst = l < 3 ? &B->d_tasks2[l] : &B->d_tasks1[l - 3];
    rc = rc ? rc : dalloc(dst, (size_t)pa.list[l].ntasks);
    pa.list[l].units = d_units[l]; pa.list[l].spans = d_spans[l]; pa.list[l].dst = *dst;
  }
  if (!rc && total) {
    pa.trace = B->trace; pa.pad = B->Kp - 1;
    pa.pairs = B->d_pairs; pa.codes = B->d_codes; pa.ptb = B->d_ptb;
    pa.rowcodes = B->d_rowcodes; pa.colcodes = B->d_colcodes;
    (void)hipGetLastError();
    hipLaunchKernelGGL(plan_tasks_kernel, dim3((unsigned)std::min((total + 3) / 4, 65536)), dim3(256), 0, st, pa, total);
    if (hipGetLastError() != hipSuccess) rc = TA_E_DEVICE;
  }
  tr.mark("uploads");
  rc = rc ? rc : dalloc(&B->d_ring, pl.ring_elems);
  rc = rc ? rc : dalloc(&B->d_tb, pl.tb_bytes);
  rc = rc ? rc : dalloc(&B->d_fo, (size_t)std::max(n, 1));
  rc = rc ? rc : dalloc(&B->d_res, (size_t)std::max(n, 1));
  rc = rc ? rc : dalloc(&B->d_cig, B->cig_bytes);
  rc = rc ? rc : dalloc(&B->d_lring, B->lring_n);
  rc = rc ? rc : dalloc(&B->d_sring, B->sring_n);
  rc = rc ? rc : dalloc(&B->d_splanes, B->splanes_n);
  rc = rc ? rc : dalloc(&B->d_sbest, B->spairs.size());
  rc = rc ? rc : dalloc(&B->d_sscore, B->spairs.size());
  rc = rc ? rc : dalloc(&B->d_wpl, LPLANES * B->long_wgs);
  if (!rc && B->lahead) {
    rc = dalloc(&B->d_lcross, B->litems.size());
    if (!rc && dalloc(&B->d_lahead, LPLANES * B->lahead)) B->lahead = 0;  // (not needed for the result)
  }
  for (auto &e : B->ev)
    if (!rc && hipEventCreate(&e) != hipSuccess) rc = TA_E_DEVICE;
  if (p->traceback && B->lgroups.size() > 1) B->gev.assign(2 * (B->lgroups.size() - 1), nullptr);
  for (auto &e : B->gev)
    if (!rc && hipEventCreate(&e) != hipSuccess) rc = TA_E_DEVICE;
  tr.mark("allocations");
  // Drained on every path: the blocks of a failed creation go back to the
  // cache only after the copies queued into them.  The letter check comes
  // back on the way.
  if (!rc && hipMemcpyAsync(bad_letter, d_bad, sizeof(int32_t), hipMemcpyDeviceToHost, st) != hipSuccess)
    rc = TA_E_DEVICE;
  ptab.stream = st;
  ptab.queued = true;
  if (hipStreamSynchronize(st) != hipSuccess && !rc) rc = TA_E_DEVICE;
  tr.mark("drain");
  if (!rc && *bad_letter) rc = TA_E_ALPHABET;
  if (rc) {
    ta_batch_destroy(B);
    return rc;
  }
  *out = B;
  return TA_OK;
}

AdmitBytes batch_tb_estimate(const ta_params *p, const ta_pair *pairs, int32_t n) {
  AdmitBytes t;
  if (!p) return t;
  const bool trace = p->mode == TA_LOCAL || p->traceback;
  LongNeed longs;
  longs.trace = p->traceback != 0;
  for (int32_t k = 0; k < n; ++k) {
    const int la = pairs[k].la, lb = pairs[k].lb;
    if (la <= 0 || lb <= 0) continue;
    if (long_pair(*p, la, lb)) longs.add(la, lb);
    else if (trace) t.least += planes_estimate(la, lb);
  }
  t.full = t.least + longs.full();
  t.least += longs.least();
  return t;
}

int ta_batch_info(ta_batch *B, int64_t *cells, int64_t *tb_bytes, int32_t *tasks) {
  if (!B) return TA_E_INVALID;
  if (cells) *cells = B->cells;
  if (tb_bytes)
    *tb_bytes = (int64_t)(B->plan.tb_bytes + 4 * LPLANES * (B->long_wgs + B->lahead) + 8 * B->lcol_n + 4 * B->splanes_n);
  if (tasks)
    *tasks = (int32_t)(B->plan.list2[0].tasks() + B->plan.list2[1].tasks() + B->plan.list2[2].tasks() +
                       B->plan.list1[0].tasks() + B->plan.list1[1].tasks() + B->litems.size() + B->sitems.size());
  return TA_OK;
}

// ---------------------------------------------------------------------------
// Launch helpers.
namespace {

TbArgs tb_args(ta_batch *B) {
  TbArgs a;
  a.pairs = B->d_pairs; a.npairs = B->n; a.order = nullptr;
  a.fo = B->d_fo; a.ptb = B->d_ptb;
  a.codes = B->d_codes; a.table = B->d_table; a.Kp = B->Kp; a.tb = B->d_tb; a.cig = B->d_cig;
  a.res = B->d_res;
  a.local = B->p.mode == TA_LOCAL; a.open = B->p.gap_open; a.ext = B->p.gap_extend;
  a.do_cigar = B->p.traceback;
  a.guard_cap = B->guard_cap;
  a.sys = 0;
  return a;
}

// `walk`: the batch's own fill (planes in d_tb); each workgroup's walker wave
// walks the pairs its fill wave finishes.
template <int P>
int launch_fill(ta_ctx *ctx, ta_batch *B, Task *const d_tasks[3], const int ntasks[3], uint16_t *rows,
                uint16_t *cols, uint32_t *ring, uint8_t *tb, int32_t *ctr, int max_groups, bool walk = false) {
  if (ntasks[0] + ntasks[1] + ntasks[2] == 0) return TA_OK;
  const bool nib = P == 2 && !B->trace;  // score-only packed kernels keep 4-bit scores
  FillArgs a;
  for (int g = 0; g < 3; ++g) {
    a.tasks[g] = d_tasks[g];
    a.ntasks[g] = ntasks[g];
  }
  a.ctr = ctr;
  a.ctr8 = B->d_ctr + (P == 2 ? 14 : 15);  // 8-lane units come only from the batch plan
  a.table = nib ? B->d_table_nib : B->d_table; a.Kp = B->Kp;
  a.bias = -B->alph.minS;
  a.shift_base = shift_base(B->p);
  a.rowcodes = rows; a.colcodes = cols; a.ring = ring; a.tb = tb; a.out = B->d_fo;
  a.open = B->p.gap_open; a.ext = B->p.gap_extend;
  a.sat_limit = 32767 - 2 * B->alph.maxS;
  walk = walk && B->trace;
  a.walk = walk;
  if (walk) a.wk = tb_args(B);
  a.ncoop = walk ? (P == 2 ? B->ncoop2 : B->ncoop1) : 0;
  a.coop_ctr = B->d_ctr + (P == 2 ? 12 : 13);
  a.err = B->d_ctr + 10;
  a.spin_limit = B->spin_limit * 16;
  const int lds = walk ? walk_lds_bytes(P, B->Kp) : fill_lds_bytes(P, B->Kp, nib);
  const int per_cu = fill_waves_per_cu(P, B->Kp, nib, waves_wanted(B), walk);
  int groups = ntasks[0] + ntasks[1] + ntasks[2];  // one wave per whole-wave task or wave unit
  if (max_groups > 0) groups = std::min(groups, max_groups);
  groups = std::max(1, std::min(groups, ctx->cus * per_cu));
  if (walk) {  // WALK_FW fill waves per workgroup; a cooperative task takes one
    groups = a.ncoop + (groups - std::min(groups, a.ncoop) + WALK_FW - 1) / WALK_FW;
    groups = std::max(1, std::min(groups, ctx->cus));
  }
  const bool local = B->p.mode == TA_LOCAL;
  void (*k)(FillArgs) = nullptr;
  if (local) k = B->trace ? fill_kernel<P, true, true> : fill_kernel<P, true, false>;
  else k = B->trace ? fill_kernel<P, false, true> : fill_kernel<P, false, false, false>;
  if (P == 2 && B->shift) k = fill_kernel<2, false, false, true>;
  (void)hipGetLastError();  // drop an earlier, already-handled error
  hipLaunchKernelGGL(k, dim3(groups), dim3(walk ? 128 * WALK_FW : 64), lds, B->stream, a);
  HIPCHK(hipGetLastError());
  return TA_OK;
}

int launch_traceback(ta_ctx *ctx, ta_batch *B, const PairDev *pairs, const PairTB *ptb, const uint8_t *tb,
                     int first, int count) {
  if (count <= 0) return TA_OK;
  TbArgs a = tb_args(B);
  const bool whole = first == 0 && count == B->n;
  a.pairs = whole ? pairs : pairs + first; a.npairs = count;
  a.order = whole ? B->d_order : nullptr;
  a.fo = whole ? B->d_fo : B->d_fo + first;
  a.ptb = whole ? ptb : ptb + first;
  a.codes = B->d_codes; a.table = B->d_table; a.Kp = B->Kp; a.tb = tb; a.cig = B->d_cig;
  a.res = whole ? B->d_res : B->d_res + first;
  a.local = B->p.mode == TA_LOCAL; a.open = B->p.gap_open; a.ext = B->p.gap_extend;
  a.do_cigar = B->p.traceback;
  a.guard_cap = B->guard_cap;
  (void)hipGetLastError();
  hipLaunchKernelGGL(traceback_kernel<0>, dim3((count + TB_WALKERS - 1) / TB_WALKERS), dim3(TB_WALKERS), 0,
                     B->stream, a);
  HIPCHK(hipGetLastError());
  return TA_OK;
}

// Long pairs [lp0, lp0 + nlp) of the batch (queue items [it0, it0 + nit)).
LongArgs long_args(ta_batch *B, int it0, int nit, int lp0, int nlp) {
  LongArgs a{};
  a.lp = B->d_lp + lp0; a.nlp = nlp;
  a.items = B->d_litems + it0; a.nitems = nit;
  a.ctr = B->d_ctr + 8;
  a.table = B->d_table; a.Kp = B->Kp; a.codes = B->d_codes;
  a.ring = B->d_lring; a.colck = B->d_lring; a.wpl = B->d_wpl;
  a.pd = B->d_pairs; a.fo = B->d_fo; a.res = B->d_res; a.cig = B->d_cig;
  a.open = B->p.gap_open; a.ext = B->p.gap_extend;
  a.ckpt_on = B->p.traceback;
  a.spin_limit = B->spin_limit;
  a.err = B->d_ctr + 10;
  return a;
}

// Forward pass of queue items [it0, it0 + nit), whose pairs' bottom rows lie in
// entries [ring0, ring0 + ring_n): entries emptied and counters cleared, then
// one wave per workgroup pulling strips.  Items name pairs from 0.
int launch_long_fwd(ta_ctx *ctx, ta_batch *B, int it0, int nit, uint64_t ring0, uint64_t ring_n) {
  if (nit <= 0) return TA_OK;
  const uint64_t n16 = ring_n / 2;
  (void)hipGetLastError();
  hipLaunchKernelGGL(long_init_kernel<0>, dim3((unsigned)std::max<uint64_t>(1, std::min<uint64_t>(4096, (n16 + 255) / 256))),
                     dim3(256), 0, B->stream, (uint4 *)(B->d_lring + ring0), n16, B->d_ctr + 8);
  const LongArgs a = long_args(B, it0, nit, 0, (int)B->longs.size());
  const bool dna = B->Kp <= STRIP_NC_DNA;
  const int gaps = -a.open - a.ext, pad = a.ext - a.open;  // scores are kept plus gaps, the pad's as it is
  const bool bytes = B->alph.minS + gaps >= -128 && B->alph.maxS + gaps <= 127 && PAD_SCORE + gaps <= 127 &&
                     pad >= -128 && pad <= 127;
  constexpr int D = STRIP_NC_DNA, P = STRIP_NC;
  const int lds = dna ? (bytes ? long_fwd_lds<D, true> : long_fwd_lds<D, false>)
                      : (bytes ? long_fwd_lds<P, true> : long_fwd_lds<P, false>);
  void (*k)(LongArgs) = dna ? (bytes ? long_fwd_kernel<D, true> : long_fwd_kernel<D, false>)
                            : (bytes ? long_fwd_kernel<P, true> : long_fwd_kernel<P, false>);
  const int per_cu = std::max(1, std::min(LONG_WAVES, ctx->lds_max / lds));
  hipLaunchKernelGGL(k, dim3(std::max(1, std::min(nit, ctx->cus * per_cu))), dim3(64), lds, B->stream, a);
  HIPCHK(hipGetLastError());
  return TA_OK;
}

// Traceback of long pairs [lp0, lp0 + nlp): one workgroup per pair, with
// regions ahead as many pairs at a time as their memory holds.
int launch_long_tb(ta_ctx *ctx, ta_batch *B, int lp0, int nlp, bool ahead) {
  if (nlp <= 0 || !B->p.traceback) return TA_OK;
  const int end = lp0 + nlp;
  while (lp0 < end) {
    int n = ahead ? 0 : nlp, items = 0;
    while (lp0 + n < end && items + B->longs[lp0 + n].S <= B->lahead) items += B->longs[lp0 + n++].S;
    LongArgs a = long_args(B, B->longs[lp0].item0, items, 0, 0);
    (void)hipGetLastError();
    if (ahead) {
      a.ahead = B->d_lahead; a.cross = B->d_lcross; a.ahead0 = B->longs[lp0].item0;
      hipLaunchKernelGGL(long_cross_kernel<0>, dim3(items), dim3(256), 0, B->stream, a);
      hipLaunchKernelGGL(long_regions_kernel<0>, dim3(items), dim3(64 * LTW), LONG_TB_LDS, B->stream, a);
    }
    a.lp = B->d_lp + lp0; a.nlp = n;
    hipLaunchKernelGGL(long_tb_kernel<0>, dim3(std::max(1, std::min(n, B->long_wgs))), dim3(64 * LTW), LONG_TB_LDS,
                       B->stream, a);
    HIPCHK(hipGetLastError());
    lp0 += n;
  }
  return TA_OK;
}

StripsArgs strips_args(ta_batch *B) {
  StripsArgs a{};
  a.sp = B->d_spairs; a.items = B->d_sitems;
  a.nitems = (int)B->sitems.size(); a.npairs = (int)B->spairs.size();
  a.ctr = B->d_ctr + 11;
  a.table = B->d_table; a.Kp = B->Kp; a.codes = B->d_codes;
  a.ring = B->d_sring; a.planes = B->d_splanes; a.best = B->d_sbest; a.score = B->d_sscore;
  a.open = B->p.gap_open; a.ext = B->p.gap_extend;
  a.sat_limit = 32767 - 2 * B->alph.maxS;
  a.spin_limit = B->spin_limit;
  a.err = B->d_ctr + 10;
  a.tb = tb_args(B);
  a.bcode_bytes = B->strips_bcode;
  return a;
}

int launch_strips(ta_ctx *ctx, ta_batch *B) {
  if (!B->strips) return TA_OK;
  const StripsArgs a = strips_args(B);
  const uint64_t n16 = B->sring_n / 2;
  (void)hipGetLastError();
  hipLaunchKernelGGL(strips_init_kernel, dim3((unsigned)std::max<uint64_t>(1, std::min<uint64_t>(4096, (n16 + 255) / 256))),
                     dim3(256), 0, B->stream, (uint4 *)B->d_sring, n16, B->d_sbest, a.npairs);
  const int lds = strips_lds(a.bcode_bytes);
  const bool local = B->p.mode == TA_LOCAL;
  void (*k)(StripsArgs) = local ? strips_kernel<true> : strips_kernel<false>;
  // one wave per workgroup; those that do not fit at once take items as others end
  const int per_cu = std::max(1, std::min(16, ctx->lds_max / lds));
  hipLaunchKernelGGL(k, dim3(std::min(a.nitems, ctx->cus * per_cu)), dim3(64), lds, B->stream, a);
  HIPCHK(hipGetLastError());
  return TA_OK;
}

int launch_strips_walk(ta_batch *B) {
  if (!B->strips) return TA_OK;
  const StripsArgs a = strips_args(B);
  const bool local = B->p.mode == TA_LOCAL;
  void (*k)(StripsArgs) = local ? strips_walk_kernel<true> : strips_walk_kernel<false>;
  (void)hipGetLastError();
  hipLaunchKernelGGL(k, dim3(a.npairs), dim3(64), 0, B->stream, a);
  HIPCHK(hipGetLastError());
  return TA_OK;
}

// Pairs whose int16 pass saturated go through the int32 kernel.
int rerun_saturated(ta_ctx *ctx, ta_batch *B) {
  std::vector<FillOut> fo(B->n);
  HIPCHK(hipMemcpyAsync(fo.data(), B->d_fo, sizeof(FillOut) * B->n, hipMemcpyDeviceToHost, B->stream));
  HIPCHK(hipStreamSynchronize(B->stream));
  std::vector<int> bad;
  for (int k = 0; k < B->n; ++k)
    if (fo[k].flags & TA_F_RERUN) bad.push_back(k);
  free_rerun(B);
  if (bad.empty()) return TA_OK;
  Plan pl;
  pl.ptb.resize(B->n);
  std::vector<Task> wave, group;
  std::vector<Unit> u;
  for (int k : bad) {
    if (pick_gg(B->hp[k].la, B->hp[k].lb, 0.0, bad.size() <= (size_t)ctx->cus * 4) == GWAVE) {
      add_task(pl, wave, 1, GWAVE, B->trace, B->hp, k, k, true);
      wave.back().flags_or = TA_F_RERUN;
    } else {
      u.push_back(Unit{k, k, true, B->hp[k].la, B->hp[k].lb});
    }
  }
  add_units(pl, group, u, B->p.mode == TA_LOCAL, B->trace, B->hp);
  for (Task &t : group) t.flags_or = TA_F_RERUN;
  std::vector<Task> all(wave);
  all.insert(all.end(), group.begin(), group.end());
  hipStream_t st = B->stream;
  int rc = TA_OK;
  rc = rc ? rc : dalloc(&B->d_ring_r, pl.ring_elems);
  rc = rc ? rc : dalloc(&B->d_tb_r, pl.tb_bytes);
  if (rc) return rc;
  // Rerun pairs read their planes from the rerun arena: their records point
  // there by offsetting against the main arena base.  Only theirs are written
  // (10 of 65,536 pairs: rerun phase 6.87 ms with the table read back, patched
  // and sent again, 6.18 so).
  std::vector<PtbPatch> patch;
  for (int k : bad) {
    patch.push_back(PtbPatch{pl.ptb[k], k, 0});
    patch.back().d.tb_off += (uint64_t)(B->d_tb_r - B->d_tb);
  }
  rc = rc ? rc : upload(&B->d_patch_r, patch, st);
  rc = rc ? rc : upload(&B->d_tasks_r, all, st);
  // (waits: the uploads' sources may go)
  rc = rc ? rc : expand_codes(pl.cjobs, pl.rows_n, pl.cols_n, B->d_pairs, B->d_codes, B->Kp, &B->d_rowcodes_r,
                              &B->d_colcodes_r, st);
  if (rc) return rc;
  B->n_rerun = (int)bad.size();
  (void)hipGetLastError();
  hipLaunchKernelGGL(patch_ptb_kernel, dim3((unsigned)std::min<size_t>(1024, (patch.size() + 255) / 256)), dim3(256), 0,
                     st, B->d_patch_r, (int)patch.size(), B->d_ptb);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemsetAsync(B->d_ctr + 4, 0, 2 * sizeof(int32_t), st));
  Task *const tk[3] = {B->d_tasks_r, B->d_tasks_r + wave.size(), nullptr};
  const int nt[3] = {(int)wave.size(), (int)group.size() / NGW, 0};
  return launch_fill<1>(ctx, B, tk, nt, B->d_rowcodes_r, B->d_colcodes_r, B->d_ring_r, B->d_tb_r, B->d_ctr + 4, 0);
}

}  // namespace

namespace {

int launch_init(ta_batch *B) {
  (void)hipGetLastError();
  hipLaunchKernelGGL(init_kernel, dim3(std::max(1, std::min(1024, (B->n + 255) / 256))), dim3(256), 0, B->stream,
                     B->d_ctr, 16, B->d_fo, B->d_fo_init, B->n);
  HIPCHK(hipGetLastError());
  return TA_OK;
}

// `timed`: the tracebacks among them are timed by themselves (not while a
// graph is captured).
int launch_fills(ta_ctx *ctx, ta_batch *B, bool timed) {
  const Plan &pl = B->plan;
  const int n2[3] = {(int)pl.list2[0].spans.size(), (int)pl.list2[1].spans.size(), (int)pl.list2[2].spans.size()};
  const int n1[3] = {(int)pl.list1[0].spans.size(), (int)pl.list1[1].spans.size(), 0};
  int rc = launch_fill<2>(ctx, B, B->d_tasks2, n2, B->d_rowcodes, B->d_colcodes, B->d_ring, B->d_tb, B->d_ctr, 0,
                          B->walk);
  if (!rc) rc = launch_fill<1>(ctx, B, B->d_tasks1, n1, B->d_rowcodes, B->d_colcodes, B->d_ring, B->d_tb,
                               B->d_ctr + 2, 0, B->walk);
  if (!rc) rc = launch_strips(ctx, B);
  // Long pairs, group by group; the last group's traceback is launch_tracebacks'.
  for (size_t g = 0; !rc && g < B->lgroups.size(); ++g) {
    const LongGroup &L = B->lgroups[g];
    rc = launch_long_fwd(ctx, B, L.it0, L.nitems, 0, L.ring_n);
    if (rc || g + 1 == B->lgroups.size() || B->gev.empty()) continue;
    if (timed) HIPCHK(hipEventRecord(B->gev[2 * g], B->stream));
    rc = launch_long_tb(ctx, B, L.lp0, L.npairs, B->lahead > 0);
    if (timed) HIPCHK(hipEventRecord(B->gev[2 * g + 1], B->stream));
  }
  return rc;
}

int launch_tracebacks(ta_ctx *ctx, ta_batch *B) {
  int rc = TA_OK;
  if (B->strips) rc = launch_strips_walk(B);
  if (!rc && !B->walk && !B->strips) {
    rc = launch_traceback(ctx, B, B->d_pairs, B->d_ptb, B->d_tb, 0, B->n);
  } else if (!rc && B->n_rest) {  // every pair with a fill task is walked by now
    TbArgs a = tb_args(B);
    a.npairs = B->n_rest;
    a.order = B->d_order_rest;
    (void)hipGetLastError();
    hipLaunchKernelGGL(traceback_kernel<0>, dim3((B->n_rest + TB_WALKERS - 1) / TB_WALKERS), dim3(TB_WALKERS), 0,
                       B->stream, a);
    HIPCHK(hipGetLastError());
  }
  if (!rc && !B->lgroups.empty()) rc = launch_long_tb(ctx, B, B->lgroups.back().lp0, B->lgroups.back().npairs, B->lahead > 0);
  return rc;
}

// A captured run: init, fills, tracebacks -- kernels only.  Batches that may
// need the int32 rerun are not captured (the rerun is a host decision).
int run_graph(ta_ctx *ctx, ta_batch *B) {
  hipStream_t st = B->stream;
  if (!B->gexec) {
    HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    int rc = launch_init(B);
    if (!rc) rc = launch_fills(ctx, B, false);
    if (!rc) rc = launch_tracebacks(ctx, B);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(st, &g);
    if (rc || e != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return rc ? rc : TA_E_DEVICE;
    }
    B->graph = g;
    HIPCHK(hipGraphInstantiate(&B->gexec, g, nullptr, nullptr, 0));
  }
  HIPCHK(hipEventRecord(B->ev[0], st));
  HIPCHK(hipGraphLaunch(B->gexec, st));
  HIPCHK(hipEventRecord(B->ev[3], st));
  B->phases_timed = false;
  return TA_OK;
}

}  // namespace

int ta_batch_run(ta_ctx *ctx, ta_batch *B) {
  if (!ctx || !B) return TA_E_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  if (B->graph_on && !B->may_saturate) return run_graph(ctx, B);
  hipStream_t st = B->stream;
  int rc = launch_init(B);
  if (rc) return rc;
  HIPCHK(hipEventRecord(B->ev[0], st));
  rc = launch_fills(ctx, B, true);
  if (rc) return rc;
  HIPCHK(hipEventRecord(B->ev[1], st));
  if (B->may_saturate) {
    rc = rerun_saturated(ctx, B);
    if (rc) return rc;
  } else if (B->n_rerun) {
    free_rerun(B);
  }
  HIPCHK(hipEventRecord(B->ev[2], st));
  rc = launch_tracebacks(ctx, B);
  if (rc) return rc;
  HIPCHK(hipEventRecord(B->ev[3], st));
  B->phases_timed = B->gev_timed = true;
  return TA_OK;
}

int ta_batch_graph(ta_batch *B, int32_t on) {
  if (!B) return TA_E_INVALID;
  B->graph_on = on != 0;
  return TA_OK;
}

int ta_batch_wait(ta_ctx *ctx, ta_batch *B) {
  if (!ctx || !B) return TA_E_INVALID;
  HIPCHK(hipStreamSynchronize(B->stream));
  float t = 0;
  B->ms[0] = B->ms[1] = B->ms[2] = -1.0;  // a captured run is timed as a whole only
  if (B->phases_timed) {
    if (hipEventElapsedTime(&t, B->ev[0], B->ev[1]) == hipSuccess) B->ms[0] = t;
    if (hipEventElapsedTime(&t, B->ev[1], B->ev[2]) == hipSuccess) B->ms[1] = t;
    if (hipEventElapsedTime(&t, B->ev[2], B->ev[3]) == hipSuccess) B->ms[2] = t;
    // long groups but the last are walked back among the fills
    for (size_t g = 0; B->gev_timed && g + 1 < B->gev.size(); g += 2) {
      if (hipEventElapsedTime(&t, B->gev[g], B->gev[g + 1]) != hipSuccess) continue;
      B->ms[0] -= t;
      B->ms[2] += t;
    }
  }
  if (hipEventElapsedTime(&t, B->ev[0], B->ev[3]) == hipSuccess) B->ms[3] = t;
  if (!B->longs.empty() || B->ncoop2 || B->ncoop1 || B->strips) {
    int32_t err = 0;
    HIPCHK(hipMemcpyAsync(&err, B->d_ctr + 10, sizeof(err), hipMemcpyDeviceToHost, B->stream));
    HIPCHK(hipStreamSynchronize(B->stream));
    if (err) {
      fprintf(stderr, "tweakalign: a wait on another wave's progress gave up (code %d)\n", err);
      return TA_E_DEVICE;
    }
  }
  return TA_OK;
}

int ta_batch_timings(ta_batch *B, double *ms, int32_t cap) {
  if (!B || !ms) return TA_E_INVALID;
  int k = 0;
  for (; k < cap && k < 4; ++k) ms[k] = B->ms[k];
  return k;
}

// Binary runs ((len << 2) | op, op 0 M / 1 D / 2 I) -> CIGAR text.
int64_t cigar_text(const uint32_t *runs, int n, char *out) {
  static const char ops[4] = {'M', 'D', 'I', '?'};
  int64_t pos = 0;
  char tmp[12];
  for (int k = 0; k < n; ++k) {
    uint32_t len = runs[k] >> 2;
    int d = 0;
    do { tmp[d++] = (char)('0' + len % 10); len /= 10; } while (len);
    if (out)
      while (d) out[pos++] = tmp[--d];
    else
      pos += d;
    if (out) out[pos] = ops[runs[k] & 3];
    ++pos;
  }
  return pos;
}
namespace {
int64_t format_runs(const uint32_t *runs, int n, char *out) { return cigar_text(runs, n, out); }
}  // namespace

namespace {

// Gathers every pair's CIGAR runs (written backwards at the end of its
// region) into one dense array: one wave per pair, dword copies.
__global__ void gather_runs_kernel(const uint32_t *cig, const ResultDev *res, const int64_t *dst_off, uint32_t *dst,
                                   int n) {
  const int p = blockIdx.x;
  if (p >= n) return;
  const int nr = res[p].cigar_len / 4;
  if (nr <= 0) return;
  const uint32_t *src = cig + res[p].cigar_off / 4;
  uint32_t *d = dst + dst_off[p] / 4;
  for (int k = threadIdx.x; k < nr; k += blockDim.x) d[k] = src[k];
}

// Results and CIGAR runs of a finished batch on the host, in pinned staging
// blocks: `res` per pair, pair k's runs at runs[off[k] / 4 ...] (cigar_len
// bytes).  Of large batches only the runs cross PCIe (gathered, dense), not
// the per-pair worst-case regions.
struct Fetched {
  StageHold resb, runsb;
  const ResultDev *res = nullptr;
  const uint32_t *runs = nullptr;
  std::vector<int64_t> off;
};

int fetch_results(ta_batch *B, Fetched &F) {
  std::vector<int64_t> &off = F.off;
  hipStream_t st = B->stream;
  if (B->n) {
    F.resb.s = stage_take(sizeof(ResultDev) * B->n);
    if (!F.resb.s.p) return TA_E_NOMEM;
    F.resb.stream = st;
    F.resb.queued = true;
    HIPCHK(hipMemcpyAsync(F.resb.s.p, B->d_res, sizeof(ResultDev) * B->n, hipMemcpyDeviceToHost, st));
    F.res = (const ResultDev *)F.resb.s.p;
  }
  // Where the pairs' regions take 1 MB at most they come back whole, in one
  // go with the results: 20 us of link at most, against an upload, a kernel,
  // a copy and a second wait (35 us) for the runs alone.
  const bool small = B->p.traceback && B->n && B->cig_bytes && B->cig_bytes <= (1 << 20);
  if (small) {
    F.runsb.s = stage_take(B->cig_bytes);
    if (!F.runsb.s.p) return TA_E_NOMEM;
    F.runsb.stream = st;
    F.runsb.queued = true;
    HIPCHK(hipMemcpyAsync(F.runsb.s.p, B->d_cig, B->cig_bytes, hipMemcpyDeviceToHost, st));
  }
  HIPCHK(hipStreamSynchronize(st));
  if (!B->p.traceback) return TA_OK;
  const ResultDev *res = F.res;
  off.assign(B->n, 0);
  if (small) {
    for (int32_t k = 0; k < B->n; ++k) off[k] = res[k].cigar_off;
    F.runs = (const uint32_t *)F.runsb.s.p;
    return TA_OK;
  }
  int64_t total = 0;
  for (int32_t k = 0; k < B->n; ++k) {
    off[k] = total;
    if (res[k].cigar_len > 0) total += res[k].cigar_len;
  }
  if (!total) return TA_OK;
  F.runsb.s = stage_take((size_t)total);
  if (!F.runsb.s.p) return TA_E_NOMEM;
  F.runsb.stream = st;
  F.runsb.queued = true;
  F.runs = (const uint32_t *)F.runsb.s.p;
  int64_t *d_off = nullptr;
  uint32_t *d_runs = nullptr;
  int rc = upload(&d_off, off, st);
  rc = rc ? rc : dalloc(&d_runs, (size_t)(total / 4));
  if (!rc) {
    (void)hipGetLastError();
    hipLaunchKernelGGL(gather_runs_kernel, dim3(B->n), dim3(64), 0, st, (const uint32_t *)B->d_cig, B->d_res,
                       d_off, d_runs, B->n);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(F.runsb.s.p, d_runs, (size_t)total, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      rc = TA_E_DEVICE;
  }
  (void)hipStreamSynchronize(st);  // nothing in flight reads the buffers once they return to the cache
  dfree(d_off);
  dfree(d_runs);
  return rc;
}

void fill_result(ta_result &o, const ResultDev &r) {
  o.score = r.score; o.a_begin = r.a_begin; o.a_end = r.a_end; o.b_begin = r.b_begin; o.b_end = r.b_end;
  o.flags = r.flags;
  o.cigar_off = 0;
  o.cigar_len = 0;
}

}  // namespace

int ta_batch_results(ta_ctx *ctx, ta_batch *B, ta_result *out, char *cigar_buf, int64_t cap, int64_t *used) {
  if (!ctx || !B || (B->n && !out)) return TA_E_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  PhaseTrace tr("results");
  Fetched F;
  int rc = fetch_results(B, F);
  tr.mark("fetch");
  if (rc) return rc;
  const ResultDev *res = F.res;
  const uint32_t *runs = F.runs;
  const std::vector<int64_t> &off = F.off;
  // CIGAR text lengths, their offsets, then the text, the first and last
  // passes on the host threads.
  const bool tb = B->p.traceback != 0;
  parallel_for((size_t)B->n, [&](size_t k) {
    const ResultDev &r = res[k];
    fill_result(out[k], r);
    if (tb && r.cigar_len > 0) out[k].cigar_len = (int32_t)format_runs(runs + off[k] / 4, r.cigar_len / 4, nullptr);
  });
  int64_t pos = 0;
  for (int32_t k = 0; k < B->n; ++k) {
    out[k].cigar_off = pos;
    pos += out[k].cigar_len;
  }
  if (used) *used = pos;
  if (pos > 0 && (!cigar_buf || pos > cap)) return TA_E_SPACE;
  if (pos > 0) parallel_for((size_t)B->n, [&](size_t k) {
    if (out[k].cigar_len > 0)
      format_runs(runs + off[k] / 4, res[k].cigar_len / 4, cigar_buf + out[k].cigar_off);
  });
  tr.mark("format");
  for (int32_t k = 0; k < B->n; ++k)
    if (out[k].flags & TA_F_WALK_FAILED) return TA_E_WALK;
  return rc;
}

int batch_results_text(ta_ctx *ctx, ta_batch *B, std::vector<ta_result> &out, std::string &text) {
  if (!ctx || !B) return TA_E_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  PhaseTrace tr("results");
  Fetched F;
  const int rc = fetch_results(B, F);
  tr.mark("fetch");
  if (rc) return rc;
  const ResultDev *res = F.res;
  const uint32_t *runs = F.runs;
  const std::vector<int64_t> &off = F.off;
  // lengths, offsets, then the text, as ta_batch_results
  out.resize(B->n);
  const bool tb = B->p.traceback != 0;
  parallel_for((size_t)B->n, [&](size_t k) {
    const ResultDev &r = res[k];
    fill_result(out[k], r);
    if (tb && r.cigar_len > 0) out[k].cigar_len = (int32_t)format_runs(runs + off[k] / 4, r.cigar_len / 4, nullptr);
  });
  int64_t pos = 0;
  for (int32_t k = 0; k < B->n; ++k) {
    out[k].cigar_off = pos;
    pos += out[k].cigar_len;
  }
  text.assign((size_t)pos, '\0');
  parallel_for((size_t)B->n, [&](size_t k) {
    if (out[k].cigar_len > 0) format_runs(runs + off[k] / 4, res[k].cigar_len / 4, &text[out[k].cigar_off]);
  });
  tr.mark("format");
  return TA_OK;
}

int ta_align_batch(ta_ctx *ctx, const ta_params *p, const ta_pair *pairs, int32_t n, ta_result *out,
                   char *cigar_buf, int64_t cap, int64_t *used) {
  ta_batch *B = nullptr;
  int rc = ta_batch_create(ctx, p, pairs, n, &B);
  if (rc) return rc;
  rc = ta_batch_run(ctx, B);
  if (!rc) rc = ta_batch_wait(ctx, B);
  if (!rc) rc = ta_batch_results(ctx, B, out, cigar_buf, cap, used);
  ta_batch_destroy(B);
  return rc;
}

// ---------------------------------------------------------------------------
// Resident sequences: codes encoded on the host once, appended to the
// context's device arena (grown by copying into a larger one; batches and
// served requests that still read the old arena hold it until they are
// freed), aligned by handle.  Codes added since the last upload wait in host
// memory and go up in one copy (seq_flush) when a call resolves handles, or
// before an add once 64 MB are pending.

// Uploads the pending codes (the caller holds seq_mu).
static int seq_flush(ta_ctx *ctx) {
  if (ctx->seq_pending.empty()) return TA_OK;
  if (hipMemcpy(ctx->seq_arena.get() + ctx->seq_flushed, ctx->seq_pending.data(), ctx->seq_pending.size(),
                hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipGetLastError();
    return TA_E_DEVICE;
  }
  ctx->seq_flushed = ctx->seq_used;  // the 32 zero bytes after it are on the device too
  ctx->seq_pending.clear();
  return TA_OK;
}

int ta_seq_add(ta_ctx *ctx, int32_t alphabet, const char *letters, int32_t len, ta_seq *out) {
  if (!ctx || !out || len < 0 || len > 1000000 || (len > 0 && !letters)) return TA_E_INVALID;
  if (alphabet != TA_PROTEIN && alphabet != TA_DNA) return TA_E_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  const Alphabet A = make_alphabet(alphabet, 1, -1);
  // the codes, code 0 up to the next 16-byte start, then the walkers' slack
  const size_t span = ((size_t)len + 15) & ~(size_t)15;
  int32_t cnt[32] = {0};
  for (int32_t i = 0; i < len; ++i) {
    const int c = A.map[(unsigned char)letters[i]];
    if (c < 0) return TA_E_ALPHABET;
    ++cnt[c];
  }
  std::lock_guard<std::mutex> g(ctx->seq_mu);
  if (ctx->seq_pending.size() >= ((size_t)64 << 20) && seq_flush(ctx)) return TA_E_DEVICE;
  const size_t off = ctx->seq_used, need = off + span + 32;
  if (need > ctx->seq_cap) {
    // a larger arena with the uploaded contents (the pending ones follow at
    // the next flush); the old one is freed once no batch holds it
    const size_t cap = std::max(need, std::max(2 * ctx->seq_cap, (size_t)16 << 20));
    uint8_t *d = nullptr;
    if (hipMalloc((void **)&d, cap) != hipSuccess) {
      (void)hipGetLastError();
      return TA_E_NOMEM;
    }
    std::shared_ptr<uint8_t> arena(d, [](uint8_t *q) { (void)hipFree(q); });
    if (ctx->seq_flushed &&
        hipMemcpy(d, ctx->seq_arena.get(), ctx->seq_flushed, hipMemcpyDeviceToDevice) != hipSuccess) {
      (void)hipGetLastError();
      return TA_E_DEVICE;
    }
    ctx->seq_arena = std::move(arena);
    ctx->seq_cap = cap;
  }
  // pending bytes [seq_flushed, off + span + 32): this sequence's codes
  // replace the previous one's trailing slack
  std::vector<uint8_t> &pend = ctx->seq_pending;
  const size_t at = off - ctx->seq_flushed;
  pend.resize(at + span + 32);
  std::fill(pend.begin() + at, pend.end(), (uint8_t)0);
  for (int32_t i = 0; i < len; ++i) pend[at + i] = (uint8_t)A.map[(unsigned char)letters[i]];
  ctx->seq_used = off + span;
  ctx->seqs.push_back(ta_ctx::SeqRec{off, len, alphabet});
  ctx->seq_counts.insert(ctx->seq_counts.end(), cnt, cnt + 32);
  *out = (ta_seq)(ctx->seqs.size() - 1);
  return TA_OK;
}

int ta_seq_reset(ta_ctx *ctx) {
  if (!ctx) return TA_E_INVALID;
  std::lock_guard<std::mutex> g(ctx->seq_mu);
  ctx->seq_arena.reset();  // freed now, or when the last batch that holds it is
  ctx->seq_cap = ctx->seq_used = ctx->seq_flushed = 0;
  ctx->seq_pending.clear();
  ctx->seq_pending.shrink_to_fit();
  ctx->seqs.clear();
  ctx->seq_counts.clear();
  return TA_OK;
}

int resident_resolve(ta_ctx *ctx, const ta_params *p, const ta_seq_pair *pairs, int32_t n, ResidentBatch &out) {
  if (!ctx || !p || n < 0 || (n > 0 && !pairs) || params_check(p)) return TA_E_INVALID;
  const Alphabet A = make_alphabet(p->alphabet, p->match, p->mismatch);
  int best[32] = {0};  // best score of each residue against any letter (0 if none is positive)
  for (int r = 0; r < A.K; ++r)
    for (int c = 0; c < A.K; ++c) best[r] = std::max<int>(best[r], A.S[r * A.K + c]);
  std::lock_guard<std::mutex> g(ctx->seq_mu);
  const int64_t ns = (int64_t)ctx->seqs.size();
  auto bound = [&](ta_seq h) {
    const int32_t *cnt = ctx->seq_counts.data() + 32 * (size_t)h;
    int64_t sum = 0;
    for (int r = 0; r < A.K; ++r) sum += (int64_t)cnt[r] * best[r];
    return sum;
  };
  out = ResidentBatch();
  out.a_off.resize(n); out.b_off.resize(n);
  out.la.resize(n); out.lb.resize(n);
  out.a_bound.resize(n); out.b_bound.resize(n);
  for (int32_t k = 0; k < n; ++k) {
    const ta_seq a = pairs[k].a, b = pairs[k].b;
    if (a < 0 || b < 0 || a >= ns || b >= ns || ctx->seqs[a].alphabet != p->alphabet ||
        ctx->seqs[b].alphabet != p->alphabet)
      return TA_E_INVALID;
    out.a_off[k] = ctx->seqs[a].off; out.b_off[k] = ctx->seqs[b].off;
    out.la[k] = ctx->seqs[a].len; out.lb[k] = ctx->seqs[b].len;
    out.a_bound[k] = bound(a); out.b_bound[k] = bound(b);
  }
  if (n > 0 && !ctx->seq_arena) return TA_E_INVALID;
  if (n > 0 && seq_flush(ctx)) return TA_E_DEVICE;
  out.arena = ctx->seq_arena;
  return TA_OK;
}

int ta_align_resident(ta_ctx *ctx, const ta_params *p, const ta_seq_pair *pairs, int32_t n, ta_result *out,
                      char *cigar_buf, int64_t cap, int64_t *used) {
  if (!ctx || n < 0 || (n > 0 && (!pairs || !out))) return TA_E_INVALID;
  ResidentBatch rb;
  int rc = resident_resolve(ctx, p, pairs, n, rb);
  if (rc) return rc;
  ta_batch *B = nullptr;
  rc = batch_create_on(ctx, p, nullptr, n, ctx->stream, &B, nullptr, &rb);
  if (rc) return rc;
  rc = ta_batch_run(ctx, B);
  if (!rc) rc = ta_batch_wait(ctx, B);
  if (!rc) rc = ta_batch_results(ctx, B, out, cigar_buf, cap, used);
  ta_batch_destroy(B);
  return rc;
}

// ---------------------------------------------------------------------------
// Plain form: one fill launch (one group, one task) and one traceback launch
// per pair, serialised on the stream -- the baseline batching is measured
// against.
int ta_batch_run_plain(ta_ctx *ctx, ta_batch *B, int32_t first, int32_t count) {
  if (!ctx || !B || first < 0 || count < 0 || first + count > B->n) return TA_E_INVALID;
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = B->stream;
  if (!B->plain_ready) {
    Plan pl;
    pl.ptb.assign(B->n, PairTB{0, 0, 0, 0, 0, 0, 0});
    uint64_t max_tb = 0, max_ring = 0;
    // NGW entries per pair: the task, then fillers for the other groups of
    // its wave (a group task runs in a wave of NGW groups; fillers write
    // nothing).
    std::vector<Task> tasks, rtasks;
    std::vector<PairTB> ptb_r(B->n, PairTB{0, 0, 0, 0, 0, 0, 0});
    std::vector<int32_t> rerun_of(B->n, -1);
    auto fill_unit = [&](std::vector<Task> &v) {
      Task f = v.back();
      f.single = 2;
      for (int q = 1; q < NGW; ++q) v.push_back(f);
    };
    for (int k = 0; k < B->n; ++k) {
      const HostPair &h = B->hp[k];
      const int P = h.path == 1 ? 1 : 2;
      const uint64_t tb0 = pl.tb_bytes, r0 = pl.ring_elems;
      if (h.path == 0 || h.path == 3) {
        if (h.path == 3) pl.ptb[k].P = 3;  // the long-pair kernels write its result
        tasks.push_back(Task{});
        fill_unit(tasks);
        continue;
      }
      const int GG = pick_gg(h.la, h.lb, 0.0, true);
      // Every plain launch reuses the same scratch: rebase to 0.
      auto rebase = [&](std::vector<Task> &v) {
        Task &T = v.back();
        max_tb = std::max(max_tb, pl.tb_bytes - tb0);
        max_ring = std::max(max_ring, pl.ring_elems - r0);
        T.tb_off = 0; T.ring_off = 0;
        pl.ptb[k].tb_off = 0;
        pl.tb_bytes = tb0; pl.ring_elems = r0;
        fill_unit(v);
      };
      add_task(pl, tasks, P, GG, B->trace, B->hp, k, k, true);
      rebase(tasks);
      if (h.maysat) {  // the int32 task a saturated int16 fill reruns as
        const PairTB p16 = pl.ptb[k];
        rerun_of[k] = (int32_t)rtasks.size();
        add_task(pl, rtasks, 1, GG, B->trace, B->hp, k, k, true);
        rtasks.back().flags_or = TA_F_RERUN;
        rebase(rtasks);
        ptb_r[k] = pl.ptb[k];
        pl.ptb[k] = p16;
      }
    }
    int rc = TA_OK;
    rc = rc ? rc : upload(&B->d_plain_tasks, tasks, st);
    rc = rc ? rc : upload(&B->d_plain_rtasks, rtasks, st);
    rc = rc ? rc : upload(&B->d_pptb_r, ptb_r, st);
    rc = rc ? rc : expand_codes(pl.cjobs, pl.rows_n, pl.cols_n, B->d_pairs, B->d_codes, B->Kp, &B->d_prow,
                                &B->d_pcol, st);
    rc = rc ? rc : upload(&B->d_pptb, pl.ptb, st);
    rc = rc ? rc : dalloc(&B->d_pring, max_ring);
    rc = rc ? rc : dalloc(&B->d_ptbuf, max_tb);
    if (rc) return rc;
    B->plain_tasks = tasks;
    B->plain_rerun = rerun_of;
    B->plain_ready = true;
  }
  B->gev_timed = false;
  HIPCHK(hipEventRecord(B->ev[0], st));
  // the counters and the error word (d_ctr[10]) start at 0, as init_kernel
  // leaves them for a batch run
  HIPCHK(hipMemsetAsync(B->d_ctr, 0, 16 * sizeof(int32_t), st));
  if (B->n > 0)
    HIPCHK(hipMemcpyAsync(B->d_fo, B->d_fo_init, sizeof(FillOut) * B->n, hipMemcpyDeviceToDevice, st));
  std::vector<int> lp_of(B->n, -1);
  for (size_t q = 0; q < B->longs.size(); ++q) lp_of[B->longs[q].pid] = (int)q;
  for (int k = first; k < first + count; ++k) {
    const HostPair &h = B->hp[k];
    if (h.path == 3) {
      const int q = lp_of[k];
      const LongPair &L = B->longs[q];
      int rc = launch_long_fwd(ctx, B, L.item0, L.S, L.ring, (uint64_t)(L.S - 1) * (L.T + 8));
      if (!rc) rc = launch_traceback(ctx, B, B->d_pairs, B->d_pptb, B->d_ptbuf, k, 1);
      if (!rc) rc = launch_long_tb(ctx, B, q, 1, false);
      if (rc) return rc;
      continue;
    }
    const PairTB *ptb = B->d_pptb;
    if (h.path) {
      HIPCHK(hipMemsetAsync(B->d_ctr + 6, 0, 2 * sizeof(int32_t), st));
      const bool wave = B->plain_tasks[NGW * k].S && pick_gg(h.la, h.lb, 0.0, true) == GWAVE;
      Task *const tk[3] = {B->d_plain_tasks + NGW * k, B->d_plain_tasks + NGW * k, nullptr};
      const int nt[3] = {wave ? 1 : 0, wave ? 0 : 1, 0};
      int rc = h.path == 1 ? launch_fill<1>(ctx, B, tk, nt, B->d_prow, B->d_pcol, B->d_pring, B->d_ptbuf, B->d_ctr + 6, 1)
                           : launch_fill<2>(ctx, B, tk, nt, B->d_prow, B->d_pcol, B->d_pring, B->d_ptbuf, B->d_ctr + 6, 1);
      if (rc) return rc;
      if (B->plain_rerun[k] >= 0) {
        // The int16 fill may have saturated: as the batched form, rerun the
        // pair in int32 when it flagged so (a host round trip per such pair).
        FillOut fo{};
        HIPCHK(hipMemcpyAsync(&fo, B->d_fo + k, sizeof(FillOut), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        if (fo.flags & TA_F_RERUN) {
          HIPCHK(hipMemsetAsync(B->d_ctr + 6, 0, 2 * sizeof(int32_t), st));
          Task *const rt[3] = {B->d_plain_rtasks + B->plain_rerun[k], B->d_plain_rtasks + B->plain_rerun[k], nullptr};
          rc = launch_fill<1>(ctx, B, rt, nt, B->d_prow, B->d_pcol, B->d_pring, B->d_ptbuf, B->d_ctr + 6, 1);
          if (rc) return rc;
          ptb = B->d_pptb_r;
        }
      }
    }
    int rc = launch_traceback(ctx, B, B->d_pairs, ptb, B->d_ptbuf, k, 1);
    if (rc) return rc;
  }
  HIPCHK(hipEventRecord(B->ev[1], st));
  HIPCHK(hipEventRecord(B->ev[2], st));
  HIPCHK(hipEventRecord(B->ev[3], st));
  return TA_OK;
}

// ---------------------------------------------------------------------------
// Autotuner: candidate launch shapes timed on the caller's pairs, the fastest
// kept per kind of batch on the context.
int ta_tune_bucket(const ta_pair *pairs, int32_t n) {
  if (!pairs || n <= 0) return 0;
  // The median (element n / 2 in sorted order) is below a limit exactly when
  // more than n / 2 lengths are: counts against the three limits, no sort.
  int32_t c[3] = {0, 0, 0};
  for (int32_t k = 0; k < n; ++k) {
    const int32_t v = std::max(pairs[k].la, pairs[k].lb);
    c[0] += v < 256;
    c[1] += v < 1024;
    c[2] += v < 4096;
  }
  const int32_t h = n / 2;
  return c[0] > h ? 0 : (c[1] > h ? 1 : (c[2] > h ? 2 : 3));
}

int ta_tune_set(ta_ctx *ctx, const ta_params *p, int32_t bucket, const ta_tuning *t) {
  if (!ctx || !p || !t || bucket < 0 || bucket > 3 || t->waves_per_cu < 0 || t->waves_per_cu > 32) return TA_E_INVALID;
  if (t->lanes != TA_LANES_AUTO && t->lanes != TA_LANES_I16 && t->lanes != TA_LANES_I32) return TA_E_INVALID;
  std::lock_guard<std::mutex> g(ctx->tune_mu);
  ctx->tune[tune_key(p, bucket)] = *t;
  return TA_OK;
}

int ta_tune_get(ta_ctx *ctx, const ta_params *p, int32_t bucket, ta_tuning *t) {
  if (!ctx || !p || !t || bucket < 0 || bucket > 3) return TA_E_INVALID;
  std::lock_guard<std::mutex> g(ctx->tune_mu);
  auto it = ctx->tune.find(tune_key(p, bucket));
  if (it == ctx->tune.end()) return TA_E_INVALID;
  *t = it->second;
  return TA_OK;
}

int ta_autotune(ta_ctx *ctx, const ta_params *p, const ta_pair *pairs, int32_t n, int32_t repeats, ta_tuning *best,
                double *best_ms) {
  if (!ctx || !p || !pairs || n <= 0) return TA_E_INVALID;
  repeats = std::max(1, std::min(repeats, 50));
  std::vector<int32_t> lanes_c;
  if (p->lanes == TA_LANES_AUTO) lanes_c = {TA_LANES_I16, TA_LANES_I32};
  else lanes_c = {p->lanes};
  const int Kp = make_alphabet(p->alphabet, p->match, p->mismatch).K + 1;
  ta_tuning win{0, TA_LANES_AUTO, 0};
  double win_ms = 1e300;
  for (int32_t lanes : lanes_c) {
    const int P = lanes == TA_LANES_I32 ? 1 : 2;
    int last_eff = -1;
    bool walk_done[2] = {false, false};  // walking fills ignore the wave count: measure one
    for (int waves : {4, 8, 12}) {
      const int eff = fill_waves_per_cu(P, Kp, P == 2 && !(p->mode == TA_LOCAL || p->traceback), waves);
      if (eff == last_eff) continue;
      last_eff = eff;
      for (int wt = 0; wt < 2; ++wt) {
        const ta_tuning cand{waves, lanes, wt};
        ta_batch *B = nullptr;
        int rc = batch_create_on(ctx, p, pairs, n, ctx->stream, &B, &cand);
        if (rc) return rc;
        if (B->walk && walk_done[wt]) {
          ta_batch_destroy(B);
          continue;
        }
        if (B->walk) walk_done[wt] = true;
        double ms = 1e300;
        for (int r = 0; r <= repeats && !rc; ++r) {  // first run warms up
          rc = ta_batch_run(ctx, B);
          if (!rc) rc = ta_batch_wait(ctx, B);
          if (!rc && r > 0) ms = std::min(ms, B->ms[3]);
        }
        ta_batch_destroy(B);
        if (rc) return rc;
        if (ms < win_ms) { win_ms = ms; win = cand; }
      }
    }
  }
  {
    std::lock_guard<std::mutex> g(ctx->tune_mu);
    ctx->tune[tune_key(p, ta_tune_bucket(pairs, n))] = win;
  }
  if (best) *best = win;
  if (best_ms) *best_ms = win_ms;
  return TA_OK;
}
