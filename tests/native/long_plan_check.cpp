// Memory plans of long pairs (tweakseq_amd/csrc/longplan.h) over random
// batches: what a plan takes stays within what its requests were admitted
// for.  Prints "long plan ok" (built and run by tests/test_long_plan.py).
#include <cmath>
#include <cstdio>
#include <random>

#include "../../tweakseq_amd/csrc/longplan.h"

using namespace ta;
typedef std::vector<std::pair<int32_t, int32_t>> Shapes;

#define CHECK(c)                                                      \
  do {                                                                \
    if (!(c)) {                                                       \
      fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); \
      return 1;                                                       \
    }                                                                 \
  } while (0)

static LongNeed need_of(const Shapes &v, bool trace) {
  LongNeed n;
  n.trace = trace;
  for (auto &s : v) n.add(s.first, s.second);
  return n;
}

// Every pair's rows and columns in the block, apart from those of its group.
static int well_formed(const LongPlan &P, const Shapes &v, bool trace) {
  int lp = 0, it = 0;
  CHECK(P.at.size() == v.size());
  for (const LongGroup &g : P.groups) {
    CHECK(g.lp0 == lp && g.it0 == it && g.npairs > 0);
    uint64_t ring = 0, col = g.ring_n;
    for (int k = g.lp0; k < g.lp0 + g.npairs; ++k) {
      CHECK(P.at[k].ring == ring && P.at[k].col == col && P.at[k].item0 == it);
      ring += (uint64_t)long_rows(v[k].first, v[k].second);
      col += (uint64_t)long_cols(v[k].first, v[k].second, trace);
      it += long_strips(v[k].first);
    }
    CHECK(ring == g.ring_n && col <= P.entries);
    lp += g.npairs;
    CHECK(g.nitems == it - g.it0);
  }
  CHECK(lp == (int)v.size());
  return 0;
}

int main() {
  std::mt19937 rng(1);
  for (int t = 0; t < 4000; ++t) {
    const bool trace = t % 3 != 0;
    const int hi = t % 2 ? 1000000 : 100000, nreq = 1 + (int)(rng() % 5);
    auto len = [&] { return std::max(1, (int)std::exp2(std::uniform_real_distribution<>(0, std::log2((double)hi))(rng))); };
    Shapes all;
    int64_t least = 0, full = 0, most = 0;
    for (int r = 0; r < nreq; ++r) {
      Shapes v;
      for (int k = (int)(rng() % (t % 5 ? 8 : 300)); k >= 0; --k) v.push_back({len(), len()});
      const LongNeed n = need_of(v, trace);
      CHECK(n.least() <= n.full() && (trace ? n.least() >= n.share : n.least() == 0));
      least += n.least();
      full += n.full();
      most = std::max(most, n.most);
      all.insert(all.end(), v.begin(), v.end());
    }
    const LongNeed n = need_of(all, trace);
    CHECK(n.least() <= least && n.full() <= full);
    const LongPlan free = long_plan(all, trace, 256, -1);
    if (well_formed(free, all, trace)) return 1;
    CHECK(8 * (int64_t)free.entries <= std::max(std::max(LONG_ROOM, n.share), most));
    // within what the requests are admitted for, whatever that is
    for (int q = 0; q < 4; ++q) {
      const int64_t limit = q == 0 ? least : q == 1 ? full : least + (int64_t)((full - least) * (rng() % 1000 / 1000.0));
      const LongPlan P = long_plan(all, trace, 256, limit);
      if (well_formed(P, all, trace)) return 1;
      CHECK(P.bytes() <= std::max(limit, trace ? 0 : most));
      if (q == 1) CHECK(P.ahead == free.ahead);
    }
  }
  printf("long plan ok\n");
  return 0;
}
