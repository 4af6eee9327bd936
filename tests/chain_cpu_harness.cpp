// The kernels that build a net's rule books from the output side
// (csrc/scn_pyr_body.h, scn_pyr_dev.h) on the host: the text the device runs, with
// an executor that does the lanes of a workgroup one after the other.  Built with
// the undefined-behaviour sanitizer by tests/test_chain_cpu.py, which compares what
// comes out with the oracle: every index the kernels compute is computed here
// first, on the CPU.  What the planning in csrc/scn_chain.hip does with a chain
// is done here by the same functions.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include "scn_pyr_body.h"

namespace {

// An executor of scn_pyr_body.h.  Backwards: the lanes and wavefronts in descending
// order (between two barriers none may matter to another).
struct HostLanes {
  static constexpr int T = 0;
  int nLanes;
  bool backwards;
  int windows = 0;
  HostLanes(int lanes, bool backwards) : nLanes(lanes), backwards(backwards) {}
  template <typename V> struct Lane { // (of the lanes that have a layer)
    V v[PYR_MAX_LEVELS + 1];
    V &operator[](int t) {
      if (t < 0 || t > PYR_MAX_LEVELS)
        abort();
      return v[t];
    }
  };
  template <typename V> struct Wave {
    V v[64];
    V &operator[](int t) { return v[t]; }
    const V &operator[](int t) const { return v[t]; }
  };
  int threads() const { return nLanes; }
  template <typename F> void each(int n, F f) const {
    for (int i = 0; i < n; ++i)
      f(backwards ? n - 1 - i : i);
  }
  template <typename F> void lanes(F f) const { each(nLanes, f); }
  template <typename F> void waves(int n, F f) const { each(n, f); }
  template <typename F> void wave(F f) const { each(64, f); }
  template <typename F> unsigned sum(F f) const {
    unsigned n = 0;
    each(64, [&](int lane) { n += f(lane); });
    return n;
  }
  template <typename F> int max(F f) const {
    int n = 0;
    each(64, [&](int lane) { n = f(lane) > n ? f(lane) : n; });
    return n;
  }
  template <typename F> Wave<unsigned> scan(F f) const {
    Wave<unsigned> w;
    unsigned n = 0;
    for (int lane = 0; lane < 64; ++lane)
      w[lane] = n += f(lane);
    return w;
  }
  template <typename F> int count(F f) const {
    int n = 0;
    each(64, [&](int lane) { n += f(lane) ? 1 : 0; });
    return n;
  }
  template <typename V> int at(const Wave<V> &w, int lane) const { return (int)w[lane]; }
  int uniform(int x) const { return x; }
  void sync() const {}
  int row(const PyrArgs &a, long long p) const { return a.dense[p]; }
  void check(bool holds) const {
    if (!holds) {
      fprintf(stderr, "a workgroup's own check does not hold\n");
      abort();
    }
  }
  void window() { ++windows; }
};

// Memory with something behind it that has to stay as it is
struct Guarded {
  std::vector<pyr_u64> v;
  size_t words;
  explicit Guarded(size_t words) : v(words + 16, 0xA5A5A5A5A5A5A5A5ull), words(words) {}
  pyr_u64 *words64() { return v.data(); }
  unsigned char *bytes() { return reinterpret_cast<unsigned char *>(v.data()); }
  ~Guarded() {
    for (size_t i = words; i < v.size(); ++i)
      if (v[i] != 0xA5A5A5A5A5A5A5A5ull) {
        fprintf(stderr, "written beyond a buffer's end\n");
        abort();
      }
  }
};

#ifndef PYR_HARNESS_PLAN
// whole samples (n: the mean sites of the levels)
void plan(PyrArgs &a, const long long *n) { pyr_plan_parts(a, n, 1); }
#endif

template <int D, int RW> void levels(const PyrArgs &a, long long words) {
  for (int y = 0; y < a.nSlabs; ++y)
    for (int b = 0; b < a.batch; ++b) {
      Guarded lds((size_t)words + 2);
      HostLanes e(64, y & 1);
      pyr_levels_body<D, RW>(e, a, lds.bytes(), b, y);
    }
}

// Both kinds of pass A, which have to agree; what they leave is then in a.pyramid
// and a.counts as the library would have it
template <int D> void pass_a(PyrArgs &a, std::vector<int> &counts) {
  const size_t all = (size_t)a.batch * (size_t)a.maskWords;
  long long words = pyr_plan_whole(a);
  for (int b = 0; b < a.batch; ++b) {
    Guarded lds((size_t)words + 2);
    HostLanes e(64, b & 1);
    pyr_masks_body<D>(e, a, lds.bytes(), b);
  }
  const int RW = pyr_set_fold(a);
  if (D == 1 || !RW)
    return;
  const std::vector<int> whole(counts);
  const std::vector<pyr_u64> masks(a.pyramid, a.pyramid + all);
  std::fill(counts.begin(), counts.end(), -1);
  std::fill(a.pyramid, a.pyramid + all, 0x3C3C3C3C3C3C3C3Cull);
  words = pyr_plan_slabs(a, RW);
  if (D == 3)
    levels<3, 1>(a, words);
  else if (RW == 1)
    levels<2, 1>(a, words);
  else if (RW == 2)
    levels<2, 2>(a, words);
  else
    levels<2, 4>(a, words);
  bool same = !memcmp(masks.data(), a.pyramid, 8 * all);
  for (int x = 0; x < a.nMasks; ++x)
    for (int b = 0; b < a.batch; ++b) {
      int n = 0;
      for (int z = 0; z < pyr_slabs(D, a.lv[0].nOut, a.lv[x], a.slabs); ++z)
        n += counts[((size_t)x * a.batch + b) * a.slabs + z];
      same = same && n == whole[(size_t)x * a.batch + b];
    }
  if (!same) {
    fprintf(stderr, "levels from the source differ\n");
    abort();
  }
}

// report: [nLevels + 1][4]
template <int D> int run(PyrArgs &a, int T, std::vector<int> &counts, long long *report) {
  pass_a<D>(a, counts);
  long long mean[PYR_MAX_LEVELS + 1];
  for (int x = 0; x < a.nMasks; ++x) {
    mean[x] = 0;
    for (int b = 0; b < a.batch; ++b)
      for (int z = 0; z < (a.slabs == 1 ? 1 : pyr_slabs(D, a.lv[0].nOut, a.lv[x], a.slabs)); ++z)
        mean[x] += counts[((size_t)x * a.batch + b) * a.slabs + z];
    mean[x] = mean[x] / a.batch + 1;
  }
  plan(a, mean);
  int over = 0;
  for (int block = a.batch * a.nParts; block >= 0; --block) {
    Guarded lds((size_t)a.ldsBytesB / 8);
    HostLanes e(T, block & 1);
    pyr_rules_body<D>(e, a, lds.bytes(), block);
    over |= reinterpret_cast<PyrHdr *>(lds.bytes())->over;
    report[0] = e.windows > report[0] ? e.windows : report[0]; // (the most windows a part took)
  }
  for (int l = 1; l <= a.nLevels; ++l)
    memcpy(report + 4 * l, a.scalars + 16 + 4 * a.lv[l].slot, 32);
  return (over & 2 ? 1 : 0) | (over & 1 ? 2 : 0);
}

long long ipow(long long a, int d) {
  long long r = 1;
  for (int i = 0; i < d; ++i)
    r *= a;
  return r;
}

} // namespace

// geo: per recorded layer {kind, nIn, nOut, size, stride}.  Source grids as
// scn_grids_build takes them.  Per layer l (1-based) rules[l - 1] (capacity
// rulesCap[l - 1] ints, may be null), ekey / erow / bgOut [l - 1]; bounds
// [l - 1][2] = {rows, active}.  report: [nLevels + 1][4] = sites, active sites,
// outgrew, terminal width or largest sample; report[0][0] = the most windows of
// levels a sample was built in.  Returns 0, or 1 | 2 when a sample
// outgrew the LDS or a layer its bounds (nothing is written then).
extern "C" int pyr_cpu_chain(int d, int batch, int n0, int nLevels, const int *geo, const int *sample,
                             const long long *key, const int *row, long long nActive, const int *bg,
                             int **rules, const long long *rulesCap, long long **ekey, int **erow, int **bgOut,
                             const long long *bounds, long long *report, int ldsBytesB, int T) {
  PyrArgs a;
  memset(&a, 0, sizeof(a));
  const long long vol0 = ipow(n0, d);
  std::vector<pyr_u64> bits((size_t)((batch * vol0 + 63) / 64 + 2), 0);
  std::vector<int> dense((size_t)(batch * vol0), -7);
  for (long long i = 0; i < nActive; ++i) {
    const long long p = (long long)sample[i] * vol0 + key[i];
    bits[(size_t)(p >> 6)] |= 1ull << (p & 63);
    dense[(size_t)p] = row[i];
  }
  a.nLevels = nLevels;
  a.batch = batch;
  a.d = d;
  a.dense = dense.data();
  a.bits = bits.data();
  a.bg = bg;
  std::vector<long long> meta((size_t)nLevels * 4), scalars((size_t)(16 + 4 * nLevels));
  const long long badSites = 0;
  a.scalars = scalars.data();
  a.badSites = &badSites;
  pyr_add_level(a, 0, PYR_REGIONS, n0, n0, 1, 1, 1, vol0, vol0 + 1);
  for (int l = 1; l <= nLevels; ++l) {
    const int *g = geo + 5 * (l - 1);
    const bool terminal = g[0] == PYR_TERMINAL;
    const long long vol = terminal ? 1 : ipow(g[2], d);
    pyr_add_level(a, l, g[0], g[1], g[2], g[3], g[4], terminal ? 1 : (int)ipow(g[3], d), vol, vol);
    PyrLevel &L = a.lv[l];
    L.rules = rules[l - 1];
    L.capacity = rulesCap[l - 1];
    L.ekey = ekey[l - 1];
    L.erow = erow[l - 1];
    L.bg = bgOut[l - 1];
    L.meta = meta.data() + 4 * (l - 1);
    L.slot = l - 1;
    L.boundRows = bounds[2 * (l - 1)];
    L.boundActive = bounds[2 * (l - 1) + 1];
  }
  if (!pyr_set_layout(a) || pyr_fixed_lds(a) + 4 * a.nChunks > ldsBytesB)
    return 4;
  a.ldsBytesB = ldsBytesB;
  Guarded pyramid((size_t)batch * (size_t)a.maskWords);
  std::vector<int> counts((size_t)a.nMasks * batch * 8, -1);
  a.pyramid = pyramid.words64();
  a.counts = counts.data();
  switch (d) {
  case 1:
    return run<1>(a, T, counts, report);
  case 2:
    return run<2>(a, T, counts, report);
  default:
    return run<3>(a, T, counts, report);
  }
}
