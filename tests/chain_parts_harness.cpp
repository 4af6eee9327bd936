// Host harness for what csrc/scn_pyr_dev.h gained beside the sweeps over whole
// samples: levels made from the source directly (a wavefront per level), and
// samples shared out among workgroups, by layers and by slabs of a layer.  The
// arguments, the entry point and the check of the masks are chain_cpu_harness.cpp's.
#include "scn_pyr_dev.h"
namespace {
template <int D> int run(PyrArgs &a, int T, long long *report);
template <> int run<1>(PyrArgs &a, int T, long long *report);
template <> int run<2>(PyrArgs &a, int T, long long *report);
template <> int run<3>(PyrArgs &a, int T, long long *report);
} // namespace
#include "chain_cpu_harness.cpp"

namespace {
int wantParts = 1, maxF = 0, mostParts = 0;

template <int D, int RW> void level(const PyrArgs &a, int b, int x, int T, pyr_u64 *out) {
  const PyrLevel &L = a.lv[x];
  const int n0 = a.lv[0].nOut, plane = D == 3 ? n0 : 1;
  const bool deep = D == 3 && L.foldW > PYR_FOLD_DIRECT;
  // (as many slabs as the masks' words, more than the device would take, included)
  const int slabs = 1 + (b + x) % 4 < L.words ? 1 + (b + x) % 4 : L.words;
  for (int i = 0; i < slabs; ++i) {
    const PyrSlab z = pyr_slab(D, L, L.magicN, i, slabs);
    std::vector<pyr_u64> lds((size_t)pyr_slab_words(D, RW, n0, L, z), 0);
    pyr_u64 *rows = lds.data(), *mid = rows + RW * plane * (z.p1 - z.p0);
    pyr_u64 *mask = mid + (deep ? RW * (z.p1 - z.p0) * L.nOut : 0);
    if (mask + (z.w1 - z.w0) != lds.data() + lds.size() || z.p1 > n0 || z.p0 < 0) {
      fprintf(stderr, "a slab's LDS\n");
      abort();
    }
    for (int t = 0; t < T; ++t)
      pyr_sweep_stage<RW>(a.bits, (long long)b * a.lv[0].volOut + (long long)z.p0 * plane * n0, n0,
                          plane * (z.p1 - z.p0), rows, t, T);
    if (deep)
      for (int t = 0; t < T; ++t)
        pyr_sweep_mid<RW>(rows, mid, z.p1 - z.p0, n0, L.nOut, L.magicN, L.foldW, L.foldS, t, T);
    for (int t = 0; t < T; ++t)
      pyr_sweep_fold<D, RW>(rows, mid, mask, z, n0, L.nOut, L.magicN, L.foldW, L.foldS, t, T);
    memcpy(out + z.w0, mask, 8 * (size_t)(z.w1 - z.w0));
  }
}

// every level from the source has to be what level after level gives
template <int D> void check_levels(PyrArgs &a, int b, int T) {
  const int RW = pyr_set_fold(a);
  for (int x = 1; x < a.nMasks && RW; ++x) {
    const PyrLevel &L = a.lv[x];
    std::vector<pyr_u64> got((size_t)L.words + 2);
    if (D == 3)
      level<3, 1>(a, b, x, T, got.data());
    else if (RW == 1)
      level<2, 1>(a, b, x, T, got.data());
    else if (RW == 2)
      level<2, 2>(a, b, x, T, got.data());
    else
      level<2, 4>(a, b, x, T, got.data());
    if (memcmp(got.data(), a.pyramid + (long long)b * a.pyrStride + L.maskOff, 8 * (size_t)(L.words + 2))) {
      fprintf(stderr, "level %d from the source differs\n", x);
      abort();
    }
  }
}

// k_pyr_rules, one part of sample b
template <int D> void part_b(const PyrArgs &a, int b, const PyrPart &part, int T) {
  std::vector<unsigned char> ldsv((size_t)a.ldsBytesB, 0xA5);
  unsigned char *lds = ldsv.data();
  PyrHdr *h = reinterpret_cast<PyrHdr *>(lds);
  h->over = 0;
  h->cut = part.F > 1;
  h->emitFrom = part.la;
  h->slab = part.f;
  h->plane[0] = part.f ? a.lv[part.la].nOut : 0;
  h->plane[1] = a.lv[part.la].nOut;
  for (int t = 0; t <= PYR_MAX_LEVELS; ++t)
    h->before[t] = 0;
  memcpy(lds + PYR_HDR_BYTES, a.pyramid + (long long)b * a.pyrStride, 8ll * a.pyrStride);
  for (int x = 0; x < a.nMasks; ++x) {
    const int *cnt = a.counts + (long long)x * a.batch * 2;
    h->actBefore[x] = h->bgBefore[x] = h->actAll[x] = h->bgAll[x] = h->maxAct[x] = 0;
    for (int s = 0; s < a.batch; ++s) {
      h->actBefore[x] += s < b ? cnt[2 * s] : 0;
      h->bgBefore[x] += s < b ? cnt[2 * s + 1] : 0;
      h->maxAct[x] = cnt[2 * s] > h->maxAct[x] ? cnt[2 * s] : h->maxAct[x];
    }
    h->n[x] = cnt[2 * b];
    h->hasBg[x] = cnt[2 * b + 1];
  }
  if (part.F > 1) {
    const PyrLds all = pyr_lds_view(a, lds, 0, 0);
    for (int t = 0; t < T; ++t)
      pyr_sweep_planes(a, all, part, t, T);
    for (int t = 0; t < T; ++t)
      pyr_fill_cut(a, all, part, t);
    pyr_fix_cut(h, part);
    if (part.F > maxF)
      maxF = part.F;
  }
  for (int xa = part.la >= 3 ? part.la - 2 : 0;;) {
    const int xb = pyr_window_end(a, h->cut ? h->held : h->n, xa, part.lb);
    const int la = xa + 1, lb = xb;
    const bool last = xb == part.lb;
    for (int t = 0; t <= a.nMasks; ++t)
      pyr_fill_offsets(h, xa, xb, t);
    for (int t = 0; t < a.nMasks; ++t)
      pyr_fill_en(a.lv[t], lds, t, h->siteOff[t]);
    const PyrLds s = pyr_lds_view(a, lds, h->total, pyr_held(h, xa));
    if (s.kOf + h->total > lds + a.ldsBytesB) {
      fprintf(stderr, "a window takes more LDS than pass B was launched with\n");
      abort();
    }
    for (int t = 1; t <= a.nLevels; ++t)
      if ((t >= la && t <= lb) || (last && lb == a.nMasks - 1 && t == a.nLevels && t > lb))
        pyr_fill_level(a.lv[t], a.lv[t - 1].maskOff, a.bg[b], s, t, xa);
    for (int t = 0; t < T; ++t)
      pyr_sweep_clear(s, t, T);
    for (int t = 0; t < T; ++t)
      pyr_sweep_enumerate<D>(a, s, xa, xb, t, T);
    if (xa == 0 && part.la == 1)
      for (int r = 0; r < pyr_held(h, 0); ++r) {
        int c[D];
        pyr_unpack<D>(s.key[r], c);
        s.srcRow[r] = (unsigned)a.dense[(long long)b * a.lv[0].volOut + pyr_key<D>(c, a.lv[0].nOut)];
      }
    for (int t = 0; t < T; ++t)
      pyr_sweep_owners<D>(s, la, lb, t, T);
    for (int x = xa; x < xb; ++x) {
      const int from = h->cut ? h->own[x] : 0, to = h->cut ? h->ownEnd[x] : h->n[x];
      unsigned carry = (unsigned)pyr_base_start(h, x);
      for (int r = from; r < to; ++r) {
        const int at = h->siteOff[x] + r - pyr_lo(h, x);
        s.base[at] = (unsigned short)carry;
        carry += (unsigned)pyr_popc32(pyr_own_mask(s, (unsigned)at));
      }
    }
    for (int t = 0; t < T; ++t)
      pyr_sweep_rows<D>(s, la, lb, b, t, T);
    for (int t = 0; t < T; ++t)
      pyr_sweep_rules<D>(s, la, lb, t, T);
    for (int t = 0; t < T; ++t)
      pyr_sweep_tail(a, s, la, lb, b, t, T);
    if (last)
      break;
    for (int t = 0; t < T; ++t)
      pyr_sweep_carry(s, lds, a, xb, t, T);
    xa = xb;
  }
}

template <int D> int run_parts(PyrArgs &a, int T, long long *report) {
  bool gaveUp = false, over = false;
  for (int b = 0; b < a.batch; ++b) {
    pass_a<D>(a, b, T / 2 > 0 ? T / 2 : 1, &gaveUp);
    if (D > 1)
      check_levels<D>(a, b, T);
  }
  for (int b = 0; b < a.batch; ++b) { // (whole samples: the reports)
    pass_b<D>(a, b, T, gaveUp, report, &over);
    if (over)
      return (gaveUp ? 1 : 0) | 2;
  }
  for (int l = 1; l <= a.nLevels; ++l) { // now again, by parts
    const PyrReport r = {report[4 * l], report[4 * l + 1], 0, report[4 * l + 3]};
    const PyrLevel &L = a.lv[l];
    const long long rules = L.kind == PYR_TERMINAL ? r.extra * a.batch : r.nSites * L.width;
    if (L.rules)
      memset(L.rules, 0x77, 4 * (size_t)rules);
    memset(L.ekey, 0x77, 8 * (size_t)r.nActive);
    memset(L.erow, 0x77, 4 * (size_t)r.nActive);
    memset(L.bg, 0x77, 4 * (size_t)a.batch);
  }
  long long n[PYR_MAX_LEVELS + 1] = {0};
  for (int x = 0; x < a.nMasks; ++x)
    for (int b = 0; b < a.batch; ++b)
      n[x] += a.counts[((long long)x * a.batch + b) * 2];
  // (every site as costly as some hundred: the parts of real fields from small ones)
  for (int x = 0; x < a.nMasks; ++x)
    n[x] = n[x] * 200 / a.batch + 1;
  pyr_plan_parts(a, n, wantParts);
  mostParts = a.nParts > mostParts ? a.nParts : mostParts;
  for (int b = 0; b < a.batch; ++b)
    for (int p = a.nParts - 1; p >= 0; --p)
      part_b<D>(a, b, a.parts[p], T);
  return 0;
}
template <> int run<1>(PyrArgs &a, int T, long long *report) { return run_parts<1>(a, T, report); }
template <> int run<2>(PyrArgs &a, int T, long long *report) { return run_parts<2>(a, T, report); }
template <> int run<3>(PyrArgs &a, int T, long long *report) { return run_parts<3>(a, T, report); }
} // namespace

// how many parts a sample is cut into at most from now on; returns the most that one has been cut into, or
// (want < 0) the most slabs of a layer
extern "C" int pyr_cpu_parts(int want) {
  if (want < 0)
    return maxF;
  wantParts = want;
  return mostParts;
}
