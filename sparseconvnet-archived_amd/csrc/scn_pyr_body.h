// The kernels that build a net's rule books from the output side, written
// once for the device and for the host: scn_pyr_dev.h has what a lane does in
// each sweep, here is what a workgroup does with the sweeps.  An executor E runs
// it, on the device the workgroup that was launched (scn_chain.hip), in the tests
// a loop over its lanes (tests/chain_cpu_harness.cpp):
//
//   T                     lanes of the workgroup
//   lanes(f)              f(t) for every lane t
//   waves(n, f)           f(i) for i < n, a wavefront each
//   wave(f)               f(lane) for the 64 lanes of a wavefront
//   sum(f), max(f)        over the wavefront, of f(lane)
//   scan(f)               Wave<unsigned> of the sums up to and with each lane
//   count(f), at(w, lane) lanes for which f holds; what that lane has in w
//   Lane<T>, Wave<T>      a T for every lane of the workgroup, of a wavefront
//   uniform(x)            x, the same for all lanes of the wavefront
//   sync()                what the lanes have written to LDS is there for all
//   row(a, p)             the source's row at position p of the batch
//   check(x), window()    for the host: x has to hold; another window of levels
#pragma once
#include "scn_pyr_dev.h"

#if defined(__HIPCC__)
#define PYR_BODY __device__ __forceinline__
#define PYR_UNROLL _Pragma("unroll")
#define PYR_UNROLL4 _Pragma("unroll 4")
#else
#define PYR_BODY static inline
#define PYR_UNROLL
#define PYR_UNROLL4
#endif

enum { PYR_META_SITES, PYR_META_ACTIVE, PYR_META_OVERFLOW, PYR_META_WIDTH }; // of a level's meta words

// ------------------------------------------------------------------- pass A
// A layer's geometry as k_pyr_masks keeps it in LDS: one broadcast read a layer
// instead of trips to the kernel arguments
struct PyrGeoA {
  int nIn, nOut, size, stride;
  int words, offIn, offOut;
  unsigned magicN, seg, segs, magicSegs;
  int pad;
};
static_assert(sizeof(PyrGeoA) == 48, "three 16-byte reads");
#define PYR_A_GEO ((PYR_MAX_LEVELS + 1) * (int)sizeof(PyrGeoA)) // geometry: after the masks
// Whole samples to k_pyr_masks.  Returns the words of LDS that takes.
PYR_FN long long pyr_plan_whole(PyrArgs &a) {
  a.slabs = 1;
  a.nSlabs = 0;
  return (8ll * a.maskWords + 15) / 16 * 2 + PYR_A_GEO / 8;
}

// Sample b's masks, layer after layer, by one wavefront
template <int D, typename E> PYR_BODY void pyr_masks_body(E &e, const PyrArgs &a, unsigned char *lds, int b) {
  pyr_u64 *masks = reinterpret_cast<pyr_u64 *>(lds);
  PyrGeoA *geo = reinterpret_cast<PyrGeoA *>(lds + (8ll * a.maskWords + 15) / 16 * 16);
  int *const counts = a.counts + (long long)b * a.slabs; // (slabs: 1)
  typename E::template Wave<unsigned> n;
  e.wave([&](int t) {
    if (t >= 1 && t < a.nMasks) {
      const PyrLevel &L = a.lv[t];
      PyrGeoA g;
      g.nIn = L.nIn;
      g.nOut = L.nOut;
      g.size = L.size;
      g.stride = L.stride;
      g.words = L.words;
      g.offIn = a.lv[t - 1].maskOff;
      g.offOut = L.maskOff;
      g.magicN = L.magicN;
      g.seg = L.seg;
      g.segs = L.segs;
      g.magicSegs = L.magicSegs;
      g.pad = 0;
      geo[t] = g;
    }
    // level 0: the sample's slice of the source mask, four words a lane at a time
    const PyrLevel &L = a.lv[0];
    const int words = L.words;
    const long long vol = L.volOut;
    n[t] = 0;
    for (int w0 = 0; w0 < words + 2; w0 += 256) {
      pyr_u64 v[4];
      PYR_UNROLL
      for (int u = 0; u < 4; ++u) {
        const int w = w0 + 64 * u + t;
        v[u] = w < words ? pyr_source_word(a.bits, vol, b, (unsigned)w) : 0ull;
      }
      PYR_UNROLL
      for (int u = 0; u < 4; ++u) {
        const int w = w0 + 64 * u + t;
        n[t] += (unsigned)pyr_popc64(v[u]);
        if (w < words + 2)
          masks[w] = v[u];
      }
    }
    // the other levels start empty: their pieces are OR-ed in
    for (int w = words + 2 + t; w < a.maskWords; w += 64)
      masks[w] = 0ull;
  });
  const unsigned sites = e.sum([&](int t) { return n[t]; });
  e.wave([&](int t) {
    if (t == 0)
      counts[0] = (int)sites;
  });
  e.sync();
  for (int x = 1; x < a.nMasks; ++x) {
    // (wavefront-uniform values, told to the compiler: the loops over a window's
    // rows then branch on scalars)
    PyrGeoA g = geo[x];
    g.nIn = e.uniform(g.nIn);
    g.nOut = e.uniform(g.nOut);
    g.size = e.uniform(g.size);
    g.stride = e.uniform(g.stride);
    g.words = e.uniform(g.words);
    g.offIn = e.uniform(g.offIn);
    g.offOut = e.uniform(g.offOut);
    g.magicN = (unsigned)e.uniform((int)g.magicN);
    g.seg = (unsigned)e.uniform((int)g.seg);
    g.segs = (unsigned)e.uniform((int)g.segs);
    g.magicSegs = (unsigned)e.uniform((int)g.magicSegs);
    e.wave([&](int t) {
      pyr_sweep_dilate<D>(masks + g.offIn, masks + g.offOut, g.nIn, g.nOut, g.size, g.stride, g.magicN, g.seg, g.segs,
                          g.magicSegs, t, 64);
    });
    e.sync();
    e.wave([&](int t) {
      n[t] = 0;
      for (int w = t; w < g.words; w += 64)
        n[t] += (unsigned)pyr_popc64(masks[g.offOut + w]);
    });
    const unsigned here = e.sum([&](int t) { return n[t]; });
    e.wave([&](int t) {
      if (t == 0)
        counts[(long long)x * a.batch * a.slabs] = (int)here;
    });
  }
  e.wave([&](int t) {
    pyr_u64 *dst = a.pyramid + (long long)b * a.maskWords;
    for (int i = t; i < a.maskWords; i += 64)
      dst[i] = masks[i];
  });
}

// The mask of sample b at the level of pair y of a.slab, one slab of it, by one wavefront
template <int D, int RW, typename E>
PYR_BODY void pyr_levels_body(E &e, const PyrArgs &a, unsigned char *lds, int b, int y) {
  const PyrPair of = pyr_pair(a.slab, y);
  const int x = of.a, slab = of.b;
  const PyrLevel &L = a.lv[x];
  const int nOut = L.nOut, n0 = a.lv[0].nOut;
  const long long vol0 = a.lv[0].volOut;
  int *const count = a.counts + ((long long)x * a.batch + b) * a.slabs + slab;
  const PyrSlab z = pyr_slab(D, L, L.magicN, slab, pyr_slabs(D, n0, L, a.slabs));
  const int words = z.w1 - z.w0;
  pyr_u64 *const out = a.pyramid + (long long)b * a.maskWords + L.maskOff + z.w0;
  pyr_u64 *const rows = reinterpret_cast<pyr_u64 *>(lds);
  const int plane = D == 3 ? n0 : 1;
  const bool deep = D == 3 && L.foldW > PYR_FOLD_DIRECT;
  pyr_u64 *const mid = rows + RW * plane * (z.p1 - z.p0);
  pyr_u64 *const mask = mid + (deep ? RW * (z.p1 - z.p0) * nOut : 0);
  e.check(x == 0 || (mask + words == rows + pyr_slab_words(D, RW, n0, L, z) && z.p0 >= 0 && z.p1 <= n0));
  if (x > 0) {
    e.wave([&](int t) {
      for (int w = t; w < words; w += 64)
        mask[w] = 0ull;
      pyr_sweep_stage<RW>(a.bits, (long long)b * vol0 + (long long)z.p0 * plane * n0, n0, plane * (z.p1 - z.p0), rows,
                          t, 64);
    });
    e.sync();
    if (deep) {
      e.wave([&](int t) {
        pyr_sweep_mid<RW>(rows, mid, z.p1 - z.p0, n0, nOut, L.magicN, L.foldW, L.foldS, t, 64);
      });
      e.sync();
    }
    e.wave([&](int t) {
      pyr_sweep_fold<D, RW>(rows, mid, mask, z, n0, nOut, L.magicN, L.foldW, L.foldS, t, 64);
    });
    e.sync();
  }
  typename E::template Wave<unsigned> n;
  e.wave([&](int t) {
    n[t] = 0;
    PYR_UNROLL4
    for (int w = t; w < words; w += 64) {
      const pyr_u64 v = x > 0 ? mask[w] : pyr_source_word(a.bits, vol0, b, (unsigned)(z.w0 + w));
      n[t] += (unsigned)pyr_popc64(v);
      out[w] = v;
    }
    if (z.w1 == L.words && t < 2) // (two spare words)
      out[words + t] = 0ull;
  });
  const unsigned sites = e.sum([&](int t) { return n[t]; });
  e.wave([&](int t) {
    if (t == 0)
      *count = (int)sites;
  });
}

// ------------------------------------------------------------------- pass B
struct PyrSums { // of a level, over the samples a lane looks at
  unsigned before, bgBefore, all, bgAll, own;
  int most;
};
struct PyrFour {
  unsigned v[4];
};

// A part of a sample; the last workgroup has no sample: it reports the counts to
// the host
template <int D, typename E> PYR_BODY void pyr_rules_body(E &e, const PyrArgs &a, unsigned char *lds, int block) {
  constexpr int T0 = E::T;
  const int T = T0 ? T0 : e.threads();
  PyrHdr *h = reinterpret_cast<PyrHdr *>(lds);
  const bool reports = block == a.batch * a.nParts;
  const int b = reports ? 0 : block % a.batch;
  const PyrPart part = a.parts[reports ? 0 : block / a.batch];
  // lane t keeps layer t's arguments from here on: fetched while the masks
  // come in, not when the level table wants them
  typename E::template Lane<PyrLevel> mine;
  typename E::template Lane<int> inMaskOff;
  const int bgSource = a.bg[b];
  const int xFirst = part.la >= 3 ? part.la - 2 : 0, xLast = part.lb;
  pyr_u64 *const masks = reinterpret_cast<pyr_u64 *>(lds + PYR_HDR_BYTES);
  unsigned short *const pref = reinterpret_cast<unsigned short *>(masks + a.maskWords);
  e.lanes([&](int t) {
    if (t <= a.nLevels) {
      mine[t] = a.lv[t];
      inMaskOff[t] = a.lv[t > 0 ? t - 1 : 0].maskOff;
    }
    if (t == 0) {
      h->over = 0;
      h->cut = part.F > 1;
      h->emitFrom = part.la;
      h->slab = part.f;
      h->plane[0] = part.f ? a.lv[part.la].nOut : 0;
      h->plane[1] = a.lv[part.la].nOut;
    }
    if (t < a.nMasks) {
      h->before[t] = 0;
      h->words[t] = mine[t].words + 2;
      h->maskOff[t] = mine[t].maskOff;
    }
    // the masks of the part's levels and of the two before it
    const pyr_u64 *src = a.pyramid + (long long)b * a.maskWords;
    const int end = xLast + 1 < a.nMasks ? a.lv[xLast + 1].maskOff : a.maskWords;
    for (int i = a.lv[xFirst].maskOff + t; i < end; i += T)
      masks[i] = src[i];
  });
  // sums over the samples, a wavefront per level
  e.waves(a.nMasks, [&](int x) {
    const int *cnt = a.counts + (long long)x * a.batch * a.slabs;
    const long long full = a.lv[x].fullSize;
    const int slabs = a.slabs == 1 ? 1 : pyr_slabs(a.d, a.lv[0].nOut, a.lv[x], a.slabs);
    typename E::template Wave<PyrSums> v;
    e.wave([&](int lane) {
      // (a batch's rows are numbered in 32 bits, so these sums fit)
      PyrSums m = {0, 0, 0, 0, 0, 0};
      for (int s = lane; s < a.batch; s += 64) {
        int n = 0;
        for (int z = 0; z < slabs; ++z)
          n += cnt[s * a.slabs + z];
        const int hb = n < full;
        if (s < b) {
          m.before += n;
          m.bgBefore += hb;
        }
        m.own = s == b ? n : m.own;
        m.all += n;
        m.bgAll += hb;
        m.most = n > m.most ? n : m.most;
      }
      v[lane] = m;
    });
    const unsigned before = e.sum([&](int lane) { return v[lane].before; });
    const unsigned bgBefore = e.sum([&](int lane) { return v[lane].bgBefore; });
    const unsigned all = e.sum([&](int lane) { return v[lane].all; });
    const unsigned bgAll = e.sum([&](int lane) { return v[lane].bgAll; });
    const unsigned own = e.sum([&](int lane) { return v[lane].own; });
    const int most = e.max([&](int lane) { return v[lane].most; });
    e.wave([&](int lane) {
      if (lane == 0) {
        h->n[x] = (int)own;
        h->hasBg[x] = (int)own < full;
        h->actBefore[x] = before;
        h->bgBefore[x] = bgBefore;
        h->actAll[x] = all;
        h->bgAll[x] = bgAll;
        h->maxAct[x] = most;
      }
    });
  });
  e.sync();
  e.lanes([&](int t) {
    if (t >= 1 && t <= a.nLevels && pyr_report(a, mine[t], h, t).over)
      PYR_ATOMIC_OR(&h->over, 1);
    // (a sample that does not fit: the whole batch is planned another way.  The
    // largest counts of two levels need not be one sample's: they only say whether
    // the samples have to be asked)
    if (t < a.nMasks && (h->maxAct[t] > PYR_ROWS_MAX ||
                         !pyr_pair_fits(a, h->maxAct[t], t + 1 < a.nMasks ? h->maxAct[t + 1] : 0)))
      PYR_ATOMIC_OR(&h->over, 4);
  });
  // rank prefixes, a wavefront per chunk of 256 words of a level: within the
  // chunk now, what lies before it once the chunks' sums are there
  unsigned *const sums = reinterpret_cast<unsigned *>(lds + PYR_HDR_BYTES + 8ll * a.pyrStride);
  e.waves(a.nChunks, [&](int i) {
    const PyrPair of = pyr_pair(a.chunk, i);
    const int x = of.a;
    if (x < xFirst || x > xLast)
      return;
    const int words = h->words[x], at = h->maskOff[x], w0 = PYR_CHUNK * of.b;
    typename E::template Wave<PyrFour> pc;
    e.wave([&](int lane) {
      PYR_UNROLL
      for (int u = 0; u < 4; ++u)
        pc[lane].v[u] = w0 + 4 * lane + u < words ? (unsigned)pyr_popc64(masks[at + w0 + 4 * lane + u]) : 0u;
    });
    auto four = [&](int lane) { return pc[lane].v[0] + pc[lane].v[1] + pc[lane].v[2] + pc[lane].v[3]; };
    auto incl = e.scan(four);
    e.wave([&](int lane) {
      unsigned run = incl[lane] - four(lane);
      PYR_UNROLL
      for (int u = 0; u < 4; ++u) {
        if (w0 + 4 * lane + u < words)
          pref[at + w0 + 4 * lane + u] = (unsigned short)run;
        run += pc[lane].v[u];
      }
      if (lane == 63)
        sums[i] = incl[lane];
    });
  });
  e.sync();
  e.waves(a.nChunks, [&](int i) {
    const PyrPair of = pyr_pair(a.chunk, i);
    const int x = of.a, c = of.b;
    if (c == 0 || x < xFirst || x > xLast)
      return;
    const unsigned before = e.sum([&](int lane) {
      unsigned s = 0;
      for (int k = lane; k < c; k += 64)
        s += sums[i - c + k];
      return s;
    });
    const int words = h->words[x], at = h->maskOff[x];
    e.wave([&](int lane) {
      const int w0 = PYR_CHUNK * c + 4 * lane;
      PYR_UNROLL
      for (int u = 0; u < 4; ++u)
        if (w0 + u < words)
          pref[at + w0 + u] = (unsigned short)(pref[at + w0 + u] + before);
    });
  });
  if (h->over & 4)
    e.lanes([&](int t) {
      for (int sample = t; sample < a.batch; sample += T) {
        const int *c = a.counts + (long long)sample * a.slabs;
        auto sites = [&](int x) {
          int n = 0;
          for (int z = 0; z < pyr_slabs(a.d, a.lv[0].nOut, a.lv[x], a.slabs); ++z)
            n += c[(long long)x * a.batch * a.slabs + z];
          return n;
        };
        bool fits = pyr_fits_of(a, sites);
        for (int x = 0; x < a.nMasks; ++x)
          fits = fits && sites(x) <= PYR_ROWS_MAX;
        if (!fits)
          PYR_ATOMIC_OR(&h->over, 2);
      }
    });
  e.sync();
  const bool over = (h->over & 3) != 0;
  e.lanes([&](int t) {
    if (reports && t >= 1 && t <= a.nLevels) {
      const PyrLevel &L = mine[t];
      const PyrReport r = pyr_report(a, mine[t], h, t);
      L.meta[PYR_META_SITES] = over ? 0 : r.nSites;
      L.meta[PYR_META_ACTIVE] = over ? 0 : r.nActive;
      L.meta[PYR_META_OVERFLOW] = over;
      L.meta[PYR_META_WIDTH] = L.kind == PYR_TERMINAL ? r.extra : 0;
      volatile long long *slot = a.scalars + 16 + 4 * L.slot;
      slot[0] = r.nSites;
      slot[1] = r.nActive;
      slot[2] = over;
      slot[3] = r.extra;
    }
    if (reports && t == 0) {
      a.scalars[15] = *a.badSites;
      a.scalars[13] = h->maxAct[0];
    }
  });
  if (over || reports)
    return;
  if (part.F > 1) {
    const PyrLds all = pyr_lds_view(a, lds, 0, 0);
    e.lanes([&](int t) { pyr_sweep_planes(a, all, part, t, T); });
    e.sync();
    e.lanes([&](int t) { pyr_fill_cut(a, all, part, t); });
    e.sync();
    e.lanes([&](int t) {
      if (t == 0)
        pyr_fix_cut(h, part);
    });
    e.sync();
  }
  // the part's layers a window of levels at a time: as many as the LDS holds (all
  // of them, for all but the largest samples); the rows of the layer before the
  // first of them are worked out here once more
  for (int xa = part.la >= 3 ? part.la - 2 : 0;;) {
    e.window();
    // where the window's levels start, and how many of them fit (at least one
    // behind xa, where there is one), a lane a level: every wavefront by itself
    typename E::template Wave<int> held;
    e.wave([&](int x) { held[x] = x >= xa && x <= part.lb ? pyr_held(h, x) : 0; });
    auto to = e.scan([&](int x) { return (unsigned)held[x]; });
    const int firstSites = e.at(held, xa);
    const long long room = a.ldsBytesB - (pyr_fixed_lds(a) + 4ll * firstSites);
    const int fit = e.count([&](int x) { return x > xa + 1 && x <= part.lb && 11ll * (int)to[x] <= room; });
    const int xb = xa < part.lb ? xa + 1 + fit : xa;
    const int la = xa + 1, lb = xb;
    const bool last = xb == part.lb;
    e.lanes([&](int t) {
      if (t >= xa && t <= xb + 1) {
        const int sum = (int)to[t] - held[t];
        h->siteOff[t] = sum;
        h->itemOff[t] = t > xa ? sum - firstSites : 0;
        if (t == xb + 1)
          h->total = sum;
      }
    });
    e.sync();
    const PyrLds s = pyr_lds_view(a, lds, h->total, pyr_held(h, xa));
    e.check(s.kOf + h->total <= lds + a.ldsBytesB);
    e.lanes([&](int t) {
      if (t < a.nMasks)
        pyr_fill_en(mine[t], lds, t, h->siteOff[t]);
      if ((t >= la && t <= lb) || (last && lb == a.nMasks - 1 && t == a.nLevels && t > lb))
        pyr_fill_level(mine[t], inMaskOff[t], bgSource, s, t, xa);
      pyr_sweep_clear(s, t, T);
    });
    e.sync();
    e.lanes([&](int t) { pyr_sweep_enumerate<D>(a, s, xa, xb, t, T); });
    e.sync();
    if (xa == 0 && part.la == 1) // the batch's rows of the source's sites: their loads go out first
      e.lanes([&](int t) {
        const PyrLevel &L = a.lv[0];
        const long long p0 = (long long)b * L.volOut;
        for (int r = t; r < pyr_held(h, 0); r += T) {
          int c[D];
          pyr_unpack<D>(s.key[r], c);
          long long p = p0 + pyr_key<D>(c, L.nOut);
          p = p < (long long)a.batch * L.volOut ? p : 0; // (a mask never has a site beyond the field)
          s.srcRow[r] = (unsigned)e.row(a, p);
        }
      });
    e.lanes([&](int t) { pyr_sweep_owners<D>(s, la, lb, t, T); });
    e.sync();
    // rows owned by the sites before, a wavefront per level
    e.waves(xb - xa, [&](int i) {
      const int x = xa + i;
      const int from = h->cut ? h->own[x] : 0;
      const int n = (h->cut ? h->ownEnd[x] : h->n[x]) - from;
      const unsigned off = (unsigned)(h->siteOff[x] + from - pyr_lo(h, x));
      unsigned carry = (unsigned)pyr_base_start(h, x);
      for (int r0 = 0; r0 < n; r0 += 256) { // (four sites a lane: the chain of sums is what this takes)
        typename E::template Wave<PyrFour> owned;
        e.wave([&](int lane) {
          const int r = r0 + 4 * lane;
          PYR_UNROLL
          for (int u = 0; u < 4; ++u)
            owned[lane].v[u] = r + u < n ? (unsigned)pyr_popc32(pyr_own_mask(s, off + r + u)) : 0u;
        });
        auto four = [&](int lane) {
          return owned[lane].v[0] + owned[lane].v[1] + owned[lane].v[2] + owned[lane].v[3];
        };
        auto incl = e.scan(four);
        e.wave([&](int lane) {
          const int r = r0 + 4 * lane;
          unsigned run = carry + incl[lane] - four(lane);
          PYR_UNROLL
          for (int u = 0; u < 4; ++u) {
            if (r + u < n)
              s.base[off + r + u] = (unsigned short)run;
            run += owned[lane].v[u];
          }
        });
        carry += (unsigned)e.at(incl, 63);
      }
      e.check(h->cut || (int)carry == h->n[x + 1]); // (every site is owned once)
    });
    e.sync();
    e.lanes([&](int t) { pyr_sweep_rows<D>(s, la, lb, b, t, T); });
    e.sync();
    e.lanes([&](int t) {
      pyr_sweep_rules<D>(s, la, lb, t, T);
      pyr_sweep_tail(a, s, la, lb, b, t, T);
    });
    if (last)
      break;
    e.sync();
    e.lanes([&](int t) { pyr_sweep_carry(s, lds, a, xb, t, T); });
    e.sync();
    xa = xb;
  }
}
