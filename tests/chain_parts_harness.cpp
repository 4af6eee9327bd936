// chain_cpu_harness.cpp with samples shared out among workgroups, by layers and by
// slabs of a layer, and levels among wavefronts: as the library does it for fields
// far larger than those the tests have.
#define PYR_PART_MIN 40  // (a part is worth its while from a site or so on)
#define PYR_SLAB_ROWS 16 // (a slab from sixteen rows on)
#include "scn_pyr_body.h"
namespace {
int wantParts = 1, maxF = 0, mostParts = 0;
#define PYR_HARNESS_PLAN
void plan(PyrArgs &a, const long long *n) {
  pyr_plan_parts(a, n, wantParts);
  mostParts = a.nParts > mostParts ? a.nParts : mostParts;
  for (int p = 0; p < a.nParts; ++p)
    maxF = a.parts[p].F > maxF ? a.parts[p].F : maxF;
}
} // namespace
#include "chain_cpu_harness.cpp"

// how many parts a sample is cut into at most from now on; returns the most that one has been cut into, or
// (want < 0) the most slabs of a layer
extern "C" int pyr_cpu_parts(int want) {
  if (want < 0)
    return maxF;
  wantParts = want;
  return mostParts;
}
