// Batch containers on the CPU, without a device: what the host view of the grids leaves behind (test_batch_grids.py).
#include "SpatiallySparseBatch.h"

// `batches` batches of `samples` samples on an input interface and one behind it, each with a host view of `sites` sites
// a sample, as downloadGrids and somebody who fills them leave it; the grids that are still held after the last
// reset, and, with keep, the most that were held by the input interface meanwhile.
extern "C" int held(int batches, int samples, int sites, int keep, int *most) {
  SpatiallySparseBatchSubInterface inputSub, sub;
  SpatiallySparseBatch batch(&inputSub);
  batch.interfaces.emplace_back(&sub);
  *most = 0;
  for (int b = 0; b < batches; ++b) {
    if (keep)
      batch.interfaces[0].keepGrids(samples - b % 2);
    if ((int)batch.interfaces[0].spareGrids.size() > *most)
      *most = (int)batch.interfaces[0].spareGrids.size();
    batch.reset();
    for (auto &i : batch.interfaces) {
      i.downloadGrids(samples);
      for (auto &g : i.grids)
        for (int s = 0; s < sites; ++s)
          g.mp[s] = s;
    }
  }
  batch.reset();
  int n = 0;
  for (auto &i : batch.interfaces)
    n += (int)(i.grids.size() + i.spareGrids.size());
  return n;
}
