// The choices of scn_planes.hip on the CPU (test_planes_choice.py).
#include "scn_planes_choice.h"

extern "C" int lines_tile(int numCU, int planes, int64_t M, int K, int N, int gather) {
  int tile = -1;
  lines_choose(numCU, planes, M, K, N, gather != 0, &tile);
  return tile;
}
extern "C" float lines_tile_cost(int numCU, int planes, int tile, int64_t M, int K, int N, int gather) {
  return lines_cost(numCU, linesTiles[planes == 3][tile], planes, M, K, N, gather != 0);
}
// how the tile is launched (launch_lines): workgroups an XCD of a LONG launch, 0: a workgroup a tile
extern "C" int lines_tile_long(int numCU, int tile, int64_t M, int K, int N) {
  const LinesTile &x = linesTiles[1][tile];
  return x.tl > 0.f ? lines_long(numCU, M, K, N, 32 * x.mt * x.rw, 32 * x.nt * x.cw, x.d) : 0;
}
// which of n weight gradients go into one launch; returns how many
extern "C" int joined(int numCU, int n, const int64_t *M, const int *K, const int *N, const int *tile, const int *each, int *out) {
  AtbShape shape[64];
  bool in[64];
  for (int k = 0; k < n; ++k)
    shape[k] = {M[k], K[k], N[k], tile[k], each[k]};
  const int count = atb_join(numCU, shape, n, in);
  for (int k = 0; k < n; ++k)
    out[k] = in[k];
  return count;
}
// a weight gradient's tile; out: the rows of a range, its cost
extern "C" int atb(int numCU, int64_t M, int K, int N, int lines, int pairsA, int pairsD, int twoByTwo, int64_t *rows, double *cost) {
  const AtbChoice c = atb_choose(numCU, M, K, N, lines != 0, pairsA != 0, pairsD != 0, twoByTwo != 0);
  *rows = c.rows, *cost = c.cost;
  return c.tile;
}
extern "C" int past_caches(int64_t M, int K, int N, int gradient) { return lines_past_caches(M, K, N, gradient != 0); }
