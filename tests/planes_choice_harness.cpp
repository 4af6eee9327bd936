// The choice of k_nin_lines' tiles on the CPU (test_planes_choice.py).
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
  return x.next > 0.f ? lines_long(numCU, M, K, N, 32 * x.mt * x.rw, 32 * x.nt * x.cw, x.d) : 0;
}
