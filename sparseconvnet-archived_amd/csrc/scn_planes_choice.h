// Which of k_nin_lines' tiles a contraction takes, and which weight gradients go into one
// launch (scn_planes.hip), by measured costs: no HIP in it.
#pragma once
#include <math.h>
#include <stdint.h>

static inline int64_t tiles_of(int64_t n, int64_t each) { return (n + each - 1) / each; }

// the bytes of W laid out as planes; whether they are more than those of the rows
static inline int64_t image_bytes(int planes, int K, int N) { return tiles_of(N, 32) * 32 * K * 2 * planes; }
static inline bool image_larger(int planes, int64_t rows, int K, int N, int channels) {
  return image_bytes(planes, K, N) > rows * channels * 4;
}

// k_nin_lines' tiles.  A workgroup alone on its compute unit takes f + T t1
// microseconds for T blocks of 32 k, with `resident` of them there (LDS) a block
// takes all of them tn.  Fitted to 26 shapes (1037 to 1.36 M rows, 128 to 2592 k, 64
// to 800 columns; 10 % rms), of which it takes 25 to the fastest of these tiles or
// one within 5 %.  Taller or wider tiles, one wavefront in place of two a SIMD, and
// deeper rings gained nothing.
// LONG: a workgroup's tiles take `begin`, and each `next` and `tl` a block.  Fitted to 37
// shapes of plain rows in every tile (9000 to 400000 rows, 64 to 2560 k, 32 to 1280
// columns; 3 to 11 % rms, all a tenth less than measured, as the others' are of plain
// rows): what it takes is 1.5 % off the fastest on average.  (With t1 for tl and a smaller
// `next` 4.7 %: 70000 x 160 x 36 23.4 us and not 19, 70000 x 512 x 64 59 and not 46.)  The
// ring of six is never the fastest so: 64 x 64 tiles of which two share a compute unit
// are.  Three tiles of columns to a wavefront keep too much from one tile to the next: 35
// registers spilled, whose memory is allocated when they are first launched.
struct LinesTile {
  int mt, nt, rw, cw, d, resident;
  float f, t1, tn, begin, next, tl; // tl 0: never LONG
};
static const LinesTile linesTiles[2][6] = {
    {{1, 2, 4, 2, 3, 2, 1.9f, .53f, .92f, 0.f, 0.f, 0.f}, {1, 2, 2, 2, 4, 2, 3.f, .22f, .38f, 0.f, 0.f, 0.f}, {1, 1, 2, 2, 3, 4, 1.9f, .36f, .58f, 0.f, 0.f, 0.f}}, // one plane
    {{1, 2, 4, 2, 3, 1, 4.1f, 1.04f, 0.f, 2.5f, 2.1f, 1.12f}, {2, 1, 4, 2, 3, 1, 4.3f, 1.25f, 0.f, 1.6f, 3.f, 1.3f}, {1, 3, 4, 1, 4, 1, 4.5f, .87f, 0.f, 0.f, 0.f, 0.f},
     {1, 2, 2, 2, 4, 1, 3.4f, .68f, 0.f, 3.1f, 1.45f, .71f}, {1, 1, 2, 2, 3, 2, 2.f, .58f, .85f, 0.f, 0.f, 0.f}, {1, 1, 2, 2, 6, 1, 2.f, .5f, 0.f, 0.f, 0.f, 0.f}}};
// (One more of three planes, for plain rows of one tile of columns, which the others give 64:
// 128 x 32, two of which share a compute unit.  With the image us, 64 x 64 and this, 123606 x 768 x 32 97,
// 87; 174344 x 1728 x 32 277, 237; 43000 x 256 x 32 18.6, 15.4; 300000 x 128 x 32 46, 38.)
constexpr int LINES_NARROW = 6;
// How many workgroups an XCD has of a LONG launch, a multiple of the slices of columns
// (0: a launch of a workgroup a tile): plain rows of no less than their weights, in three
// planes, of no more than 512 k, where a compute unit that has room for one workgroup has
// more than one tile.  (Longer contractions have little of their time between the tiles:
// in the tiles that are best for them, a workgroup a tile and LONG, 5000 x 2560 x 800 144,
// 148, 26000 x 1280 x 480 168, 202; 16500 x 512 x 256 37.4, 38.1, its gradient 40, 37.
// Gathered rows: 15948 x 1280 x 480 115 us for 110, 15003 x 1920 x 640 232 for 220, with the
// rules of the next tiles under way; two workgroups to a compute unit see to that
// themselves: 139000 x 128 x 64 36 for 29.)  The launch and the choice of its tile both ask
// here: with LONG's costs for tiles that are not launched so, 2600 x 1024 x 1920 took 78 us
// and not 68, 2500 x 256 x 2048 28 and not 25.
static inline int lines_long(int numCU, int64_t M, int K, int N, int rows, int columns, int d) {
  const int cus = numCU / 8, T = K / 32;
  const int64_t splits = tiles_of(N, columns);
  return T >= d - 1 && T <= 16 && splits <= cus && !image_larger(3, M, K, N, K) && tiles_of(M, rows) * splits > numCU
             ? (int)(cus / splits * splits)
             : 0;
}
// Whether LONG's results are to go past the caches: those of a gradient, which is read
// once, and what would not be found there anyway, rows and results of more than the 256 MB
// of the Infinity Cache.  A layer's output is read at once and by windows: contraction and
// pooling, a workgroup a tile, past the caches, through them, 139000 x 384 x 128 138, 140,
// 131; 139000 x 256 x 192 161, 165, 152; 100000 x 96 x 192 68, 76, 65; 60000 x 320 x 160 70,
// 75, 67; 57000 x 256 x 96 36.5, 38.7, 36.5; 250000 x 128 x 192 229, 212, 220; 600000 x 64 x 64
// 166, 145, 158.
static inline bool lines_past_caches(int64_t M, int K, int N, bool gradient) {
  return gradient || M * ((int64_t)K + N) * 4 > (int64_t)256 << 20;
}
static inline float lines_cost(int numCU, const LinesTile &x, int planes, int64_t M, int K, int N, bool gather) {
  const int T = K / 32, rows = 32 * x.mt * x.rw, columns = 32 * x.nt * x.cw;
  const float n = (float)tiles_of(M, rows) * tiles_of(N, columns) / numCU;
  float cost;
  if (n <= x.resident) {
    const float shared = x.resident > 1 ? (fmaxf(ceilf(n), 1.f) - 1.f) / (x.resident - 1) : 0.f;
    cost = x.f + T * (x.t1 + shared * (x.tn - x.t1));
  } else if (const int per = x.tl > 0.f && !gather ? lines_long(numCU, M, K, N, rows, columns, x.d) : 0) {
    cost = x.begin + tiles_of(tiles_of(M, rows) * tiles_of(N, columns), 8 * per) * (x.next + T * x.tl);
  } else {
    const float rounds = n / x.resident <= 3.f ? ceilf(n / x.resident) : n / x.resident + .5f;
    cost = rounds * (x.f + T * (x.resident > 1 ? x.tn : x.t1));
  }
  // (rows that few workgroups share, and the clock: 130000 x 512 x 64 63 us in the
  // second tile, 58 in k_nin_planes)
  return planes == 3 && gather && n > (x.mt > 1 ? 1.f : 4.f) ? 1.12f * cost : cost;
}
static inline float lines_choose(int numCU, int planes, int64_t M, int K, int N, bool gather, int *tile) {
  float least = 1e30f;
  for (int i = 0; i < (planes == 3 ? 6 : 3); ++i) {
    const float cost = lines_cost(numCU, linesTiles[planes == 3][i], planes, M, K, N, gather);
    if (cost < least)
      least = cost, *tile = i;
  }
  return least + 4.f;
}

// k_nin_rows16: how many tiles of columns a wavefront of it takes, 0: not one for it (bf16
// rows through rules; more than 32 columns).  Slices cost what their columns do and the
// fetching of the rows.  Measured against what else there is (k_nin_planes, k_nin_lines) on 69 shapes of
// 800 to 674000 rows, 256 to 3456 k and 64 to 320 columns, by workgroups to a compute unit: two
// tiles of columns 0.73 to 1.3 of them 1.09, 2.2 to 2.3 0.93 to 0.98 (2592 k 0.95), from 3.6
// on 0.70 to 0.96; three 0.45 1.09, 0.86 to 1.1 0.91 to 0.94, from 1.6 on 0.71 to 0.95; four 0.15 to 0.3
// 1.1 to 1.3, 0.33 to 0.76 from 2016 k on 0.91 to 0.99, 1.1 to 1.4 0.84 to 1.03, then 0.77 to
// 0.94.  Shorter ones, of 256 to 864 k, have more of their time in a workgroup's start and stores:
// up to 3 workgroups 0.99 to 1.5, from 4 on 0.79 to 1.01.
static inline int rows16_tiles(int numCU, int64_t M, int K, int N) {
  int tiles = 0;
  int64_t least = INT64_MAX;
  for (int nt = 4; nt >= 2; --nt)
    if (const int64_t cost = tiles_of(N, 32 * nt) * (nt + 1); cost < least)
      least = cost, tiles = nt;
  const float n = (float)tiles_of(M, 256) * tiles_of(N, 32 * tiles) / numCU;
  return n >= (K < 896 ? 4.f : tiles == 2 ? 2.f : tiles == 4 && K >= 2000 ? .4f : .8f) ? tiles : 0;
}

// ---- a weight gradient (scn_atb_planes)
constexpr int ATB_STEP = 16; // rows that a wavefront takes at a time
// By lines, tiles of two have a step's planes made among the MFMAs of the step before, and
// three wavefronts to a SIMD.  What a 1 x 1 tile is for is over in a few steps, which
// begin and end sooner in eight wavefronts without: 400 x 384 x 128 5.4 -> 4.0 us, 1000 x
// 512 x 160 6.4 -> 5.4, 2500 x 384 x 64 6.2 -> 4.9, 8000 x 256 x 64 7.5 -> 6.3.
constexpr bool atb_ahead(int MT, int NT) { return MT * NT == 2; }
constexpr int atb_waves(int MT, int NT, bool LINES) { return LINES && atb_ahead(MT, NT) ? 12 : 8; }
// The tile and the ranges of rows that cost least: rounds of one workgroup a compute
// unit, each `ti` microseconds for every step of its wavefronts and `f` to start, to sum
// and to store, and the atomics.  By lines fitted to 25 shapes (1000 to 198759 rows, 16 to
// 1728 x 32 to 480, gathered and plain) in every tile and three to seven numbers of
// ranges, 11 % rms: what it takes is 1.2 % off the fastest of these on average
// (2.4 with the costs of eight wavefronts and ranges of 128 rows, rounded up to 192 by the
// launch: 3000 x 864 x 64 10.2 -> 7.7, 45000 x 128 x 64 13.5 -> 12.0).  Where rows are loaded
// into registers, eight wavefronts, their own costs.  Two by two tiles, us against two by one, plain rows: 126507 x 1728 x 64 175, 246;
// 53325 x 640 x 320 135, 176; 17223 x 1280 x 480 145, 187; 139000 x 384 x 128 91, 117.
// (The search is 0.1 to 2 us of the host's time, a launch some 5.)
struct AtbTile {
  int mt, nt;
  double ti[2], f[2]; // registers, lines
};
static const AtbTile atbTiles[4] = {
    {1, 1, {.8, .67}, {4., 2.2}}, {2, 1, {1.13, 1.4}, {4., 3.7}}, {1, 2, {1.13, 1.42}, {4., 4.2}}, {2, 2, {1.95, 1.36}, {6., 3.7}}};
struct AtbChoice {
  int tile;     // -1: none
  int64_t rows; // of a range, whole steps of a workgroup
  double cost;
};
static inline AtbChoice atb_choose(int numCU, int64_t M, int K, int N, bool lines, bool pairsA, bool pairsD, bool twoByTwo) {
  AtbChoice best = {-1, 0, 1e300};
  for (int i = 0; i < (twoByTwo ? 4 : 3); ++i) {
    const AtbTile &t = atbTiles[i];
    const int64_t tiles = tiles_of(K, 32 * t.mt) * tiles_of(N, 32 * t.nt), each = atb_waves(t.mt, t.nt, lines) * ATB_STEP;
    if ((t.mt == 2 && !pairsA) || (t.nt == 2 && !pairsD) || tiles > 0x7fffffffll)
      continue;
    const int64_t most = tiles_of(M, each);
    for (int64_t s = 1; s <= most && s <= 4096; s += s < 64 ? 1 : s / 32) {
      const int64_t steps = tiles_of(M, s * each), ranges = tiles_of(M, steps * each), rounds = tiles_of(tiles * ranges, numCU);
      const double cost = rounds * (steps * t.ti[lines] + t.f[lines]) + (double)tiles * ranges * t.mt * t.nt * 1024 / 2e5;
      if (cost < best.cost)
        best = {i, steps * each, cost};
      if (rounds > 8)
        break;
    }
  }
  return best;
}

// ---- weight gradients of several layers (k_atb_many)
// How a layer is taken: a first layer's few columns, two by one tiles for what is no more
// than 32 columns of dW wide, two by two.  What a step and a tile's beginning and end
// take, in sixteenths of a microsecond: these of eleven sets, by which the layers of a
// batch of drawings took 39 to 44 us and of voxel models 34 to 37.
enum { ATB_FIRST, ATB_NARROW, ATB_WIDE };
struct AtbKind {
  int mt, nt, step, tile;
};
constexpr AtbKind atbKinds[3] = {{1, 1, 16, 75}, {2, 1, 17, 75}, {2, 2, 27, 88}};
constexpr int ATB_TILE_COST = 75; // (for atb_join)
constexpr int ATB_MANY_ROWS = 128; // of a step
struct AtbShape {
  int64_t M;
  int K, N;
  int tile; // 32 rows of dW each, 0: not one for k_atb_many
  int each; // a step's cost
  int64_t tiles() const { return tile ? tiles_of(K, 32 * tile) * tiles_of(N, 32) : 0; }
  int64_t steps() const { return tiles_of(M, ATB_MANY_ROWS); }
};
// One that keeps the chip busy by itself (some 60 us) gains nothing among others, and
// two by two tiles may be better for it.  One that is left alone goes by itself, too, in
// the tile that is best for it: us, alone in k_atb_many and by itself, 1000 x 512 x 160
// 11.7, 7.4; 11400 x 384 x 128 23.5, 15.7; 28000 x 256 x 96 25.5, 18.6; 57250 x 128 x 64
// 22.2, 15.5.  Several, in launches of their own and in one: the layers of a batch of
// drawings, first and second 23.9, 20.9, second and third 29.3, 24.8, fourth and fifth
// 23.1, 25.1; second to fourth 42.5, 37.4, fourth to sixth 28.6, 25.3; all seven 73.9, 46.8.
static inline int atb_join(int numCU, const AtbShape *shape, int n, bool *joined) {
  int count = 0, last = 0;
  for (int k = 0; k < n; ++k) {
    const AtbShape &s = shape[k];
    joined[k] = s.M > 0 && s.tile > 0 && s.tiles() <= 4096 &&
                s.tiles() * (s.steps() * s.each + ATB_TILE_COST) <= (int64_t)64 * 16 * numCU;
    if (joined[k])
      ++count, last = k;
  }
  if (count != 1)
    return count;
  joined[last] = false;
  return 0;
}
