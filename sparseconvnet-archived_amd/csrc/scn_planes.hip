// NetworkInNetwork contraction on the bf16 matrix cores, in one, two or three
// bf16 planes per fp32 operand.
//
// A float has 24 significant bits and a bf16 8, so x = hi + mid + lo with
// hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid is exact (both
// subtractions are; |mid| <= 2^-9 |x|, |lo| <= 2^-17 |x|) down to bf16's smallest
// step, 2^-133: of |x| < 2^-110 up to 2^-134 is lost (bf16 subnormals count, in
// the conversion and in the MFMA).  With three planes
// of both operands the six products hi hi, hi mid, mid hi, mid mid, hi lo and
// lo hi, each exact in the MFMA's fp32 accumulator, are the product a b up to
// the 2^-25 |a b| of the three that are left out: less than the rounding of
// one fp32 multiplication, and than that of the accumulation either way.  (Sums
// of split operands in this manner: Henry, Tang and Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations",
// 2019.)  Error against 64 bits: 0.31 to 0.38 of the fp32 MFMA kernels'.
// v_mfma_f32_32x32x16_bf16 does 32768 flops in 32 cycles, v_mfma_f32_32x32x2_f32
// 4096 in 64, so six of the former are 2.7 times as fast.
//   PL 3: SCN_FP32; PL 2: SCN_BF16X3 (hi hi, hi lo, lo hi); PL 1: SCN_BF16.
#include "scn_image_dev.h"
#include "scn_planes_choice.h"
#include <math.h>
#include <utility>

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

bool scn_planes_shape(int K) { return K % 32 == 0 && K >= 64; }

// Rows that are known on the device only.  Which kernel takes a layer depends
// on their number; where either may be right both are launched, and one of them
// finds that it is not its.
struct RowRange {
  const long long *d_rows; // null: as many as the host says
  long long above, upTo;   // this kernel's: above < rows <= upTo
  __device__ __forceinline__ long long live(long long bound) const {
    if (!d_rows)
      return bound;
    const long long n = *d_rows;
    return n <= above || n > upTo ? 0 : n < bound ? n : bound;
  }
};

// An infinite operand, or one that rounds to an infinite bf16, leaves NaN in its
// other planes (x - hi), where fp32 arithmetic has an infinity or a finite sum.
// So with three planes a sum that is not finite is taken again from the operands
// themselves; the test costs an instruction a result.  The tiles that hold such
// sums are taken again whole, on the fp32 MFMA: a net whose weights have all gone
// to infinities costs a few times what a sound one does, not a serial chain of K
// a result.
template <int PL> __device__ __forceinline__ bool doubtful(float sum) {
  return PL == 3 && !(fabsf(sum) <= 3.4028235e38f);
}
struct PlainW { // W as the caller gave it
  const float *W;
  int wT; // [N x K] and not [K x N]
};
// Eight k of a 32 x 32 tile on v_mfma_f32_32x32x2_f32: lane (c, q) holds a[i] and
// b[i] of the same k for its row of A and column of W.
__device__ __forceinline__ void mfma8_f32(const float (&a)[8], const float (&b)[8], floatx16 &acc) {
#pragma unroll
  for (int i = 0; i < 8; ++i)
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i], acc, 0, 0, 0);
}

// Four channels (A16: eight) of a gathered row: columns k .. of the row that
// `rules` (in LDS, fs of them) stand for.
template <bool A16>
__device__ __forceinline__ floatx4 gathered_piece(const unsigned char *A, const GatherSource &gs,
                                                  const int *rules, int k) {
  const int f = (int)__umulhi((unsigned)k, gs.magic);
  const int rule = rules[f];
  const unsigned char *const row = rule >= 0 ? A + (long long)rule * gs.nIn * (A16 ? 2 : 4)
                                             : reinterpret_cast<const unsigned char *>(gs.zeros);
  return *reinterpret_cast<const floatx4 *>(row + (k - f * gs.nIn) * (A16 ? 2 : 4));
}

// A 32 x 32 tile on the fp32 MFMA by one wavefront: row m of A (GATHER: through
// its rules, in LDS) and column n of W are this lane's, as in mfma8_f32; `mine`
// are the registers of the result it has a use for.
template <bool GATHER>
__device__ __forceinline__ floatx16 tile_f32(const float *A, const GatherSource &gs, const int *rules,
                                             const PlainW &w, long long m, int n, int K, int N, unsigned mine) {
  const int q = (threadIdx.x & 63) >> 5;
  floatx16 sum;
#pragma unroll
  for (int v = 0; v < 16; ++v)
    sum[v] = 0.f;
  if (GATHER && gs.namedOnly) {
    // position by position, each of which the rows that it is named for take
    for (int f = 0; f < gs.fs; ++f) {
      const unsigned named = (unsigned)__ballot(rules[f] >= 0); // row by row (the upper half holds them again)
      if (!named)
        continue;
      floatx16 part;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        part[v] = 0.f;
#pragma unroll 1
      for (int t = 0; t < gs.nIn; t += 16) {
        float a[8], b[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = t + 8 * q + 4 * h;
          const bool inside = k < gs.nIn; // (in fours)
          const floatx4 x = gathered_piece<false>(reinterpret_cast<const unsigned char *>(A), gs, rules,
                                                  f * gs.nIn + (inside ? k : 0));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            a[4 * h + i] = inside ? x[i] : 0.f;
            b[4 * h + i] = inside ? w.W[(long long)(f * gs.nIn + k + i) * N + n] : 0.f;
          }
        }
        mfma8_f32(a, b, part);
      }
      bool open = false;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        sum[v] += named >> (8 * (v / 4) + 4 * q + v % 4) & 1 ? part[v] : 0.f;
        open |= (mine >> v & 1) && sum[v] == sum[v];
      }
      if (!__any(open))
        break;
    }
    return sum;
  }
#pragma unroll 1
  for (int t = 0; t < K; t += 16) { // (K is a multiple of 32)
    const int k = t + 8 * q;
    float a[8], b[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const floatx4 x = GATHER ? gathered_piece<false>(reinterpret_cast<const unsigned char *>(A), gs, rules, k + 4 * h)
                               : *reinterpret_cast<const floatx4 *>(A + m * K + k + 4 * h);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a[4 * h + i] = x[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      b[i] = w.W[w.wT ? (long long)n * K + k + i : (long long)(k + i) * N + n];
    mfma8_f32(a, b, sum);
    if (t % 128 == 112) { // a NaN stays one: through when there is nothing else
      bool open = false;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        open |= (mine >> v & 1) && sum[v] == sum[v];
      if (!__any(open))
        break;
    }
  }
  return sum;
}

enum { W_PLAIN, W_IMAGE, W_STREAM }; // how W comes: see k_nin_planes
// Of the loads a wavefront has asked for, all but the last N have landed, and its
// LDS reads too: what another wavefront asks for next may take their place.
template <int N> __device__ __forceinline__ void w_landed() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N < 63 ? N : 63) : "memory");
}
// A barrier for LDS accesses; loads under way stay so.
__device__ __forceinline__ void barrier_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A kilobyte of global memory straight into LDS, 16 bytes a lane, lane after lane
// from `lds`.  (The compiler does not know of it: see lines_landed and w_landed.)
__device__ __forceinline__ void dma_kilobyte(unsigned lds, const unsigned char *from) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds), "v"(from) : "memory", "m0");
}
// ... and 256 bytes, a word a lane.  (What is asked for behind the compiler's back
// goes to LDS and never to a register of its: one promised by an asm before the data
// is there may be copied or spilled on the way, with what it held before.)
__device__ __forceinline__ void dma_words(unsigned lds, const int *from) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(lds), "v"(from) : "memory", "m0");
}

// A workgroup of WAVES wavefronts owns 32 WAVES MT rows x 32 NT columns, a
// wavefront 32 MT rows of them, and walks k in blocks of 32, two MFMA steps.
// W passes through LDS buffers, a block each, split into planes on the way in
// (W_PLAIN) or copied from an image of it, through registers (W_IMAGE) or without
// a stop there (W_STREAM: three buffers, filled two blocks ahead), and laid out
// as the MFMA reads it, [plane][16 k][tile][lane]: every operand read is a
// contiguous kilobyte.  A goes from global memory (GATHER: through the rules of
// the workgroup's rows, staged in LDS) straight into registers, PD blocks ahead
// as W does, and is split there.
// Lane (c, q) supplies k = 8 q .. 8 q + 7 of a step's sixteen for row c of A
// and for its columns of W; it owns the NT adjacent columns NT c .. NT c + NT -
// 1 (tile j of the MFMA = columns {NT c + j}).
// The products beyond hi hi are a 2^-8 of it and go to accumulators of their
// own: added to the large ones each of them would be rounded at their scale.
//
// The matrix pipe is kept busy by what is issued between its instructions: a
// unit is one row tile's step, its 6 NT MFMAs (32 cycles each, 4 to issue) have
// the splitting of the next unit's operand (44 vector instructions) dealt out
// among them, the request for the operand a block on, and the reads of the W
// tiles of the next step, each as soon as its registers have had their last
// use.  The barrier of a block stands before its last tile's MFMAs.
//
// K is a multiple of 32.  GATHER 1: so are a gathered row's channels, and a
// block lies within one filter position; GATHER 2: they are a multiple of 4 and
// every four of them are looked up.  A16: the rows are bf16 already.
template <int PL, int MT, int NT, int PD, int GATHER, bool A16, int WM, int WAVES>
__global__ void __launch_bounds__(64 * WAVES, WAVES == 8 ? 4 : MT * NT >= 3 ? 2 : MT * NT * PD >= 2 ? 3 : 4)
    k_nin_planes(const float *__restrict__ A, const float *__restrict__ W,
                 float *__restrict__ out, long long M, int K, int N,
                 Epilogue ep, GatherSource gs, int nSplits, RowRange rows, PlainW plain) {
  M = rows.live(M);
  const unsigned tiles = (unsigned)((M + 32 * WAVES * MT - 1) / (32 * WAVES * MT)) * nSplits;
  if (blockIdx.x >= tiles)
    return;
  const unsigned tileOf = xcd_eighth(blockIdx.x, tiles);
  constexpr int ES = A16 ? 2 : 4;
  constexpr int THREADS = 64 * WAVES;
  constexpr int ROWS = 32 * MT * WAVES, NW = 32 * NT;
  constexpr int STEP_BYTES = NT * 1024;       // one plane of 16 k
  constexpr int PLANE_BYTES = 2 * STEP_BYTES; // ... of a block
  constexpr int BUF_BYTES = PL * PLANE_BYTES;
  constexpr bool STREAM = WM == W_STREAM;
  constexpr int BUFS = STREAM ? 3 : 2;
  constexpr int UNITS = 2 * MT; // of a block: (step, row tile)
  extern __shared__ __attribute__((aligned(16))) unsigned char sW[]; // [BUFS][BUF_BYTES], then the rules
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int c = lane & 31, q = lane >> 5;
  const int split = tileOf % nSplits; // workgroups that share rows are neighbours
  const long long wgRow0 = (long long)(tileOf / nSplits) * ROWS;
  const long long row0 = wgRow0 + wave * 32 * MT;
  const int n0 = split * NW;
  const int T = K / 32;

  // ---- W.  One item = V adjacent columns of two consecutive k, or 16 bytes of the
  // image.  (Every instruction occupies the vector memory path for 16 cycles or
  // more: with the eight k of a column to an item, a dword each, the (1, 2) tiles of
  // 100 drawings' layers took 15.7 us and not 14.5, the (1, 1) tiles 20.6 and not
  // 20.2.  Such an item was stored 16 bytes a plane; the dwords that this one stores
  // meet on their banks, in half of the cycles that the LDS is in use (5 % before);
  // with them that is an eighth of all.  N is a multiple of 4; a scratch matrix W may
  // be aligned to no more than a float.)
  constexpr bool IMG = WM == W_IMAGE;
  constexpr int V = NT % 2 ? 2 : 4;
  constexpr int ITEMS = IMG ? BUF_BYTES / 16 : 16 * NW / V;
  constexpr int WPER = STREAM ? 0 : (ITEMS + THREADS - 1) / THREADS;
  constexpr int WREGS = IMG ? 4 : 2 * V;
  float wv[PD][WPER + 1][WREGS];
  int wDst[WPER + 1][IMG ? 1 : V];
  const float *wSrc[WPER + 1];
#pragma unroll
  for (int u = 0; u < WPER; ++u) {
    int x = tid + THREADS * u;
    x = x < ITEMS ? x : ITEMS - 1; // past the end: the last item again (same value, same place)
    if constexpr (IMG) {
      wDst[u][0] = x * 16;
      wSrc[u] = W + (long long)split * T * (BUF_BYTES / 4) + x * 4;
    } else {
      const int kp = x / (NW / V), at = V * (x % (NW / V));
#pragma unroll
      for (int e = 0; e < V; ++e)
        wDst[u][e] = (kp / 8) * STEP_BYTES + (at + e) % NT * 1024 + (kp / 4 & 1) * 512 + (at + e) / NT * 16 + (kp & 3) * 4;
      // (columns past the end are not stored)
      wSrc[u] = W + (long long)(2 * kp) * N + (n0 + at < N ? n0 + at : N - V);
    }
  }
  auto w_load = [&](int slot, int t) {
    t = t < T ? t : T - 1;
#pragma unroll
    for (int u = 0; u < WPER; ++u) {
      if constexpr (IMG) {
        const floatx4 v = *reinterpret_cast<const floatx4 *>(wSrc[u] + (long long)t * (BUF_BYTES / 4));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          wv[slot][u][i] = v[i];
      } else {
        typedef float floatxv __attribute__((ext_vector_type(V), aligned(4)));
        const float *p = wSrc[u] + (long long)t * 32 * N;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const floatxv v = *reinterpret_cast<const floatxv *>(p + (long long)h * N);
#pragma unroll
          for (int e = 0; e < V; ++e)
            wv[slot][u][2 * e + h] = v[e];
        }
      }
    }
  };
  auto w_store = [&](int slot, int buf) {
#pragma unroll
    for (int u = 0; u < WPER; ++u) {
      if constexpr (IMG) {
        *reinterpret_cast<floatx4 *>(sW + buf * BUF_BYTES + wDst[u][0]) =
            floatx4{wv[slot][u][0], wv[slot][u][1], wv[slot][u][2], wv[slot][u][3]};
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) {
          unsigned w[PL];
          split2<PL>(wv[slot][u][2 * e], wv[slot][u][2 * e + 1], w);
#pragma unroll
          for (int l = 0; l < PL; ++l)
            *reinterpret_cast<unsigned *>(sW + buf * BUF_BYTES + l * PLANE_BYTES + wDst[u][e]) = w[l];
        }
      }
    }
  };
  // W_STREAM: a block of the image goes straight into LDS, a kilobyte an instruction,
  // each wavefront every WAVES-th of them.  (The compiler does not know of these
  // loads: what it waits for of its own, the loads being counted in order, it
  // waits a little longer for.)
  constexpr int CHUNKS = BUF_BYTES / 1024;
  const unsigned char *const image =
      reinterpret_cast<const unsigned char *>(W) + (long long)split * T * BUF_BYTES + 16 * lane;
  const int wave0 = __builtin_amdgcn_readfirstlane(wave);
  const unsigned ldsW = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)sW;
  auto w_fetch = [&](int t, int buf) {
    if constexpr (STREAM) {
      t = t < T ? t : T - 1; // (past the last block: that one again, where nobody reads)
      const unsigned char *const src = image + (long long)t * BUF_BYTES;
#pragma unroll
      for (int u = 0; u < (CHUNKS + WAVES - 1) / WAVES; ++u) {
        const int chunk = wave0 + WAVES * u;
        if ((u + 1) * WAVES <= CHUNKS || chunk < CHUNKS) {
          dma_kilobyte(ldsW + (unsigned)(buf * BUF_BYTES + chunk * 1024), src + chunk * 1024);
        }
      }
    }
  };

  // ---- A
  const unsigned char *const Ab = reinterpret_cast<const unsigned char *>(A);
  int *const sRules = reinterpret_cast<int *>(sW + BUFS * BUF_BYTES);
  const unsigned char *rowPtr[MT]; // this lane's rows at the filter position of the block to fetch
  int fetchT = 0, f = 0, ch = 0;   // the block to fetch
  auto aim = [&]() {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int rule = sRules[(wave * 32 * MT + 32 * i + c) * gs.fs + f];
      rowPtr[i] = (rule >= 0 ? Ab + (long long)rule * gs.nIn * ES
                             : reinterpret_cast<const unsigned char *>(gs.zeros)) + 8 * q * ES;
    }
  };
  auto next_block = [&]() { // (past the last block: the last one again)
    if (fetchT + 1 < T) {
      ++fetchT;
      ch += 32;
      if (GATHER == 1 && ch == gs.nIn) {
        ch = 0, ++f;
        aim();
      }
    }
  };
  floatx4 raw[PD][UNITS][A16 ? 1 : 2];
  auto a_load = [&](int slot, int u) {
    if (GATHER == 2) {
#pragma unroll
      for (int h = 0; h < (A16 ? 1 : 2); ++h)
        raw[slot][u][h] = gathered_piece<A16>(Ab, gs, sRules + (wave * 32 * MT + 32 * (u % MT) + c) * gs.fs,
                                        ch + 16 * (u / MT) + 8 * q + 4 * h);
      return;
    }
    const floatx4 *const p = reinterpret_cast<const floatx4 *>(rowPtr[u % MT] + (ch + 16 * (u / MT)) * ES);
    raw[slot][u][0] = p[0];
    if (!A16)
      raw[slot][u][A16 ? 0 : 1] = p[1];
  };
  bf16x8 ap[2][PL]; // the unit in hand and the next one
  auto a_split = [&](int slot, int u, int dst) {
    if (A16 && !STREAM) {
      ap[dst][0] = __builtin_bit_cast(bf16x8, raw[slot][u][0]);
    } else if (A16) {
      floatx4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) // (a copy that stays one: see the loads)
        asm("v_mov_b32 %0, %1" : "=v"(x[i]) : "v"(raw[slot][u][0][i]));
      ap[dst][0] = __builtin_bit_cast(bf16x8, x);
    } else {
      const floatx4 x = raw[slot][u][0], y = raw[slot][u][A16 ? 0 : 1];
      const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
      split8<PL>(v, ap[dst]);
    }
  };

  // ---- prologue
#pragma unroll
  for (int p = 0; p < PD; ++p)
    w_load(p, p);
#pragma unroll
  for (int p = 0; p < (STREAM ? 3 : 0); ++p)
    w_fetch(p, p);
  if (STREAM && !GATHER) { // (GATHER: with the rules)
    w_landed<0>();
    barrier_lds();
  }
  if (GATHER) {
    const long long first = wgRow0 * gs.fs, last = M * gs.fs - 1;
    for (int i = tid; i < ROWS * gs.fs; i += THREADS) {
      const long long r = first + i;
      sRules[i] = gs.rules[r < last ? r : last];
    }
    if (STREAM)
      w_landed<0>();
    __syncthreads();
    if (GATHER == 1)
      aim();
  } else {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      long long m = row0 + 32 * i + c;
      m = m < M ? m : M - 1; // rows past the end: read a valid row, store nothing
      rowPtr[i] = Ab + (m * K + 8 * q) * ES;
    }
  }
#pragma unroll
  for (int p = 0; p < PD; ++p) {
    if (p)
      next_block();
#pragma unroll
    for (int u = 0; u < UNITS; ++u)
      a_load(p, u);
  }
  w_store(0, 0);
  if (!STREAM)
    __syncthreads();

  constexpr int NACC = PL > 1 ? 2 : 1;
  floatx16 acc[NACC][MT][NT];
#pragma unroll
  for (int h = 0; h < NACC; ++h)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[h][i][j][v] = 0.f;

  const unsigned char *const wLane = sW + lane * 16;
  constexpr int BB = NT == 1 ? 2 : 1; // a single tile has no other's MFMAs to be read under
  bf16x8 b[BB][NT][PL];
  int cur = 0;
  auto other = [&]() { return STREAM ? (cur == 2 ? 0 : cur + 1) : cur ^ 1; };
  auto read_b = [&](int buf, int s, int j) {
#pragma unroll
    for (int l = 0; l < PL; ++l)
      b[s % BB][j][l] = *reinterpret_cast<const bf16x8 *>(wLane + buf * BUF_BYTES + l * PLANE_BYTES +
                                                          s * STEP_BYTES + j * 1024);
  };
#pragma unroll
  for (int j = 0; j < NT; ++j)
    read_b(0, 0, j);
  a_split(0, 0, 0);

  auto tile = [&](int s, int i, int j, int src) {
    // products x y with x + y < PL: the largest terms of the product of the sums
#pragma unroll
    for (int x = 0; x < PL; ++x)
#pragma unroll
      for (int y = 0; x + y < PL; ++y) {
        floatx16 &d = acc[x + y == 0 ? 0 : NACC - 1][i][j];
        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ap[src][x], b[s % BB][j][y], d, 0, 0, 0);
      }
  };
  auto deal = [&](int mfmas) {
#pragma unroll
    for (int i = 0; i < mfmas; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); // MFMA
      __builtin_amdgcn_sched_group_barrier(0x320, 1, 0); // a load, an LDS read or write
      __builtin_amdgcn_sched_group_barrier(0x002, 5, 0); // vector arithmetic
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int PRODUCTS = PL * (PL + 1) / 2;
  // (loads of A a block, and image loads that every wavefront makes)
  constexpr int A_LOADS = UNITS * (A16 ? 1 : 2), W_LOADS = CHUNKS / WAVES;
  auto block = [&](int p, int t, bool firstOfAll) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int s = u / MT, i = u % MT, src = u & 1; // (UNITS is even)
      // the next unit's operand; its registers then take a later block's
      if (u + 1 < UNITS)
        a_split(p, u + 1, src ^ 1);
      else
        a_split((p + 1) % PD, 0, src ^ 1);
      if (u == 0) {
        next_block();
        if (!STREAM)
          a_load(p, 0); // (unit 0 was split a unit ago)
      }
      // (W_STREAM: into registers whose last use lies behind the last unit's
      // scheduling barrier: were both in one region the load would get others,
      // copied back at the end of the loop, where the copy waits for a load just
      // made)
      if (STREAM)
        a_load(p, u);
      else if (u + 1 < UNITS)
        a_load(p, u + 1);
      if (u == UNITS - 1)
        w_store((p + 1) % PD, cur ^ 1);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (u == UNITS - 1 && j == (NT > 1)) { // before the first read of the next block's W
          if (NT > 1)
            deal(PRODUCTS);
          if constexpr (STREAM) {
            // The next block's W was asked for two blocks ago (the first three
            // blocks' before the loop, and waited for there); since then this
            // wavefront has asked for two blocks of A, wherever in the loop the
            // compiler has put those, and one of W, of which a block each may
            // still be under way.  Behind the barrier nobody reads this block's W
            // any more: its place takes the third.
            w_landed<A_LOADS + W_LOADS>();
            barrier_lds();
            w_fetch(t + 3, cur);
          } else {
            __syncthreads();
          }
          cur = other();
        }
        // a tile's W is read as soon as its registers are free
        if (NT == 1) {
          if (i == MT - 1)
            read_b(cur, s ^ 1, 0);
        } else if (i == MT - 1 && j > 0) {
          read_b(cur, s ^ 1, j - 1);
        } else if (i == 0 && j == 0 && !(s == 0 && firstOfAll)) {
          read_b(cur, s, NT - 1);
        }
        tile(s, i, j, src);
      }
      deal(u == UNITS - 1 && NT > 1 ? PRODUCTS * (NT - 1) : PRODUCTS * NT);
    }
  };
  for (int t = 0; t < T; t += PD) {
#pragma unroll
    for (int p = 0; p < PD; ++p)
      if (t + p < T) { // uniform
        w_load(p, t + p + PD);
        block(p, t + p, t + p == 0);
      }
  }
  if (STREAM)
    w_landed<0>(); // (before the wavefront gives its LDS back)

  // ---- epilogue: register v of a tile is row 8 (v / 4) + 4 q + v % 4
  const int n = n0 + NT * c;
  ColEpilogue col[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    col[j] = load_col(ep, n + j < N ? n + j : N - 1);
  const bool whole = n0 + NW <= N && N % NT == 0;
  unsigned long long again = 0; // results to be taken from the operands themselves
  if constexpr (PL == 3) {
    float none = 0.f; // 0 sum: NaN for a sum that is not finite
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          none = fmaf(acc[0][i][j][v] + acc[NACC - 1][i][j][v], 0.f, none);
    if (none != 0.f) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (doubtful<PL>(acc[0][i][j][v] + acc[NACC - 1][i][j][v]))
              again |= 1ull << ((i * NT + j) * 16 + v);
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const long long r0 = row0 + 32 * i + 4 * q;
    float *const o = out + r0 * N + n;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int dr = 8 * (v / 4) + v % 4;
      if (r0 + dr >= M)
        continue;
      float r[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j)
        r[j] = finish(NACC == 2 ? acc[0][i][j][v] + acc[NACC - 1][i][j][v] : acc[0][i][j][v], col[j]);
      float *const orow = o + (long long)dr * N;
      if (whole && NT == 4) {
        *reinterpret_cast<float4 *>(orow) = make_float4(r[0], r[1 % NT], r[2 % NT], r[3 % NT]);
      } else if (whole && NT == 2) {
        *reinterpret_cast<float2 *>(orow) = make_float2(r[0], r[1 % NT]);
      } else {
#pragma unroll
        for (int j = 0; j < NT; ++j)
          if (whole || n + j < N)
            orow[j] = r[j];
      }
    }
  }
  if constexpr (PL == 3) {
    if (!__any(again != 0))
      return;
#pragma unroll 1
    for (int e = 0; e < MT * NT; ++e) { // tile (i, j); uniform
      const unsigned mine = (unsigned)(again >> (16 * e)) & 0xffffu;
      if (!__any(mine != 0))
        continue;
      const int i = e / NT, j = e % NT;
      long long m = row0 + 32 * i + c;
      m = m < M ? m : M - 1;
      const int nn = n + j < N ? n + j : N - 1;
      const floatx16 sum = tile_f32<GATHER != 0>(A, gs, sRules + (m - wgRow0) * gs.fs, plain, m, nn, K, N, mine);
      const ColEpilogue last = load_col(ep, nn);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const long long r = row0 + 32 * i + 8 * (v / 4) + 4 * q + v % 4;
        if ((mine >> v & 1) && r < M && n + j < N)
          out[r * N + n + j] = finish(sum[v], last);
      }
    }
  }
}

// Few rows: a workgroup owns 32 rows x 32 columns and its eight wavefronts take
// the blocks of 32 k in turn, so that a contraction of a few hundred k is one
// or two trips to memory long, whatever it is wide: W comes straight from
// global memory (no two wavefronts want the same piece of it), and the eight
// partial tiles meet in LDS.
// GATHER 1: a gathered row's channels are a multiple of 32 (a block lies within one
// filter position), 2: of 4.
template <int PL, int GATHER, bool A16, bool WT>
__global__ void __launch_bounds__(512, GATHER == 2 && PL > 1 ? 2 : 4)
    k_nin_planes_splitk(const float *__restrict__ A, const float *__restrict__ W,
                        float *__restrict__ out, long long M, int K, int N,
                        Epilogue ep, GatherSource gs, int nSplits, RowRange rows) {
  M = rows.live(M);
  const unsigned tiles = (unsigned)((M + 31) / 32) * nSplits;
  if (blockIdx.x >= tiles)
    return;
  const unsigned tileOf = xcd_eighth(blockIdx.x, tiles);
  constexpr int ES = A16 ? 2 : 4;
  __shared__ __attribute__((aligned(16))) float sPart[8 * 16 * 64];
  __shared__ int sRules[GATHER ? 32 * GF_MAX_FS : 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, q = lane >> 5;
  const int split = tileOf % nSplits;
  const long long row0 = (long long)(tileOf / nSplits) * 32;
  const int n0 = split * 32;
  const int T = K / 32;
  const unsigned char *const Ab = reinterpret_cast<const unsigned char *>(A);
  const int n = n0 + c < N ? n0 + c : N - 1; // (a column past the end is not stored)
  // this lane's place in a step's eight rows of W, in bytes (the rows' own addresses
  // are the wavefront's)
  const unsigned wLane = WT ? 32u * q : 4u * ((unsigned)(8 * q) * N + n);
  const float *const wRow = WT ? W + (long long)n * K : W;
  struct Block {
    floatx4 a[2][A16 ? 1 : 2];
    float w[2][8];
  };
  long long m = row0 + c;
  m = m < M ? m : M - 1; // rows past the end: read a valid row, store nothing
  auto load_w = [&](Block &b, int t) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        b.w[s][i] = *reinterpret_cast<const float *>(
            reinterpret_cast<const unsigned char *>(wRow + (long long)(32 * t + 16 * s + i) * (WT ? 1 : N)) + wLane);
  };
  auto load_a = [&](Block &b, int t) {
    const unsigned char *row = nullptr;
    if (GATHER == 1) {
      const int f = (int)__umulhi((unsigned)(32 * t), gs.magic); // uniform
      const int rule = sRules[c * gs.fs + f];
      row = (rule >= 0 ? Ab + (long long)rule * gs.nIn * ES : reinterpret_cast<const unsigned char *>(gs.zeros)) +
            (32 * t - f * gs.nIn + 8 * q) * ES;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int h = 0; h < (A16 ? 1 : 2); ++h) {
        const int k = 32 * t + 16 * s + 8 * q + 4 * h;
        b.a[s][h] = GATHER == 1   ? *reinterpret_cast<const floatx4 *>(row + (16 * s + 4 * h) * ES)
                    : GATHER == 2 ? gathered_piece<A16>(Ab, gs, sRules + c * gs.fs, k)
                                  : *reinterpret_cast<const floatx4 *>(Ab + (m * K + k) * ES);
      }
  };
  constexpr int NACC = PL > 1 ? 2 : 1;
  floatx16 acc[NACC];
#pragma unroll
  for (int h = 0; h < NACC; ++h)
#pragma unroll
    for (int v = 0; v < 16; ++v)
      acc[h][v] = 0.f;
  auto compute = [&](const Block &b) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 ap[PL], bp[PL];
      if constexpr (A16) {
        ap[0] = __builtin_bit_cast(bf16x8, b.a[s][0]);
      } else {
        const floatx4 x = b.a[s][0], y = b.a[s][1];
        const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        split8<PL>(v, ap);
      }
      split8<PL>(b.w[s], bp);
#pragma unroll
      for (int x = 0; x < PL; ++x)
#pragma unroll
        for (int y = 0; x + y < PL; ++y) {
          floatx16 &d = acc[x + y == 0 ? 0 : NACC - 1];
          d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ap[x], bp[y], d, 0, 0, 0);
        }
    }
  };

  Block b0, b1;
  const int t0 = wave < T ? wave : T - 1;
  load_w(b0, t0);
  if (GATHER) {
    const long long first = row0 * gs.fs, last = M * gs.fs - 1;
    for (int i = tid; i < 32 * gs.fs; i += 512) {
      const long long r = first + i;
      sRules[i] = gs.rules[r < last ? r : last];
    }
    __syncthreads();
  }
  load_a(b0, t0);
  for (int t = wave; t < T; t += 16) {
    const int t1 = t + 8 < T ? t + 8 : T - 1;
    load_w(b1, t1);
    load_a(b1, t1);
    compute(b0);
    if (t + 8 >= T)
      break;
    const int t2 = t + 16 < T ? t + 16 : T - 1;
    load_w(b0, t2);
    load_a(b0, t2);
    compute(b1);
  }
  // (the lane's numbers anew: the loop has no registers to keep them in)
  const int at = __lane_id(), c1 = at & 31, q1 = at >> 5;
  const ColEpilogue col = load_col(ep, n0 + c1 < N ? n0 + c1 : N - 1);
#pragma unroll
  for (int v = 0; v < 16; ++v)
    sPart[(wave * 16 + v) * 64 + at] = NACC == 2 ? acc[0][v] + acc[NACC - 1][v] : acc[0][v];
  __syncthreads();
  // register v of lane (c, q) is row 8 (v / 4) + 4 q + v % 4; this wavefront's
  // are v = wave and wave + 8
  float sum[2];
  unsigned again = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int v = 8 * h + wave;
    sum[h] = sPart[v * 64 + at];
#pragma unroll
    for (int w = 1; w < 8; ++w)
      sum[h] += sPart[(w * 16 + v) * 64 + at];
    if (doubtful<PL>(sum[h]))
      again |= 1u << v;
  }
  if constexpr (PL == 3) {
    if (__any(again != 0)) {
      const long long m1 = row0 + c1 < M ? row0 + c1 : M - 1;
      const int n1 = n0 + c1 < N ? n0 + c1 : N - 1;
      const floatx16 plain =
          tile_f32<GATHER != 0>(A, gs, sRules + (GATHER ? (int)(m1 - row0) * gs.fs : 0), PlainW{W, WT}, m1, n1, K, N, again);
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (again >> v & 1)
          sum[v / 8] = plain[v];
    }
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int v = 8 * h + wave;
    const int dr = 8 * (v / 4) + 4 * q1 + v % 4;
    if (row0 + dr < M && n0 + c1 < N)
      out[(row0 + dr) * N + n0 + c1] = finish(sum[h], col);
  }
}

// Of the requests a wavefront has made, all but the last N have landed.
template <int N> __device__ __forceinline__ void lines_landed() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N < 63 ? N : 63) : "memory");
}

// The same contraction with both operands through LDS: the rows of A by whole
// lines, W from its image, by requests that need no registers (dma_kilobyte), D - 1
// blocks of 32 k ahead.  k_nin_planes fetches a row 16 bytes a lane, 32 rows to an
// instruction, and a block ahead: layers of some 10000 rows spent their time waiting
// for those loads, and wide ones went through their rows once for every 32 or 64
// columns.  Here a workgroup of RW by CW wavefronts owns 32 MT RW rows x 32 NT CW
// columns, a wavefront 32 MT x 32 NT of them.
//
// A block's slot: its rows, a line (128 bytes) each, whose eight pieces are stored
// rotated by the row (piece ^ row % 8, by what each lane asks for), so that eight
// rows' reads of one piece lie on all banks; then its chunks of the image.  Units,
// splitting under the MFMAs and the order of all sums are k_nin_planes': the same
// bits.  One barrier a block, before its second step's MFMAs: behind it the next
// block may be read and the last one's slot is asked for again.
//
// Straight code that is run once is fetched from L2 by every compute unit: an
// epilogue with a branch an element took 1.1 us a tile, and takes 0.4.
//
// Microseconds, the rows written by a kernel before, k_nin_planes with its image
// (where it takes one) -> here with the image made: three planes, through rules,
// 28400 x 256 x 96 20.6 -> 16.1, 11400 x 384 x 128 17.7 -> 14.4, 6160 x 1280 x 480
// 71 -> 45, 2250 x 1920 x 640 61 -> 43; not gathered 11434 x 512 x 96 30 -> 21,
// 139000 x 128 x 384 136 -> 116; one plane, 41600 x 640 x 320 60 -> 46, 2176 x 2560 x
// 800 46 -> 25, 140000 x 384 x 128 47 -> 37.  With the chip full k_nin_planes' (2, 2)
// tiles of three planes stay ahead on gathered rows: 1.36 M x 1728 x 64 1483 against
// 1797.

// LONG (plain rows): a workgroup goes through several tiles of the same columns, and
// asks for the next one's rows before it is done with one, D - 1 blocks ahead across the
// tiles.  Each tile by itself began with a trip to memory and ended in its stores, 4 of
// the 10 us that one of 128 x 128 x 128 took: 139000 x 128 x 128 55 us -> 37, 400000 x 96 x
// 128 116 -> 73, 139000 x 256 x 192 109 -> 92, 50000 x 320 x 1280 265 -> 244.
//   2: the results go past the caches, which the rows are wanted in (139000 x 128 x 384
// 127 -> 115, and so 95); 1: through them (lines_past_caches).
template <int PL, int MT, int NT, int RW, int CW, int D, bool GATHER, bool A16, int LONG = 0>
__global__ void __launch_bounds__(64 * RW * CW, 2)
    k_nin_lines(const float *__restrict__ A, const unsigned char *__restrict__ image, float *__restrict__ out, long long M,
                int K, int N, Epilogue ep, GatherSource gs, int nSplits, bool byColumns, RowRange rows, PlainW plain) {
  constexpr int WAVES = RW * CW, THREADS = 64 * WAVES;
  constexpr int ROWS = 32 * MT * RW, TW = NT * CW, NW = 32 * TW;
  constexpr int ES = A16 ? 2 : 4, LINE = 32 * ES, LANES = LINE / 16; // a row's part of a block, and lanes that fetch it
  constexpr int A_CHUNKS = ROWS * LINE / 1024, W_CHUNKS = TW * PL * 2;
  constexpr int A_PER = (A_CHUNKS + WAVES - 1) / WAVES, W_PER = (W_CHUNKS + WAVES - 1) / WAVES, PER = A_PER + W_PER;
  constexpr int A_BYTES = A_CHUNKS * 1024, SLOT = (A_CHUNKS + W_CHUNKS) * 1024;
  extern __shared__ __attribute__((aligned(16))) unsigned char sW[]; // [D][SLOT], then the rules
  M = rows.live(M);
  const unsigned rowTiles = (unsigned)((M + ROWS - 1) / ROWS), tiles = rowTiles * nSplits;
  // LONG: the grid is eight times a multiple of nSplits; an XCD has an eighth of the rows
  unsigned longFirst = 0, longStep = 0;
  int mine = 1; // tiles of this workgroup
  if constexpr (LONG) {
    const unsigned x = blockIdx.x & 7, per = gridDim.x >> 3, rem = rowTiles & 7;
    const unsigned group = (blockIdx.x >> 3) / nSplits, count = (rowTiles >> 3) + (x < rem);
    longStep = per / nSplits;
    if (group >= count)
      return;
    mine = (int)((count - group + longStep - 1) / longStep);
    longFirst = x * (rowTiles >> 3) + (x < rem ? x : rem) + group;
  } else {
    if (blockIdx.x >= tiles)
      return;
  }
  const unsigned tileOf = LONG ? 0 : xcd_eighth(blockIdx.x, tiles);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, q = lane >> 5;
  const int cg = wave % CW, rg = wave / CW;
  const int split = LONG ? (blockIdx.x >> 3) % nSplits : byColumns ? tileOf / rowTiles : tileOf % nSplits;
  long long wgRow0 = (long long)(LONG ? longFirst : byColumns ? tileOf % rowTiles : tileOf / nSplits) * ROWS;
  long long row0 = wgRow0 + rg * 32 * MT;
  const int n0 = split * NW + cg * 32 * NT; // this wavefront's columns
  const int T = K / 32;
  int *const sRules = reinterpret_cast<int *>(sW + D * SLOT);
  static_assert(!LONG || !GATHER, "LONG: plain rows");
  const unsigned char *const Ab = reinterpret_cast<const unsigned char *>(A);
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)sW;

  // ---- requests
  const unsigned char *wSrc[W_PER];
  unsigned wDst[W_PER];
  const int lastTile = (N + 31) / 32 - 1;
#pragma unroll
  for (int u = 0; u < W_PER; ++u) {
    int x = wave + WAVES * u;
    x = x < W_CHUNKS ? x : W_CHUNKS - 1; // (past the end: the last one again)
    int tile = split * TW + x / (2 * PL);
    tile = tile < lastTile ? tile : lastTile;
    wSrc[u] = image + ((long long)tile * T * (2 * PL) + x % (2 * PL)) * 1024 + 16 * lane;
    wDst[u] = A_BYTES + x * 1024;
  }
  const unsigned char *rowPtr[A_PER];
  int f = 0, ch = 0;
  // LONG: the tile whose rows are asked for, its first row, and the block of it
  int asked = 0, askedBlock = 0;
  long long askedRow0 = wgRow0;
  // (A16: two rows lie on all banks, so that they are rotated by pairs)
  const int piece = 16 * ((lane % LANES) ^ (A16 ? lane >> 3 & 3 : lane >> 3));
  auto aim = [&]() {
#pragma unroll
    for (int u = 0; u < A_PER; ++u) {
      const int x = wave + WAVES * u;
      const int r = 64 / LANES * (x < A_CHUNKS ? x : A_CHUNKS - 1) + lane / LANES;
      if (GATHER) {
        const int rule = sRules[r * gs.fs + f];
        rowPtr[u] = (rule >= 0 ? Ab + (long long)rule * gs.nIn * ES : reinterpret_cast<const unsigned char *>(gs.zeros)) + piece;
      } else {
        long long m = (LONG ? askedRow0 : wgRow0) + r;
        m = m < M ? m : M - 1;
        rowPtr[u] = Ab + m * K * ES + piece;
      }
    }
  };
  auto fetch_w = [&](int t, int slot, int u) {
    dma_kilobyte(lds0 + slot * SLOT + wDst[u], wSrc[u] + (long long)t * (2 * PL * 1024));
  };
  auto fetch_a = [&](int slot, int u) {
    const int x = wave + WAVES * u;
    dma_kilobyte(lds0 + slot * SLOT + (x < A_CHUNKS ? x : A_CHUNKS - 1) * 1024, rowPtr[u] + ch * ES);
  };
  auto advance = [&]() { // to the next block's rows
    if constexpr (LONG) {
      ++askedBlock;
      if (askedBlock == T) {
        askedBlock = ch = 0;
        askedRow0 += (long long)longStep * ROWS;
        if (++asked < mine)
          aim();
        return;
      }
    }
    ch += 32;
    if (GATHER && ch == gs.nIn) {
      ch = 0;
      if (++f < gs.fs)
        aim();
    }
  };

  // ---- operands
  const unsigned char *const aLane = sW + (rg * 32 * MT + c) * LINE;
  const int swizzle = A16 ? c >> 1 & 3 : c & 7;
  const unsigned char *const wLane = sW + A_BYTES + cg * NT * PL * 2048 + lane * 16;
  floatx4 raw[2];
  unsigned ap[2][PL][4]; // words of an MFMA operand: two k each
  auto read_a = [&](int slot, int u) { // unit u of a block: (step, row tile)
    const unsigned char *const p = aLane + slot * SLOT + (u % MT) * 32 * LINE;
    if constexpr (A16) {
      const uint4 w = *reinterpret_cast<const uint4 *>(p + (((2 * (u / MT) + q) ^ swizzle) * 16));
      ap[u & 1][0][0] = w.x, ap[u & 1][0][1] = w.y, ap[u & 1][0][2] = w.z, ap[u & 1][0][3] = w.w;
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        raw[h] = *reinterpret_cast<const floatx4 *>(p + (((4 * (u / MT) + 2 * q + h) ^ swizzle) * 16));
    }
  };
  auto a_split = [&](int dst, int p) { // a quarter of it
    const floatx4 x = raw[p / 2];
    unsigned w[PL];
    split2<PL>(x[2 * (p % 2)], x[2 * (p % 2) + 1], w);
#pragma unroll
    for (int l = 0; l < PL; ++l) {
      asm volatile("" : "+v"(w[l])); // (here, and not where it is used)
      ap[dst][l][p] = w[l];
    }
  };
  auto operand = [&](int src, int l) {
    return __builtin_bit_cast(bf16x8, uint4{ap[src][l][0], ap[src][l][1], ap[src][l][2], ap[src][l][3]});
  };
  constexpr int BB = NT == 1 ? 2 : 1; // a single tile has no other's MFMAs to be read under
  bf16x8 b[BB][NT][PL];
  auto read_b = [&](int slot, int s, int j) {
#pragma unroll
    for (int l = 0; l < PL; ++l)
      b[s % BB][j][l] = *reinterpret_cast<const bf16x8 *>(wLane + slot * SLOT + ((j * PL + l) * 2 + s) * 1024);
  };

  // ---- prologue
  ColEpilogue col[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + 32 * j + c;
    col[j] = load_col(ep, n < N ? n : N - 1);
  }
  const int first = T < D - 1 ? T : D - 1;
  if (GATHER) {
    const long long begin = wgRow0 * gs.fs, last = M * gs.fs - 1;
    for (int i = tid; i < ROWS * gs.fs; i += THREADS) {
      const long long r = begin + i;
      sRules[i] = gs.rules[r < last ? r : last];
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) // (asked for now: they come with the rules)
    asm volatile("" : "+v"(col[j].pb), "+v"(col[j].slope));
  __syncthreads();
  aim();
#pragma unroll 1
  for (int t = 0; t < first; ++t) {
#pragma unroll
    for (int u = 0; u < W_PER; ++u)
      fetch_w(t, t, u);
#pragma unroll
    for (int u = 0; u < A_PER; ++u)
      fetch_a(t, u);
    advance();
  }
  if (first == D - 1)
    lines_landed<PER *(D - 2)>();
  else
    lines_landed<0>();
  barrier_lds();

  constexpr int NACC = PL > 1 ? 2 : 1;
  floatx16 acc[NACC][MT][NT];
#pragma unroll
  for (int h = 0; h < NACC; ++h)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[h][i][j][v] = 0.f;

  int last = D - 1, cur = 0, next = 1; // slots of blocks t - 1, t and t + 1
  read_a(0, 0);
#pragma unroll
  for (int j = 0; j < NT; ++j)
    read_b(0, 0, j);
  if (!A16) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
      a_split(0, p);
    read_a(0, 1);
  }

  constexpr int PRODUCTS = PL * (PL + 1) / 2;
  auto tile = [&](int s, int i, int j, int src) {
#pragma unroll
    for (int x = 0; x < PL; ++x)
#pragma unroll
      for (int y = 0; x + y < PL; ++y) {
        floatx16 &d = acc[x + y == 0 ? 0 : NACC - 1][i][j];
        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(operand(src, x), b[s % BB][j][y], d, 0, 0, 0);
      }
  };
  // vector instructions to go with an MFMA: the splitting, dealt out to all tiles but the first
  constexpr int VALU = ((PL == 1 ? 4 : PL == 2 ? 24 : 44) + PRODUCTS * (NT > 1 ? NT - 1 : 1) - 1) / (PRODUCTS * (NT > 1 ? NT - 1 : 1)) + 1;
  auto deal = [&]() {
#pragma unroll
    for (int i = 0; i < PRODUCTS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x320, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int UNITS = 2 * MT, SECOND = MT; // the first unit of the second step: the barrier before it
  bool ahead = false;                        // LONG: not this workgroup's first tile
  auto block = [&](int t, auto steady) {     // steady: with a block to ask for
    const bool more = steady || t + D - 1 < T; // uniform
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int s = u / MT, i = u % MT, src = u & 1;
      if (u == SECOND) {
        // The next block has landed (those asked for behind it may be under way), and
        // nobody reads the last one any more.
        if (!(steady || t + D - 1 <= T)) // uniform
          lines_landed<0>();
        else if (LONG && ahead && t + 1 <= D - 2) // asked for before the last tile's results were stored
          lines_landed<PER *(D - 3) + MT * NT * 16>();
        else
          lines_landed<PER *(D - 3)>();
        asm volatile("s_barrier" ::: "memory");
      }
      if (A16) // (where the last unit but one's operand was)
        read_a(u + 1 < UNITS ? cur : next, (u + 1) % UNITS);
      else if (MT == 1 && u == SECOND)
        read_a(next, 0);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (NT == 1) {
          if (i == MT - 1)
            read_b(s ? next : cur, s ^ 1, 0);
        }
        tile(s, i, j, src);
        if (NT > 1 && i == MT - 1)
          read_b(s ? next : cur, s ^ 1, j);
#pragma unroll
        for (int p = 0; p < (A16 ? 0 : 4); ++p)
          if (j == (NT == 1 || !(MT == 1 && u == SECOND) ? p * NT / 4 : 1 + p * (NT - 1) / 4))
            a_split(src ^ 1, p);
        if (!A16 && j == NT - 1) { // (split: its registers take the next but one)
          if (MT > 1)
            read_a(u + 2 < UNITS ? cur : next, (u + 2) % UNITS);
          else if (u == SECOND)
            read_a(next, 1);
        }
        deal();
        if (more && u >= SECOND) {
          constexpr int G = MT * NT;
          const int g = i * NT + j;
#pragma unroll
          for (int x = g * PER / G; x < (g + 1) * PER / G; ++x) {
            if (x < W_PER)
              fetch_w(LONG ? askedBlock : t + D - 1, last, x);
            else
              fetch_a(last, x - W_PER);
          }
        }
      }
    }
    if (more)
      advance();
    last = cur, cur = next, next = next == D - 1 ? 0 : next + 1;
  };
  for (int at = 0;;) { // the tiles
  int t = 0;
#pragma unroll 1
  for (; t + (LONG && at + 1 < mine ? 0 : D - 1) < T; ++t)
    block(t, std::true_type());
#pragma unroll 1
  for (; t < T; ++t)
    block(t, std::false_type());

  // ---- epilogue: register v of a tile is row 8 (v / 4) + 4 q + v % 4
  int lane = tid & 63;
  if constexpr (LONG) // (what follows from it is not kept from one tile to the next)
    asm volatile("" : "+v"(lane));
  const int c = lane & 31, q = lane >> 5;
  if constexpr (NACC == 2) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[0][i][j][v] += acc[NACC - 1][i][j][v];
  }
  unsigned long long again = 0; // results to be taken from the operands themselves
  if constexpr (PL == 3) {
    float none[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}; // 0 sum: NaN for a sum that is not finite
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          none[v % 8] = fmaf(acc[0][i][j][v], 0.f, none[v % 8]);
    if (((none[0] + none[1]) + (none[2] + none[3])) + ((none[4] + none[5]) + (none[6] + none[7])) != 0.f) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (doubtful<PL>(acc[0][i][j][v]))
              again |= 1ull << ((i * NT + j) * 16 + v);
    }
  }
  {
    // (what lies past the last row, or in no column, is past the buffer's end: not
    // stored, without a branch to each)
    const long long left = ((M - row0) * N - n0) * 4;
    const __amdgpu_buffer_rsrc_t to =
        __builtin_amdgcn_make_buffer_rsrc(out + row0 * N + n0, 0, (int)(left < 0 ? 0 : left < 0x40000000 ? left : 0x40000000),
                                          0x00020000);
    const unsigned pitch = 4u * (unsigned)N;
    unsigned at[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
      at[j] = n0 + 32 * j + c < N ? (unsigned)(4 * q) * pitch + 128u * j + 4u * c : 0x80000000u;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(finish(acc[0][i][j][v], col[j])), to, at[j], 0, LONG == 2 ? 2 : 0);
          at[j] += v % 4 == 3 ? 5 * pitch : pitch;
        }
  }
  if constexpr (PL == 3) {
    if (__any(again != 0))
#pragma unroll 1
    for (int e = 0; e < MT * NT; ++e) {
      const unsigned mine = (unsigned)(again >> (16 * e)) & 0xffffu;
      if (!__any(mine != 0))
        continue;
      const int i = e / NT, j = e % NT;
      long long m = row0 + 32 * i + c;
      m = m < M ? m : M - 1;
      const int n = n0 + 32 * j + c, nn = n < N ? n : N - 1;
      const floatx16 exact = tile_f32<GATHER>(A, gs, sRules + (m - wgRow0) * gs.fs, plain, m, nn, K, N, mine);
      const ColEpilogue last = load_col(ep, nn);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const long long r = row0 + 32 * i + 8 * (v / 4) + 4 * q + v % 4;
        if ((mine >> v & 1) && r < M && n < N)
          out[r * N + n] = finish(exact[v], last);
      }
    }
  }
  if (!LONG || ++at == mine)
    return;
  if constexpr (LONG) {
    wgRow0 += (long long)longStep * ROWS, row0 += (long long)longStep * ROWS;
    ahead = true;
#pragma unroll
    for (int h = 0; h < NACC; ++h)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            acc[h][i][j][v] = 0.f;
    // (the first operands anew: they need no registers while results are stored)
    read_a(cur, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      read_b(cur, 0, j);
#pragma unroll
    for (int p = 0; p < 4; ++p)
      a_split(0, p);
    read_a(cur, 1);
  }
  }
}

// The split contraction where there are more rows: 64 rows x 64 columns a workgroup, whose
// eight wavefronts take the blocks of 32 k in turn, as k_nin_planes_splitk's do, with the same
// sums in the same order: the same bits.  A wavefront owns all of the tile, so that no two
// want the same piece of A or W: rows come into a ring of its own in LDS by whole lines (each
// sixteen bytes through the rule of its own position), W straight into registers, from
// k_nin_lines' image or as it stands, and there is no barrier between the first block and
// the last.  The eight partial tiles meet in the rings' place.
// What bounds it: a block is 20 KB for 48 MFMAs, and a wavefront waits once a step for what
// it asked for a step before: eight blocks take 2.5 us where the MFMAs are 1.4.  The tiles of
// k_nin_lines move half of that and leave compute units idle at so few rows: split_rows has
// both sides' times.  1037 x 2560 x 800 49 -> 32 us (W as it stands: 37), 16000 x 1728 x 64 36
// -> 24, channels in other than 32s 1037 x 1600 x 800 54 -> 26; 61 images 354 -> 337.
enum { S64_IMAGE, S64_PLAIN, S64_TURNED }; // W: its image, [K x N], [N x K]
template <int PL, bool GATHER, int WM>
__global__ void __launch_bounds__(512, 2)
    k_nin_split64(const float *__restrict__ A, const unsigned char *__restrict__ image, float *__restrict__ out, long long M,
                  int K, int N, Epilogue ep, GatherSource gs, int nSplits, bool byColumns, RowRange rows, PlainW plain) {
  constexpr int SLOT = 8192, RING = 2 * SLOT;
  extern __shared__ __attribute__((aligned(16))) unsigned char sW[]; // [8][RING], then the rules
  M = rows.live(M);
  const unsigned rowTiles = (unsigned)((M + 63) / 64), tiles = rowTiles * nSplits;
  if (blockIdx.x >= tiles)
    return;
  const unsigned tileOf = xcd_eighth(blockIdx.x, tiles);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, q = lane >> 5;
  const int split = byColumns ? tileOf / rowTiles : tileOf % nSplits;
  const long long row0 = (long long)(byColumns ? tileOf % rowTiles : tileOf / nSplits) * 64;
  const int n0 = split * 64;
  const int T = K / 32;
  int *const sRules = reinterpret_cast<int *>(sW + 8 * RING);
  unsigned char *const ring = sW + wave * RING;
  const unsigned ldsRing =
      __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring);
  const unsigned char *const Ab = reinterpret_cast<const unsigned char *>(A);

  // ---- W: a step's chunks of the image, or its eight k of a lane's two columns
  const int lastTile = (N + 31) / 32 - 1;
  const unsigned char *wSrc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tile = 2 * split + j < lastTile ? 2 * split + j : lastTile;
    wSrc[j] = image + (long long)tile * T * (2 * PL * 1024) + 16 * lane;
  }
  constexpr int WS = WM == S64_IMAGE ? 2 : 1;
  bf16x8 w[WS][2][PL]; // of a step
  float wRaw[2][WM == S64_IMAGE ? 1 : 8]; // of the next one
  auto load_w = [&](int t, int s) {
    t = t < T ? t : T - 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (WM == S64_IMAGE) {
#pragma unroll
        for (int l = 0; l < PL; ++l)
          w[s % WS][j][l] = *reinterpret_cast<const bf16x8 *>(wSrc[j] + ((long long)t * (2 * PL) + 2 * l + s) * 1024);
      } else {
        const int n = n0 + 32 * j + c < N ? n0 + 32 * j + c : N - 1, k = 32 * t + 16 * s + 8 * q;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          wRaw[j][i % (WM == S64_IMAGE ? 1 : 8)] = plain.W[WM == S64_TURNED ? (long long)n * K + k + i : (long long)(k + i) * N + n];
      }
    }
  };
  auto take_w = [&](int t, int s) { // the step whose W was asked for last, and the next one's asked for
    if constexpr (WM == S64_IMAGE) {
      load_w(t, s);
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        split8<PL>(reinterpret_cast<const float(&)[8]>(wRaw[j]), w[0][j]);
      load_w(t, s);
    }
  };
  // ---- rows: eight of them, a line each, to a request; a line's pieces are rotated by the row
  const int piece = (lane & 7) ^ (lane >> 3);
  int f = 0;         // GATHER: the position of this lane's piece, and where in a row of it
  unsigned in = 0;
  auto aim = [&](int t) {
    t = t < T ? t : T - 1;
    const unsigned k = 32 * t + 4 * piece;
    f = GATHER ? (int)__umulhi(k, gs.magic) : 0;
    in = 4 * (k - (GATHER ? f * gs.nIn : 0));
  };
  auto fetch = [&](int slot, int u) { // of the block aimed at
    int r = 8 * u + (lane >> 3);
    asm volatile("" : "+v"(r)); // (no address is kept from block to block)
    unsigned long long from;
    if (GATHER) {
      const int rule = sRules[r * gs.fs + f];
      from = rule >= 0 ? (unsigned long long)(uintptr_t)Ab + (unsigned long long)(unsigned)rule * (unsigned)(gs.nIn * 4)
                       : (unsigned long long)(uintptr_t)gs.zeros;
    } else {
      const long long m = row0 + r < M ? row0 + r : M - 1; // rows past the end: read a valid row, store nothing
      from = (unsigned long long)(uintptr_t)Ab + (unsigned long long)m * (unsigned)K * 4;
    }
    dma_kilobyte(ldsRing + slot * SLOT + u * 1024, reinterpret_cast<const unsigned char *>(from + in));
  };

  // ---- operands
  floatx4 raw[2];
  unsigned ap[2][PL][4]; // words of an MFMA operand: two k each
  auto read_a = [&](int slot, int u) { // unit u of a block: (step, row tile)
    const unsigned char *const p = ring + slot * SLOT + (u % 2) * 4096 + c * 128;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      raw[h] = *reinterpret_cast<const floatx4 *>(p + (((4 * (u / 2) + 2 * q + h) ^ (c & 7)) * 16));
  };
  auto a_split = [&](int dst, int p) { // a quarter of it
    const floatx4 x = raw[p / 2];
    unsigned v[PL];
    split2<PL>(x[2 * (p % 2)], x[2 * (p % 2) + 1], v);
#pragma unroll
    for (int l = 0; l < PL; ++l) {
      asm volatile("" : "+v"(v[l])); // (here, and not where it is used)
      ap[dst][l][p] = v[l];
    }
  };
  auto operand = [&](int src, int l) {
    return __builtin_bit_cast(bf16x8, uint4{ap[src][l][0], ap[src][l][1], ap[src][l][2], ap[src][l][3]});
  };
  constexpr int NACC = PL > 1 ? 2 : 1;
  floatx16 acc[NACC][2][2];
#pragma unroll
  for (int h = 0; h < NACC; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[h][i][j][v] = 0.f;

  // ---- the blocks
  load_w(wave, 0);
  if (GATHER) {
    const long long first = row0 * gs.fs, last = M * gs.fs - 1;
    for (int i = tid; i < 64 * gs.fs; i += 512) {
      const long long r = first + i;
      sRules[i] = gs.rules[r < last ? r : last];
    }
    __syncthreads();
  }
  if (wave < T) {
    aim(wave);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      fetch(0, u);
    lines_landed<0>();
    read_a(0, 0);
#pragma unroll
    for (int p = 0; p < 4; ++p)
      a_split(0, p);
    read_a(0, 1);
    int cur = 0;
#pragma unroll 1
    for (int t = wave; t < T; t += 8) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = u / 2, i = u % 2, src = u & 1;
        if (u == 2) // the next block's rows, and this one's other W
          lines_landed<0>();
        if (u == 0)
          take_w(t, 1);
        if (u == 2)
          take_w(t + 8, 0);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
          for (int x = 0; x < PL; ++x)
#pragma unroll
            for (int y = 0; x + y < PL; ++y) {
              floatx16 &d = acc[x + y == 0 ? 0 : NACC - 1][i][j];
              d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(operand(src, x), w[s % WS][j][y], d, 0, 0, 0);
            }
#pragma unroll
          for (int p = 2 * j; p < 2 * j + 2; ++p)
            a_split(src ^ 1, p);
          if (j == 1) // (split: its registers take the next but one)
            read_a(u + 2 < 4 ? cur : cur ^ 1, (u + 2) % 4);
          if (s == 0) { // (the next block's rows: the last one's place)
            if (u == 0 && j == 0)
              aim(t + 8);
            fetch(cur ^ 1, 4 * i + 2 * j);
            fetch(cur ^ 1, 4 * i + 2 * j + 1);
          }
#pragma unroll
          for (int x = 0; x < PL * (PL + 1) / 2; ++x) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x320, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, PL == 3 ? 8 : 16, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      cur ^= 1;
    }
  }
  lines_landed<0>(); // (nothing is on its way into the rings)

  // ---- the partial tiles
  float *const sPart = reinterpret_cast<float *>(sW); // [8][64][64]: wavefront, register, lane
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        sPart[(wave * 64 + (2 * i + j) * 16 + v) * 64 + lane] =
            NACC == 2 ? acc[0][i][j][v] + acc[NACC - 1][i][j][v] : acc[0][i][j][v];
  ColEpilogue col[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + 32 * j + c;
    col[j] = load_col(ep, n < N ? n : N - 1);
  }
  __syncthreads();
  // register v of tile (i, j), lane (c, q), is row 32 i + 8 (v / 4) + 4 q + v % 4; this
  // wavefront's are v = wave and wave + 8 of every tile
  unsigned again[4];
  float sum[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    again[e] = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int v = 8 * h + wave;
      float x = sPart[(e * 16 + v) * 64 + lane];
#pragma unroll
      for (int k = 1; k < 8; ++k)
        x += sPart[(k * 64 + e * 16 + v) * 64 + lane];
      sum[2 * e + h] = x;
      if (doubtful<PL>(x))
        again[e] |= 1u << v;
    }
  }
  if constexpr (PL == 3) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (__any(again[e] != 0)) {
        const int r = 32 * (e / 2) + c;
        const long long m = row0 + r < M ? row0 + r : M - 1;
        const int n = n0 + 32 * (e % 2) + c < N ? n0 + 32 * (e % 2) + c : N - 1;
        const floatx16 exact = tile_f32<GATHER>(A, gs, sRules + (GATHER ? (int)(m - row0) * gs.fs : 0), plain, m, n, K, N, again[e]);
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (again[e] >> v & 1)
            sum[2 * e + v / 8] = exact[v];
      }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int v = 8 * h + wave;
      const long long r = row0 + 32 * (e / 2) + 8 * (v / 4) + 4 * q + v % 4;
      const int n = n0 + 32 * (e % 2) + c;
      if (r < M && n < N)
        out[r * N + n] = finish(sum[2 * e + h], col[e % 2]);
    }
}

// Long contractions of bf16 rows through rules, one plane, with the chip full.  A wavefront
// owns 64 rows x 32 NT columns: six LDS reads to eight MFMAs (NT 4), where a tile of rows
// to four of columns reads five to four, all that LDS gives while the pipe is busy, and
// fetched its rows 32 to an instruction, all that the address unit does.  Rows come into
// LDS by requests of 16 rows' 64 bytes, into a ring of the wavefront's own, so that a
// block's place is asked for again as soon as it has been read, without a barrier: they
// have one and a half blocks' time.  W comes from k_nin_lines' image, a ring for the
// workgroup, one barrier a block.  A wavefront's rules come four positions at a time,
// while the four before are used.  A step's operands are read under the step before; sums
// in k_nin_planes' order: the same bits.
// LDS: the rows' rings, W's, the rules (two sets of four positions).
//
// Microseconds with the rounding of the rows and the image, k_nin_planes -> here: 595610 x
// 2592 x 128 423 -> 384, x 1728 x 64 225 -> 185; 389361 x 3456 x 96 336 -> 257; 116482 x
// 1728 x 96 73 -> 56; 176025 x 864 x 192 102 -> 87 (k_nin_lines).  Of the first 16 % is
// power: with zeros for data 367 -> 322.  The pipe is busy in 54 % of the cycles at 1.88 GHz
// (46 before); without its requests the loop takes 290 of 358, and half of the rows' do not
// change it by more than 6 %.  Eight wavefronts to a workgroup, half of W's requests: 387.
constexpr int ROWS16_WAVES = 4;
template <int NT>
__global__ void __launch_bounds__(64 * ROWS16_WAVES, 2)
    k_nin_rows16(const unsigned char *__restrict__ A, const unsigned char *__restrict__ image, float *__restrict__ out,
                 long long M, int K, int N, Epilogue ep, GatherSource gs, int nSplits, RowRange rows) {
  constexpr int WAVES = ROWS16_WAVES, MT = 2, D = 3, ROWS = 32 * MT * WAVES;
  constexpr int A_BLOCK = 32 * MT * 64, W_BLOCK = NT * 2048; // of a wavefront, of the workgroup
  constexpr int A_PER = A_BLOCK / 1024, W_PER = (2 * NT + WAVES - 1) / WAVES;
  extern __shared__ __attribute__((aligned(16))) unsigned char sW[];
  M = rows.live(M);
  const unsigned tiles = (unsigned)((M + ROWS - 1) / ROWS) * nSplits;
  if (blockIdx.x >= tiles)
    return;
  const unsigned tileOf = xcd_eighth(blockIdx.x, tiles);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, q = lane >> 5;
  const int split = tileOf % nSplits;
  const long long row0 = (long long)(tileOf / nSplits) * ROWS + wave * 32 * MT;
  const int n0 = split * 32 * NT;
  const int T = K / 32, perPosition = gs.nIn / 32;
  unsigned char *const sA = sW + wave * D * A_BLOCK, *const sB = sW + WAVES * D * A_BLOCK;
  int *const sRules = reinterpret_cast<int *>(sB + D * W_BLOCK) + wave * 2 * 128 * MT;
  auto lds_at = [](const void *p) {
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const unsigned char *)p;
  };
  const unsigned ldsA = __builtin_amdgcn_readfirstlane(lds_at(sA)), ldsB = __builtin_amdgcn_readfirstlane(lds_at(sB)),
                 ldsRules = __builtin_amdgcn_readfirstlane(lds_at(sRules));

  // ---- requests
  const unsigned char *wSrc[W_PER];
  const int lastTile = (N + 31) / 32 - 1;
#pragma unroll
  for (int u = 0; u < W_PER; ++u) {
    int x = wave + WAVES * u;
    x = x < 2 * NT ? x : 2 * NT - 1; // (past the end: the last one again)
    int tile = split * NT + x / 2;
    tile = tile < lastTile ? tile : lastTile;
    wSrc[u] = image + ((long long)tile * T * 2 + x % 2) * 1024 + 16 * lane;
  }
  auto fetch_w = [&](int t, int slot, int u) {
    const int x = wave + WAVES * u;
    dma_kilobyte(ldsB + slot * W_BLOCK + (x < 2 * NT ? x : 2 * NT - 1) * 1024, wSrc[u] + (long long)t * 2048);
  };
  // sixteen rows' rules of four positions, a word a lane (rows and positions past the end:
  // the last ones)
  auto fetch_rules = [&](int group, int u) {
    long long m = row0 + 16 * u + lane / 4;
    m = m < M ? m : M - 1;
    const int f = 4 * group + lane % 4;
    dma_words(ldsRules + ((group & 1) * 2 * MT + u) * 256, gs.rules + m * gs.fs + (f < gs.fs ? f : gs.fs - 1));
  };
  // (two rows lie on 32 banks and four on all: a row's four pieces are rotated by pairs of
  // rows, and again every eight)
  const int piece = 16 * ((lane & 3) ^ (lane >> 3 & 3) ^ (lane >> 5));
  const unsigned char *rowPtr[A_PER];
  int f = 0, ch = 0; // the block to ask for
  int rule[A_PER];
  auto look_up = [&]() { // (rules that have landed; before the first block of a position)
#pragma unroll
    for (int u = 0; u < A_PER; ++u)
      rule[u] = sRules[((f >> 2 & 1) * 2 * MT + u) * 64 + (lane & ~3) + (f & 3)];
  };
  auto aim = [&]() {
#pragma unroll
    for (int u = 0; u < A_PER; ++u)
      asm volatile("" : "+v"(rule[u])); // (all of them waited for at once)
#pragma unroll
    for (int u = 0; u < A_PER; ++u) {
      const unsigned long long from = (unsigned long long)(uintptr_t)A + (unsigned long long)(unsigned)rule[u] * (unsigned)(gs.nIn * 2);
      rowPtr[u] = reinterpret_cast<const unsigned char *>(rule[u] >= 0 ? from : (unsigned long long)(uintptr_t)gs.zeros) + piece;
    }
    // (a quarter of the next four, ahead of the rows: landed when all but those have)
    if (4 * (f / 4 + 1) < gs.fs)
      fetch_rules(f / 4 + 1, f & 3);
  };
  auto fetch_a = [&](int slot, int u) {
    dma_kilobyte(ldsA + slot * A_BLOCK + u * 1024, rowPtr[u] + ch * 64);
  };
  auto advance = [&]() {
    if (++ch == perPosition)
      ch = 0, ++f;
  };

  // ---- operands
  const unsigned char *const aLane = sA + c * 64;
  const int swizzle = (c >> 1 & 3) ^ (c >> 3 & 1);
  const unsigned char *const wLane = sB + lane * 16;
  bf16x8 a[2][MT], b[2][NT]; // of a step
  auto read = [&](int slot, int s, int x) { // the x'th operand of a step
    if (x < MT)
      a[s][x] = *reinterpret_cast<const bf16x8 *>(aLane + slot * A_BLOCK + x * 2048 + (((2 * s + q) ^ swizzle) * 16));
    else if (x < MT + NT)
      b[s][x - MT] = *reinterpret_cast<const bf16x8 *>(wLane + slot * W_BLOCK + ((x - MT) * 2 + s) * 1024);
  };

  // ---- prologue
  ColEpilogue col[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + 32 * j + c;
    col[j] = load_col(ep, n < N ? n : N - 1);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) // (asked for now: nothing the compiler waits for is left for the loop)
    asm volatile("" : "+v"(col[j].pb), "+v"(col[j].slope));
#pragma unroll
  for (int u = 0; u < 2 * MT; ++u)
    fetch_rules(0, u);
#pragma unroll
  for (int t = 0; t < D - 1; ++t) // (T is at least two)
#pragma unroll
    for (int u = 0; u < W_PER; ++u)
      fetch_w(t, t, u);
  lines_landed<(D - 1) * W_PER>();
#pragma unroll 1
  for (int t = 0; t < D && t < T; ++t) {
    if (ch == 0) {
      look_up();
      aim();
    }
#pragma unroll
    for (int u = 0; u < A_PER; ++u)
      fetch_a(t, u);
    advance();
  }
  lines_landed<0>();
  barrier_lds();

  floatx16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[i][j][v] = 0.f;
  int cur = 0, next = 1, last = 2; // slots of blocks t, t + 1 and t - 1 (or t + 2)
#pragma unroll
  for (int x = 0; x < MT + NT; ++x)
    read(0, 0, x);

  constexpr int G = MT * NT, SPREAD = G / 4; // MFMAs of a step; the next step's operands are read behind the first of them
  auto step = [&](int s, int slot, auto &&between) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int i = g / NT, j = g % NT;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s][i], b[s][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      read(slot, s ^ 1, g);
      if (g == G - 1)
#pragma unroll
        for (int x = G; x < MT + NT; ++x)
          read(slot, s ^ 1, x);
      between(g);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // A block's requests, among the MFMAs: in its second step the W of block t + 2 and the
  // first half of block t + 3's rows, in the next block's first step the other half.
  auto block = [&](int t, auto steady) { // steady: with blocks to ask for
    const bool rest = steady || t + D - 1 < T; // uniform: the last block's other half
    const int before = last;
    step(0, cur, [&](int g) {
#pragma unroll
      for (int u = A_PER / 2; u < A_PER; ++u)
        if (g == (u - A_PER / 2) * SPREAD && rest && t > 0)
          fetch_a(before, u);
      if (g == SPREAD * A_PER / 2 && rest && t > 0)
        advance();
    });
    // Of what this wavefront has asked for, all but the rows of block t + 2 has landed,
    // and behind the barrier the others' parts of block t + 1's W too; nobody reads
    // block t - 1's any more, whose place block t + 2's takes.
    if (steady)
      lines_landed<A_PER>();
    else
      lines_landed<0>();
    asm volatile("s_barrier" ::: "memory");
    const bool more = steady || t + D < T, turn = more && ch == 0; // uniform
    if (turn)
      look_up();
    step(1, next, [&](int g) {
#pragma unroll
      for (int u = 0; u < W_PER; ++u)
        if (g == u * SPREAD && (steady || t + 2 < T))
          fetch_w(t + 2, last, u);
      // (this block's rows are in registers since this step's first MFMAs: its place is
      // asked for again)
      if (g == G / 2 - 1 && turn)
        aim();
#pragma unroll
      for (int u = 0; u < A_PER / 2; ++u)
        if (g == G / 2 + u * SPREAD && more)
          fetch_a(cur, u);
    });
    const int was = cur;
    cur = next, next = last, last = was;
  };
  int t = 0;
#pragma unroll 1
  for (; t + D < T; ++t)
    block(t, std::true_type());
#pragma unroll 1
  for (; t < T; ++t)
    block(t, std::false_type());

  // ---- epilogue: register v of a tile is row 8 (v / 4) + 4 q + v % 4
  // (what lies past the last row, or in no column, is past the buffer's end: not stored)
  const long long left = ((M - row0) * N - n0) * 4;
  const __amdgpu_buffer_rsrc_t to =
      __builtin_amdgcn_make_buffer_rsrc(out + row0 * N + n0, 0, (int)(left < 0 ? 0 : left < 0x40000000 ? left : 0x40000000),
                                        0x00020000);
  const unsigned pitch = 4u * (unsigned)N;
  unsigned at[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    at[j] = n0 + 32 * j + c < N ? (unsigned)(4 * q) * pitch + 128u * j + 4u * c : 0x80000000u;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(finish(acc[i][j][v], col[j])), to, at[j], 0, 0);
        at[j] += v % 4 == 3 ? 5 * pitch : pitch;
      }
}

// The image of W that k_nin_planes reads: for every slice of 32 NT
// columns and every block of 32 k what w_store leaves in LDS, in that order.
template <int PL, int NT>
__global__ void __launch_bounds__(256)
    k_planes_image(const float *__restrict__ W, unsigned char *__restrict__ image,
                   int K, int N, int nSplits) {
  constexpr int NW = 32 * NT, BUF_BYTES = PL * 2 * NT * 1024;
  const int T = K / 32;
  const long long item = (long long)blockIdx.x * 256 + threadIdx.x; // (slice, block, 8 k, column)
  if (item >= (long long)nSplits * T * 4 * NW)
    return;
  const int x = (int)(item % (4 * NW));
  const long long st = item / (4 * NW); // slice * T + block
  const int t = (int)(st % T), split = (int)(st / T);
  const int kg = x / NW, tile = (x % NW) / 32, cc = x % 32;
  int n = split * NW + NT * cc + tile;
  n = n < N ? n : N - 1;
  const float *const src = W + (long long)(32 * t + 8 * kg) * N + n;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    v[i] = src[(long long)i * N];
  bf16x8 p[PL];
  split8<PL>(v, p);
#pragma unroll
  for (int l = 0; l < PL; ++l)
    *reinterpret_cast<bf16x8 *>(image + st * BUF_BYTES + l * 2 * NT * 1024 + (kg / 2) * NT * 1024 + tile * 1024 +
                                (kg & 1) * 512 + cc * 16) = p[l];
}

__global__ void __launch_bounds__(256) k_weight_images(ImageList l) { weight_images_block(l, blockIdx.x); }
// What k_nin_lines takes: three planes or one, blocks within one filter position, 64
// rows of the output within the gigabyte that its stores reach (columns that there are
// none of lie from 2 GB on, and have to stay there).
static bool lines_shape(int planes, int K, int N, int nIn) {
  return planes != 2 && scn_planes_shape(K) && nIn % 32 == 0 && N <= 1 << 22;
}

// False: convert on the way instead -- the stream is being captured (a graph may
// be replayed beside the context's own calls, whose weights the room holds), or
// the context has no such room.
static bool planes_image(scn_ctx *ctx) {
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(ctx->stream, &capturing) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return ctx->d_image && capturing == hipStreamCaptureStatusNone;
}

// Blocks ahead: two where the registers allow it (a wavefront alone on its SIMD
// waits for the trip to L2 in every block otherwise: one tile, three planes at
// one workgroup a compute unit 0.79 -> 0.64 us a block; with three planes of
// wider tiles it spills and loses).
constexpr int planes_depth(int PL, int MT, int NT) {
  return PL * MT * NT <= 4 || (PL < 3 && MT == 1) ? 2 : 1;
}
// (W_STREAM: gathered rows, with one plane bf16 ones.  W_IMAGE: gathered rows, with
// two planes any; k_nin_lines takes the others.)
template <int PL, int MT, int NT, int WM, bool FINE = false, int WAVES = 4>
static int launch_planes(scn_ctx *ctx, const float *A, const float *W,
                         float *out, long long M, int K, int N,
                         const Epilogue &ep, const GatherSource *gs, bool a16, const RowRange &rows) {
  const int nSplits = scn_ceil_div(N, 32 * NT);
  const size_t lds = (size_t)(WM == W_STREAM ? 3 : 2) * PL * 2 * NT * 1024 +
                     (gs ? (size_t)32 * WAVES * MT * gs->fs * 4 : 0);
  constexpr int G = FINE ? 2 : 1, PD = planes_depth(PL, MT, NT);
  // (what a launch may ask for without saying so: saying it costs 0.1 ms and more a kernel)
  SCN_REQUIRE(lds <= 64 * 1024, SCN_ERR_ARG, "planes: %d filter positions", gs ? gs->fs : 0);
  const PlainW plain = {W, 0};
  constexpr bool GATHERED = WM == W_STREAM || (WM == W_IMAGE && PL != 2);
  SCN_REQUIRE(gs || !GATHERED, SCN_ERR_ARG, "planes: no rules");
  if (WM != W_PLAIN) {
    const long long items = (long long)nSplits * (K / 32) * 4 * 32 * NT;
    hipLaunchKernelGGL((k_planes_image<PL, NT>), dim3(scn_ceil_div(items, 256)), dim3(256), 0, ctx->stream, W, ctx->d_image,
                       K, N, nSplits);
    W = reinterpret_cast<const float *>(ctx->d_image);
  }
  const dim3 grid((unsigned)(scn_ceil_div(M, 32 * WAVES * MT) * (long long)nSplits));
#define SCN_PLANES_GO(G, H, src)                                               \
  hipLaunchKernelGGL((k_nin_planes<PL, MT, NT, PD, G, H, WM, WAVES>), grid,   \
                     dim3(64 * WAVES), lds, ctx->stream, A, W, out, M, K, N,   \
                     ep, src, nSplits, rows, plain)
  if constexpr (!GATHERED)
    if (!gs) {
      SCN_PLANES_GO(0, false, GatherSource());
      return SCN_OK;
    }
  if (WM == W_STREAM || (PL == 1 && a16))
    SCN_PLANES_GO(G, PL == 1, *gs);
  else if constexpr (WM != W_STREAM)
    SCN_PLANES_GO(G, false, *gs);
#undef SCN_PLANES_GO
  return SCN_OK;
}
static int weight_images(scn_ctx *ctx, const ImageList &l) {
  if (l.firstBlock[l.count] == 0)
    return SCN_OK;
  hipLaunchKernelGGL(k_weight_images, dim3(l.firstBlock[l.count]), dim3(256), 0, ctx->stream, l);
  return SCN_OK;
}
static void add_image(ImageList &l, const float *W, unsigned char *image, int planes, int K, int N, int fs) {
  const int i = l.count++;
  l.W[i] = W, l.image[i] = image, l.K[i] = K, l.N[i] = N, l.fs[i] = fs, l.planes[i] = planes;
  l.firstBlock[i + 1] = l.firstBlock[i] + (unsigned)scn_ceil_div((int64_t)K / 8 * ((N + 31) / 32 * 32), 256);
}
template <int PL, int MT, int NT, int RW, int CW, int D, bool A16 = false>
static int launch_lines(scn_ctx *ctx, const float *A, const float *W, float *out, long long M, int K, int N,
                        const Epilogue &ep, const GatherSource *gs, bool wT, const RowRange &rows,
                        const unsigned char *image) {
  if (!image) {
    ImageList l;
    l.count = 0, l.firstBlock[0] = 0;
    add_image(l, W, ctx->d_image, PL, K, N, wT ? -1 : 0);
    SCN_TRY(weight_images(ctx, l));
    image = ctx->d_image;
  }
  constexpr int ROWS = 32 * MT * RW, COLUMNS = 32 * NT * CW;
  const size_t lds = (size_t)D * (ROWS / (A16 ? 16 : 8) + NT * CW * PL * 2) * 1024 + (gs ? (size_t)ROWS * gs->fs * 4 : 0);
  SCN_REQUIRE(lds <= 160 * 1024, SCN_ERR_ARG, "planes: %d filter positions", gs ? gs->fs : 0);
  const int nSplits = scn_ceil_div(N, COLUMNS);
  const dim3 grid((unsigned)(scn_ceil_div(M, ROWS) * (long long)nSplits));
  // An XCD takes neighbouring tiles: rows with all their columns, so that they come
  // to its L2 once, or, where the image is the larger part, columns with all rows.
  const bool byColumns = image_larger(PL, scn_rows_hint(ctx, M), K, N, gs ? gs->nIn : K);
  if constexpr (PL == 3 && !A16 && D <= 4 && NT < 3 && 2 * D * (ROWS / 8 + NT * CW * PL * 2) > 160) // (as linesTiles' tl)
    if (const int per = gs ? 0 : lines_long(ctx->numCU, scn_rows_hint(ctx, M), K, N, ROWS, COLUMNS, D)) {
      // (W turned: a gradient)
      hipLaunchKernelGGL((lines_past_caches(scn_rows_hint(ctx, M), K, N, wT) ? k_nin_lines<PL, MT, NT, RW, CW, D, false, false, 2> : k_nin_lines<PL, MT, NT, RW, CW, D, false, false, 1>),
                         dim3(8 * per), dim3(64 * RW * CW), lds, ctx->stream, A, image, out, M, K, N, ep, GatherSource(), nSplits,
                         byColumns, rows, PlainW{W, wT});
      return SCN_OK;
    }
  if (gs)
    hipLaunchKernelGGL((k_nin_lines<PL, MT, NT, RW, CW, D, true, A16>), grid, dim3(64 * RW * CW), lds, ctx->stream, A, image,
                       out, M, K, N, ep, *gs, nSplits, byColumns, rows, PlainW{W, wT});
  else if constexpr (!A16)
    hipLaunchKernelGGL((k_nin_lines<PL, MT, NT, RW, CW, D, false, false>), grid, dim3(64 * RW * CW), lds, ctx->stream, A, image,
                       out, M, K, N, ep, GatherSource(), nSplits, byColumns, rows, PlainW{W, wT});
  return SCN_OK;
}
template <int PL, int WM>
static int launch_split64(scn_ctx *ctx, const float *A, const float *W, float *out, long long M, int K, int N,
                          const Epilogue &ep, const GatherSource *gs, const RowRange &rows, const unsigned char *image) {
  const int nSplits = scn_ceil_div(N, 64);
  const size_t lds = 128 * 1024 + (gs ? (size_t)64 * gs->fs * 4 : 0);
  const dim3 grid((unsigned)(scn_ceil_div(M, 64) * (long long)nSplits));
  const bool byColumns = image_larger(PL, scn_rows_hint(ctx, M), K, N, gs ? gs->nIn : K);
  const PlainW plain = {W, WM == S64_TURNED};
  if (!gs)
    hipLaunchKernelGGL((k_nin_split64<PL, false, WM>), grid, dim3(512), lds, ctx->stream, A, image, out, M, K, N, ep,
                       GatherSource(), nSplits, byColumns, rows, plain);
  else if constexpr (WM != S64_TURNED)
    hipLaunchKernelGGL((k_nin_split64<PL, true, WM>), grid, dim3(512), lds, ctx->stream, A, image, out, M, K, N, ep, *gs,
                       nSplits, byColumns, rows, plain);
  return SCN_OK;
}
// (nIn in 32s; an image made by the call where there is none)
template <int NT>
static int launch_rows16(scn_ctx *ctx, const void *A, const float *W, float *out, long long M, int K, int N,
                         const Epilogue &ep, const GatherSource &gs, const RowRange &rows, const unsigned char *image) {
  if (!image) {
    ImageList l;
    l.count = 0, l.firstBlock[0] = 0;
    add_image(l, W, ctx->d_image, 1, K, N, 0);
    SCN_TRY(weight_images(ctx, l));
    image = ctx->d_image;
  }
  const int nSplits = scn_ceil_div(N, 32 * NT);
  const size_t lds = ROWS16_WAVES * (3 * 4096 + 2048) + 3 * NT * 2048; // (NT 4: two workgroups to a compute unit, just)
  hipLaunchKernelGGL((k_nin_rows16<NT>), dim3((unsigned)(scn_ceil_div(M, 64 * ROWS16_WAVES) * (long long)nSplits)),
                     dim3(64 * ROWS16_WAVES), lds, ctx->stream, (const unsigned char *)A, image, out, M, K, N, ep, gs, nSplits, rows);
  return SCN_OK;
}
template <int PL>
static int launch_splitk(scn_ctx *ctx, const float *A, const float *W,
                         float *out, long long M, int K, int N,
                         const Epilogue &ep, const GatherSource *gs, bool a16, bool wT,
                         const RowRange &rows) {
  const int nSplits = scn_ceil_div(N, 32);
  const dim3 grid((unsigned)(scn_ceil_div(M, 32) * (long long)nSplits));
#define SCN_SPLITK_GO(G, H, T, src)                                            \
  hipLaunchKernelGGL((k_nin_planes_splitk<PL, G, H, T>), grid, dim3(512), 0,   \
                     ctx->stream, A, W, out, M, K, N, ep, src, nSplits, rows)
  if (PL == 3 && wT)
    SCN_SPLITK_GO(0, false, PL == 3, GatherSource());
  else if (!gs)
    SCN_SPLITK_GO(0, false, false, GatherSource());
  else if (PL == 1 && a16)
    SCN_SPLITK_GO(2, PL == 1, false, *gs);
  else if (gs->nIn % 32 == 0)
    SCN_SPLITK_GO(1, false, false, *gs);
  else
    SCN_SPLITK_GO(2, false, false, *gs);
#undef SCN_SPLITK_GO
  return SCN_OK;
}

// Which tile.  With n workgroups on every compute unit a block of 32 k takes tn
// n microseconds, and no less than t1 (its chain: request, split, barrier).
// Three planes: measured on contractions of 256 and 1152 k at 256 to 2048
// workgroups, with W converted on the way and from its image.  A wavefront of
// two row tiles and two column tiles (2, 2) is the fastest per flop (232
// TFLOP/s from the image with the chip full, (1, 1) 173; 1.36 M x 1728 x 64
// through its rules 222) and the first to leave the chip idle, so
// the row count decides.
// One plane: fitted to 148 shapes (2800 to 200000 rows, 256 to 2592 k, 64 to 640
// columns), fp32 and bf16 rows, which it gives within 1 % of the best tile on
// average.  What bounds it is the fetching of A, once for every slice of
// columns, so the tile is one row tile by up to four column tiles: from the
// image, with bf16 rows, 596000 x 2592 x 128 511 -> 433 us (913 TFLOP/s) against
// (2, 2), which goes twice through A; 5900 x 1920 x 640 with fp32 rows 57 -> 38
// against (1, 2).  Five and eight column tiles, or two by four, gain no more.
// Every choice gives the same bits.  The start and the stores of a workgroup
// cost by its tiles, the image 5 us.
struct PlanesCost {
  float t1, tn;
};
static const int planesTiles[2][4][2] = {{{1, 1}, {1, 2}, {1, 3}, {1, 4}},  // row tiles, column tiles of a wavefront:
                                         {{1, 1}, {1, 2}, {1, 3}, {2, 2}}}; // one plane, more
static const PlanesCost planesCost[3][4][2] = {
    // one plane: converted, image
    {{{.5f, .5f}, {.44f, .44f}}, {{.67f, .66f}, {.43f, .43f}}, {{.81f, .81f}, {.48f, .48f}}, {{1.21f, 1.21f}, {.46f, .46f}}},
    // ... of bf16 rows
    {{{.36f, .26f}, {.22f, .22f}}, {{.44f, .44f}, {.24f, .24f}}, {{.6f, .6f}, {.28f, .28f}}, {{.95f, .95f}, {.3f, .3f}}},
    // three planes
    {{{.64f, .46f}, {.54f, .39f}}, {{.96f, .72f}, {.95f, .64f}}, {{1.6f, 1.16f}, {1.23f, .99f}}, {{1.36f, 1.29f}, {1.22f, 1.16f}}}};

// The split contraction takes up to this many rows: one or two trips to memory
// while its workgroups are up to so many a compute unit.  Two fit (with 158
// registers, until the rows of whole blocks were looked up once and W's addresses
// left to the scalar unit, it was one: 2600 x 512 x 160 11.0 us, now 8.4).  Measured
// against k_nin_lines with its image made, us at so many a compute unit: three
// planes, 512 k 2.4 11.2, 12.2, and 3.1 14.5, 12.8; 768 k 2.5 15.0, 17.0, and 3.2
// 19.4, 17.6; 256 k 1.8 6.2, 7.7, and 2.4 8.5, 8.0; 2560 k 2.2 41.7, 45.9, and 3.1
// 51.7, 46.5; one plane, 512 k 1.6 6.9, 7.2, and 2.0 9.3, 7.4; 256 k 1.8 5.4, 5.4.
static long long few_rows(scn_ctx *ctx, int planes, int K, int N) {
  if (N > 1 << 26) // (a lane's place in nine rows of W has 32 bits)
    return 0;
  const float perCU = planes == 1 ? 2.f : fminf(1.f + K / 230.f, planes == 2 ? 3.1f : 2.6f);
  const long long rows = (long long)(perCU * ctx->numCU / scn_ceil_div(N, 32));
  return 32 * (rows < 1 ? 1 : rows);
}
// Beyond those k_nin_split64 takes it while its workgroups are no more than the compute
// units: what one takes is its wavefronts' blocks, 2.5 us each in three planes and 1.1 in one,
// and 5 to 7, and a second round as long again (2257 x 1920 x 640, 360 of them, 45.5 us
// where tiles take 46, and 21.7 where they take 17.7). us, rows through rules, images made
// before, the tiles and here: three planes, 1037 x 2560 x 800 49.5, 31.8; 2257 x 1920 x 448 37.4,
// 26.1; 8000 x 1024 x 128 22.1, 16.4; 3000 x 768 x 320 17.3, 13.2; 5000 x 512 x 192 13.0,
// 10.9; one plane 22.0, 15.2; 17.1, 12.1; 11.7, 9.3; 9.5, 8.3; 7.9, 7.4; W as it stands,
// with nothing made before, 12383 x 448 x 64 14.4, 13.5, but 3909 x 256 x 160 9.7, 11.8:
// below 448 k there is no more than a block or two to a wavefront.  One plane from 1024 k on:
// below, it gains a microsecond or two (1152 x 800 x 800 12.8, 11.0), and a batch near the line
// pays 4.6 for the launch that finds nothing.
static long long split_rows(scn_ctx *ctx, int planes, int K, int N) {
  const long long few = few_rows(ctx, planes, K, N), more = 64ll * (ctx->numCU / scn_ceil_div(N, 64));
  return planes != 2 && K >= (planes == 1 ? 1024 : 448) && few > 0 && more > few ? more : few;
}

struct PlanesChoice {
  int tile; // index into planesTiles, -1: split contraction
  bool image;
  float cost; // microseconds, about
  int lines = -1; // k_nin_lines, a tile of its own: index into linesTiles
  int rows16 = 0; // k_nin_rows16, of so many tiles of columns
  const unsigned char *weights = nullptr; // the image it reads, null: to be made
  const unsigned char *given = nullptr;   // the image there is, for the split contraction
};
// images: of the tiles only those from the image (scn_planes_abt: whether there is one), or
// only the others
enum { TILES_ALL, TILES_IMAGE, TILES_CONVERT };
static PlanesChoice planes_choose(scn_ctx *ctx, int planes, long long M, int K, int N, bool a16, int images = TILES_ALL) {
  if (M <= split_rows(ctx, planes, K, N))
    return {-1, false, 0.f};
  const int T = K / 32;
  PlanesChoice best = {0, false, 0.f};
  float least = 1e30f;
  for (int i = 0; i < 4; ++i) {
    const int mt = planesTiles[planes > 1][i][0], nt = planesTiles[planes > 1][i][1];
    const long long nSplits = scn_ceil_div(N, 32 * nt);
    const float wgs = (float)(scn_ceil_div(M, 128 * mt) * nSplits) / ctx->numCU;
    const float n = wgs <= 4.f ? ceilf(wgs) : wgs + .5f;
    const int units = 4 * mt * nt;
    for (int img = images == TILES_IMAGE; img < (images == TILES_CONVERT ? 1 : 2); ++img) {
      if (img && (size_t)nSplits * T * planes * 2 * nt * 1024 > SCN_IMAGE_BYTES)
        continue;
      const PlanesCost &c = planesCost[planes > 1 ? 2 : a16][i][img];
      const float cost = T * fmaxf(c.t1, c.tn * n) + 3.f + units * (.2f + .17f * n) + (img ? 5.f : 0.f);
      if (cost < least)
        least = cost, best = {i, img != 0, cost};
    }
  }
  return best;
}
// The same of bf16 rows, whose tile goes by the columns, and with the image where it
// is not made yet.  Fitted to 49 shapes (3500 to 120000 rows, 256 to 1152 k, 64 to
// 320 columns).  Making the image is what small layers would lose by: us in
// k_nin_planes -> here, 9000 x 576 x 160 11.1 -> 13.9, 30000 x 256 x 64 8.7 -> 9.1;
// 9000 x 1024 x 320 30 -> 21, 60000 x 512 x 128 25 -> 21, 120000 x 576 x 160 61 -> 54.
static float lines_rows16(scn_ctx *ctx, long long M, int K, int N, bool image) {
  const float n = (float)scn_ceil_div(M, 128) * scn_ceil_div(N, N <= 64 ? 64 : 128) / ctx->numCU;
  const float x = fmaxf(n - .5f, 0.f), T = K / 32;
  return (N <= 64 ? 3.f + 2.6f * x + T * (.2f + .15f * x) : 2.3f + 1.6f * x + T * (.37f + .22f * x)) +
         (image ? 0.f : 3.f + (float)K * N / 150000.f);
}
bool scn_planes_splitk(scn_ctx *ctx, int planes, long long M, int K, int N) {
  return M <= few_rows(ctx, planes, K, N);
}

// The split contraction, in the kernel for so many rows.  (bf16 rows: k_nin_split64 rounds
// the fp32 ones, the same bits.)
template <int PL>
static int launch_split(scn_ctx *ctx, const float *A, const float *A32, const float *W, float *out, long long M, int K, int N,
                        const Epilogue &ep, const GatherSource *gs, bool a16, bool wT, const RowRange &rows,
                        const unsigned char *image) {
  const long long few = few_rows(ctx, PL, K, N);
  if constexpr (PL != 2)
    if (split_rows(ctx, PL, K, N) > few && scn_rows_hint(ctx, M) > few) {
      const float *const from = a16 ? A32 : A;
      if (image)
        return launch_split64<PL, S64_IMAGE>(ctx, from, W, out, M, K, N, ep, gs, rows, image);
      if constexpr (PL == 3)
        if (wT)
          return launch_split64<PL, S64_TURNED>(ctx, from, W, out, M, K, N, ep, gs, rows, nullptr);
      return launch_split64<PL, S64_PLAIN>(ctx, from, W, out, M, K, N, ep, gs, rows, nullptr);
    }
  return launch_splitk<PL>(ctx, A, W, out, M, K, N, ep, gs, a16, wT, rows);
}

template <int PL>
static int planes_forward(scn_ctx *ctx, const float *A, const float *A32, const float *W,
                          float *out, long long M, int K, int N,
                          const Epilogue &ep, const GatherSource *gs, bool a16,
                          const PlanesChoice &choice, bool wT = false) {
  RowRange rows = {ctx->d_meta ? ctx->d_meta + META_SITES : nullptr, -1, 1ll << 62};
  if (rows.d_rows) {
    // Near the line both are launched, each for its numbers of rows; away from
    // it the guess decides, and is held against the counts when they are known.
    // A kernel launched by itself is launched for every row there may be: where
    // the guess was wrong its rows are rounded otherwise, not left out.
    // (A launch that finds nothing to do is 4 to 5 us, a pass queued again hundreds: of the
    // larger matrices that k_nin_split64 takes, whose batches vary less, within a fifteenth.)
    const long long split = split_rows(ctx, PL, K, N), hint = scn_rows_hint(ctx, M);
    const int near = split > few_rows(ctx, PL, K, N) ? 15 : 5;
    if (M > split && (near + 1) * hint > near * split && near * hint < (near + 1) * split) {
      RowRange upper = rows;
      rows.upTo = upper.above = split;
      SCN_TRY(launch_split<PL>(ctx, A, A32, W, out, split, K, N, ep, gs, a16, wT, rows, choice.given));
      rows = upper;
    } else if (hint <= split) {
      scn_rows_chosen(ctx, -1, split);
      return launch_split<PL>(ctx, A, A32, W, out, M, K, N, ep, gs, a16, wT, rows, choice.given);
    } else {
      scn_rows_chosen(ctx, split, 1ll << 62);
    }
  } else if (choice.tile < 0) {
    return launch_split<PL>(ctx, A, A32, W, out, M, K, N, ep, gs, a16, wT, rows, choice.given);
  }
  if constexpr (PL == 1)
    switch (choice.rows16) {
    case 2:
      return launch_rows16<2>(ctx, A, W, out, M, K, N, ep, *gs, rows, choice.weights);
    case 3:
      return launch_rows16<3>(ctx, A, W, out, M, K, N, ep, *gs, rows, choice.weights);
    case 4:
      return launch_rows16<4>(ctx, A, W, out, M, K, N, ep, *gs, rows, choice.weights);
    }
#define SCN_LINES_CASE(I, MT, NT, RW, CW, D)                                                                             \
  case I:                                                                                                               \
    return launch_lines<PL, MT, NT, RW, CW, D>(ctx, A, W, out, M, K, N, ep, gs, wT, rows, choice.weights);
  if constexpr (PL == 3) {
    switch (choice.lines) { // (as in linesTiles)
      SCN_LINES_CASE(0, 1, 2, 4, 2, 3)
      SCN_LINES_CASE(1, 2, 1, 4, 2, 3)
      SCN_LINES_CASE(2, 1, 3, 4, 1, 4)
      SCN_LINES_CASE(3, 1, 2, 2, 2, 4)
      SCN_LINES_CASE(4, 1, 1, 2, 2, 3)
      SCN_LINES_CASE(5, 1, 1, 2, 2, 6)
      SCN_LINES_CASE(LINES_NARROW, 1, 1, 4, 1, 3)
    }
  } else if constexpr (PL == 1) {
    switch (choice.lines) {
      SCN_LINES_CASE(0, 1, 2, 4, 2, 3)
      SCN_LINES_CASE(1, 1, 2, 2, 2, 4)
      SCN_LINES_CASE(2, 1, 1, 2, 2, 3)
    case 3: // (of bf16 rows)
      return launch_lines<PL, 1, 2, 4, 2, 3, true>(ctx, A, W, out, M, K, N, ep, gs, wT, rows, choice.weights);
    case 4:
      return launch_lines<PL, 1, 1, 4, 2, 4, true>(ctx, A, W, out, M, K, N, ep, gs, wT, rows, choice.weights);
    }
  }
#undef SCN_LINES_CASE
  // (channels in other than 32s, seldom met: one tile)
  if (gs && gs->nIn % 32 != 0)
    return launch_planes<PL, 1, 2, W_PLAIN, true>(ctx, A, W, out, M, K, N, ep, gs, a16, rows);
  // W_STREAM where the chip is full and the contraction long: the widest tile, W
  // from its image, rows gathered (by no more than 27 positions: with the third
  // buffer two workgroups still fit a compute unit's LDS).  The registers it frees
  // let bf16 rows go eight wavefronts to a workgroup, half the reading of W:
  // 596000 x 2592 x 128 433 -> 406 us, and of ten layers of 57 to 395 GFLOP 0.99 to
  // 1.10 times as fast.  In three planes it is 1 % of layers of 1728 k and more,
  // whose loop is all they are (1.36 M x 1728 x 64 1422 -> 1398 us, 596000 x 2592 x
  // 128 1808 -> 1788, 3456 k 889 -> 876: means of each side's runs, in turn on one
  // card), and nothing that shows on shorter ones (512 to 1280 k, 66 to 970 us: 0.97
  // to 1.03).  Everywhere else what the third buffer costs is not made good: (3, 1, 1)
  // 58.8 -> 61.6 us, one plane (1, 2) 40 -> 47, rows that are not gathered 141 -> 148.
  if constexpr (PL != 2)
    if (choice.tile == 3 && choice.image && gs && (PL > 1 || a16))
      return launch_planes<PL, (PL > 1 ? 2 : 1), (PL > 1 ? 2 : 4), W_STREAM, false, (PL > 1 ? 4 : 8)>(
          ctx, A, W, out, M, K, N, ep, gs, a16, rows);
#define SCN_PLANES_CASE(I, MT, NT)                                             \
  case I:                                                                      \
    return choice.image                                                        \
               ? launch_planes<PL, MT, NT, W_IMAGE>(ctx, A, W, out, M, K, N, ep, gs, a16, rows) \
               : launch_planes<PL, MT, NT, W_PLAIN>(ctx, A, W, out, M, K, N, ep, gs, a16, rows);
  switch (choice.tile) {
    SCN_PLANES_CASE(0, 1, 1)
    SCN_PLANES_CASE(1, 1, 2)
    SCN_PLANES_CASE(2, 1, 3)
    SCN_PLANES_CASE(3, (PL > 1 ? 2 : 1), (PL > 1 ? 2 : 4))
  }
#undef SCN_PLANES_CASE
  return SCN_ERR_ARG;
}

// k_nin_lines where it is the faster (the same bits): for rows that are not gathered
// wherever it can run, as k_nin_planes' costs are too low for those.
static void lines_instead(scn_ctx *ctx, int planes, long long M, int K, int N, const GatherSource *gs, const void *image,
                          bool room, bool unlikely, bool wT, PlanesChoice &choice) {
  if (!lines_shape(planes, K, N, gs ? gs->nIn : K) ||
      !(image || (room && image_bytes(planes, K, N) <= (int64_t)SCN_IMAGE_BYTES)))
    return;
  // Plain rows of up to four tiles of 32 x 32 to a compute unit, in three planes: what
  // the image's launch takes is a third of all. us, from an image made by the call and converted on the
  // way, 5760 x 256 x 160 13.6, 9.9; 10474 x 256 x 96 13.6, 9.7; 9307 x 128 x 64 9.3, 7.1; 3810 x 544 x 256 16.8, 14.7;
  // at 4.3 to a unit 11818 x 224 x 96 12.9, 12.7, at 4.8 4872 x 608 x 256 20.1, 25.1.
  if (!gs && !image && !wT && planes == 3 && tiles_of(M, 32) * tiles_of(N, 32) <= 4ll * ctx->numCU) {
    choice = planes_choose(ctx, 3, M, K, N, false, TILES_CONVERT);
    return;
  }
  int tile = 0;
  const float cost = lines_choose(ctx->numCU, planes, M, K, N, gs != nullptr, &tile) + (image ? 0.f : 4.f);
  // (2: what the other's leave out of a launch; unlikely: for rows there probably are not, without
  // a launch for an image where there is one)
  if (gs && cost >= choice.cost + 2.f && !(unlikely && image))
    return;
  if (!gs && planes == 3 && N <= 32) // (gathered rows of one tile of columns are k_nin_planes')
    tile = LINES_NARROW;
  choice.lines = tile;
  choice.weights = (const unsigned char *)image;
}

int scn_planes_forward(scn_ctx *ctx, int planes, const float *A, const float *W,
                       float *out, long long M, int K, int N,
                       const Epilogue &ep, const GatherSource *gs, bool a16,
                       const void *image, const float *A32) {
  // (rows guessed: a tile in any case, they may be more)
  const long long split = split_rows(ctx, planes, K, N), hint = scn_rows_hint(ctx, M);
  const long long rows = M > split && hint <= split ? split + 1 : hint;
  PlanesChoice choice = planes_choose(ctx, planes, rows, K, N, a16);
  choice.given = (const unsigned char *)image;
  const bool room = planes_image(ctx);
  choice.image = choice.image && room;
  // (bf16 rows: a block takes half a line of each.  k_nin_planes' cost is 2 too high where
  // it converts W on the way, of layers that small.  Long contractions of few rows: 8000 x
  // 1536 x 256 23.4 -> 17.1 us, 6000 x 1920 x 640 40 -> 27.6, 20000 x 1728 x 128 38 -> 21.)
  if (a16 && choice.tile >= 0 && N > 32 && lines_shape(1, K, N, gs->nIn) &&
      (image || (room && image_bytes(1, K, N) <= (int64_t)SCN_IMAGE_BYTES))) {
    choice.rows16 = rows16_tiles(ctx->numCU, rows, K, N);
    if (choice.rows16 == 0 &&
        lines_rows16(ctx, rows, K, N, image != nullptr) < choice.cost - (choice.image ? 0.f : 2.f))
      choice.lines = N <= 64 ? 4 : 3;
    if (choice.rows16 || choice.lines >= 0)
      choice.weights = (const unsigned char *)image;
  }
  if (choice.tile >= 0 && !a16)
    lines_instead(ctx, planes, rows, K, N, gs, image, room, hint <= split, false, choice);
  return planes == 3   ? planes_forward<3>(ctx, A, A32, W, out, M, K, N, ep, gs, a16, choice)
         : planes == 2 ? planes_forward<2>(ctx, A, A32, W, out, M, K, N, ep, gs, a16, choice)
                       : planes_forward<1>(ctx, A, A32, W, out, M, K, N, ep, gs, a16, choice);
}

// The planes of a call of that precision, 0: none that take an image
static int image_planes(int precision) {
  return precision == SCN_FP32_PLANES ? 3 : precision == SCN_BF16 ? 1 : 0;
}
extern "C" int64_t scn_weight_image_bytes(scn_ctx *ctx, int64_t M, int K, int N, int nIn, int precision) {
  const int planes = image_planes(precision);
  if (!ctx || M < 1 || K < 1 || N < 1 || nIn < 1 || planes == 0 || N % 4 != 0 || !lines_shape(planes, K, N, nIn))
    return 0;
  const long long hint = scn_rows_hint(ctx, M), few = few_rows(ctx, planes, K, N), split = split_rows(ctx, planes, K, N);
  if (split > few ? hint <= few : 6 * hint <= 5 * split)
    return 0;
  if (split > few && hint <= split) // (k_nin_split64)
    return image_bytes(planes, K, N);
  int tile;
  const PlanesChoice choice = planes_choose(ctx, planes, hint > split ? hint : split + 1, K, N, false);
  if (nIn != K && lines_choose(ctx->numCU, planes, hint, K, N, true, &tile) >= choice.cost + 2.f)
    return 0;
  return image_bytes(planes, K, N);
}
// Rows that a pooling has rounded on the way (2 bytes more of the some 24 to 44 that it
// moves for a feature), us of fp32 rows and of these, with the image: 41600 x 640 x 320 36, 31;
// 10500 x 1280 x 480 29.5, 24.7; 26000 x 1280 x 480 60, 39; 110000 x 512 x 160 60, 39; 60000 x
// 256 x 96 12.8, 11.1; 90000 x 512 x 96 of eight positions 30, 19.7.  Below 2e9 products it is a
// microsecond or none (26000 x 384 x 128 10.3, 9.3; 6000 x 896 x 256 11.3, 11.8), and longer ones
// need the rows for k_nin_rows16 (10500 x 1920 x 640 46, 33; 8000 42, 32.5; 6000 26, 28; 6000 x
// 2560 x 800 50, 40; 4500 33, 39; 30000 x 2592 x 128 37, 42).
extern "C" int scn_rounded_rows_pay(scn_ctx *ctx, int64_t M, int fs, int nIn, int N) {
  if (!ctx || M < 1 || fs < 1 || nIn < 1 || N < 1 || !lines_shape(1, fs * nIn, N, nIn))
    return 0;
  const long long rows = scn_rows_hint(ctx, M), K = (long long)fs * nIn;
  return (double)rows * K * N >= 2e9 && (K <= 1280 || tiles_of(rows, 256) * tiles_of(N, 128) >= .6 * ctx->numCU);
}
static int image_list(scn_ctx *ctx, const scn_image_item *items, int nItems, ImageList &l) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_weight_images_many: null context");
  SCN_REQUIRE(nItems >= 0 && nItems <= SCN_IMAGES_MAX && (items || nItems == 0), SCN_ERR_ARG,
              "scn_weight_images_many: %d items (at most %d)", nItems, SCN_IMAGES_MAX);
  static_assert(SCN_IMAGES_MAX <= 64, "a lane an item");
  l.count = 0, l.firstBlock[0] = 0;
  long long blocks = 0;
  for (int k = 0; k < nItems; ++k) {
    const scn_image_item &it = items[k];
    const int planes = image_planes(it.precision);
    SCN_REQUIRE(it.d_W && it.d_image && planes && scn_planes_shape(it.K) && it.N >= 1 && it.fs >= 0 &&
                    (it.fs == 0 || (it.K % it.fs == 0 && it.K / it.fs % 8 == 0)) && ((uintptr_t)it.d_image & 15) == 0,
                SCN_ERR_ARG, "scn_weight_images_many: item %d K %d N %d fs %d precision %d", k, it.K, it.N, it.fs,
                it.precision);
    blocks += scn_ceil_div((int64_t)it.K / 8 * (((int64_t)it.N + 31) / 32 * 32), 256);
    SCN_REQUIRE(blocks <= 0x7fffffffll, SCN_ERR_CAPACITY, "scn_weight_images_many: %lld workgroups", blocks);
    add_image(l, it.d_W, (unsigned char *)it.d_image, planes, it.K, it.N, it.fs);
  }
  return SCN_OK;
}
extern "C" int scn_weight_images_many(scn_ctx *ctx, const scn_image_item *items, int nItems) {
  ImageList l;
  SCN_TRY(image_list(ctx, items, nItems, l));
  ProfScope prof(ctx, SCN_K_NIN);
  SCN_TRY(weight_images(ctx, l));
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}
// (what an earlier call left and nobody has asked for is given up: its images may be
// gone)
extern "C" int scn_weight_images_later(scn_ctx *ctx, const scn_image_item *items, int nItems) {
  if (ctx)
    ctx->imagesLater.count = 0;
  if (ctx && ctx->prof) // (a launch of its own, which is no layer's, where layers are timed)
    return nItems == 0 ? SCN_OK : scn_weight_images_many(ctx, items, nItems);
  ImageList l;
  SCN_TRY(image_list(ctx, items, nItems, l));
  ctx->imagesLater = l;
  return SCN_OK;
}
int scn_images_now(scn_ctx *ctx) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_conv_nin_forward: null context");
  ImageList &l = ctx->imagesLater;
  if (l.count == 0)
    return SCN_OK;
  const int n = l.count;
  l.count = 0;
  ImageList now = l;
  now.count = n;
  SCN_TRY(weight_images(ctx, now));
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// out = A Wt^T for Wt [N x K].  False: nothing has been launched; not a shape for
// it, or (transpose) one that scn_planes_forward takes to the same bits from the
// transpose, because the image may not be used now.
bool scn_planes_abt(scn_ctx *ctx, const float *A, const float *Wt, float *out,
                    long long M, int K, int N, const Epilogue &ep, int *rc, bool *transpose) {
  *transpose = false;
  if (!scn_planes_shape(K) || ((uintptr_t)A & 15) || ((uintptr_t)out & 15) || N % 4 != 0)
    return false;
  PlanesChoice choice = planes_choose(ctx, 3, M, K, N, false, TILES_IMAGE);
  const bool room = planes_image(ctx);
  if (choice.tile >= 0)
    lines_instead(ctx, 3, M, K, N, nullptr, nullptr, room, false, true, choice);
  if (choice.tile >= 0 && choice.lines < 0) {
    *transpose = choice.image;
    return false;
  }
  ProfScope prof(ctx, SCN_K_BACKWARD);
  *rc = planes_forward<3>(ctx, A, A, Wt, out, M, K, N, ep, nullptr, false, choice, true);
  return true;
}

// out = A W^T for A [M x n], W [K x n] of no more than 32 columns: a gradient by a layer
// of few outputs.  What bounds it is writing out.  A wavefront has 64 rows of A as planes
// in its registers and goes through the rows of W, 32 at a time, which are split as they
// come, the next ones under way; twelve MFMAs make 4 KB of out.
// Behind it the fp32 kernel for short contractions, which keeps to vector instructions, us:
// 118144 x 896 of 32 249 -> 105 (4.0 TB/s), 30000 x 864 67 -> 28, 100000 x 128 36 -> 16, 9000 x 64 8.5 -> 7.1,
// 40000 x 512 of 16 35 -> 21; of 1000 rows 8.8, 10.0 (the line: 2048).  The error against 64 bits
// is 0.4 of its.  The results go past the caches (through them 114).
constexpr int NARROW_MT = 2, NARROW_WAVES = 4;
__global__ void __launch_bounds__(64 * NARROW_WAVES, 2)
    k_abt_narrow(const float *__restrict__ A, const float *__restrict__ W, float *__restrict__ out, long long M, int n, int K,
                 int tiles) { // (of columns, to a workgroup)
  constexpr int PL = 3, MT = NARROW_MT;
  const int lane = threadIdx.x & 63, c = lane & 31, q = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned at = xcd_eighth(blockIdx.x, gridDim.x);
  const long long row0 = ((long long)at * NARROW_WAVES + wave) * 32 * MT;
  if (row0 >= M) // (no barrier below)
    return;
  bf16x8 a[MT][2][PL];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const long long r = row0 + 32 * i + c < M ? row0 + 32 * i + c : M - 1; // (not stored)
      const int k = 16 * s + 8 * q;
      float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (k < n) {
        const floatx4 x = *reinterpret_cast<const floatx4 *>(A + r * n + k), y = *reinterpret_cast<const floatx4 *>(A + r * n + k + 4);
        v[0] = x[0], v[1] = x[1], v[2] = x[2], v[3] = x[3], v[4] = y[0], v[5] = y[1], v[6] = y[2], v[7] = y[3];
      }
      split8<PL>(v, a[i][s]);
    }
  const int t0 = blockIdx.y * tiles, all = (K + 31) / 32, t1 = t0 + tiles < all ? t0 + tiles : all;
  const bool whole = row0 + 32 * MT <= M; // uniform
  const unsigned place = 4 * q * (unsigned)K + c; // this lane's in a tile
  floatx4 raw[2][2];
  auto load = [&](int t) {
    const int row = 32 * t + c < K ? 32 * t + c : K - 1; // (not stored)
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = 16 * s + 8 * q;
        raw[s][h] = k < n ? *reinterpret_cast<const floatx4 *>(W + (long long)row * n + k + 4 * h) : floatx4{0.f, 0.f, 0.f, 0.f};
      }
  };
  load(t0);
#pragma unroll 1
  for (int t = t0; t < t1; ++t) {
    bf16x8 b[2][PL];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const float v[8] = {raw[s][0][0], raw[s][0][1], raw[s][0][2], raw[s][0][3], raw[s][1][0], raw[s][1][1], raw[s][1][2], raw[s][1][3]};
      split8<PL>(v, b[s]);
    }
    load(t + 1 < t1 ? t + 1 : t);
    floatx16 acc[2][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[h][i][v] = 0.f;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int x = 0; x < PL; ++x)
#pragma unroll
        for (int y = 0; x + y < PL; ++y)
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            floatx16 &d = acc[x + y == 0 ? 0 : 1][i];
            d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][s][x], b[s][y], d, 0, 0, 0);
          }
    float none[4] = {0.f, 0.f, 0.f, 0.f}; // 0 sum: NaN for a sum that is not finite
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[0][i][v] += acc[1][i][v];
        none[v % 4] = fmaf(acc[0][i][v], 0.f, none[v % 4]);
      }
    const int col = 32 * t + c;
    if (__any((none[0] + none[1]) + (none[2] + none[3]) != 0.f)) { // these rows and columns as fp32 has them
      for (int x = 0; x < 16 * MT && col < K; ++x) {
        const long long row = row0 + 2 * x + q;
        if (row >= M)
          break;
        float sum = 0.f;
        for (int k = 0; k < n; ++k)
          sum = fmaf(A[row * n + k], W[(long long)col * n + k], sum);
        out[row * K + col] = sum;
      }
      continue;
    }
    if (col < K) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int r = 32 * i + 8 * (v / 4) + v % 4; // uniform
          if (whole || row0 + r + 4 * q < M)
            __builtin_nontemporal_store(acc[0][i][v], out + (row0 + r) * K + 32 * t + place);
        }
    }
  }
}
// Whether it is one for this; then it has been launched
bool scn_abt_narrow(scn_ctx *ctx, const float *A, const float *W, float *out, long long M, int n, int K) {
  if (n > 32 || n % 8 || (((uintptr_t)A | (uintptr_t)W) & 15) || M < 2048 || M >= 1ll << 32 || K < 64 || K > 1 << 24)
    return false;
  const long long groups = (M + 32 * NARROW_MT * NARROW_WAVES - 1) / (32 * NARROW_MT * NARROW_WAVES);
  const int all = (K + 31) / 32;
  // (two workgroups a compute unit, of four tiles of columns at least)
  int parts = (int)std::max<long long>(1, std::min<long long>((2 * ctx->numCU + groups - 1) / groups, all / 4));
  const int tiles = (all + parts - 1) / parts;
  parts = (all + tiles - 1) / tiles;
  ProfScope prof(ctx, SCN_K_BACKWARD);
  hipLaunchKernelGGL(k_abt_narrow, dim3((unsigned)groups, (unsigned)parts), dim3(64 * NARROW_WAVES), 0, ctx->stream, A, W, out,
                     M, n, K, tiles);
  return true;
}

// ------------------------------------------------------- dW = A^T D in planes
// The contraction runs over the rows of both matrices, so an MFMA operand is
// eight consecutive rows of one column: dword loads (pairs of columns for two
// tiles) that 32 lanes make of 32 neighbouring columns, whole lines, and no
// turning in LDS.  A workgroup owns 32 MT x 32 NT of dW and a range of rows; its
// wavefronts, eight or twelve, take sixteen rows each in turn and their sums meet in LDS.
// The workgroups of one tile add to dW with float atomics, some 200 of which
// retire in a nanosecond: few workgroups (one a compute unit), each with as many
// rows as that leaves it (29827 x 256 x 96 in 23 us, where the fp32 MFMA with a
// thousand workgroups took 32; 200000 x 1728 x 64 in 350, 470).
// GATHER: the rows of A through rules, which lie position by position, so that
// a lane's eight are two loads (eight of them through row by row rules: 17.8 us
// where this is 15.6 and a gathered matrix 14.5, and 8.2 to gather it).
// LINES: the rows come into LDS by whole lines, a ring of steps for each wavefront,
// which waits for nobody: a kilobyte to a request, where the loads above take 256 or
// 512 bytes and every request occupies the path for 16 cycles or more, twice what the
// splitting takes.  A backward layer with dW of 139000 x 384 x 128 384 -> 370 us;
// dW of 28000 x 256 x 96 and its like 16.5 -> 15.6, of which some 5 are the start and
// the atomics; 35461 x 256 x 96 20, 198759 x 1728 x 64 328 (A from HBM at 4.2 TB/s).
// In tiles of two a step's planes are made among the MFMAs of the step before, by three
// wavefronts to a SIMD: the two together 55 -> 50 us for six layers of a batch of drawings
// in one launch.
constexpr int atb_ring(int MT, int NT) { return MT * NT >= 2 ? 2 : 3; }
// (one tile of dW, of the rows from m0 to m1: m0 a multiple of ATB_STEP; GM wavefronts)
template <int MT, int NT, bool GATHER, bool LINES, int GM>
__device__ __forceinline__ void atb_tile(const float *__restrict__ A, const float *__restrict__ D, float *__restrict__ dW,
                                         float *__restrict__ db, long long M, int K, int N, int nTiles,
                                         GatherSource gs, const float *zeros, unsigned tile, long long m0,
                                         long long m1, int nBase = 0) {
  constexpr int PL = 3;
  constexpr int TILE = 32 * MT * 32 * NT; // floats of a wavefront's tile
  extern __shared__ __attribute__((aligned(16))) float sTile[]; // [GM][TILE], [GM][32 NT], a flag
  float *const sBias = sTile + GM * TILE;
  int *const sAgain = reinterpret_cast<int *>(sBias + GM * 32 * NT);
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid)); // (what follows from it is not kept from one tile to the next)
  const int lane = tid & 63, wave = tid >> 6;
  const int c = lane & 31, q = lane >> 5;
  const int k0 = (int)(tile / nTiles) * 32 * MT;
  const int n0 = nBase + (int)(tile % nTiles) * 32 * NT;
  // this lane's columns (past the end: the last ones, not stored)
  int ka = k0 + MT * c, na = n0 + NT * c;
  ka = ka + MT <= K ? ka : K - MT;
  na = na + NT <= N ? na : N - NT;
  const unsigned offA = (unsigned)(8 * q) * K + ka, offD = (unsigned)(8 * q) * N + na;
  // GATHER: this lane's filter position and channel, the same for all rows
  const int f = GATHER ? ka / gs.nIn : 0, ch = GATHER ? ka - f * gs.nIn : 0;

  struct Step {
    float a[8][MT], d[8][NT];
    int rule[GATHER ? 8 : 1];
  };
  // GATHER: the rules of a step are asked for a step before its rows are
  auto look_up = [&](Step &s, long long m) {
#pragma unroll
    for (int h = 0; h < (GATHER ? 2 : 0); ++h) {
      // (the positions' pitch: the last rows of one are padded with none)
      const long long pitch = (M + ATB_STEP - 1) / ATB_STEP * ATB_STEP;
      const long long at = m + 8 * q + 4 * h;
      const int4 v = *reinterpret_cast<const int4 *>(gs.rules + f * pitch + (at < pitch ? at : pitch - 4));
      s.rule[(4 * h) % (GATHER ? 8 : 1)] = v.x, s.rule[(4 * h + 1) % (GATHER ? 8 : 1)] = v.y;
      s.rule[(4 * h + 2) % (GATHER ? 8 : 1)] = v.z, s.rule[(4 * h + 3) % (GATHER ? 8 : 1)] = v.w;
    }
  };
  auto load = [&](Step &s, long long m, bool guard) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float *pa, *pd;
      if (guard) {
        long long r = m + 8 * q + i;
        r = r < m1 ? r : m1 - 1;
        pa = A + r * K + ka;
        pd = D + r * N + na;
      } else {
        pa = A + (m + i) * K + offA;
        pd = D + (m + i) * N + offD;
      }
      if constexpr (GATHER)
        pa = s.rule[i] >= 0 ? A + (long long)s.rule[i] * gs.nIn + ch : gs.zeros;
      if constexpr (MT == 2) {
        const floatx2 v = *reinterpret_cast<const floatx2 *>(pa);
        s.a[i][0] = v[0], s.a[i][1] = v[1];
      } else {
        s.a[i][0] = *pa;
      }
      if constexpr (NT == 2) {
        const floatx2 v = *reinterpret_cast<const floatx2 *>(pd);
        s.d[i][0] = v[0], s.d[i][1] = v[1];
      } else {
        s.d[i][0] = *pd;
      }
      if (guard && m + 8 * q + i >= m1) {
#pragma unroll
        for (int j = 0; j < MT; ++j)
          s.a[i][j] = 0.f;
#pragma unroll
        for (int j = 0; j < NT; ++j)
          s.d[i][j] = 0.f;
      }
    }
  };
  floatx16 acc[2][MT][NT];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[h][i][j][v] = 0.f;
  // the column sums of D, by the workgroups of the first tile of K
  // (not by two by two tiles without LINES, whose registers are full)
  const bool sums = (LINES || MT * NT < 4) && db && k0 == 0;
  float ds[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    ds[j] = 0.f;
  struct Planes {
    bf16x8 a[MT][PL], d[NT][PL];
  };
  auto split = [&](const Step &s, Planes &p, bool counts) { // (counts: whether the step's D is to be summed)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const float sum =
          ((s.d[0][j] + s.d[1][j]) + (s.d[2][j] + s.d[3][j])) + ((s.d[4][j] + s.d[5][j]) + (s.d[6][j] + s.d[7][j]));
      ds[j] += counts ? sum : 0.f;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const float v[8] = {s.a[0][i], s.a[1][i], s.a[2][i], s.a[3][i], s.a[4][i], s.a[5][i], s.a[6][i], s.a[7][i]};
      split8<PL>(v, p.a[i]);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const float v[8] = {s.d[0][j], s.d[1][j], s.d[2][j], s.d[3][j], s.d[4][j], s.d[5][j], s.d[6][j], s.d[7][j]};
      split8<PL>(v, p.d[j]);
    }
  };
  auto multiply = [&](const Planes &p) {
#pragma unroll
    for (int x = 0; x < PL; ++x)
#pragma unroll
      for (int y = 0; x + y < PL; ++y)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            floatx16 &d = acc[x + y == 0 ? 0 : 1][i][j];
            d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(p.a[i][x], p.d[j][y], d, 0, 0, 0);
          }
  };
  auto compute = [&](const Step &s) {
    Planes p;
    split(s, p, sums);
    multiply(p);
  };
  if constexpr (LINES) {
    constexpr int RING = atb_ring(MT, NT), AU = 2 * MT, DU = 2 * NT, FETCH = AU + DU;
    constexpr int SLOT = FETCH * 1024;
    const int wave0 = __builtin_amdgcn_readfirstlane(wave);
    unsigned char *const ring = reinterpret_cast<unsigned char *>(sTile) + wave0 * RING * SLOT;
    const unsigned ldsRing = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring;
    const long long pitch = (M + ATB_STEP - 1) / ATB_STEP * ATB_STEP;
    // what this lane asks for: four columns of every 8 / MT-th (8 / NT-th) row
    int ca = k0 + 4 * (lane % (8 * MT)), cd = n0 + 4 * (lane % (8 * NT));
    ca = ca < K ? ca : K - 4, cd = cd < N ? cd : N - 4; // (past the end: not stored)
    const int ra = lane / (8 * MT), rd = lane / (8 * NT);
    const int f4 = GATHER ? ca / gs.nIn : 0, ch4 = GATHER ? ca - f4 * gs.nIn : 0;
    const int steps = (int)((m1 - m0 - ATB_STEP * wave0 + ATB_STEP * GM - 1) / (ATB_STEP * GM));
    auto place = [&](int t) { return m0 + ATB_STEP * (wave0 + (long long)GM * (t < steps ? t : steps - 1)); };
    // Rules: a word a lane for each request of rows, behind the rings of all wavefronts
    struct Rules {
      int r[GATHER ? AU : 1];
    };
    int *const sRule = reinterpret_cast<int *>(reinterpret_cast<unsigned char *>(sTile) + GM * RING * SLOT) + wave0 * AU * 64;
    auto ask = [&](int t, int *to) { // (the positions' pitch: whole steps)
      const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int *)to;
#pragma unroll
      for (int u = 0; u < (GATHER ? AU : 0); ++u)
        dma_words(lds + u * 256, gs.rules + f4 * pitch + place(t) + 8 / MT * u + ra);
    };
    auto look = [&](Rules &x, const int *from) { // (read before the next ones take their place)
#pragma unroll
      for (int u = 0; u < (GATHER ? AU : 0); ++u)
        x.r[u % (GATHER ? AU : 1)] = from[u * 64 + lane];
#pragma unroll
      for (int u = 0; u < (GATHER ? AU : 0); ++u)
        asm volatile("" : "+v"(x.r[u % (GATHER ? AU : 1)]) : : "memory");
    };
    // (byte addresses: a multiplication a request of gathered rows, none of plain ones)
    typedef unsigned long long u64;
    const u64 none = (u64)(uintptr_t)(GATHER ? gs.zeros : zeros);
    const u64 fromA = (u64)(uintptr_t)(GATHER ? A + ch4 : A + (m0 + ra) * K + ca);
    const u64 fromD = (u64)(uintptr_t)(D + (m0 + rd) * N + cd);
    const unsigned rowA = (GATHER ? gs.nIn : K) * 4u;
    const int left = (int)(m1 - m0);
    auto fetch = [&](const Rules &x, int t, int slot) {
      const int m = (int)(place(t) - m0); // uniform
      const unsigned lds = ldsRing + slot * SLOT;
      const u64 stepA = fromA + (u64)m * K * 4, stepD = fromD + (u64)m * N * 4;
      // (chosen, not jumped to: the MFMAs beside are dealt out in one block of code)
      auto request = [&](int u, bool live, u64 from) {
        asm volatile("" : "+v"(from));
        dma_kilobyte(lds + u * 1024, reinterpret_cast<const unsigned char *>((uintptr_t)(live ? from : none)));
      };
#pragma unroll
      for (int u = 0; u < AU; ++u) {
        const int rule = x.r[GATHER ? u % AU : 0];
        if constexpr (GATHER)
          request(u, rule >= 0, fromA + (u64)(unsigned)rule * rowA);
        else
          request(u, m + 8 / MT * u + ra < left, stepA + (u64)(8 / MT * u) * K * 4);
      }
#pragma unroll
      for (int u = 0; u < DU; ++u)
        request(AU + u, m + 8 / NT * u + rd < left, stepD + (u64)(8 / NT * u) * N * 4);
    };
    auto take = [&](Step &s, int slot) {
      const unsigned char *const at = ring + slot * SLOT;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float *const pa = reinterpret_cast<const float *>(at) + (8 * q + i) * 32 * MT + MT * c;
        const float *const pd = reinterpret_cast<const float *>(at + AU * 1024) + (8 * q + i) * 32 * NT + NT * c;
        if constexpr (MT == 2) {
          const floatx2 v = *reinterpret_cast<const floatx2 *>(pa);
          s.a[i][0] = v[0], s.a[i][1] = v[1];
        } else {
          s.a[i][0] = *pa;
        }
        if constexpr (NT == 2) {
          const floatx2 v = *reinterpret_cast<const floatx2 *>(pd);
          s.d[i][0] = v[0], s.d[i][1] = v[1];
        } else {
          s.d[i][0] = *pd;
        }
      }
    };
    if (steps > 0) { // uniform
      // Rules are asked for a step before their rows, in front of the rows asked for
      // then: what has landed when all but the last step's rows have holds a step's
      // rows and the next request's rules.
      if constexpr (atb_ahead(MT, NT)) {
        // A step's planes are made while the MFMAs of the one before run, dealt out
        // among them.  So a slot is free when its planes have been made, and RING steps
        // are under way.
        Rules first[RING];
        int *const spare = reinterpret_cast<int *>(ring + (RING - 1) * SLOT); // (nothing is asked for there yet)
        static_assert(RING * AU * 256 <= SLOT, "a slot holds the first rules");
#pragma unroll
        for (int r = 0; r < RING; ++r)
          ask(r, spare + r * AU * 64);
        ask(RING, sRule);
        w_landed<0>();
#pragma unroll
        for (int r = 0; r < RING; ++r)
          look(first[r], spare + r * AU * 64);
        w_landed<0>(); // (the words have been read: their place is asked for again)
#pragma unroll
        for (int r = 0; r < RING; ++r)
          fetch(first[r], r, r);
        int slot = 1, into = 0;
        Planes even, odd;
        Rules x;
        {
          Step s;
          w_landed<(RING - 1) * FETCH>();
          take(s, 0);
          split(s, even, true);
        }
        auto step = [&](const Planes &now, Planes &next, int t) {
          w_landed<(RING - 2) * FETCH>(); // (and this wavefront's reads of the slot that is asked for again)
          look(x, sRule);
          Step s;
          take(s, slot);
          ask(t + RING + 1, sRule);
          fetch(x, t + RING, into);
          split(s, next, t + 1 < steps);
          multiply(now);
#pragma unroll
          for (int k = 0; k < 6 * MT * NT; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                                   // MFMA
            __builtin_amdgcn_sched_group_barrier(0x2, (44 * (MT + NT) + 6 * MT * NT - 1) / (6 * MT * NT), 0); // VALU
          }
          // (here and not where they are used)
#pragma unroll
          for (int l = 0; l < PL; ++l) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
              asm volatile("" : "+v"(next.a[i][l]));
#pragma unroll
            for (int j = 0; j < NT; ++j)
              asm volatile("" : "+v"(next.d[j][l]));
          }
          slot = slot == RING - 1 ? 0 : slot + 1, into = into == RING - 1 ? 0 : into + 1;
        };
#pragma unroll 1
        for (int t = 0; t < steps; ++t) {
          step(even, odd, t);
          if (++t == steps)
            break;
          step(odd, even, t);
        }
      } else {
        static_assert(!GATHER || RING <= 3, "the first two steps' rules come together");
        Rules x;
        {
          Rules second;
          int *const spare = reinterpret_cast<int *>(ring + (RING - 1) * SLOT); // (nothing is asked for there yet)
          ask(0, spare);
          ask(1, spare + AU * 64);
          ask(RING - 1, sRule);
          w_landed<0>();
          look(x, spare);
          look(second, spare + AU * 64);
          fetch(x, 0, 0);
          if (RING == 3)
            fetch(second, 1, 1);
        }
        int slot = 0, into = RING - 1;
#pragma unroll 1
        for (int t = 0; t < steps; ++t) {
          w_landed<RING == 3 ? FETCH : 0>(); // (and this wavefront's reads of the slot that is asked for again)
          look(x, sRule);
          ask(t + RING, sRule);
          fetch(x, t + RING - 1, into);
          Step s;
          take(s, slot);
          compute(s);
          slot = slot == RING - 1 ? 0 : slot + 1, into = into == RING - 1 ? 0 : into + 1;
        }
      }
      w_landed<0>();
    }
    __syncthreads(); // (the sums take the rings' place)
  } else {
    const long long whole = m1 - ATB_STEP; // last start of a step without a guard
    Step s0, s1;
    long long m = m0 + ATB_STEP * wave; // a step in GM is this wavefront's
    auto fetch = [&](Step &s, long long at) {
      if (at <= whole)
        load(s, at, false);
      else
        load(s, at < m1 ? at : m1 - 1, true);
    };
    if (m < m1) {
      look_up(s0, m);
      look_up(s1, m + ATB_STEP * GM);
      fetch(s0, m);
      look_up(s0, m + 2 * ATB_STEP * GM);
      for (;;) {
        const long long ma = m + ATB_STEP * GM;
        if (ma < m1) {
          fetch(s1, ma);
          look_up(s1, ma + 2 * ATB_STEP * GM);
        }
        compute(s0);
        if (ma >= m1)
          break;
        const long long mb = ma + ATB_STEP * GM;
        if (mb < m1) {
          fetch(s0, mb);
          look_up(s0, mb + 2 * ATB_STEP * GM);
        }
        compute(s1);
        if (mb >= m1)
          break;
        m = mb;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        sTile[wave * TILE + ((i * NT + j) * 16 + v) * 64 + lane] = acc[0][i][j][v] + acc[1][i][j][v];
  if (tid == 0)
    *sAgain = 0;
  if (sums)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const float both = ds[j] + __shfl_xor(ds[j], 32);
      if (q == 0)
        sBias[wave * 32 * NT + NT * c + j] = both;
    }
  __syncthreads();
  if (sums && tid < 32 * NT && n0 + tid < N) {
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < GM; ++g)
      sum += sBias[g * 32 * NT + tid];
    unsafeAtomicAdd(db + n0 + tid, sum);
  }
  // element e of the tile: register v of lane l of sub-tile (i, j): row (of dW)
  // MT (8 (v / 4) + 4 (l / 32) + v % 4) + i, column NT (l % 32) + j
  auto add = [&](int e) {
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < GM; ++g)
      sum += sTile[g * TILE + e];
    return sum;
  };
  auto put = [&](int e, float sum) {
    const int l = e & 63, v = (e >> 6) & 15, ij = e >> 10;
    const int kk = k0 + MT * (8 * (v / 4) + 4 * (l >> 5) + v % 4) + ij / NT;
    const int nn = n0 + NT * (l & 31) + ij % NT;
    if (kk < K && nn < N)
      unsafeAtomicAdd(dW + (long long)kk * N + nn, sum);
  };
  unsigned again = 0; // this lane's elements that are to be taken again
  for (int e = tid; e < TILE; e += 64 * GM) {
    const float sum = add(e);
    if (doubtful<PL>(sum))
      again |= 1u << (e / (64 * GM));
    else
      put(e, sum);
  }
  if (again)
    *sAgain = 1;
  __syncthreads();
  if (*sAgain) { // the workgroup's rows on the fp32 MFMA, two a step
    floatx16 plain[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          plain[i][j][v] = 0.f;
#pragma unroll 4
    for (long long r0 = m0 + 2 * wave; r0 < m1; r0 += 2 * GM) {
      const int l = __lane_id(); // (anew: its columns need no registers until here)
      const long long r = r0 + (l >> 5);
      int ka = k0 + MT * (l & 31), na = n0 + NT * (l & 31);
      ka = ka + MT <= K ? ka : K - MT;
      na = na + NT <= N ? na : N - NT;
      float a[MT], d[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if constexpr (GATHER) {
          const int rule = r < m1 ? gs.rules[ka / gs.nIn * ((M + ATB_STEP - 1) / ATB_STEP * ATB_STEP) + r] : -1;
          a[i] = rule >= 0 ? A[(long long)rule * gs.nIn + ka % gs.nIn + i] : 0.f;
        } else {
          a[i] = r < m1 ? A[r * K + ka + i] : 0.f;
        }
#pragma unroll
      for (int j = 0; j < NT; ++j)
        d[j] = r < m1 ? D[r * N + na + j] : 0.f;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          plain[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], d[j], plain[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          sTile[wave * TILE + ((i * NT + j) * 16 + v) * 64 + lane] = plain[i][j][v];
    __syncthreads();
    for (int e = tid; e < TILE; e += 64 * GM)
      if (again >> (e / (64 * GM)) & 1)
        put(e, add(e));
  }
}

template <int MT, int NT, bool GATHER, bool LINES>
__global__ void __launch_bounds__(64 * atb_waves(MT, NT, LINES), atb_waves(MT, NT, LINES) / 4)
    k_atb_planes(const float *__restrict__ A, const float *__restrict__ D,
                 float *__restrict__ dW, float *__restrict__ db, long long M, int K, int N, int nTiles,
                 long long rowsPerSplit, GatherSource gs, const float *zeros) {
  // (the tiles of a range of rows, which read the same, to one XCD)
  const unsigned at = xcd_eighth(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const long long m0 = at / gridDim.x * rowsPerSplit, m1 = m0 + rowsPerSplit < M ? m0 + rowsPerSplit : M;
  atb_tile<MT, NT, GATHER, LINES, atb_waves(MT, NT, LINES)>(A, D, dW, db, M, K, N, nTiles, gs, zeros, at % gridDim.x,
                                                            m0, m1);
}
constexpr size_t atb_lds(int MT, int NT, bool GATHER, bool LINES, int GM) {
  const size_t sums = ((size_t)GM * 32 * MT * 32 * NT + GM * 32 * NT + 1) * sizeof(float);
  const size_t rings = (size_t)GM * (atb_ring(MT, NT) * 2048 * (MT + NT) + (GATHER ? 2 * MT * 256 : 0));
  return LINES && rings > sums ? rings : sums;
}

template <int MT, int NT, bool GATHER, bool LINES>
static int launch_atb(scn_ctx *ctx, const float *A, const float *D, float *dW, float *db,
                      long long M, int K, int N, long long rows, const GatherSource &gs) {
  constexpr int GM = atb_waves(MT, NT, LINES);
  constexpr size_t lds = atb_lds(MT, NT, GATHER, LINES, GM);
  static OncePerDevice configured;
  const int rc = configured.run(ctx->device, [&]() {
    return hipFuncSetAttribute(reinterpret_cast<const void *>(k_atb_planes<MT, NT, GATHER, LINES>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess
               ? SCN_OK
               : SCN_ERR_HIP;
  });
  SCN_REQUIRE(rc == SCN_OK, SCN_ERR_HIP, "hipFuncSetAttribute failed");
  const int nTiles = scn_ceil_div(N, 32 * NT);
  const long long tiles = (long long)scn_ceil_div(K, 32 * MT) * nTiles;
  hipLaunchKernelGGL((k_atb_planes<MT, NT, GATHER, LINES>), dim3((unsigned)tiles, (unsigned)((M + rows - 1) / rows)),
                     dim3(64 * GM), lds, ctx->stream, A, D, dW, db, M, K, N, nTiles, rows, gs, ctx->d_zeros);
  return SCN_OK;
}
template <int MT, int NT>
static int launch_atb(scn_ctx *ctx, const float *A, const float *D, float *dW, float *db, long long M, int K, int N,
                      long long rows, const GatherSource *gs, bool lines) {
  if constexpr (MT == 2 && NT == 2) // (gathered by lines only: see below)
    return gs      ? launch_atb<MT, NT, true, true>(ctx, A, D, dW, db, M, K, N, rows, *gs)
           : lines ? launch_atb<MT, NT, false, true>(ctx, A, D, dW, db, M, K, N, rows, GatherSource())
                   : launch_atb<MT, NT, false, false>(ctx, A, D, dW, db, M, K, N, rows, GatherSource());
  else if (gs)
    return lines ? launch_atb<MT, NT, true, true>(ctx, A, D, dW, db, M, K, N, rows, *gs)
                 : launch_atb<MT, NT, true, false>(ctx, A, D, dW, db, M, K, N, rows, *gs);
  else
    return lines ? launch_atb<MT, NT, false, true>(ctx, A, D, dW, db, M, K, N, rows, GatherSource())
                 : launch_atb<MT, NT, false, false>(ctx, A, D, dW, db, M, K, N, rows, GatherSource());
}

int scn_atb_planes(scn_ctx *ctx, const float *A, const float *D, float *dW, float *db,
                   long long M, int K, int N, const GatherSource *gs) {
  // (requests of four columns, in one filter position each)
  const bool lines = K % 4 == 0 && N % 4 == 0 && (!gs || gs->nIn % 4 == 0) && (((uintptr_t)A | (uintptr_t)D) & 15) == 0;
  // Pairs of columns are loaded as one: K (N) even for two row (column) tiles.  (Two by two
  // tiles not by lines, of gathered rows or with sums: 264 bytes a lane spilled)
  const bool pairsA = (gs ? gs->nIn : K) % 2 == 0 && ((uintptr_t)A & 7) == 0, pairsD = N % 2 == 0 && ((uintptr_t)D & 7) == 0;
  AtbChoice c = atb_choose(ctx->numCU, M, K, N, lines, pairsA, pairsD, !gs && (!db || lines));
  // (through rules they take a quarter longer than of plain rows: us, two by one and two by
  // two, 150000 x 1728 x 64 257, 209; 139000 x 384 x 128 118, 96; 12000 x 1152 x 128 38, 33.5;
  // 30000 x 256 x 128, which costs 20.3 and 19.5 by atb_choose, 22, 25; 60000 x 256 x 64 22, 24.7)
  if (gs && lines) {
    const AtbChoice two = atb_choose(ctx->numCU, M, K, N, true, pairsA, pairsD, true);
    if (1.25 * two.cost < c.cost)
      c = two;
  }
  SCN_REQUIRE(c.tile >= 0, SCN_ERR_CAPACITY, "scn_sgemm_AtB: K %d N %d", K, N);
  switch (c.tile) { // (as in atbTiles)
  case 1:
    return launch_atb<2, 1>(ctx, A, D, dW, db, M, K, N, c.rows, gs, lines);
  case 2:
    return launch_atb<1, 2>(ctx, A, D, dW, db, M, K, N, c.rows, gs, lines);
  case 3:
    return launch_atb<2, 2>(ctx, A, D, dW, db, M, K, N, c.rows, gs, lines);
  }
  return launch_atb<1, 1>(ctx, A, D, dW, db, M, K, N, c.rows, gs, lines);
}

// ---- the weight gradients of all layers of a net in one launch.  Each by itself is
// a wave of workgroups that begins (some 4 us of trips to memory and of sums), has
// a few microseconds of rows and ends in as many atomics again.  Here the tiles of
// all of them, cut into ranges of rows, lie end to end, and every compute unit has
// one workgroup that takes an equal part of that line: the end of one tile's range,
// whole ones, the beginning of another.  So all end together, which workgroups of
// one range each do not: their number is that of the compute units only by chance,
// and a layer's ranges are shorter or longer than the next one's.  The seven layers of
// a batch of 100 drawings (83597 x 12 x 32 to 100 x 192 x 100): 81 us in launches of
// their own, 57 with workgroups of one range each, 51 so; without the first layer 65,
// 50, 48.  12 batches of drawings 6515 -> 6260 us, of voxel models 5430 -> 5285.
// The tiles are two by two where dW has the columns, by eight wavefronts: its rows and
// D's are then read half as often, and split into planes two thirds as often, as for tiles
// of two by one by twelve wavefronts, which a step took for as long as all its requests,
// vector instructions and MFMAs one after the other (0.13 us a wavefront on a compute
// unit; with any one of them left out 0.11): seven layers of drawings 47 -> 39 us, six of
// voxel models 39.5 -> 34.  Wider tiles shared by the wavefronts would end in more
// atomics, of which 256 workgroups of 4096 each are some 5 us.
// What is left of up to half a tile at the end of dW's columns is two by one; rows that
// are no whole requests, a net's first layer, one by one.
constexpr int ATB_ENTRIES = 2 * SCN_ATB_MAX; // (a layer may be two of them)
struct AtbList {
  const float *A[ATB_ENTRIES], *D[ATB_ENTRIES];
  float *dW[ATB_ENTRIES], *db[ATB_ENTRIES];
  const int *rules[ATB_ENTRIES]; // null: plain rows
  const float *zeros;
  int M[ATB_ENTRIES], K[ATB_ENTRIES], N[ATB_ENTRIES], fs[ATB_ENTRIES];
  int steps[ATB_ENTRIES]; // of a range, ATB_MANY ATB_STEP rows each
  int first[ATB_ENTRIES]; // place in the line
  // the first of its columns of dW, tiles of columns, of what kind.  (Words, not bytes: with
  // an array of bytes beside them the compiler takes its index into the base of the
  // pointers' scalar loads, whose address loses the last two bits of each of its parts.)
  int column[ATB_ENTRIES], nTiles[ATB_ENTRIES], kind[ATB_ENTRIES];
  int count, length, part; // of the line; of a workgroup
};
constexpr int ATB_MANY = 8; // wavefronts
static_assert(ATB_MANY * ATB_STEP == ATB_MANY_ROWS, "a step of a range");
static_assert(sizeof(AtbList) <= 4096, "a kernel's arguments");
__global__ void __launch_bounds__(64 * ATB_MANY, ATB_MANY / 4) k_atb_many(AtbList l) {
  static_assert(ATB_ENTRIES <= 64, "a lane an entry");
  int pos = (int)xcd_eighth(blockIdx.x, gridDim.x) * l.part; // (neighbours to one XCD)
  const int end = pos + l.part < l.length ? pos + l.part : l.length;
#pragma unroll 1
  while (pos < end) { // uniform
    const int lane = __lane_id(); // (anew)
    const int t = __popcll(__ballot(lane < l.count && pos >= l.first[lane < ATB_ENTRIES ? lane : 0])) - 1;
    const int K = l.K[t], N = l.N[t], steps = l.steps[t], M = l.M[t], kind = l.kind[t];
    GatherSource gs = GatherSource();
    gs.rules = l.rules[t];
    gs.fs = l.fs[t];
    gs.nIn = K / gs.fs;
    gs.zeros = l.zeros;
    const int cost = atbKinds[kind].step, begin = atbKinds[kind].tile, whole = begin + steps * cost;
    // the range of a tile that this is in, tile after tile of one range of rows
    const unsigned unit = (unsigned)(pos - l.first[t]) / whole;
    const int from = pos - l.first[t] - (int)unit * whole;
    const int to = whole - from < end - pos ? whole : from + end - pos;
    auto step = [&](int place) { return place <= begin ? 0 : (place - begin + cost - 1) / cost; };
    pos += to - from;
    const int nTiles = l.nTiles[t];
    const unsigned tiles = (unsigned)(K + 32 * atbKinds[kind].mt - 1) / (32 * atbKinds[kind].mt) * nTiles;
    const long long r0 = (long long)(unit / tiles) * steps;
    const long long m0 = (r0 + step(from)) * ATB_MANY_ROWS, m1 = (r0 + step(to)) * ATB_MANY_ROWS;
    if (m0 >= (m1 < M ? m1 : M))
      continue;
    __syncthreads(); // (the one before is done with LDS)
#define SCN_ATB_TILE(MT, NT, GATHER, LINES)                                                                   \
  atb_tile<MT, NT, GATHER, LINES, ATB_MANY>(l.A[t], l.D[t], l.dW[t], l.db[t], M, K, N, nTiles, gs, l.zeros, \
                                            unit % tiles, m0, m1 < M ? m1 : M, l.column[t])
    if (kind == ATB_WIDE && gs.rules)
      SCN_ATB_TILE(2, 2, true, true);
    else if (kind == ATB_WIDE)
      SCN_ATB_TILE(2, 2, false, true);
    else if (kind == ATB_FIRST)
      SCN_ATB_TILE(1, 1, true, false);
    else if (gs.rules)
      SCN_ATB_TILE(2, 1, true, true);
    else
      SCN_ATB_TILE(2, 1, false, true);
#undef SCN_ATB_TILE
  }
}
// how an item is taken among many: -1: not one for it
static int atb_many_kind(const scn_atb_item &it) {
  const int K = it.fs * it.nIn;
  if (it.M > (1 << 30) || it.N % 4 || (((uintptr_t)it.d_in | (uintptr_t)it.d_D) & 15))
    return -1;
  if (it.d_positions && it.nIn % 4)
    return K <= 32 ? ATB_FIRST : -1;
  return K % 4 ? -1 : it.N > 32 ? ATB_WIDE : ATB_NARROW;
}
int scn_atb_planes_many(scn_ctx *ctx, const scn_atb_item *items, int nItems) {
  AtbList l;
  l.count = 0;
  l.zeros = ctx->d_zeros;
  AtbShape shape[SCN_ATB_MAX];
  bool joined[SCN_ATB_MAX];
  int kinds[SCN_ATB_MAX];
  for (int k = 0; k < nItems; ++k) {
    kinds[k] = atb_many_kind(items[k]);
    shape[k] = {items[k].M, items[k].fs * items[k].nIn, items[k].N, kinds[k] < 0 ? 0 : atbKinds[kinds[k]].mt,
                kinds[k] < 0 ? 0 : atbKinds[kinds[k]].step / atbKinds[kinds[k]].nt};
  }
  atb_join(ctx->numCU, shape, nItems, joined);
  long long tiles[ATB_ENTRIES], steps[ATB_ENTRIES], work = 0;
  auto enter = [&](const scn_atb_item &it, int kind, int column, int columns) {
    const int c = l.count++, K = it.fs * it.nIn;
    const AtbKind &x = atbKinds[kind];
    l.A[c] = it.d_in, l.D[c] = it.d_D, l.dW[c] = it.d_dW, l.db[c] = it.d_db, l.rules[c] = it.d_positions;
    l.M[c] = (int)it.M, l.K[c] = K, l.N[c] = it.N, l.fs[c] = it.fs, l.kind[c] = kind;
    l.column[c] = column, l.nTiles[c] = (int)scn_ceil_div(columns, 32 * x.nt);
    tiles[c] = scn_ceil_div(K, 32 * x.mt) * l.nTiles[c], steps[c] = scn_ceil_div(it.M, ATB_MANY_ROWS);
    work += tiles[c] * steps[c] * x.step;
  };
  for (int k = 0; k < nItems; ++k) {
    const scn_atb_item &it = items[k];
    if (it.M > 0 && !joined[k]) {
      GatherSource gs = GatherSource();
      gs.rules = it.d_positions;
      gs.fs = it.fs;
      gs.nIn = it.nIn;
      gs.zeros = ctx->d_zeros;
      SCN_TRY(scn_atb_planes(ctx, it.d_in, it.d_D, it.d_dW, it.d_db, it.M, shape[k].K, it.N, it.d_positions ? &gs : nullptr));
    }
    if (!joined[k])
      continue;
    const int rest = kinds[k] == ATB_WIDE && (it.N - 1) % 64 < 32 ? (it.N - 1) % 64 + 1 : 0; // (columns of half a tile)
    enter(it, kinds[k], 0, it.N - rest);
    if (rest)
      enter(it, ATB_NARROW, it.N - rest, rest);
  }
  if (l.count == 0)
    return SCN_OK;
  // ranges about as long as a workgroup's part, all tiles of one side by side: they
  // read the same rows
  const long long part = scn_ceil_div(work, ctx->numCU);
  long long length = 0;
  for (int c = 0; c < l.count; ++c) {
    const AtbKind &x = atbKinds[l.kind[c]];
    long long ranges = (steps[c] * x.step + part / 2) / part;
    ranges = ranges < 1 ? 1 : ranges > steps[c] ? steps[c] : ranges;
    l.steps[c] = (int)scn_ceil_div(steps[c], ranges);
    l.first[c] = (int)length;
    length += tiles[c] * scn_ceil_div(steps[c], l.steps[c]) * (x.tile + (long long)l.steps[c] * x.step);
  }
  l.length = (int)length; // (at most SCN_ATB_MAX times what an item may be, and a range more of each)
  l.part = scn_ceil_div(length, ctx->numCU);
  constexpr size_t lds = atb_lds(2, 2, true, true, ATB_MANY);
  static_assert(lds <= 160 << 10 && lds >= atb_lds(2, 2, false, true, ATB_MANY) && lds >= atb_lds(2, 1, true, true, ATB_MANY) &&
                    lds >= atb_lds(2, 1, false, true, ATB_MANY) && lds >= atb_lds(1, 1, true, false, ATB_MANY),
                "one size for all");
  static OncePerDevice configured;
  const int rc = configured.run(ctx->device, [&]() {
    return hipFuncSetAttribute(reinterpret_cast<const void *>(k_atb_many), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds) == hipSuccess
               ? SCN_OK
               : SCN_ERR_HIP;
  });
  SCN_REQUIRE(rc == SCN_OK, SCN_ERR_HIP, "hipFuncSetAttribute failed");
  hipLaunchKernelGGL(k_atb_many, dim3((unsigned)scn_ceil_div(length, l.part)), dim3(64 * ATB_MANY), lds, ctx->stream, l);
  return SCN_OK;
}
