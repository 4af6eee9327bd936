// The planes of a float, and the images of weights made of them: scn_planes.hip, and
// scn_nin.hip where images are made beside a net's first layer.
#pragma once
#include "scn_nin_dev.h"

// The PL planes of two floats, a word each.
template <int PL> __device__ __forceinline__ void split2(float a, float b, unsigned (&w)[PL]) {
#pragma unroll
  for (int l = 0; l < PL; ++l) {
    w[l] = pack_bf16x2(a, b);
    if (l + 1 < PL) {
      a -= __uint_as_float(w[l] << 16);
      b -= __uint_as_float(w[l] & 0xffff0000u);
    }
  }
}
// The PL planes of eight floats, each as an MFMA operand.
template <int PL>
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&p)[PL]) {
  unsigned w[4][PL];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    split2<PL>(x[2 * i], x[2 * i + 1], w[i]);
#pragma unroll
  for (int l = 0; l < PL; ++l)
    p[l] = __builtin_bit_cast(bf16x8, uint4{w[0][l], w[1][l], w[2][l], w[3][l]});
}

// The image of W that k_nin_lines reads: a chunk of 1 KB for every tile of 32
// columns, block of 32 k, plane and step of 16 k, in that order.  Those of several
// layers in one launch (each by itself takes 3 us, whatever it holds).
//   fs 0: W is [K x N]; -1: [N x K]; more: the filters of the layer whose input's
//   gradient this is, [fs N x K / fs], its rule positions in the same order.
template <int PL>
__device__ __forceinline__ void weight_image(const float *__restrict__ W, unsigned char *__restrict__ image, int K, int N,
                                             int fs, long long item) {
  const int T = K / 32, columns = (N + 31) / 32 * 32;
  if (item >= (long long)T * 4 * columns)
    return;
  const int column = (int)(item % columns), kg = (int)(item / columns); // (eight k, column)
  const int n = column < N ? column : N - 1, k = 8 * kg;
  float v[8];
  if (fs == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = W[(long long)(k + i) * N + n];
  } else {
    const int width = fs < 0 ? K : K / fs, f = k / width; // (a multiple of 8)
    const float *const src = W + ((long long)f * N + n) * width + (k - f * width);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = src[i];
  }
  bf16x8 p[PL];
  split8<PL>(v, p);
#pragma unroll
  for (int l = 0; l < PL; ++l)
    *reinterpret_cast<bf16x8 *>(image + ((((long long)(column / 32) * T + kg / 4) * PL + l) * 2 + kg / 2 % 2) * 1024 +
                                (kg & 1) * 512 + (column & 31) * 16) = p[l];
}
// a workgroup of 256 lanes, the block'th of the list's
__device__ __forceinline__ void weight_images_block(const ImageList &l, unsigned block) {
  const int lane = threadIdx.x & 63;
  const int x = __popcll(__ballot(lane < l.count && block >= l.firstBlock[lane < SCN_IMAGES_MAX ? lane : 0])) - 1;
  const long long item = (long long)(block - l.firstBlock[x]) * 256 + threadIdx.x;
  if (l.planes[x] == 3)
    weight_image<3>(l.W[x], l.image[x], l.K[x], l.N[x], l.fs[x], item);
  else
    weight_image<1>(l.W[x], l.image[x], l.K[x], l.N[x], l.fs[x], item);
}
