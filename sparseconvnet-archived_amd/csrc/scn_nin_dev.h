// What the NetworkInNetwork kernels of several files share: the epilogue's
// constants, the source of a gathered matrix, bf16 conversions.
#pragma once
#include "scn_common.h"

struct Epilogue {
  const float *bias;
  const float *prelu;
  float p;
  float slope;
  int act;
};

// Bias, p and activation of one column, branch-free: every supported activation is v > 0 ? v : v * slope with slope
// 1 (none), 0 (ReLU), a constant (leaky) or PReLU's learnt per-column value.
struct ColEpilogue {
  float pb;    // p * bias[n]
  float p;
  float slope;
};
__device__ __forceinline__ ColEpilogue load_col(const Epilogue &e, int n) {
  ColEpilogue c;
  c.p = e.p;
  c.pb = e.p * e.bias[n];
  c.slope = e.act == SCN_PRELU
                ? e.prelu[n]
                : (e.act == SCN_RELU ? 0.f
                                     : (e.act == SCN_LEAKYRELU || e.act == SCN_VLEAKYRELU ? e.slope : 1.f));
  return c;
}
__device__ __forceinline__ float finish(float acc, const ColEpilogue &c) {
  const float v = c.p * acc + c.pb;
  const float neg = c.slope == 0.f ? 0.f : v * c.slope;
  return v > 0.f ? v : neg;
}

//
// GATHER: A is never materialised.  Row m of A is the receptive field of
// output site m, column q * nIn + c = channel c of input row
// rules[m * fs + q] (what scn_gather_rows would have written).
#define GF_MAX_FS 27
struct GatherSource {
  const int *rules;   // [M x fs]
  int fs;             // rule-row width
  int nIn;            // channels of the gathered matrix, nIn % 4 == 0
  unsigned magic;     // floor(2^32 / nIn) + 1: k / nIn == mulhi(k, magic) for k nIn < 2^32
  const float *zeros; // at least nIn zeros: the row a negative rule stands for
  // a negative rule adds nothing, and not 0 times its weights: the same but for
  // weights that are not finite (scn_planes_forward with three planes only)
  int namedOnly;
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned pack_bf16x2(float a, float b) {
  floatx2 f = {a, b};
  bf16x2 h = __builtin_convertvector(f, bf16x2);
  return __builtin_bit_cast(unsigned, h);
}

// scn_nin.hip: nin_forward takes the fused convolution of SCN_FP32_PLANES to
// scn_planes_forward, whatever the rows
bool scn_conv_takes_planes(const float *A, const float *W, const float *out, int K, int N);
// scn_conv_nin_forward_image without bias and activation, in SCN_FP32_PLANES;
// with scn_conv_takes_planes, GatherSource::namedOnly
int scn_conv_named(scn_ctx *ctx, const float *d_in, const int32_t *d_rules, int fs, int nIn, const float *d_W,
                   const void *d_image, float *d_out, int64_t M, int N);
// scn_planes.hip: the contraction with fp32 operands as `planes` bf16 planes
bool scn_planes_shape(int K);
// ... takes the split contraction: few rows
bool scn_planes_splitk(scn_ctx *ctx, int planes, long long M, int K, int N);
// (image: W as scn_weight_images_many leaves it, or null; a16: A holds bf16 rows, those
// of A32 rounded)
int scn_planes_forward(scn_ctx *ctx, int planes, const float *A, const float *W,
                       float *out, long long M, int K, int N,
                       const Epilogue &ep, const GatherSource *gs, bool a16,
                       const void *image = nullptr, const float *A32 = nullptr);
// dW += A^T D, db (may be null) += the column sums of D (gs: the rows of A through
// rules, position by position)
int scn_atb_planes(scn_ctx *ctx, const float *A, const float *D, float *dW, float *db,
                   long long M, int K, int N, const GatherSource *gs = nullptr);
// what scn_weight_images_later left, made now
int scn_images_now(scn_ctx *ctx);
int scn_atb_planes_many(scn_ctx *ctx, const scn_atb_item *items, int nItems);
// out = A Wt^T; false: the caller's other way, or (transpose) scn_planes_forward
// on the transpose
bool scn_abt_narrow(scn_ctx *ctx, const float *A, const float *W, float *out, long long M, int n, int K);
bool scn_planes_abt(scn_ctx *ctx, const float *A, const float *Wt, float *out,
                    long long M, int K, int N, const Epilogue &ep, int *rc, bool *transpose);
