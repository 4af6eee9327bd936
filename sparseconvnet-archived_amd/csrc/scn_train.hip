// The backward pass and the weight update behind the C ABI: what the layers'
// backwards() call in the reference, one entry point per free function there.
//   softmax + NLL gradient     SoftmaxClassifier.cu:7-14
//   activation derivatives     SigmoidLayer.cu:23-177, NetworkInNetworkPReLULayer.cu:25-47
//   bias gradient              columnSum, NetworkInNetworkLayer.cu:84-105
//   weight gradient  A^T D     d_rowMajorSGEMM_alphaAtB_betaC, utilities.cu:144-155
//   input gradient   D W^T     d_rowMajorSGEMM_alphaABt_betaC, utilities.cu:157-168
//   weight update              dGradientDescent(KeepPositive), NetworkInNetworkLayer.cu:27-41
//   convolution                dPropBackwardFromMatrixMultiplyOutput, ConvolutionalLayer.cu:42-63
//   max-pooling                dMaxPoolBackProp, MaxPoolingLayer.cu:74-82
//   terminal pooling           dTerminalPoolBackProp, TerminalPoolingLayer.cu:48-62
#include <mutex>
#include "scn_grids_dev.h"
#include "scn_nin_dev.h"
#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

typedef float floatx4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- softmax
__global__ void k_softmax_grad(const float *__restrict__ probs,
                               const int *__restrict__ labels,
                               float *__restrict__ delta, long long total,
                               int N, float *copy) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total)
    return;
  long long k = i / N;
  int c = (int)(i - k * N);
  const float p = probs[i];
  delta[i] = p - (c == labels[k] ? 1.f : 0.f);
  if (copy) // (the host's memory, perhaps)
    copy[i] = p;
}

static int softmax_grad(scn_ctx *ctx, const float *d_probs,
                        const int32_t *d_labels, float *d_delta,
                        int64_t batch, int N, float *copy) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_softmax_grad: null context");
  SCN_REQUIRE(batch >= 0 && N >= 1, SCN_ERR_ARG,
              "scn_softmax_grad: batch %lld N %d", (long long)batch, N);
  if (batch == 0)
    return SCN_OK;
  SCN_REQUIRE(d_probs && d_labels && d_delta, SCN_ERR_ARG,
              "scn_softmax_grad: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  long long total = batch * N;
  hipLaunchKernelGGL(k_softmax_grad, dim3(scn_ceil_div(total, 256)), dim3(256),
                     0, ctx->stream, d_probs, d_labels, d_delta, total, N, copy);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}
extern "C" int scn_softmax_grad(scn_ctx *ctx, const float *d_probs,
                                const int32_t *d_labels, float *d_delta,
                                int64_t batch, int N) {
  return softmax_grad(ctx, d_probs, d_labels, d_delta, batch, N, nullptr);
}
// ... and the probabilities to `copy` (device or pinned host memory), which would be
// a launch of its own (2.9 us of a training batch)
extern "C" int scn_softmax_grad_copy(scn_ctx *ctx, const float *d_probs,
                                     const int32_t *d_labels, float *d_delta,
                                     int64_t batch, int N, float *copy) {
  SCN_REQUIRE(copy || batch == 0, SCN_ERR_ARG, "scn_softmax_grad_copy: null copy");
  return softmax_grad(ctx, d_probs, d_labels, d_delta, batch, N, copy);
}

// ------------------------------------------------- activation derivatives
// One pass over the [M x N] gradient: multiplies it in place by the
// derivative of the activation (expressed through the layer's output, as the
// reference does), and leaves the column sums of the result in db (the bias
// gradient) and, for PReLU, the slope gradient in dprelu.  A lane owns V
// neighbouring columns (four where the rows are 16-byte aligned) and takes four
// rows per trip, so that eight 16-byte loads are in flight; the lanes of a row
// lie side by side, as many rows to a workgroup as fit.
__device__ __forceinline__ float act_derivative(int act, float b, float d,
                                                float alpha, float &t) {
  switch (act) {
  case SCN_RELU:
    return b > 0 ? d : 0.f;
  case SCN_LEAKYRELU:
  case SCN_VLEAKYRELU:
    return b > 0 ? d : d * alpha;
  case SCN_TANH:
    return d * (1 + b) * (1 - b);
  case SCN_SIGMOID:
    return d * b * (1 - b);
  case SCN_PRELU:
    t += d * (b > 0 ? 0.f : b / alpha);
    return b > 0 ? d : d * alpha;
  default: // SOFTMAX (folded into the classifier's gradient), NOSIGMOID
    return d;
  }
}
#define ACTB_THREADS 512
template <int V>
__global__ __launch_bounds__(ACTB_THREADS) void k_act_backward(
    const float *__restrict__ out, const float *delta, float *dst, long long M,
    int N, int act, const float *__restrict__ prelu, float *__restrict__ db,
    float *__restrict__ dprelu, int P) {
  typedef float vec __attribute__((ext_vector_type(V)));
  __shared__ float sS[ACTB_THREADS * V], sT[ACTB_THREADS * V];
  // P lanes a row, rows of lanes; lanes beyond the last whole row idle
  const int rows = ACTB_THREADS / P;
  const int tx = threadIdx.x % P, ty = threadIdx.x / P;
  const int c = (blockIdx.x * P + tx) * V;
  float s[V], t[V];
#pragma unroll
  for (int i = 0; i < V; ++i)
    s[i] = t[i] = 0.f;
  if (c < N && ty < rows) {
    float alpha[V];
#pragma unroll
    for (int i = 0; i < V; ++i)
      alpha[i] = act == SCN_PRELU ? prelu[c + i] : act == SCN_LEAKYRELU ? 0.01f : 0.333f;
    const long long step = (long long)rows * gridDim.y;
    long long r = (long long)blockIdx.y * rows + ty;
    for (; r + 3 * step < M; r += 4 * step) {
      vec b[4], d[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        b[u] = *reinterpret_cast<const vec *>(out + (r + u * step) * N + c);
        d[u] = *reinterpret_cast<const vec *>(delta + (r + u * step) * N + c);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int i = 0; i < V; ++i) {
          d[u][i] = act_derivative(act, b[u][i], d[u][i], alpha[i], t[i]);
          s[i] += d[u][i];
        }
        *reinterpret_cast<vec *>(dst + (r + u * step) * N + c) = d[u];
      }
    }
    for (; r < M; r += step) {
      vec d = *reinterpret_cast<const vec *>(delta + r * N + c);
      const vec b = *reinterpret_cast<const vec *>(out + r * N + c);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        d[i] = act_derivative(act, b[i], d[i], alpha[i], t[i]);
        s[i] += d[i];
      }
      *reinterpret_cast<vec *>(dst + r * N + c) = d;
    }
  }
#pragma unroll
  for (int i = 0; i < V; ++i) {
    sS[threadIdx.x * V + i] = s[i];
    sT[threadIdx.x * V + i] = t[i];
  }
  __syncthreads();
  // column x of the workgroup's P V: the sum over its rows of lanes
  for (int x = threadIdx.x; x < P * V; x += ACTB_THREADS) {
    const int col = blockIdx.x * P * V + x;
    if (col >= N)
      continue;
    float sum = 0.f, sumT = 0.f;
    for (int k = 0; k < rows; ++k) {
      sum += sS[k * P * V + x];
      sumT += sT[k * P * V + x];
    }
    unsafeAtomicAdd(db + col, sum);
    if (act == SCN_PRELU)
      unsafeAtomicAdd(dprelu + col, sumT);
  }
}

static int activation_backward(scn_ctx *ctx, const float *d_out,
                               const float *d_delta, float *d_dst, int64_t M, int N, int act,
                               const float *d_prelu, float *d_db,
                               float *d_dprelu, bool clear) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_activation_backward: null context");
  SCN_REQUIRE(M >= 0 && N >= 1, SCN_ERR_ARG,
              "scn_activation_backward: M %lld N %d", (long long)M, N);
  SCN_REQUIRE(act >= SCN_NOSIGMOID && act <= SCN_SIGMOID, SCN_ERR_ARG,
              "scn_activation_backward: activation %d", act);
  SCN_REQUIRE(d_db, SCN_ERR_ARG, "scn_activation_backward: null d_db");
  SCN_REQUIRE(act != SCN_PRELU || (d_prelu && d_dprelu), SCN_ERR_ARG,
              "scn_activation_backward: PReLU needs slopes and their gradient");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  if (clear) {
    SCN_TRY(scn_fill32(ctx, d_db, 0, (size_t)N));
    if (act == SCN_PRELU)
      SCN_TRY(scn_fill32(ctx, d_dprelu, 0, (size_t)N));
  }
  if (M == 0)
    return SCN_OK;
  SCN_REQUIRE(d_out && d_delta && d_dst, SCN_ERR_ARG,
              "scn_activation_backward: null buffer");
  const int V = N % 4 == 0 && (((uintptr_t)d_out | (uintptr_t)d_delta | (uintptr_t)d_dst) & 15) == 0 ? 4 : 1;
  // (a row of up to 64 lanes: with fewer rows of lanes the sums below are short)
  const int colBlocks = scn_ceil_div(N, V * 64);
  const int P = scn_ceil_div(N / V, colBlocks);
  // every workgroup ends with one atomic per column onto the same N addresses,
  // and those serialise (about 25 ns each): few, long-lived workgroups, one per
  // compute unit (60478 x 64: 11.4 -> 8.2 us)
  const int rows = ACTB_THREADS / P;
  int rowBlocks = scn_ceil_div(M, 4 * rows); // at least four rows per lane
  const int cap = scn_ceil_div(ctx->numCU, colBlocks);
  if (rowBlocks > cap)
    rowBlocks = cap;
  hipLaunchKernelGGL((V == 4 ? k_act_backward<4> : k_act_backward<1>), dim3(colBlocks, rowBlocks),
                     dim3(ACTB_THREADS), 0, ctx->stream, d_out, d_delta, d_dst, (long long)M, N, act,
                     d_prelu, d_db, d_dprelu, P);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

extern "C" int scn_activation_backward(scn_ctx *ctx, const float *d_out,
                                       float *d_delta, int64_t M, int N,
                                       int act, const float *d_prelu,
                                       float *d_db, float *d_dprelu) {
  return activation_backward(ctx, d_out, d_delta, d_delta, M, N, act, d_prelu,
                             d_db, d_dprelu, true);
}

extern "C" int scn_activation_backward_acc(scn_ctx *ctx, const float *d_out,
                                           float *d_delta, int64_t M, int N,
                                           int act, const float *d_prelu,
                                           float *d_db, float *d_dprelu) {
  return activation_backward(ctx, d_out, d_delta, d_delta, M, N, act, d_prelu,
                             d_db, d_dprelu, false);
}
extern "C" int scn_activation_backward_to(scn_ctx *ctx, const float *d_out,
                                          const float *d_delta, float *d_dst,
                                          int64_t M, int N, int act,
                                          const float *d_prelu, float *d_db,
                                          float *d_dprelu, int accumulate) {
  return activation_backward(ctx, d_out, d_delta, d_dst, M, N, act, d_prelu,
                             d_db, d_dprelu, !accumulate);
}

// The number of rows is the caller's, whatever scn_ctx_rows_from says to the
// forward calls, whose kernels run in some of the backward ones
struct OwnRows {
  scn_ctx *ctx;
  const long long *meta;
  explicit OwnRows(scn_ctx *c) : ctx(c), meta(c->d_meta) { c->d_meta = nullptr; }
  ~OwnRows() { ctx->d_meta = meta; }
};

// ---------------------------------------------- dW = A^T D (scn_planes.hip)
static int sgemm_AtB(scn_ctx *ctx, const float *d_A, const float *d_D,
                     float *d_dW, float *d_db, int64_t M, int K, int N, bool clear) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_sgemm_AtB: null context");
  SCN_REQUIRE(M >= 0 && K >= 1 && N >= 1, SCN_ERR_ARG,
              "scn_sgemm_AtB: M %lld K %d N %d", (long long)M, K, N);
  SCN_REQUIRE(d_dW, SCN_ERR_ARG, "scn_sgemm_AtB: null d_dW");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  if (clear)
    SCN_TRY(scn_fill32(ctx, d_dW, 0, (size_t)K * N));
  if (clear && d_db)
    SCN_TRY(scn_fill32(ctx, d_db, 0, (size_t)N));
  if (M == 0)
    return SCN_OK;
  SCN_REQUIRE(d_A && d_D, SCN_ERR_ARG, "scn_sgemm_AtB: null buffer");
  SCN_TRY(scn_atb_planes(ctx, d_A, d_D, d_dW, d_db, (long long)M, K, N));
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

extern "C" int scn_sgemm_AtB(scn_ctx *ctx, const float *d_A, const float *d_D,
                             float *d_dW, int64_t M, int K, int N) {
  return sgemm_AtB(ctx, d_A, d_D, d_dW, nullptr, M, K, N, true);
}

// the kernels only ever add to dW, so beta = 1 is the same launch without the
// clearing one before it
extern "C" int scn_sgemm_AtB_acc(scn_ctx *ctx, const float *d_A,
                                 const float *d_D, float *d_dW, int64_t M,
                                 int K, int N) {
  return sgemm_AtB(ctx, d_A, d_D, d_dW, nullptr, M, K, N, false);
}
// with the bias gradient, the column sums of D, which passes by anyway,
// summed as the floats they are: 0.4 to 0.95 times as far from 64 bits as
// k_act_backward's sums of the same matrix (57250 x 64: 1.2e-7
// against 2.2e-7, 82400 x 32: 2.2e-7 against 2.3e-7)
extern "C" int scn_sgemm_AtB_sums(scn_ctx *ctx, const float *d_A, const float *d_D, float *d_dW, float *d_db,
                                  int64_t M, int K, int N, int accumulate) {
  SCN_REQUIRE(d_db, SCN_ERR_ARG, "scn_sgemm_AtB_sums: null d_db");
  return sgemm_AtB(ctx, d_A, d_D, d_dW, d_db, M, K, N, !accumulate);
}

// The same product with A left ungathered: row m of it is what scn_gather_rows
// would make of the rules of output row m, given position by position.
extern "C" int scn_conv_AtB(scn_ctx *ctx, const float *d_in, const int32_t *d_positions, int fs, int nIn,
                            const float *d_D, float *d_dW, float *d_db, int64_t M, int N, int accumulate) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_conv_AtB: null context");
  SCN_REQUIRE(M >= 0 && fs >= 1 && nIn >= 1 && nIn <= SCN_ZERO_FLOATS && (int64_t)fs * nIn <= 0x7fffffff && N >= 1,
              SCN_ERR_ARG, "scn_conv_AtB: M %lld fs %d nIn %d N %d", (long long)M, fs, nIn, N);
  SCN_REQUIRE(d_dW, SCN_ERR_ARG, "scn_conv_AtB: null d_dW");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  if (!accumulate)
    SCN_TRY(scn_fill32(ctx, d_dW, 0, (size_t)fs * nIn * N));
  if (!accumulate && d_db)
    SCN_TRY(scn_fill32(ctx, d_db, 0, (size_t)N));
  if (M == 0)
    return SCN_OK;
  // (d_in may be null: an input without rows, every rule negative)
  SCN_REQUIRE(d_positions && d_D, SCN_ERR_ARG, "scn_conv_AtB: null buffer");
  SCN_REQUIRE(((uintptr_t)d_positions & 15) == 0, SCN_ERR_ARG, "scn_conv_AtB: positions start on 16 bytes");
  GatherSource gs = GatherSource();
  gs.rules = d_positions;
  gs.fs = fs;
  gs.nIn = nIn;
  gs.zeros = ctx->d_zeros;
  SCN_TRY(scn_atb_planes(ctx, d_in, d_D, d_dW, d_db, (long long)M, fs * nIn, N, &gs));
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

extern "C" int scn_AtB_many(scn_ctx *ctx, const scn_atb_item *items, int nItems) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_AtB_many: null context");
  SCN_REQUIRE(nItems >= 0 && nItems <= SCN_ATB_MAX && (items || nItems == 0), SCN_ERR_ARG,
              "scn_AtB_many: %d items (at most %d)", nItems, SCN_ATB_MAX);
  for (int k = 0; k < nItems; ++k) {
    const scn_atb_item &it = items[k];
    SCN_REQUIRE(it.M >= 0 && it.fs >= 1 && it.nIn >= 1 && (int64_t)it.fs * it.nIn <= 0x7fffffff && it.N >= 1 &&
                    (it.d_positions ? it.nIn <= SCN_ZERO_FLOATS : it.fs == 1 || it.M == 0),
                SCN_ERR_ARG, "scn_AtB_many: item %d M %lld fs %d nIn %d N %d", k, (long long)it.M, it.fs, it.nIn, it.N);
    // (d_in may be null where there are rules, all negative)
    SCN_REQUIRE(it.M == 0 || (it.d_dW && it.d_D && (it.d_in || it.d_positions)), SCN_ERR_ARG,
                "scn_AtB_many: item %d null buffer", k);
    SCN_REQUIRE(((uintptr_t)it.d_positions & 15) == 0, SCN_ERR_ARG, "scn_AtB_many: positions start on 16 bytes");
  }
  ProfScope prof(ctx, SCN_K_BACKWARD);
  SCN_TRY(scn_atb_planes_many(ctx, items, nItems));
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// ------------------------------------- the gradient of a convolution's input
// dA = D W^T scattered through the rules is itself a convolution: row r of the
// input gets, for every filter position f at which an output row o names it,
// D[o] W_f^T.  There is one such o at most, unless r is a background row, which
// any number of windows names.  So a layer's rules are turned round once
// (inverse[r * fs + f] = o, negative: none); the rows of D that name a sample's
// background row (background[o]: at which positions) are summed per position
// (k_background_sums) into rows behind D's own, which the background row's
// inverse names; and the forward kernels do
// the rest on W with every position's block transposed: no matrix of M x K is
// written and read again, none is cleared, and no float is added atomically but
// those few.  (A position that no row names adds nothing, as in the scatter, and
// not 0 times its weights, which may be infinite: GatherSource::namedOnly, and
// k_input_gradient_again for the shapes that the planes do not take.)
// Of a batch of 100 drawings the backward kernels of the layer 57000 x 128 -> 64
// take 4.4 + 17.2 + 22.5 + 14.7 us with the matrix (image, dW, dA, scatter; 8.2
// for the gathering besides) and 15.6 + 6.3 + 19.3 without (dW, sums, gradient);
// 12 batches 7570 -> 6620 us of kernels, of voxel models 5650 -> 5000.  Turning
// the rules round, on the producers' streams, is 10 us of a batch.
#define POSITIONS_PITCH(rows) (((rows) + 15) & ~15ll)
struct InverseList {
  const int *rules[SCN_INVERSE_MAX], *bg[SCN_INVERSE_MAX];
  int *inverse[SCN_INVERSE_MAX], *positions[SCN_INVERSE_MAX];
  int *background[SCN_INVERSE_MAX];
  int rows[SCN_INVERSE_MAX], inRows[SCN_INVERSE_MAX];
  unsigned firstBlock[SCN_INVERSE_MAX + 1];
  int fs[SCN_INVERSE_MAX], batch[SCN_INVERSE_MAX];
  int count;
};
// a workgroup an item
__global__ __launch_bounds__(256) void k_inverse_background(InverseList l) {
  const int t = blockIdx.x, fs = l.fs[t];
  if (l.background[t])
    for (int s = threadIdx.x; s < l.batch[t]; s += 256) {
      l.background[t][l.rows[t] + 2 * s] = 0x7fffffff;
      l.background[t][l.rows[t] + 2 * s + 1] = -1;
    }
  if (!l.inverse[t]) // (not wanted, or an input without rows)
    return;
  // (-2 - x: a background row's, until a row that names it is met)
  for (int x = threadIdx.x; x < l.batch[t] * fs; x += 256) {
    const int r = l.bg[t][x / fs];
    if (r >= 0 && r < l.inRows[t])
      l.inverse[t][(long long)r * fs + x % fs] = -2 - x;
  }
}
// a lane a row of the output
__global__ __launch_bounds__(256) void k_inverse_rules(InverseList l) {
  static_assert(SCN_INVERSE_MAX <= 64, "a lane an item");
  const int lane = threadIdx.x & 63;
  const int t =
      __popcll(__ballot(lane < l.count && blockIdx.x >= l.firstBlock[lane < SCN_INVERSE_MAX ? lane : 0])) - 1;
  const long long o = (long long)(blockIdx.x - l.firstBlock[t]) * 256 + threadIdx.x;
  const int rows = l.rows[t], inRows = l.inRows[t], fs = l.fs[t];
  const long long pitch = POSITIONS_PITCH((long long)rows);
  const int *const rules = l.rules[t];
  int *const inverse = l.inverse[t], *const positions = l.positions[t];
  if (o >= pitch)
    return;
  unsigned mask = 0;
  int sample = 0;
  for (int f = 0; f < fs; ++f) {
    const int r = o < rows ? rules[o * fs + f] : -1;
    if (positions)
      positions[f * pitch + o] = r;
    if (!inverse || r < 0 || r >= inRows)
      continue;
    int *const at = inverse + (long long)r * fs + f;
    const int was = *at;
    if (was >= -1 && was < rows) {
      *at = (int)o;
    } else { // (a background row's; those that find it unnamed all store the same)
      mask |= 1u << f;
      sample = (was < 0 ? -2 - was : was - rows) / fs;
      if (was < 0)
        *at = rows - 2 - was;
    }
  }
  if (!l.background[t])
    return;
  if (o < rows)
    l.background[t][o] = (int)mask;
  // the first and the last row of a sample that name its background: of the rows of
  // a wavefront only those at the ends of a sample's run (all of them: 22 us a batch
  // of 100 drawings and not 8, some 400 atomics on a line)
  int *const ends = l.background[t] + rows;
  const unsigned long long named = __ballot(mask != 0);
  const unsigned long long below = named & ((1ull << lane) - 1), above = named & ~((2ull << lane) - 1);
  const int before = __shfl(sample, below ? 63 - __builtin_clzll(below) : lane);
  const int behind = __shfl(sample, above ? __builtin_ctzll(above) : lane);
  if (!mask)
    return;
  if (!below || before != sample)
    atomicMin(&ends[2 * sample], (int)o);
  if (!above || behind != sample)
    atomicMax(&ends[2 * sample + 1], (int)o);
}
extern "C" int64_t scn_positions_pitch(int64_t rows) { return POSITIONS_PITCH(rows); }
extern "C" int scn_rules_inverse_many(scn_ctx *ctx, const scn_inverse_item *items, int nItems) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_rules_inverse_many: null context");
  SCN_REQUIRE(nItems >= 0 && nItems <= SCN_INVERSE_MAX && (items || nItems == 0), SCN_ERR_ARG,
              "scn_rules_inverse_many: %d items (at most %d)", nItems, SCN_INVERSE_MAX);
  InverseList l;
  void *fill[SCN_INVERSE_MAX];
  size_t words[SCN_INVERSE_MAX];
  long long blocks = 0; // (16 items of no more than 2^23 workgroups)
  int fills = 0;
  bool ends = false;
  l.count = 0;
  for (int k = 0; k < nItems; ++k) {
    const scn_inverse_item &it = items[k];
    SCN_REQUIRE(it.input && it.rows >= 0 && it.inputRows >= 0 && it.inputRows <= 0x7fffffffll && it.fs >= 1 &&
                    it.fs <= 32,
                SCN_ERR_ARG, "scn_rules_inverse_many: item %d rows %lld of %lld fs %d", k, (long long)it.rows,
                (long long)it.inputRows, it.fs);
    SCN_REQUIRE(!it.input->pending, SCN_ERR_STATE, "scn_rules_inverse_many: item %d: counts not settled", k);
    SCN_REQUIRE(it.rows + (int64_t)it.input->batch * it.fs <= 0x7fffffffll, SCN_ERR_CAPACITY,
                "scn_rules_inverse_many: item %d: %lld rows", k, (long long)it.rows);
    SCN_REQUIRE((it.d_rules || it.rows == 0) && (it.d_inverse || !it.d_background), SCN_ERR_ARG,
                "scn_rules_inverse_many: item %d null buffer", k);
    const int c = l.count++;
    l.rules[c] = it.d_rules;
    l.bg[c] = it.input->bg.p;
    l.inverse[c] = it.inputRows ? it.d_inverse : nullptr;
    l.positions[c] = it.d_positions;
    l.background[c] = it.d_background;
    l.rows[c] = (int)it.rows;
    l.inRows[c] = (int)it.inputRows;
    l.fs[c] = it.fs;
    l.batch[c] = it.input->batch;
    l.firstBlock[c] = (unsigned)blocks;
    blocks += scn_ceil_div(scn_positions_pitch(it.rows), 256);
    ends |= it.d_background != nullptr;
    if (l.inverse[c]) {
      fill[fills] = it.d_inverse;
      words[fills++] = (size_t)it.inputRows * it.fs;
    }
  }
  if (l.count == 0)
    return SCN_OK;
  l.firstBlock[l.count] = (unsigned)blocks;
  ProfScope prof(ctx, SCN_K_RULES);
  if (fills)
    SCN_TRY(scn_fill32_many(ctx, fill, words, fills, 0xffffffffu));
  if (fills || ends)
    hipLaunchKernelGGL(k_inverse_background, dim3(l.count), dim3(256), 0, ctx->stream, l);
  if (blocks)
    hipLaunchKernelGGL(k_inverse_rules, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, l);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// A workgroup takes a part of the rows of D between the first and the last that
// name a sample's background.  A lane keeps the sums of V columns at FS positions
// over every rows-th row, as the row's mask says, the workgroup's lanes of one
// column are put together in LDS, and each sum is added to memory once.  (Ranges
// of rows without regard to samples, with the sums given up where the sample
// changes: 9.4 us a layer of 100 drawings on average.)
template <int V, int FS>
__global__ __launch_bounds__(256) void k_background_sums(float *delta, long long M, int N,
                                                         const int *__restrict__ background, int fs, int parts,
                                                         int P) {
  typedef float vec __attribute__((ext_vector_type(V)));
  __shared__ float sSum[256 * V * FS];
  const int tid = threadIdx.x;
  const int rows = 256 / P; // lanes beyond the last whole row idle
  const int tx = tid % P, ty = tid / P;
  const int c = (blockIdx.y * P + tx) * V;
  const unsigned at = xcd_eighth(blockIdx.x, gridDim.x);
  const int sample = (int)(at / parts), part = (int)(at % parts);
  int first = background[M + 2 * sample], end = background[M + 2 * sample + 1] + 1;
  const int range = (end - first + parts - 1) / parts;
  if (end <= first || first + part * range >= end)
    return;
  first += part * range;
  end = first + range < end ? first + range : end;
  for (int f0 = 0; f0 < fs; f0 += FS) {
    vec acc[FS];
#pragma unroll
    for (int f = 0; f < FS; ++f)
      acc[f] = vec(0.f);
    // (the rows are asked for before it is known whether they are wanted: most are)
    constexpr int AHEAD = 4;
    if (c < N && ty < rows)
      for (int r = first + ty; r < end; r += AHEAD * rows) {
        unsigned mask[AHEAD];
        vec d[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
          const int ru = r + u * rows < end ? r + u * rows : end - 1;
          mask[u] = r + u * rows < end ? (unsigned)background[ru] >> f0 : 0;
          d[u] = *reinterpret_cast<const vec *>(delta + (long long)ru * N + c);
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
#pragma unroll
          for (int f = 0; f < FS; ++f)
            acc[f] += mask[u] >> f & 1 ? d[u] : vec(0.f);
      }
#pragma unroll
    for (int f = 0; f < FS; ++f)
#pragma unroll
      for (int v = 0; v < V; ++v)
        sSum[(f * V + v) * 256 + tid] = acc[f][v];
    __syncthreads();
    for (int x = tid; x < P * V * FS; x += 256) {
      const int f = x / (P * V), col = x % (P * V), lane = col / V, v = col % V;
      const int n = (blockIdx.y * P + lane) * V + v;
      if (n >= N || f0 + f >= fs)
        continue;
      float sum = 0.f;
      for (int k = 0; k < rows; ++k)
        sum += sSum[(f * V + v) * 256 + k * P + lane];
      unsafeAtomicAdd(delta + (M + (long long)sample * fs + f0 + f) * N + n, sum);
    }
    __syncthreads();
  }
}
extern "C" int scn_background_sums(scn_ctx *ctx, float *d_delta, int64_t M, int N, const int32_t *d_background,
                                   int fs, int batch) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_background_sums: null context");
  SCN_REQUIRE(M >= 0 && M <= 0x7fffffffll && N >= 1 && fs >= 1 && fs <= 32 && batch >= 0, SCN_ERR_ARG,
              "scn_background_sums: M %lld N %d fs %d batch %d", (long long)M, N, fs, batch);
  if (M == 0 || batch == 0)
    return SCN_OK;
  SCN_REQUIRE(d_delta && d_background, SCN_ERR_ARG, "scn_background_sums: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  const int V = N % 4 == 0 && ((uintptr_t)d_delta & 15) == 0 ? 4 : 1;
  const int colBlocks = scn_ceil_div(N, V * 64);
  const int P = scn_ceil_div(scn_ceil_div(N, V), colBlocks);
  // two workgroups a compute unit, of 32 rows at least: what it costs to begin and to end
  long long parts = scn_ceil_div(2 * ctx->numCU, (int64_t)batch * colBlocks);
  const long long most = scn_ceil_div(M, 32ll * batch);
  parts = parts < most ? parts : most;
  SCN_REQUIRE(batch * parts <= 0x7fffffffll, SCN_ERR_CAPACITY, "scn_background_sums: batch %d", batch);
  const dim3 grid((unsigned)(batch * parts), (unsigned)colBlocks);
#define SCN_BGS_GO(V, FS)                                                                                     \
  hipLaunchKernelGGL((k_background_sums<V, FS>), grid, dim3(256), 0, ctx->stream, d_delta, (long long)M, N,   \
                     d_background, fs, (int)parts, P)
  if (V == 4 && fs <= 4)
    SCN_BGS_GO(4, 4);
  else if (V == 4)
    SCN_BGS_GO(4, 8);
  else
    SCN_BGS_GO(1, 8);
#undef SCN_BGS_GO
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// (buffers cleared and filters turned round in one launch: the two are what a backward
// pass begins with, 2.3 to 4 and 4.6 us a launch. With the classifier's copy beside its
// gradient, two launches of a batch less: 12 batches with their updates 5.30 -> 5.21 ms for 100
// drawings, 4.38 -> 4.29 for 32 fields of 3-D)
__global__ __launch_bounds__(256) void k_transpose_filters(BeginList l) {
  __shared__ float tile[32][33];
  begin_list_block(l, blockIdx.x, threadIdx.x, tile);
}
extern "C" int scn_transpose_filters_many(scn_ctx *ctx, const scn_filter_item *items, int nItems) {
  return scn_gradients_begin(ctx, nullptr, nullptr, 0, items, nItems);
}
int scn_begin_list(scn_ctx *ctx, void *const *d_clear, const size_t *nWords, int nClear, const scn_filter_item *items,
                   int nItems, BeginList *list) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_transpose_filters_many: null context");
  SCN_REQUIRE(nItems >= 0 && nItems <= SCN_FILTERS_MAX && (items || nItems == 0), SCN_ERR_ARG,
              "scn_transpose_filters_many: %d items (at most %d)", nItems, SCN_FILTERS_MAX);
  static_assert(SCN_FILTERS_MAX <= 64, "a lane an item");
  FilterList &l = list->filters;
  long long blocks = 0;
  for (int k = 0; k < nItems; ++k) {
    const scn_filter_item &it = items[k];
    SCN_REQUIRE(it.d_W && it.d_Wt && it.fs >= 1 && it.nIn >= 1 && it.N >= 1, SCN_ERR_ARG,
                "scn_transpose_filters_many: item %d fs %d nIn %d N %d", k, it.fs, it.nIn, it.N);
    l.W[k] = it.d_W;
    l.Wt[k] = it.d_Wt;
    l.nIn[k] = it.nIn;
    l.N[k] = it.N;
    l.firstBlock[k] = (unsigned)blocks;
    blocks += (long long)it.fs * scn_ceil_div(it.N, 32) * scn_ceil_div(it.nIn, 32);
    SCN_REQUIRE(blocks <= 0x7fffffffll, SCN_ERR_CAPACITY, "scn_transpose_filters_many: %lld workgroups", blocks);
  }
  l.count = nItems;
  l.firstBlock[nItems] = (unsigned)blocks;
  SCN_TRY(scn_fill_list(ctx, d_clear, nWords, nClear, &list->fill, &list->fillBlocks));
  SCN_REQUIRE(blocks + list->fillBlocks <= 0x7fffffffll, SCN_ERR_CAPACITY, "scn_gradients_begin: %lld workgroups",
              blocks + list->fillBlocks);
  list->blocks = (unsigned)blocks + list->fillBlocks;
  return SCN_OK;
}
extern "C" int scn_gradients_begin(scn_ctx *ctx, void *const *d_clear, const size_t *nWords, int nClear,
                                   const scn_filter_item *items, int nItems) {
  BeginList l;
  SCN_TRY(scn_begin_list(ctx, d_clear, nWords, nClear, items, nItems, &l));
  if (l.blocks == 0)
    return SCN_OK;
  ProfScope prof(ctx, SCN_K_BACKWARD);
  hipLaunchKernelGGL(k_transpose_filters, dim3(l.blocks), dim3(256), 0, ctx->stream, l);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// Where the planes do not take the product (few shapes: rows in other than 32s): the
// elements that are not finite again, without the positions that no row names.  A
// sum of fs N products each, one after the other.
__global__ __launch_bounds__(256) void k_input_gradient_again(const float *__restrict__ delta,
                                                              const int *__restrict__ inverse, int fs, int N,
                                                              const float *__restrict__ Wt, float *__restrict__ din,
                                                              long long count, int nIn) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < count; i += (long long)gridDim.x * 256) {
    if (fabsf(din[i]) <= 3.4028235e38f)
      continue;
    const long long r = i / nIn;
    const int c = (int)(i - r * nIn);
    float sum = 0.f;
    for (int f = 0; f < fs; ++f) {
      const int o = inverse[r * fs + f];
      for (int n = 0; n < (o < 0 ? 0 : N); ++n)
        sum = fmaf(delta[(long long)o * N + n], Wt[((long long)f * N + n) * nIn + c], sum);
    }
    din[i] = sum;
  }
}
extern "C" int scn_conv_input_gradient(scn_ctx *ctx, const float *d_delta, const int32_t *d_inverse, int fs, int N,
                                       const float *d_Wt, const void *d_image, float *d_din, int64_t inputRows,
                                       int nIn) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_conv_input_gradient: null context");
  SCN_REQUIRE(inputRows >= 0 && nIn >= 1 && nIn <= SCN_ZERO_FLOATS && N <= SCN_ZERO_FLOATS, SCN_ERR_ARG,
              "scn_conv_input_gradient: %lld rows nIn %d N %d", (long long)inputRows, nIn, N);
  if (inputRows == 0)
    return SCN_OK;
  OwnRows ownRows(ctx);
  SCN_REQUIRE(d_inverse, SCN_ERR_ARG, "scn_conv_input_gradient: null rules");
  SCN_TRY(scn_conv_named(ctx, d_delta, d_inverse, fs, N, d_Wt, d_image, d_din, inputRows, nIn));
  if (!scn_conv_takes_planes(d_delta, d_Wt, d_din, fs * N, nIn)) {
    ProfScope prof(ctx, SCN_K_BACKWARD);
    const long long count = (long long)inputRows * nIn, most = 16ll * ctx->numCU, blocks = (count + 255) / 256;
    hipLaunchKernelGGL(k_input_gradient_again, dim3((unsigned)(blocks < most ? blocks : most)), dim3(256), 0,
                       ctx->stream, d_delta, d_inverse, fs, N, d_Wt, d_din, count, nIn);
    SCN_HIP_CHECK(hipGetLastError());
  }
  return SCN_OK;
}

// ------------------------------------------------------------ dA = D W^T
// The forward contraction with W transposed.  The planes make their image from W
// as it stands, or read it so; other shapes, and calls that may not use the
// context's room (under capture), take a transposed copy in the caller's
// workspace, where the zero bias of a wide result is too.
__global__ void k_transpose(const float *__restrict__ W, float *__restrict__ Wt,
                            int K, int N) {
  __shared__ float tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5; // 32 x 8
  const int k0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  for (int i = ty; i < 32; i += 8)
    if (k0 + i < K && n0 + tx < N)
      tile[i][tx] = W[(long long)(k0 + i) * N + n0 + tx];
  __syncthreads();
  for (int i = ty; i < 32; i += 8)
    if (n0 + i < N && k0 + tx < K)
      Wt[(long long)(n0 + i) * K + k0 + tx] = tile[tx][i];
}

extern "C" int64_t scn_sgemm_ABt_workspace(int N, int K) {
  return (int64_t)N * K + K;
}

extern "C" int scn_sgemm_ABt(scn_ctx *ctx, const float *d_D, const float *d_W,
                             float *d_dA, int64_t M, int N, int K,
                             float *d_workspace) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_sgemm_ABt: null context");
  SCN_REQUIRE(M >= 0 && K >= 1 && N >= 1, SCN_ERR_ARG,
              "scn_sgemm_ABt: M %lld N %d K %d", (long long)M, N, K);
  if (M == 0)
    return SCN_OK;
  SCN_REQUIRE(d_D && d_W && d_dA && d_workspace, SCN_ERR_ARG,
              "scn_sgemm_ABt: null buffer");
  OwnRows ownRows(ctx);
  bool transpose = false;
  Epilogue ep = Epilogue();
  ep.bias = ctx->d_zeros;
  ep.p = 1.f;
  ep.act = SCN_NOSIGMOID;
  if (scn_abt_narrow(ctx, d_D, d_W, d_dA, (long long)M, N, K)) {
    SCN_HIP_CHECK(hipGetLastError());
    return SCN_OK;
  }
  if (K <= SCN_ZERO_FLOATS) { // the planes read W [K x N] as it stands
    int rc = SCN_OK;
    if (scn_planes_abt(ctx, d_D, d_W, d_dA, (long long)M, N, K, ep, &rc, &transpose)) {
      SCN_TRY(rc);
      SCN_HIP_CHECK(hipGetLastError());
      return SCN_OK;
    }
  }
  // the zero bias: the context's own zeros when they are enough of them
  float *Wt = d_workspace, *zeros = d_workspace + (size_t)N * K;
  {
    ProfScope prof(ctx, SCN_K_BACKWARD);
    hipLaunchKernelGGL(k_transpose, dim3(scn_ceil_div(N, 32), scn_ceil_div(K, 32)),
                       dim3(256), 0, ctx->stream, d_W, Wt, K, N);
    SCN_HIP_CHECK(hipGetLastError());
    if (K <= SCN_ZERO_FLOATS)
      zeros = ctx->d_zeros;
    else
      SCN_TRY(scn_fill32(ctx, zeros, 0, (size_t)K));
  }
  if (transpose) {
    ProfScope prof(ctx, SCN_K_BACKWARD);
    SCN_TRY(scn_planes_forward(ctx, 3, d_D, Wt, d_dA, (long long)M, N, K, ep, nullptr, false));
    SCN_HIP_CHECK(hipGetLastError());
    return SCN_OK;
  }
  return scn_nin_forward(ctx, d_D, Wt, zeros, nullptr, d_dA, M, N, K, 1.0f,
                         SCN_NOSIGMOID, SCN_FP32);
}

// dA = D W^T for callers that may not allocate (code under HIP graph capture,
// serving loops, harnesses that forbid hipMalloc): the transposed weights and
// the zero bias live in a file-scope device array instead of a caller's
// workspace.  Every device the library runs on holds its own copy of the array
// at its own address; host code reaches it only through the pointer that
// hipGetSymbolAddress returned for that device.
#define ABT_STATIC_FLOATS (1 << 20) // 4 MiB per device
static __device__ __align__(256) float scratch[ABT_STATIC_FLOATS];
#define ABT_MAX_DEVICES 64
// per device, set once by scn_ctx_create: the array's address, an event that
// marks the end of the last call that used it, and whose call that was
static float *g_abtScratch[ABT_MAX_DEVICES];
static hipEvent_t g_abtDone[ABT_MAX_DEVICES];
static const scn_ctx *g_abtUser[ABT_MAX_DEVICES];
static std::mutex g_abtMutex;

int scn_abt_static_setup(int device) {
  SCN_REQUIRE(device >= 0 && device < ABT_MAX_DEVICES, SCN_ERR_ARG,
              "device %d: at most %d devices", device, ABT_MAX_DEVICES);
  std::lock_guard<std::mutex> lock(g_abtMutex); // (contexts are made by several threads)
  if (g_abtScratch[device])
    return SCN_OK;
  float *ptr = nullptr;
  SCN_HIP_CHECK(hipSetDevice(device));
  SCN_HIP_CHECK(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
  SCN_REQUIRE(ptr != nullptr, SCN_ERR_HIP,
              "hipGetSymbolAddress returned no address for the static scratch");
  SCN_HIP_CHECK(hipEventCreateWithFlags(&g_abtDone[device], hipEventDisableTiming));
  g_abtScratch[device] = ptr;
  return SCN_OK;
}

// a context that is destroyed gives the array up
void scn_abt_static_forget(const scn_ctx *ctx) {
  std::lock_guard<std::mutex> lock(g_abtMutex);
  for (int d = 0; d < ABT_MAX_DEVICES; ++d)
    if (g_abtUser[d] == ctx)
      g_abtUser[d] = nullptr;
}

extern "C" int64_t scn_sgemm_ABt_static_limit(void) { return ABT_STATIC_FLOATS; }

extern "C" int scn_sgemm_ABt_static(scn_ctx *ctx, const float *d_D,
                                    const float *d_W, float *d_dA, int64_t M,
                                    int N, int K) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_sgemm_ABt_static: null context");
  SCN_REQUIRE(M >= 0 && K >= 1 && N >= 1, SCN_ERR_ARG,
              "scn_sgemm_ABt_static: M %lld N %d K %d", (long long)M, N, K);
  SCN_REQUIRE(scn_sgemm_ABt_workspace(N, K) <= ABT_STATIC_FLOATS,
              SCN_ERR_CAPACITY,
              "scn_sgemm_ABt_static: N %d x K %d weights need %lld floats of "
              "scratch, the static array holds %d; use scn_sgemm_ABt with a "
              "workspace",
              N, K, (long long)scn_sgemm_ABt_workspace(N, K), ABT_STATIC_FLOATS);
  const int dev = ctx->device;
  float *ptr = dev >= 0 && dev < ABT_MAX_DEVICES ? g_abtScratch[dev] : nullptr;
  SCN_REQUIRE(ptr, SCN_ERR_STATE,
              "scn_sgemm_ABt_static: no scratch address for device %d", dev);
  if (M == 0)
    return SCN_OK;
  // One array a device: calls of one context follow each other on its stream;
  // a call of another context while the last one has not finished is refused.
  // (a stream under capture records and queries nothing: its owner has to
  // keep other users of the array away for as long as the graph may run)
  std::lock_guard<std::mutex> lock(g_abtMutex);
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  SCN_HIP_CHECK(hipStreamIsCapturing(ctx->stream, &capturing));
  if (g_abtUser[dev] && g_abtUser[dev] != ctx) {
    const hipError_t busy = hipEventQuery(g_abtDone[dev]);
    SCN_REQUIRE(busy != hipErrorNotReady, SCN_ERR_STATE,
                "scn_sgemm_ABt_static: the device's static array is still in "
                "use by a call of another context");
    SCN_HIP_CHECK(busy);
  }
  // (the kernels clear and fill what they use of the array: nothing of an
  // earlier call is read)
  SCN_TRY(scn_sgemm_ABt(ctx, d_D, d_W, d_dA, M, N, K, ptr));
  if (capturing == hipStreamCaptureStatusNone) {
    SCN_HIP_CHECK(hipEventRecord(g_abtDone[dev], ctx->stream));
    g_abtUser[dev] = ctx;
  }
  return SCN_OK;
}

// ---------------------------------------------------------- weight update
__global__ void k_nag_update(const float *__restrict__ delta,
                             float *__restrict__ mom, float *__restrict__ wts,
                             long long n, float lr, float mu, int keepPositive) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  float w = wts[i], m = mom[i];
  const float d = delta[i];
  w -= m * mu;
  m = mu * m - lr * (1 - mu) * d;
  w += m * (1 + mu);
  if (keepPositive)
    w = w > 0.001f ? w : 0.001f;
  wts[i] = w;
  mom[i] = m;
}

extern "C" int scn_nag_update(scn_ctx *ctx, const float *d_delta,
                              float *d_momentum, float *d_weights, int64_t n,
                              float learningRate, float momentum,
                              int keepPositive) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_nag_update: null context");
  SCN_REQUIRE(n >= 0, SCN_ERR_ARG, "scn_nag_update: n %lld", (long long)n);
  if (n == 0)
    return SCN_OK;
  SCN_REQUIRE(d_delta && d_momentum && d_weights, SCN_ERR_ARG,
              "scn_nag_update: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  hipLaunchKernelGGL(k_nag_update, dim3(scn_ceil_div(n, 256)), dim3(256), 0,
                     ctx->stream, d_delta, d_momentum, d_weights, (long long)n,
                     learningRate, momentum, keepPositive);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// The momentum step of several tensors (all layers' W, B and PReLU slopes) in
// one launch: a workgroup finds its tensor from the running workgroup counts (a
// lane a count: a walk over them in the arguments is a trip a cache line).
// With `clear` the gradient is left zero, so the next batch's accumulating
// products need no clearing launch.
struct NagList {
  float *delta[SCN_NAG_MAX];
  float *mom[SCN_NAG_MAX];
  float *wts[SCN_NAG_MAX];
  long long n[SCN_NAG_MAX];
  unsigned firstBlock[SCN_NAG_MAX + 1];
  int keepPositive[SCN_NAG_MAX];
  int count;
};

__global__ __launch_bounds__(256) void k_nag_update_many(NagList l, float lr,
                                                         float mu, int clear) {
  static_assert(SCN_NAG_MAX <= 64, "a lane an item");
  const int lane = threadIdx.x & 63;
  const int t = __popcll(__ballot(lane < l.count && blockIdx.x >= l.firstBlock[lane < SCN_NAG_MAX ? lane : 0])) - 1;
  const long long i =
      (long long)(blockIdx.x - l.firstBlock[t]) * blockDim.x + threadIdx.x;
  if (i >= l.n[t])
    return;
  float w = l.wts[t][i], m = l.mom[t][i];
  const float d = l.delta[t][i];
  w -= m * mu;
  m = mu * m - lr * (1 - mu) * d;
  w += m * (1 + mu);
  if (l.keepPositive[t])
    w = w > 0.001f ? w : 0.001f;
  l.wts[t][i] = w;
  l.mom[t][i] = m;
  if (clear)
    l.delta[t][i] = 0.f;
}

extern "C" int scn_nag_update_many(scn_ctx *ctx, const scn_nag_item *items,
                                   int nItems, float learningRate,
                                   float momentum, int clearGradients) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_nag_update_many: null context");
  SCN_REQUIRE(nItems >= 0 && nItems <= SCN_NAG_MAX && (items || nItems == 0),
              SCN_ERR_ARG, "scn_nag_update_many: %d items (at most %d)",
              nItems, SCN_NAG_MAX);
  NagList l;
  l.count = 0;
  long long blocks = 0;
  for (int k = 0; k < nItems; ++k) {
    const scn_nag_item &it = items[k];
    SCN_REQUIRE(it.n >= 0, SCN_ERR_ARG, "scn_nag_update_many: item %d n %lld",
                k, (long long)it.n);
    if (it.n == 0)
      continue;
    SCN_REQUIRE(it.d_delta && it.d_momentum && it.d_weights, SCN_ERR_ARG,
                "scn_nag_update_many: item %d null buffer", k);
    const int c = l.count++;
    l.delta[c] = it.d_delta;
    l.mom[c] = it.d_momentum;
    l.wts[c] = it.d_weights;
    l.n[c] = it.n;
    l.keepPositive[c] = it.keepPositive;
    l.firstBlock[c] = (unsigned)blocks;
    blocks += scn_ceil_div(it.n, 256);
    SCN_REQUIRE(blocks <= 0x7fffffffll, SCN_ERR_CAPACITY,
                "scn_nag_update_many: %lld workgroups", blocks);
  }
  if (l.count == 0)
    return SCN_OK;
  l.firstBlock[l.count] = (unsigned)blocks;
  ProfScope prof(ctx, SCN_K_BACKWARD);
  hipLaunchKernelGGL(k_nag_update_many, dim3((unsigned)blocks), dim3(256), 0,
                     ctx->stream, l, learningRate, momentum, clearGradients);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// ------------------------------------------------- scatter-add through rules
// A float atomic costs by the 64-byte pieces it touches, some 20 of which retire
// in a nanosecond however many of their lanes are live, and pieces of one line
// follow one another at 2 ns: a matrix of two and a half inputs a row, a fifth of
// them background, was added at a quarter of the rate it can be read at.  So a
// workgroup takes EN consecutive entries, whose neighbouring windows share most
// of their input rows, sorts them by row in LDS (a hash table, then a scan over
// its slots) and adds every row to memory once.  An item is up to eight entries
// of a row, summed in registers by a lane per channel, two items in flight; a
// row of more items (the background row of a sample, named by a fifth to a half
// of the entries) is put together in LDS first.
// 94264 x 4 x 96: 39 us (97 with runs of eight entries and no sorting; it takes
// 36 to read), 249376 x 8 x 32 74 (540), 60448 x 8 x 64 32 (211), 121924 x 27 x
// 64 255 (3078), 34485 x 4 x 64 15.5 (36), 1858 x 4 x 128 6.1 (9).
#define GB_RUN 8  // entries of one item
#define GB_FLIGHT 2 // items of a lane in flight
#define GB_LONG 4 // rows of more than one item that are summed in LDS
#define GB_LONG_WIDTH 512
struct GbItem {
  int row; // -1 - l: the l-th long row
  unsigned short start, len;
};
template <int T, int EN>
__global__ __launch_bounds__(T) void k_gather_backward(
    float *__restrict__ din, const float *__restrict__ dconv,
    const int *__restrict__ rules, long long count, int nIn, int channels,
    int splits) {
  constexpr int SLOTS = 2 * EN;
  __shared__ int sRow[SLOTS];   // hash table of the tile's rows
  __shared__ int sCount[SLOTS]; // entries of each; then where they begin
  __shared__ unsigned short sEntry[EN]; // entries, row by row
  __shared__ GbItem sItem[EN];
  __shared__ int sWave[3][T / 64];
  __shared__ int sLongRow[GB_LONG];
  __shared__ float sLong[GB_LONG * GB_LONG_WIDTH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long long e0 = (long long)(blockIdx.x / splits) * EN;
  const int c0 = (int)(blockIdx.x % splits) * channels;
  const int width = nIn - c0 < channels ? nIn - c0 : channels;
  const int longRows = width <= GB_LONG_WIDTH ? GB_LONG : 0;
  for (int i = tid; i < SLOTS; i += T)
    sRow[i] = -1, sCount[i] = 0;
  for (int i = tid; i < longRows * width; i += T)
    sLong[i] = 0.f;
  const int r = tid < EN && e0 + tid < count ? rules[e0 + tid] : -1;
  __syncthreads();
  int slot = 0, place = 0;
  if (r >= 0) {
    unsigned h = ((unsigned)r * 2654435761u) >> 7 & (SLOTS - 1);
    while (true) { // (twice as many slots as entries: ends)
      const int was = atomicCAS(&sRow[h], -1, r);
      if (was == -1 || was == r)
        break;
      h = (h + 1) & (SLOTS - 1);
    }
    slot = (int)h;
    place = atomicAdd(&sCount[h], 1);
  }
  __syncthreads();
  // entries, items and long rows before every slot (a thread has one or two)
  constexpr int SPT = SLOTS > T ? SLOTS / T : 1;
  int n[SPT], entries = 0, items = 0, longs = 0;
#pragma unroll
  for (int u = 0; u < SPT; ++u) {
    n[u] = tid * SPT + u < SLOTS ? sCount[tid * SPT + u] : 0;
    entries += n[u];
    items += (n[u] + GB_RUN - 1) / GB_RUN;
    longs += n[u] > GB_RUN;
  }
  int pe = entries, pi = items, pl = longs;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int ve = __shfl_up(pe, d), vi = __shfl_up(pi, d), vl = __shfl_up(pl, d);
    if (lane >= d)
      pe += ve, pi += vi, pl += vl;
  }
  if (lane == 63)
    sWave[0][wave] = pe, sWave[1][wave] = pi, sWave[2][wave] = pl;
  __syncthreads();
  int total = 0, nLong = 0;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) {
    if (w < wave)
      pe += sWave[0][w], pi += sWave[1][w], pl += sWave[2][w];
    total += sWave[1][w];
    nLong += sWave[2][w];
  }
  nLong = nLong < longRows ? nLong : longRows;
  pe -= entries;
  pi -= items;
  pl -= longs;
#pragma unroll
  for (int u = 0; u < SPT; ++u) {
    if (n[u] == 0)
      continue;
    GbItem it;
    it.row = sRow[tid * SPT + u];
    sCount[tid * SPT + u] = pe;
    if (n[u] > GB_RUN) {
      if (pl < longRows) {
        sLongRow[pl] = it.row;
        it.row = -1 - pl;
      }
      ++pl;
    }
    for (int k = 0; k < n[u]; k += GB_RUN) {
      it.start = (unsigned short)(pe + k);
      it.len = (unsigned short)(n[u] - k < GB_RUN ? n[u] - k : GB_RUN);
      sItem[pi++] = it;
    }
    pe += n[u];
  }
  __syncthreads();
  if (r >= 0)
    sEntry[sCount[slot] + place] = (unsigned short)tid;
  __syncthreads();
  const float *const src = dconv + e0 * nIn + c0;
  float *const dst = din + c0;
  const unsigned work = (unsigned)total * width;
  const unsigned magic = 0xffffffffu / width + 1; // (x / width, exact for 2^32 / width of them)
  auto of = [&](unsigned x) {
    return width > 1024 ? x / (unsigned)width : width == 1 ? x : __umulhi(x, magic);
  };
  for (unsigned x = tid; x < work; x += GB_FLIGHT * T) {
    float v[GB_FLIGHT][GB_RUN];
    GbItem it[GB_FLIGHT];
    unsigned j[GB_FLIGHT];
#pragma unroll
    for (int h = 0; h < GB_FLIGHT; ++h) {
      const unsigned xh = x + h * T;
      const unsigned i = of(xh);
      j[h] = xh - i * width;
      it[h].len = 0;
      if (xh < work)
        it[h] = sItem[i];
#pragma unroll
      for (int u = 0; u < GB_RUN; ++u) {
        v[h][u] = 0.f;
        if (u < it[h].len)
          v[h][u] = src[(long long)sEntry[it[h].start + u] * nIn + j[h]];
      }
    }
#pragma unroll
    for (int h = 0; h < GB_FLIGHT; ++h) {
      if (it[h].len == 0)
        continue;
      float acc = v[h][0];
#pragma unroll
      for (int u = 1; u < GB_RUN; ++u)
        acc += v[h][u];
      if (it[h].row >= 0)
        unsafeAtomicAdd(dst + (long long)it[h].row * nIn + j[h], acc);
      else
        unsafeAtomicAdd(&sLong[(-1 - it[h].row) * width + j[h]], acc);
    }
  }
  if (nLong == 0)
    return;
  __syncthreads();
  for (int i = tid; i < nLong * width; i += T)
    unsafeAtomicAdd(dst + (long long)sLongRow[i / width] * nIn + i % width, sLong[i]);
}

extern "C" int scn_gather_rows_backward(scn_ctx *ctx, float *d_din,
                                        const float *d_dconv,
                                        const int32_t *d_rules, int64_t count,
                                        int nIn) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_gather_rows_backward: null context");
  SCN_REQUIRE(count >= 0 && nIn >= 1, SCN_ERR_ARG,
              "scn_gather_rows_backward: count %lld nIn %d", (long long)count,
              nIn);
  if (count == 0)
    return SCN_OK;
  SCN_REQUIRE(d_din && d_dconv && d_rules, SCN_ERR_ARG,
              "scn_gather_rows_backward: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  // Tiles of 512 entries while there are two and a half for every compute unit
  // (60448 x 8 x 64: 32 us, 36 with 256), of 64 while there is no more than one
  // of 128 (6041 x 4 x 96: 7.7 us, 9.1 with 256), and where tiles are few, each
  // is given to several workgroups by its channels.
  const int most = scn_ceil_div(nIn, 32);
  const int EN = count >= 1280ll * ctx->numCU ? 512 : count > 128ll * ctx->numCU ? 256 : 64;
  const long long tiles = scn_ceil_div(count, EN);
  int splits = scn_ceil_div(EN == 64 ? 4 * ctx->numCU : 3 * ctx->numCU / 2, tiles);
  const int channels = 32 * scn_ceil_div(most, splits < most ? splits : most);
  splits = scn_ceil_div(nIn, channels);
  SCN_REQUIRE(tiles * splits <= 0x7fffffffll, SCN_ERR_CAPACITY,
              "scn_gather_rows_backward: %lld workgroups", tiles * splits);
#define SCN_GB_GO(T, EN)                                                       \
  hipLaunchKernelGGL((k_gather_backward<T, EN>),                               \
                     dim3((unsigned)(tiles * splits)), dim3(T), 0,             \
                     ctx->stream, d_din, d_dconv, d_rules, (long long)count,   \
                     nIn, channels, splits)
  if (EN == 512)
    SCN_GB_GO(512, 512);
  else if (EN == 256)
    SCN_GB_GO(512, 256);
  else
    SCN_GB_GO(256, 64);
#undef SCN_GB_GO
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// dMaxPoolBackProp.  What a float atomic costs (above) is the number of 64-byte
// pieces touched, and a row of the input is chosen by some of its channels in
// most of the windows that it is in.  So a workgroup takes the entries of 16 EPT
// consecutive output rows, whose windows overlap, in 16 channels (C below 16:
// the power of two that covers them, more rows), puts together in LDS what goes
// to a row and adds it to memory once.  Rows are found through a hash table;
// entries that find no room there go to memory by themselves.  A target is keyed
// by its offset from the entry's channel, so any choice is added where it says.
// 71426 x 128 of 150000 rows, side 3: 76 us (162 with runs of eight output rows
// in registers: 4.3 pieces for 16 entries, now 2.3), of which 39 are the part in
// LDS; the layers of a training batch of 2-D characters 20.6 -> 12.6 us on
// average, of 3-D models 12.0 -> 8.9.
template <int EPT>
__global__ __launch_bounds__(256) void k_maxpool_backward(
    float *__restrict__ din, const float *__restrict__ dout, long long count,
    int C, const int *__restrict__ choice, int shift, int slices,
    const float *__restrict__ out, int act) {
  constexpr int T = 256, SLOTS = 128 * EPT, PROBES = 3, ROOM = 1024 * EPT;
  constexpr int NONE = -2147483647 - 1;
  __shared__ int sKey[SLOTS], sId[SLOTS], sTarget[SLOTS];
  __shared__ float sSum[ROOM];
  __shared__ int sRows;
  const int tid = threadIdx.x, P = 1 << shift;
  const unsigned tileOf = xcd_eighth(blockIdx.x, gridDim.x);
  const long long r0 = (long long)(tileOf / slices) * (T * EPT >> shift);
  const int j = (int)(tileOf % slices) * P + (tid & (P - 1)); // (P divides T)
  int tg[EPT], slot[EPT];
  float dv[EPT];
#pragma unroll
  for (int u = 0; u < EPT; ++u) {
    const long long r = r0 + (tid >> shift) * EPT + u;
    const bool live = r < count && j < C;
    tg[u] = live ? choice[r * C + j] : -1;
    dv[u] = live ? dout[r * C + j] : 0.f;
    if (out) { // what was chosen: the output of the layer below
      float none = 0.f;
      dv[u] = act_derivative(act, live ? out[r * C + j] : 0.f, dv[u], act == SCN_LEAKYRELU ? 0.01f : 0.333f, none);
    }
  }
#pragma unroll
  for (int v = 1; v < EPT; ++v)
#pragma unroll
    for (int u = 0; u < v; ++u)
      if (tg[u] == tg[v] && tg[v] >= 0) {
        dv[v] += dv[u];
        tg[u] = -1;
      }
  for (int i = tid; i < SLOTS; i += T)
    sKey[i] = NONE;
  if (tid == 0)
    sRows = 0;
  __syncthreads();
  // The keys claim their slots in rounds: whoever finds a slot empty writes to
  // it, and after the barrier all see who has it.  (A slot that is taken stays
  // so: a barrier a round is enough.  With compare-and-swap, lane after lane on
  // one address, this part took 96 us of 71426 x 128.)
  unsigned placed = 0;
#pragma unroll
  for (int u = 0; u < EPT; ++u) {
    slot[u] = (int)(((unsigned)(tg[u] - j) * 2654435761u) >> 11 & (SLOTS - 1));
    placed |= tg[u] < 0 ? 1u << u : 0;
  }
#pragma unroll 1
  for (int k = 0; k < PROBES; ++k) {
    int was[EPT];
#pragma unroll
    for (int u = 0; u < EPT; ++u)
      was[u] = __hip_atomic_load(&sKey[slot[u]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
    for (int u = 0; u < EPT; ++u)
      if (was[u] == NONE && !(placed >> u & 1))
        __hip_atomic_store(&sKey[slot[u]], tg[u] - j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < EPT; ++u)
      was[u] = __hip_atomic_load(&sKey[slot[u]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
    for (int u = 0; u < EPT; ++u)
      if (!(placed >> u & 1)) {
        if (was[u] == tg[u] - j)
          placed |= 1u << u;
        else
          slot[u] = (slot[u] + 1) & (SLOTS - 1);
      }
  }
  __syncthreads();
  // rows of the sums, in order of arrival
  const int most = ROOM >> shift < SLOTS ? ROOM >> shift : SLOTS;
#pragma unroll
  for (int i = tid; i < SLOTS; i += T) { // (a multiple of 64 slots: whole wavefronts)
    const int key = sKey[i];
    const unsigned long long taken = __ballot(key != NONE);
    int first = 0;
    if ((tid & 63) == 0)
      first = atomicAdd(&sRows, __popcll(taken));
    first = __shfl(first, 0);
    const int id = first + __popcll(taken & ((1ull << (tid & 63)) - 1));
    sId[i] = id;
    if (key != NONE)
      sTarget[id] = key;
  }
  __syncthreads();
  const int sums = (sRows < most ? sRows : most) << shift;
  for (int i = tid; i < sums; i += T)
    sSum[i] = 0.f;
  __syncthreads();
  // An atomic add of a float to LDS takes 3 cycles a lane (46 of the 74 us that
  // 71426 x 128 took with one for every entry).  So of the entries of a sum one,
  // whose mark is seen there, stores, and only the others add.
  int *const sMark = reinterpret_cast<int *>(sSum);
  int cell[EPT];
#pragma unroll
  for (int u = 0; u < EPT; ++u) {
    cell[u] = -1;
    if (tg[u] < 0)
      continue;
    const int id = placed >> u & 1 ? sId[slot[u]] : most;
    if (id < most) {
      cell[u] = (id << shift) + (tid & (P - 1));
      __hip_atomic_store(&sMark[cell[u]], tid * EPT + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
      unsafeAtomicAdd(din + tg[u], dv[u]);
    }
  }
  __syncthreads();
  unsigned stores = 0;
#pragma unroll
  for (int u = 0; u < EPT; ++u)
    if (cell[u] >= 0 && sMark[cell[u]] == tid * EPT + u)
      stores |= 1u << u;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < EPT; ++u)
    if (stores >> u & 1)
      sSum[cell[u]] = dv[u];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < EPT; ++u)
    if (cell[u] >= 0 && !(stores >> u & 1))
      unsafeAtomicAdd(&sSum[cell[u]], dv[u]);
  __syncthreads();
  for (int i = tid; i < sums; i += T) { // (T is a multiple of P: j is this lane's channel here too)
    const float sum = sSum[i];
    if (sum != 0.f)
      unsafeAtomicAdd(din + sTarget[i >> shift] + j, sum);
  }
}

static int maxpool_backward(scn_ctx *ctx, float *d_din, const float *d_dout, int64_t count, int C,
                            const int32_t *d_choice, const float *d_out, int act) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_maxpool_backward: null context");
  SCN_REQUIRE(count >= 0 && C >= 1, SCN_ERR_ARG,
              "scn_maxpool_backward: count %lld C %d", (long long)count, C);
  if (count == 0)
    return SCN_OK;
  SCN_REQUIRE(d_din && d_dout && d_choice, SCN_ERR_ARG,
              "scn_maxpool_backward: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  int shift = 0;
  while (shift < 4 && (1 << shift) < C)
    ++shift;
  const int slices = scn_ceil_div(C, 1 << shift);
  // four entries a lane while that leaves four workgroups a compute unit (two
  // there: 76 -> 86 us; a wave of workgroups that is nearly empty below)
  int ept = 4;
  auto tiles = [&]() { return scn_ceil_div(count, 256 * ept >> shift) * (long long)slices; };
  if (tiles() < 4ll * ctx->numCU)
    ept = 2;
  SCN_REQUIRE(tiles() <= 0x7fffffffll, SCN_ERR_CAPACITY,
              "scn_maxpool_backward: %lld workgroups", tiles());
  auto *const kernel = ept == 4 ? k_maxpool_backward<4> : k_maxpool_backward<2>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiles()), dim3(256), 0, ctx->stream,
                     d_din, d_dout, (long long)count, C, d_choice, shift,
                     slices, d_out, act);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}
extern "C" int scn_maxpool_backward(scn_ctx *ctx, float *d_din,
                                    const float *d_dout, int64_t count, int C,
                                    const int32_t *d_choice) {
  return maxpool_backward(ctx, d_din, d_dout, count, C, d_choice, nullptr, SCN_NOSIGMOID);
}
// An output of the pooling is the activation it chose: the derivative is taken on
// the way, where there are fewer of them than the layer below has (a pass of its
// own over the pooling's outputs: 10 us of a layer of 36000 x 64, 36 of a batch
// of 100 drawings).
extern "C" int scn_maxpool_backward_through(scn_ctx *ctx, float *d_din, const float *d_dout, int64_t count, int C,
                                            const int32_t *d_choice, const float *d_out, int act) {
  SCN_REQUIRE(act >= SCN_NOSIGMOID && act <= SCN_SIGMOID && act != SCN_PRELU, SCN_ERR_ARG,
              "scn_maxpool_backward_through: activation %d", act);
  SCN_REQUIRE(d_out || count == 0, SCN_ERR_ARG, "scn_maxpool_backward_through: null d_out");
  return maxpool_backward(ctx, d_din, d_dout, count, C, d_choice, d_out, act);
}

// ------------------------------------ the gradient of a pooling's input, by rows
// The scatter above adds, where a row of the input has a window or a few: with the
// pooling's rules turned round (inverse[r slots + j] = the window in which row r lies
// at the j-th of the offsets that a row may have in a window; negative: none) every
// row is read together and written once, nothing is cleared and no float is added
// atomically.  A sample's background row may lie in any of its windows: those are
// walked by one to eight wavefronts a sample and 16 channels, which also sums, where the layer
// before the pooling is a convolution, what goes to the rows that name that
// convolution's background, per position (what k_background_sums makes of din), from
// the same windows: an output of the pooling has one row that it chose.
//
// A row's slot: ceil(size / stride) of them an axis.
static int pool_slots(int dimension, int size, int stride, int *perAxis) {
  *perAxis = stride >= 1 ? (size + stride - 1) / stride : 0;
  int n = 1;
  for (int a = 0; a < dimension; ++a)
    n *= *perAxis;
  return n == 1 || n == 2 || n == 4 || n == 8 ? n : 0;
}
extern "C" int scn_pool_inverse_slots(int dimension, int size, int stride) {
  int k;
  double width = 1; // (positions of a window)
  for (int a = 0; a < dimension; ++a)
    width *= size;
  return dimension >= 1 && dimension <= 8 && size >= 1 && stride >= 1 && width <= 1024 ? pool_slots(dimension, size, stride, &k) : 0;
}
struct PoolInverseList {
  const int *rules[SCN_INVERSE_MAX], *bg[SCN_INVERSE_MAX], *outBg[SCN_INVERSE_MAX];
  int *inverse[SCN_INVERSE_MAX], *samples[SCN_INVERSE_MAX], *copy[SCN_INVERSE_MAX]; // copy: null, or the host's memory
  long long volume[SCN_INVERSE_MAX];
  int rows[SCN_INVERSE_MAX], inRows[SCN_INVERSE_MAX], batch[SCN_INVERSE_MAX];
  int dimension[SCN_INVERSE_MAX], size[SCN_INVERSE_MAX], stride[SCN_INVERSE_MAX], slots[SCN_INVERSE_MAX];
  unsigned firstBlock[SCN_INVERSE_MAX + 1];
  int count;
};
// a workgroup an item: where the samples' windows begin, and the background rows' marks
__global__ __launch_bounds__(256) void k_pool_samples(PoolInverseList l) {
  const int t = blockIdx.x, batch = l.batch[t], slots = l.slots[t];
  int *const copy = l.copy[t];
  // A sample's rows are its sites and then, if it is not full, a background row: its
  // last row follows from that row of the last sample up to it that has one, and the
  // full ones since.  (The last such sample by a running maximum; each looking back by
  // itself: 18 us where the small fields of a batch of 100 drawings are full.)
  __shared__ int sLast[256];
  const int lane = threadIdx.x;
  int carry = -1;
  if (lane == 0) {
    l.samples[t][0] = 0;
    if (copy)
      copy[0] = 0;
  }
  for (int base = 0; base < batch; base += 256) { // uniform
    const int s = base + lane, row = s < batch ? l.outBg[t][s] : -1;
    int last = row >= 0 ? s : carry;
    sLast[lane] = last;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      const int other = lane >= off ? sLast[lane - off] : -1;
      last = other > last ? other : last;
      __syncthreads();
      sLast[lane] = last;
      __syncthreads();
    }
    carry = sLast[255];
    __syncthreads();
    if (s < batch) {
      const long long e = last >= 0 ? l.outBg[t][last] + 1 + (s - last) * l.volume[t] : (s + 1) * l.volume[t];
      const int to = (int)(e < l.rows[t] ? e : l.rows[t]);
      l.samples[t][s + 1] = to;
      if (copy)
        copy[s + 1] = to;
    }
  }
  for (int s = threadIdx.x; s < batch; s += 256) {
    const int r = l.bg[t][s], mine = r >= 0 && r < l.inRows[t] ? r : -1;
    l.samples[t][batch + 1 + s] = mine;
    if (mine >= 0)
      for (int j = 0; j < slots; ++j)
        l.inverse[t][(long long)mine * slots + j] = -2;
  }
}
// a lane a window
__global__ __launch_bounds__(256) void k_pool_inverse(PoolInverseList l) {
  static_assert(SCN_INVERSE_MAX <= 64, "a lane an item");
  const int lane = threadIdx.x & 63;
  const int t =
      __popcll(__ballot(lane < l.count && blockIdx.x >= l.firstBlock[lane < SCN_INVERSE_MAX ? lane : 0])) - 1;
  const long long o = (long long)(blockIdx.x - l.firstBlock[t]) * 256 + threadIdx.x;
  if (o >= l.rows[t])
    return;
  const int dimension = l.dimension[t], size = l.size[t], stride = l.stride[t], slots = l.slots[t], inRows = l.inRows[t];
  const int perAxis = (size + stride - 1) / stride;
  int width = 1;
  for (int a = 0; a < dimension; ++a)
    width *= size;
  int *const inverse = l.inverse[t];
  for (int f = 0; f < width; ++f) { // (uniform; offsets along the last axis first)
    int j = 0;
    for (int a = 0, x = f, each = 1; a < dimension; ++a, x /= size, each *= perAxis)
      j += x % size / stride * each;
    const int r = l.rules[t][o * width + f];
    if (r < 0 || r >= inRows)
      continue;
    int *const at = inverse + (long long)r * slots + j;
    if (*at != -2)
      *at = (int)o;
  }
}
extern "C" int scn_pool_inverse_many(scn_ctx *ctx, const scn_pool_inverse_item *items, int nItems) {
  return scn_pool_inverse_many_copy(ctx, items, nItems, nullptr);
}
extern "C" int scn_pool_inverse_many_copy(scn_ctx *ctx, const scn_pool_inverse_item *items, int nItems, int32_t *copy) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_pool_inverse_many: null context");
  SCN_REQUIRE(nItems >= 0 && nItems <= SCN_INVERSE_MAX && (items || nItems == 0), SCN_ERR_ARG,
              "scn_pool_inverse_many: %d items (at most %d)", nItems, SCN_INVERSE_MAX);
  PoolInverseList l;
  void *fill[SCN_INVERSE_MAX];
  size_t words[SCN_INVERSE_MAX];
  long long blocks = 0; // (16 items of no more than 2^23 workgroups)
  int fills = 0;
  l.count = 0;
  for (int k = 0; k < nItems; ++k) {
    const scn_pool_inverse_item &it = items[k];
    SCN_REQUIRE(it.input && it.output && it.rows >= 0 && it.rows <= 0x7fffffffll && it.inputRows >= 0, SCN_ERR_ARG,
                "scn_pool_inverse_many: item %d rows %lld of %lld", k, (long long)it.rows, (long long)it.inputRows);
    const int slots = scn_pool_inverse_slots(it.input->d, it.size, it.stride);
    SCN_REQUIRE(slots > 0, SCN_ERR_ARG, "scn_pool_inverse_many: item %d size %d stride %d", k, it.size, it.stride);
    SCN_REQUIRE(it.inputRows * slots <= 0x7fffffffll, SCN_ERR_CAPACITY, "scn_pool_inverse_many: item %d: %lld rows", k,
                (long long)it.inputRows);
    SCN_REQUIRE(!it.input->pending && !it.output->pending, SCN_ERR_STATE,
                "scn_pool_inverse_many: item %d: counts not settled", k);
    SCN_REQUIRE(it.input->batch == it.output->batch && it.input->d == it.output->d, SCN_ERR_ARG,
                "scn_pool_inverse_many: item %d: grids of another pooling", k);
    SCN_REQUIRE((it.d_rules || it.rows == 0) && (it.d_inverse || it.inputRows == 0) && it.d_samples, SCN_ERR_ARG,
                "scn_pool_inverse_many: item %d null buffer", k);
    const int c = l.count++;
    l.rules[c] = it.d_rules;
    l.bg[c] = it.input->bg.p;
    l.outBg[c] = it.output->bg.p;
    l.volume[c] = it.output->vol;
    l.inverse[c] = it.d_inverse;
    l.samples[c] = it.d_samples;
    l.copy[c] = copy;
    if (copy)
      copy += it.input->batch + 1;
    l.rows[c] = (int)it.rows;
    l.inRows[c] = (int)it.inputRows;
    l.batch[c] = it.input->batch;
    l.dimension[c] = it.input->d;
    l.size[c] = it.size;
    l.stride[c] = it.stride;
    l.slots[c] = slots;
    l.firstBlock[c] = (unsigned)blocks;
    blocks += scn_ceil_div(it.rows, 256);
    if (it.inputRows) {
      fill[fills] = it.d_inverse;
      words[fills++] = (size_t)it.inputRows * slots;
    }
  }
  if (l.count == 0)
    return SCN_OK;
  l.firstBlock[l.count] = (unsigned)blocks;
  ProfScope prof(ctx, SCN_K_RULES);
  if (fills)
    SCN_TRY(scn_fill32_many(ctx, fill, words, fills, 0xffffffffu));
  hipLaunchKernelGGL(k_pool_samples, dim3(l.count), dim3(256), 0, ctx->stream, l);
  if (blocks)
    hipLaunchKernelGGL(k_pool_inverse, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, l);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

struct PoolGradient {
  float *din;
  const float *dout, *out; // out: the derivative of act is taken through it (null: has been)
  const int *choice, *inverse, *samples, *background;
  int rows, inRows, C, batch, act, fs, chunks;
  int waves; // wavefronts to a sample and 16 channels: 1, 2, 4 or 8
  unsigned sampleBlocks, magic; // choice / C = (choice * magic >> 32) >> shift
  int shift;
};
// the sum over the two lanes of a row of sixteen that lie eight apart
__device__ __forceinline__ float sum_eights(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false)); // row_ror:8
}
// (the activation is the same for all: one branch)
template <int V>
__device__ __forceinline__ void pool_gradient_of(const PoolGradient &g, float (&d)[V], const float (&o)[V]) {
  float none = 0.f;
  if (!g.out)
    return;
  if (g.act == SCN_RELU) {
#pragma unroll
    for (int k = 0; k < V; ++k)
      d[k] = act_derivative(SCN_RELU, o[k], d[k], 0.f, none);
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k)
      d[k] = act_derivative(g.act, o[k], d[k], g.act == SCN_LEAKYRELU ? 0.01f : 0.333f, none);
  }
}
// Bound by the lines it asks for: of a row the windows that are there and no others
// (asked for all the same: rows alone 20.8 us and not 11.8), of a sample's windows 64
// bytes a request (32: 19 us for the samples alone and not 12).  57456 x 32 of 116619
// rows of 100 samples, side 3: 16.9 us, with 4 sums, where clearing, scattering and
// k_background_sums take 7 + 23 + 7; 27157 x 64 of 57508 16.9, 31; 39071 x 32 of 203375
// voxels of 32 samples, side 2, with 8 sums, 22, 42.
template <int W, int FS>
__global__ __launch_bounds__(512, W == 8 ? 4 : 8) void k_maxpool_gradient(PoolGradient g) {
  constexpr int T = 512;
  const int tid = threadIdx.x, C = g.C;
  if (blockIdx.x < g.sampleBlocks) { // samples, eight lanes of two channels
    constexpr int SUMS = 2 * (FS + 1), AHEAD = 4;
    __shared__ float sSum[T / 16][8][SUMS]; // [row of sixteen lanes][lane][position, channel]
    const int waves = g.waves, STEP = 8 * waves;
    // (a wavefront's item is the same in all its lanes)
    const int item = __builtin_amdgcn_readfirstlane((int)blockIdx.x * (T / 64 / waves) + (tid >> 6) / waves);
    const int sample = item / g.chunks, j = tid & 7;
    const int c = item % g.chunks * 16 + 2 * j;
    const bool there = sample < g.batch;
    const int first = there ? g.samples[sample] : 0, end = there ? g.samples[sample + 1] : 0;
    const int bg = there ? g.samples[g.batch + 1 + sample] : -1;
    float acc[FS + 1][2] = {};
    if (c < C)
      for (int w = first + (tid % (64 * waves) >> 3); w < end; w += AHEAD * STEP) {
        int ch[AHEAD][2];
        float d[AHEAD][2], o[AHEAD][2];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
          const int wu = w + u * STEP < end ? w + u * STEP : w;
          const size_t at = (size_t)wu * C + c;
          const int2 cc = *reinterpret_cast<const int2 *>(g.choice + at);
          const float2 dd = *reinterpret_cast<const float2 *>(g.dout + at);
          const float2 oo = g.out ? *reinterpret_cast<const float2 *>(g.out + at) : dd;
          ch[u][0] = w + u * STEP < end ? cc.x : -1, ch[u][1] = w + u * STEP < end ? cc.y : -1;
          d[u][0] = dd.x, d[u][1] = dd.y, o[u][0] = oo.x, o[u][1] = oo.y;
        }
        int mask[AHEAD][2];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int row = ch[u][k] >= 0 ? (int)(__umulhi((unsigned)ch[u][k], g.magic) >> g.shift) : -1;
            ch[u][k] = row;
            if (FS > 0) {
              const bool in = row >= 0 && row < g.inRows;
              const int m = g.background[in ? row : 0];
              mask[u][k] = in ? m : 0;
            }
          }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
          pool_gradient_of<2>(g, d[u], o[u]);
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            acc[FS][k] += ch[u][k] >= 0 && ch[u][k] == bg ? d[u][k] : 0.f;
#pragma unroll
            for (int f = 0; f < FS; ++f)
              acc[f][k] += mask[u][k] >> f & 1 ? d[u][k] : 0.f;
          }
        }
      }
#pragma unroll
    for (int f = 0; f <= FS; ++f)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const float v = sum_eights(acc[f][k]);
        if ((tid & 15) < 8)
          sSum[tid >> 4][j][2 * f + k] = v;
      }
    __syncthreads();
    // a sum to a lane: the item's wavefronts share them
    for (int x = tid % (64 * waves); x < 8 * SUMS; x += 64 * waves) {
      const int k = x & 1, q = x >> 1 & 7, f = x >> 4;
      const int cc = item % g.chunks * 16 + 2 * q + k;
      if (!there || cc >= C || (f < FS && f >= g.fs) || (f == FS && bg < 0))
        continue;
      const int row0 = (tid >> 6) / waves * waves * 4;
      float sum = 0.f;
      for (int y = 0; y < 4 * waves; ++y)
        sum += sSum[row0 + y][q][2 * f + k];
      const long long row = f == FS ? bg : g.inRows + (long long)sample * g.fs + f;
      g.din[row * C + cc] = sum;
    }
    return;
  }
  // a row and four channels to a lane
  const unsigned quads = C / 4;
  const unsigned at = xcd_eighth(blockIdx.x - g.sampleBlocks, gridDim.x - g.sampleBlocks) * T + tid;
  const unsigned r = at / quads;
  if (r >= (unsigned)g.inRows)
    return;
  const int c = (int)(at - r * quads) * 4, flat = (int)(r * C) + c;
  int w[W];
  const int *const from = g.inverse + (size_t)r * W;
  if constexpr (W % 4 == 0) {
#pragma unroll
    for (int j = 0; j < W; j += 4) {
      const int4 x = *reinterpret_cast<const int4 *>(from + j);
      w[j] = x.x, w[j + 1] = x.y, w[j + 2] = x.z, w[j + 3] = x.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < W; ++j)
      w[j] = from[j];
  }
  if (w[0] == -2) // a background row
    return;
  // (all windows are asked for together)
  int4 ch[W];
  float4 d[W], o[W];
#pragma unroll
  for (int j = 0; j < W; ++j) {
    ch[j] = make_int4(-1, -1, -1, -1);
    if (w[j] >= 0) {
      const size_t x = (size_t)(unsigned)(w[j] * C + c);
      ch[j] = *reinterpret_cast<const int4 *>(g.choice + x);
      d[j] = *reinterpret_cast<const float4 *>(g.dout + x);
      if (g.out)
        o[j] = *reinterpret_cast<const float4 *>(g.out + x);
    }
  }
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < W; ++j) {
    float v[4] = {d[j].x, d[j].y, d[j].z, d[j].w};
    const float y[4] = {o[j].x, o[j].y, o[j].z, o[j].w};
    pool_gradient_of<4>(g, v, y);
    const int t[4] = {ch[j].x, ch[j].y, ch[j].z, ch[j].w};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      sum[k] += t[k] == flat + k ? v[k] : 0.f;
  }
  *reinterpret_cast<float4 *>(g.din + (size_t)r * C + c) = make_float4(sum[0], sum[1], sum[2], sum[3]);
}
extern "C" int scn_maxpool_gradient(scn_ctx *ctx, float *d_din, int64_t inputRows, const float *d_dout, int64_t rows,
                                    int C, const int32_t *d_choice, const float *d_out, int act,
                                    const int32_t *d_inverse, int slots, const int32_t *d_samples, int batch,
                                    const int32_t *d_background, int fs) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_maxpool_gradient: null context");
  SCN_REQUIRE(rows >= 0 && inputRows >= 0 && C >= 4 && C % 4 == 0 && batch >= 0, SCN_ERR_ARG,
              "scn_maxpool_gradient: rows %lld of %lld C %d batch %d", (long long)rows, (long long)inputRows, C, batch);
  SCN_REQUIRE(slots == 1 || slots == 2 || slots == 4 || slots == 8, SCN_ERR_ARG, "scn_maxpool_gradient: %d slots", slots);
  SCN_REQUIRE(!d_background || (fs >= 1 && fs <= 8), SCN_ERR_ARG, "scn_maxpool_gradient: fs %d", fs);
  SCN_REQUIRE(act >= SCN_NOSIGMOID && act <= SCN_SIGMOID && act != SCN_PRELU, SCN_ERR_ARG,
              "scn_maxpool_gradient: activation %d", act);
  SCN_REQUIRE(inputRows * C <= 0x7fffffffll && rows * C <= 0x7fffffffll, SCN_ERR_CAPACITY,
              "scn_maxpool_gradient: %lld x %d", (long long)inputRows, C);
  const int64_t sums = d_background ? (int64_t)batch * fs : 0;
  if (inputRows + sums == 0)
    return SCN_OK;
  SCN_REQUIRE(d_din, SCN_ERR_ARG, "scn_maxpool_gradient: null d_din");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  if (rows == 0)
    return scn_fill32(ctx, d_din, 0, (size_t)(inputRows + sums) * C);
  SCN_REQUIRE(d_dout && d_choice && d_samples && (d_inverse || inputRows == 0), SCN_ERR_ARG,
              "scn_maxpool_gradient: null buffer");
  SCN_REQUIRE((((uintptr_t)d_din | (uintptr_t)d_dout | (uintptr_t)d_choice | (uintptr_t)d_out | (uintptr_t)d_inverse) & 15) == 0,
              SCN_ERR_ARG, "scn_maxpool_gradient: buffers start on 16 bytes");
  PoolGradient g = {d_din, d_dout, d_out, d_choice, d_inverse, d_samples, d_background, (int)rows, (int)inputRows, C,
                    batch, act, d_background ? fs : 0, scn_ceil_div(C, 16), 1, 0u, 0u, 0};
  SCN_REQUIRE((int64_t)batch * g.chunks <= 0x3fffffffll, SCN_ERR_CAPACITY, "scn_maxpool_gradient: batch %d", batch);
  // (32 windows to a wavefront and round)
  while (g.waves < 8 && rows > 32ll * g.waves * batch)
    g.waves *= 2;
  g.sampleBlocks = (unsigned)scn_ceil_div((int64_t)batch * g.chunks, 8 / g.waves);
  // x / C for x < 2^31: ceil(2^(31 + s) / C), s = ceil(log2 C)
  int s = 0;
  while ((1ll << s) < C)
    ++s;
  g.magic = (unsigned)(((1ull << (31 + s)) + C - 1) / C);
  g.shift = s - 1;
  const dim3 grid(g.sampleBlocks + (unsigned)scn_ceil_div(inputRows * (C / 4), 512));
#define SCN_PG_GO(W, FS) hipLaunchKernelGGL((k_maxpool_gradient<W, FS>), grid, dim3(512), 0, ctx->stream, g)
#define SCN_PG_FS(W)     \
  if (g.fs == 0)         \
    SCN_PG_GO(W, 0);     \
  else if (g.fs <= 4)    \
    SCN_PG_GO(W, 4);     \
  else                   \
    SCN_PG_GO(W, 8)
  if (slots == 1) {
    SCN_PG_FS(1);
  } else if (slots == 2) {
    SCN_PG_FS(2);
  } else if (slots == 4) {
    SCN_PG_FS(4);
  } else {
    SCN_PG_FS(8);
  }
#undef SCN_PG_FS
#undef SCN_PG_GO
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// dTerminalPoolBackProp: every row listed for a sample receives (not
// accumulates) the sample's gradient divided by the number of rows listed.
__global__ void k_terminal_backward(float *__restrict__ din,
                                    const float *__restrict__ dout,
                                    const int *__restrict__ rules, int C,
                                    int S) {
  const long long b = blockIdx.x;
  const int *rr = rules + b * S;
  int maxP = 0;
  while (maxP < S && rr[maxP] >= 0)
    ++maxP;
  for (int j = threadIdx.x; j < C; j += blockDim.x) {
    const float t = dout[b * C + j] / (float)maxP;
    for (int p = 0; p < maxP; ++p)
      din[(long long)rr[p] * C + j] = t;
  }
}

extern "C" int scn_terminal_pool_backward(scn_ctx *ctx, float *d_din,
                                          const float *d_dout,
                                          const int32_t *d_rules,
                                          int64_t count, int C, int S) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_terminal_pool_backward: null context");
  SCN_REQUIRE(count >= 0 && C >= 1 && S >= 1, SCN_ERR_ARG,
              "scn_terminal_pool_backward: count %lld C %d S %d",
              (long long)count, C, S);
  if (count == 0)
    return SCN_OK;
  SCN_REQUIRE(count <= 0x7fffffffll, SCN_ERR_CAPACITY,
              "scn_terminal_pool_backward: %lld samples", (long long)count);
  SCN_REQUIRE(d_din && d_dout && d_rules, SCN_ERR_ARG,
              "scn_terminal_pool_backward: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  hipLaunchKernelGGL(k_terminal_backward, dim3((unsigned)count),
                     dim3(C >= 256 ? 256 : 64), 0, ctx->stream, d_din, d_dout,
                     d_rules, C, S);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// The backward pass of a net's end in one launch: the classifier's d input = D W^T,
// spread by the terminal pooling over its rows, times the derivative of the activation
// that made them, with the sums of a PReLU's slopes.  Every launch of such a batch is 4
// us whatever it holds (100 drawings: W transposed 2.7, the product 5.5, spread 3.6,
// derivative 6.0 us and a gap each -> 7.3).  A workgroup has two samples, as k_classifier;
// 32 lanes take a row of W, its products with both are summed across them.  Then a lane
// has four channels of a sample: its rows four at a time.  Code that is run once is
// fetched by every compute unit, which is most of what is left: with the derivative's
// cases and eight rows laid out one after the other it took 10 to 14 us.
#define TG_ROWS 2
#define TG_THREADS 512
#define TG_DEPTH 12
#define TG_MAX_K 1024
#define TG_MAX_N 128
struct TerminalGradient {
  const float *delta, *W; // [M x N], [K x N]
  float *dpooled;         // [M x K]
  const int *rules;       // [M x S]
  float *din;
  const float *features; // of the rows that are pooled
  const float *prelu;
  float *dprelu;
  long long M;
  int S, K, N, act;
};
// the sum over 32 lanes, in all of them
__device__ __forceinline__ float sum32(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));  // 1 0 3 2
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));  // 2 3 0 1
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true)); // eight turned round
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true)); // sixteen
  return v + __shfl_xor(v, 16, 64);
}
__global__ __launch_bounds__(TG_THREADS) void k_terminal_gradient(TerminalGradient g) {
  __shared__ __attribute__((aligned(16))) float sD[TG_ROWS][TG_MAX_N], sT[TG_ROWS][TG_MAX_K];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long long m0 = (long long)blockIdx.x * TG_ROWS;
  const int K = g.K, N = g.N, S = g.S;
  static_assert(TG_THREADS == TG_ROWS * TG_MAX_K / 4, "a lane four channels");
  const int row = tid / (TG_MAX_K / 4), k = 4 * (tid % (TG_MAX_K / 4));
  const long long m = m0 + row;
  constexpr int RULES = 4; // at a time
  int rule[RULES];
  auto load_rules = [&](int p0) {
#pragma unroll
    for (int u = 0; u < RULES; ++u)
      rule[u] = m < g.M && p0 + u < S ? g.rules[m * S + p0 + u] : -1;
  };
  load_rules(0);
  if (tid < TG_ROWS * TG_MAX_N) {
    const int r = tid / TG_MAX_N, j = tid % TG_MAX_N;
    sD[r][j] = m0 + r < g.M && j < N ? g.delta[(m0 + r) * N + j] : 0.f;
  }
  // rows of W: two a wavefront and load, sixteen a workgroup
  const int j4 = 4 * (lane & 31), c0 = 2 * wave + (lane >> 5);
  const float *const w = g.W + (j4 < N ? j4 : 0); // (past the end: times zero)
  float4 wv[TG_DEPTH];
  auto load_w = [&](int from) {
#pragma unroll
    for (int i = 0; i < TG_DEPTH; ++i) {
      const int c = from + 16 * i < K ? from + 16 * i : K - 1; // (not stored)
      wv[i] = *reinterpret_cast<const float4 *>(w + (long long)c * N);
    }
  };
  load_w(c0);
  __syncthreads();
  float4 d[TG_ROWS];
#pragma unroll
  for (int r = 0; r < TG_ROWS; ++r)
    d[r] = j4 < N ? *reinterpret_cast<const float4 *>(&sD[r][j4]) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 1
  for (int from = c0;; from += 16 * TG_DEPTH) {
    float t[TG_ROWS][TG_DEPTH];
#pragma unroll
    for (int i = 0; i < TG_DEPTH; ++i)
#pragma unroll
      for (int r = 0; r < TG_ROWS; ++r)
        t[r][i] = j4 < N ? fmaf(wv[i].x, d[r].x, wv[i].y * d[r].y) + fmaf(wv[i].z, d[r].z, wv[i].w * d[r].w) : 0.f;
    const bool more = from - c0 + 16 * TG_DEPTH < K; // uniform
    if (more)
      load_w(from + 16 * TG_DEPTH);
#pragma unroll
    for (int i = 0; i < TG_DEPTH; ++i)
#pragma unroll
      for (int r = 0; r < TG_ROWS; ++r) {
        t[r][i] = sum32(t[r][i]);
        if ((lane & 31) == 0 && from + 16 * i < K)
          sT[r][from + 16 * i] = t[r][i];
      }
    if (!more)
      break;
  }
  __syncthreads();
  float slope[4] = {0.f, 0.f, 0.f, 0.f};
  if (m < g.M && k < K) {
    const float4 t4 = *reinterpret_cast<const float4 *>(&sT[row][k]);
    *reinterpret_cast<float4 *>(g.dpooled + m * K + k) = t4;
    // the rows up to the first negative rule
    int count = 0;
    bool more = true;
#pragma unroll 1
    for (int p0 = 0; p0 < S && more; p0 += RULES) {
      if (p0)
        load_rules(p0);
#pragma unroll
      for (int u = 0; u < RULES; ++u) {
        more = more && rule[u] >= 0;
        count += more;
      }
    }
    const bool curved = g.act == SCN_TANH || g.act == SCN_SIGMOID;
    float t[4] = {t4.x / (float)count, t4.y / (float)count, t4.z / (float)count, t4.w / (float)count}, neg[4], alpha[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { // (as act_derivative)
      alpha[i] = g.act == SCN_PRELU ? g.prelu[k + i] : g.act == SCN_LEAKYRELU ? 0.01f : 0.333f;
      neg[i] = g.act == SCN_RELU ? 0.f : g.act == SCN_NOSIGMOID || g.act == SCN_SOFTMAX ? t[i] : t[i] * alpha[i];
    }
#pragma unroll 1
    for (int p0 = 0; p0 < count; p0 += RULES) {
      if (S > RULES)
        load_rules(p0);
      float4 y[RULES];
#pragma unroll
      for (int u = 0; u < RULES; ++u) // (past the last: that one again)
        y[u] = *reinterpret_cast<const float4 *>(g.features + (long long)(p0 + u < count ? rule[u] : rule[0]) * K + k);
#pragma unroll
      for (int u = 0; u < RULES; ++u) {
        const float v[4] = {y[u].x, y[u].y, y[u].z, y[u].w};
        float r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          r[i] = v[i] > 0 ? t[i] : neg[i];
        if (curved) { // uniform
#pragma unroll
          for (int i = 0; i < 4; ++i)
            r[i] = g.act == SCN_TANH ? t[i] * (1 + v[i]) * (1 - v[i]) : t[i] * v[i] * (1 - v[i]);
        }
        if (p0 + u < count) {
          *reinterpret_cast<float4 *>(g.din + (long long)rule[u] * K + k) = make_float4(r[0], r[1], r[2], r[3]);
          if (g.act == SCN_PRELU) // uniform
#pragma unroll
            for (int i = 0; i < 4; ++i)
              slope[i] += v[i] > 0 ? 0.f : t[i] * (v[i] / alpha[i]);
        }
      }
    }
  }
  if (g.act != SCN_PRELU) // uniform
    return;
  __syncthreads(); // (sT has been read)
  if (k < K)
    *reinterpret_cast<float4 *>(&sT[row][k]) = make_float4(slope[0], slope[1], slope[2], slope[3]);
  __syncthreads();
  for (int c = tid; c < K; c += TG_THREADS)
    unsafeAtomicAdd(g.dprelu + c, sT[0][c] + sT[1][c]);
}
extern "C" int scn_terminal_gradient_supported(int K, int N) {
  return K >= 4 && K <= TG_MAX_K && K % 4 == 0 && N >= 4 && N <= TG_MAX_N && N % 4 == 0;
}
extern "C" int scn_terminal_gradient(scn_ctx *ctx, const float *d_delta, const float *d_W, float *d_dpooled,
                                     const int32_t *d_rules, int64_t M, int S, float *d_din, const float *d_features,
                                     int act, const float *d_prelu, float *d_dprelu, int K, int N) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_terminal_gradient: null context");
  SCN_REQUIRE(M >= 0 && S >= 1 && scn_terminal_gradient_supported(K, N) && act >= SCN_NOSIGMOID && act <= SCN_SIGMOID,
              SCN_ERR_ARG, "scn_terminal_gradient: M %lld S %d K %d N %d activation %d", (long long)M, S, K, N, act);
  if (M == 0)
    return SCN_OK;
  SCN_REQUIRE(scn_ceil_div(M, TG_ROWS) <= 0x7fffffffll, SCN_ERR_CAPACITY, "scn_terminal_gradient: %lld samples", (long long)M);
  // (d_din and d_features may be null: no rows, every rule negative)
  SCN_REQUIRE(d_delta && d_W && d_dpooled && d_rules && (act != SCN_PRELU || (d_prelu && d_dprelu)), SCN_ERR_ARG,
              "scn_terminal_gradient: null buffer");
  SCN_REQUIRE((((uintptr_t)d_W | (uintptr_t)d_dpooled | (uintptr_t)d_din | (uintptr_t)d_features) & 15) == 0, SCN_ERR_ARG,
              "scn_terminal_gradient: matrices start on 16 bytes");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  const TerminalGradient g = {d_delta, d_W, d_dpooled, d_rules, d_din, d_features, d_prelu, d_dprelu, M, S, K, N, act};
  hipLaunchKernelGGL(k_terminal_gradient, dim3((unsigned)scn_ceil_div(M, TG_ROWS)), dim3(TG_THREADS), 0, ctx->stream, g);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// ------------------------------------------------ dropout during training
// A training batch keeps a random subset of every layer's features
// (featuresPresent); the layer then works on the sub-matrix of its weights
// that joins the kept inputs to the kept outputs.
__global__ void k_shrink_matrix(const float *__restrict__ W,
                                float *__restrict__ w,
                                const int *__restrict__ inPresent,
                                const int *__restrict__ outPresent, int nOut,
                                long long total, int nOutP) {
  long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total)
    return;
  const long long i = idx / nOutP;
  const int j = (int)(idx - i * nOutP);
  const long long row = inPresent ? inPresent[i] : i;
  w[idx] = W[row * nOut + outPresent[j]];
}

extern "C" int scn_shrink_matrix(scn_ctx *ctx, const float *d_W, float *d_w,
                                 const int32_t *d_inPresent,
                                 const int32_t *d_outPresent, int nOut,
                                 int nInPresent, int nOutPresent) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_shrink_matrix: null context");
  SCN_REQUIRE(nOut >= 1 && nInPresent >= 0 && nOutPresent >= 0 &&
                  nOutPresent <= nOut,
              SCN_ERR_ARG, "scn_shrink_matrix: nOut %d present %d x %d", nOut,
              nInPresent, nOutPresent);
  const long long total = (long long)nInPresent * nOutPresent;
  if (total == 0)
    return SCN_OK;
  SCN_REQUIRE(d_W && d_w && d_outPresent, SCN_ERR_ARG,
              "scn_shrink_matrix: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  hipLaunchKernelGGL(k_shrink_matrix, dim3(scn_ceil_div(total, 256)), dim3(256),
                     0, ctx->stream, d_W, d_w, d_inPresent, d_outPresent, nOut,
                     total, nOutPresent);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// dGradientDescentShrunkMatrix: the momentum step on the entries of W (and MW)
// that the batch used; delta is the gradient of the shrunk matrix.
__global__ void k_nag_update_shrunk(const float *__restrict__ delta,
                                    float *__restrict__ mom,
                                    float *__restrict__ wts,
                                    const int *__restrict__ inPresent,
                                    const int *__restrict__ outPresent,
                                    int nOut, long long total, int nOutP,
                                    float lr, float mu) {
  long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total)
    return;
  const long long i = idx / nOutP;
  const int j = (int)(idx - i * nOutP);
  const long long row = inPresent ? inPresent[i] : i;
  const long long at = row * nOut + outPresent[j];
  float w = wts[at], m = mom[at];
  const float d = delta[idx];
  w -= m * mu;
  m = mu * m - lr * (1 - mu) * d;
  w += m * (1 + mu);
  wts[at] = w;
  mom[at] = m;
}

extern "C" int scn_nag_update_shrunk(scn_ctx *ctx, const float *d_delta,
                                     float *d_momentum, float *d_weights,
                                     const int32_t *d_inPresent,
                                     const int32_t *d_outPresent, int nOut,
                                     int nInPresent, int nOutPresent,
                                     float learningRate, float momentum) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_nag_update_shrunk: null context");
  SCN_REQUIRE(nOut >= 1 && nInPresent >= 0 && nOutPresent >= 0 &&
                  nOutPresent <= nOut,
              SCN_ERR_ARG, "scn_nag_update_shrunk: nOut %d present %d x %d",
              nOut, nInPresent, nOutPresent);
  const long long total = (long long)nInPresent * nOutPresent;
  if (total == 0)
    return SCN_OK;
  SCN_REQUIRE(d_delta && d_momentum && d_weights && d_outPresent, SCN_ERR_ARG,
              "scn_nag_update_shrunk: null buffer");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  hipLaunchKernelGGL(k_nag_update_shrunk, dim3(scn_ceil_div(total, 256)),
                     dim3(256), 0, ctx->stream, d_delta, d_momentum, d_weights,
                     d_inPresent, d_outPresent, nOut, total, nOutPresent,
                     learningRate, momentum);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// ------------------------------------------------ weight rescaling passes
// What a RESCALEBATCH needs of vectorCUDA<float>: meanAbs() and
// multiplicativeRescale() (vectorCUDA.cu:121-170).
__global__ __launch_bounds__(256) void k_sum_abs(const float *__restrict__ x,
                                                 long long n, double *out) {
  __shared__ double part[4];
  double s = 0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    s += fabsf(x[i]);
  for (int o = 32; o > 0; o >>= 1)
    s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0)
    part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0)
    unsafeAtomicAdd(out, part[0] + part[1] + part[2] + part[3]);
}

extern "C" int scn_sum_abs(scn_ctx *ctx, const float *d_x, int64_t n,
                           double *h_sum) {
  SCN_REQUIRE(ctx && h_sum, SCN_ERR_ARG, "scn_sum_abs: null argument");
  SCN_REQUIRE(n >= 0, SCN_ERR_ARG, "scn_sum_abs: n %lld", (long long)n);
  *h_sum = 0;
  if (n == 0)
    return SCN_OK;
  SCN_REQUIRE(d_x, SCN_ERR_ARG, "scn_sum_abs: null buffer");
  double *acc = (double *)(ctx->d_scalars + 8); // words 8..9: free for this
  SCN_TRY(scn_fill32(ctx, acc, 0u, 2));
  int blocks = scn_ceil_div(n, 256 * 16);
  if (blocks > ctx->numCU * 8)
    blocks = ctx->numCU * 8;
  hipLaunchKernelGGL(k_sum_abs, dim3(blocks), dim3(256), 0, ctx->stream, d_x,
                     (long long)n, acc);
  SCN_HIP_CHECK(hipGetLastError());
  return scn_d2h(ctx, h_sum, acc, sizeof(double));
}

__global__ void k_scale(float *__restrict__ x, long long n, float m) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    x[i] *= m;
}

extern "C" int scn_scale(scn_ctx *ctx, float *d_x, int64_t n,
                         float multiplier) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_scale: null context");
  SCN_REQUIRE(n >= 0, SCN_ERR_ARG, "scn_scale: n %lld", (long long)n);
  if (n == 0)
    return SCN_OK;
  SCN_REQUIRE(d_x, SCN_ERR_ARG, "scn_scale: null buffer");
  hipLaunchKernelGGL(k_scale, dim3(scn_ceil_div(n, 256)), dim3(256), 0,
                     ctx->stream, d_x, (long long)n, multiplier);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}
