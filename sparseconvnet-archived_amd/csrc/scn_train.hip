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
#include "scn_nin_dev.h"
#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

typedef float floatx4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- softmax
__global__ void k_softmax_grad(const float *__restrict__ probs,
                               const int *__restrict__ labels,
                               float *__restrict__ delta, long long total,
                               int N) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total)
    return;
  long long k = i / N;
  int c = (int)(i - k * N);
  delta[i] = probs[i] - (c == labels[k] ? 1.f : 0.f);
}

extern "C" int scn_softmax_grad(scn_ctx *ctx, const float *d_probs,
                                const int32_t *d_labels, float *d_delta,
                                int64_t batch, int N) {
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
                     0, ctx->stream, d_probs, d_labels, d_delta, total, N);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
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

// ---------------------------------------------- dW = A^T D (scn_planes.hip)
static int sgemm_AtB(scn_ctx *ctx, const float *d_A, const float *d_D,
                     float *d_dW, int64_t M, int K, int N, bool clear) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_sgemm_AtB: null context");
  SCN_REQUIRE(M >= 0 && K >= 1 && N >= 1, SCN_ERR_ARG,
              "scn_sgemm_AtB: M %lld K %d N %d", (long long)M, K, N);
  SCN_REQUIRE(d_dW, SCN_ERR_ARG, "scn_sgemm_AtB: null d_dW");
  ProfScope prof(ctx, SCN_K_BACKWARD);
  if (clear)
    SCN_TRY(scn_fill32(ctx, d_dW, 0, (size_t)K * N));
  if (M == 0)
    return SCN_OK;
  SCN_REQUIRE(d_A && d_D, SCN_ERR_ARG, "scn_sgemm_AtB: null buffer");
  SCN_TRY(scn_atb_planes(ctx, d_A, d_D, d_dW, (long long)M, K, N));
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

extern "C" int scn_sgemm_AtB(scn_ctx *ctx, const float *d_A, const float *d_D,
                             float *d_dW, int64_t M, int K, int N) {
  return sgemm_AtB(ctx, d_A, d_D, d_dW, M, K, N, true);
}

// the kernels only ever add to dW, so beta = 1 is the same launch without the
// clearing one before it
extern "C" int scn_sgemm_AtB_acc(scn_ctx *ctx, const float *d_A,
                                 const float *d_D, float *d_dW, int64_t M,
                                 int K, int N) {
  return sgemm_AtB(ctx, d_A, d_D, d_dW, M, K, N, false);
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
  // (M is the caller's number of rows, whatever scn_ctx_rows_from says to the
  // forward calls, whose kernels run here)
  struct OwnRows {
    scn_ctx *ctx;
    const long long *meta;
    explicit OwnRows(scn_ctx *c) : ctx(c), meta(c->d_meta) { c->d_meta = nullptr; }
    ~OwnRows() { ctx->d_meta = meta; }
  } ownRows(ctx);
  bool transpose = false;
  Epilogue ep = Epilogue();
  ep.bias = ctx->d_zeros;
  ep.p = 1.f;
  ep.act = SCN_NOSIGMOID;
  if (K <= SCN_ZERO_FLOATS) { // the planes read W [K x N] as it stands
    int rc = SCN_OK;
    ProfScope prof(ctx, SCN_K_BACKWARD);
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
    int C, const int *__restrict__ choice, int shift, int slices) {
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

extern "C" int scn_maxpool_backward(scn_ctx *ctx, float *d_din,
                                    const float *d_dout, int64_t count, int C,
                                    const int32_t *d_choice) {
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
                     slices);
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
