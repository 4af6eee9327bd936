// Rule-driven feature kernels: gather, max-pool with argmax, terminal
// average, softmax.  All of them move bytes: they are sized and indexed for
// HBM bandwidth (128-bit accesses wherever the channel count allows, rule
// offsets staged in LDS, 64-bit element offsets).
#include "scn_nin_dev.h"
#include "scn_common.h"

#define GATHER_TILE 256 // rules per block iteration at most
#define GATHER_THREADS 256

// out[c * nIn + j] = in[rules[c] * nIn + j]   (ConvolutionalLayer.cu:12-31)
// The output is one contiguous run per tile, so consecutive lanes write
// consecutive 16-byte chunks; reads are contiguous per rule.  A negative rule
// (the reference reads out of bounds on one) gathers a row of zeros.
// `tile`: rules a workgroup takes at a time.  What it waits for is a trip to the rules and
// one to the rows for every four loads of a lane: fewer rules, halved while a lane has more
// than four loads (so down to between two and four), where there are not as many
// workgroups as compute units (us, with 256 and so: 2000 rows of 8 x
// 128 6.6, 4.9; 60 of 8 x 160 6.5, 4.8; with more workgroups it loses: 30000 of 4 x 64 7.9, 8.5).
template <typename VecT, int VEC>
__global__ void __launch_bounds__(GATHER_THREADS)
    k_gather(const float *__restrict__ in, float *__restrict__ out,
             const int *__restrict__ rules, long long count, int nIn,
             int chunks, const long long *dRows, int perRow, int tile) {
  if (dRows)
    count = live_rows(count / perRow, dRows) * perRow;
  __shared__ long long roff[GATHER_TILE];
  const int tid = threadIdx.x;
  const int q0 = tid / chunks, ch0 = tid - q0 * chunks;
  const int dq = GATHER_THREADS / chunks, dch = GATHER_THREADS - dq * chunks;
  for (long long c0 = (long long)blockIdx.x * tile; c0 < count; c0 += (long long)gridDim.x * tile) {
    long long left = count - c0;
    const int n = left < tile ? (int)left : tile;
    if (tid < n) {
      int rule = rules[c0 + tid];
      roff[tid] = rule < 0 ? -1 : (long long)rule * nIn;
    }
    __syncthreads();
    const int items = n * chunks;
    VecT *dst = reinterpret_cast<VecT *>(out + c0 * nIn);
    int q = q0, ch = ch0;
    int idx = tid;
    // four independent loads in flight per lane
    for (; idx + 3 * GATHER_THREADS < items; idx += 4 * GATHER_THREADS) {
      VecT v[4];
      int qq = q, cc = ch;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        long long ro = roff[qq];
        v[u] = ro < 0 ? VecT{} : *reinterpret_cast<const VecT *>(in + ro + cc * VEC);
        qq += dq;
        cc += dch;
        if (cc >= chunks) {
          cc -= chunks;
          ++qq;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        dst[idx + u * GATHER_THREADS] = v[u];
      q = qq;
      ch = cc;
    }
    for (; idx < items; idx += GATHER_THREADS) {
      long long ro = roff[q];
      dst[idx] = ro < 0 ? VecT{} : *reinterpret_cast<const VecT *>(in + ro + ch * VEC);
      q += dq;
      ch += dch;
      if (ch >= chunks) {
        ch -= chunks;
        ++q;
      }
    }
    __syncthreads();
  }
}

// Rows of one word: four rules to a lane and nothing in LDS (21.5 M rules 46 us, 69 beside what
// a layer does before it, -> 30; 900000 5.5 -> 5.2)
__global__ void __launch_bounds__(256)
    k_gather_words(const float *__restrict__ in, float *__restrict__ out, const int *__restrict__ rules, long long count,
                   const long long *dRows, int perRow) {
  if (dRows)
    count = live_rows(count / perRow, dRows) * perRow;
  const long long at = 4 * ((long long)xcd_eighth(blockIdx.x, gridDim.x) * 256 + threadIdx.x);
  if (at + 4 <= count) {
    const int4 r = *reinterpret_cast<const int4 *>(rules + at);
    *reinterpret_cast<float4 *>(out + at) = make_float4(r.x < 0 ? 0.f : in[r.x], r.y < 0 ? 0.f : in[r.y], r.z < 0 ? 0.f : in[r.z],
                                                        r.w < 0 ? 0.f : in[r.w]);
  } else {
    for (long long i = at; i < count; ++i)
      out[i] = rules[i] < 0 ? 0.f : in[rules[i]];
  }
}

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

extern "C" int scn_gather_rows(scn_ctx *ctx, const float *d_in, float *d_out,
                               const int32_t *d_rules, int64_t count,
                               int nIn) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_gather_rows: null context");
  SCN_REQUIRE(count >= 0 && nIn >= 1, SCN_ERR_ARG,
              "scn_gather_rows: count %lld nIn %d", (long long)count, nIn);
  if (count == 0)
    return SCN_OK;
  SCN_REQUIRE(d_in && d_out && d_rules, SCN_ERR_ARG,
              "scn_gather_rows: null buffer");
  ProfScope ps(ctx, SCN_K_GATHER);
  // (rows not known on the host yet: count is their bound times the rule width)
  const long long *dRows = ctx->d_meta ? ctx->d_meta + META_SITES : nullptr;
  const int perRow = dRows && ctx->rowsBound > 0 ? (int)(count / ctx->rowsBound) : 1;
  // (a launch has fewer than 2^32 lanes, and four rules to a lane: far more rules are the
  // other kernel's, whose workgroups go round)
  if (nIn == 1 && aligned16(d_rules) && aligned16(d_out) && count < (long long)1 << 32) {
    hipLaunchKernelGGL(k_gather_words, dim3((unsigned)((count + 1023) / 1024)), dim3(256), 0, ctx->stream, d_in, d_out, d_rules,
                       (long long)count, dRows, perRow);
    SCN_HIP_CHECK(hipGetLastError());
    return SCN_OK;
  }
  const bool wide = nIn % 4 == 0 && aligned16(d_in) && aligned16(d_out);
  const int chunks = wide ? nIn / 4 : nIn;
  const long long maxBlocks = (long long)ctx->numCU * 16;
  int tile = GATHER_TILE;
  while (tile > 16 && tile * chunks > 4 * GATHER_THREADS && (count + tile - 1) / tile < ctx->numCU)
    tile /= 2;
  const long long tiles = (count + tile - 1) / tile;
  int blocks = (int)(tiles < maxBlocks ? tiles : maxBlocks);
  if (wide) {
    hipLaunchKernelGGL((k_gather<float4, 4>), dim3(blocks),
                       dim3(GATHER_THREADS), 0, ctx->stream, d_in, d_out,
                       d_rules, (long long)count, nIn, chunks, dRows, perRow, tile);
  } else {
    hipLaunchKernelGGL((k_gather<float, 1>), dim3(blocks),
                       dim3(GATHER_THREADS), 0, ctx->stream, d_in, d_out,
                       d_rules, (long long)count, nIn, chunks, dRows, perRow, tile);
  }
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// dMaxPool (MaxPoolingLayer.cu:9-35): strict '<' so the first maximum wins,
// negative rules skipped.  One lane owns VEC channels of one output row.
// A workgroup's rules come in one request a lane through LDS where they fit, and a
// row is told from a lane by a multiplication (a 64-bit division is some 100
// instructions): windows of 3 x 3 from 88000 x 32 7.1 -> 6.7 us, from 57500 x 64 7.9 ->
// 7.3, few of them 3.7 -> 3.5, 246000 x 64 at a copy's rate either way (86.4, 87.8);
// beside a contraction, whose path to memory has nine requests less a window to share,
// more (a layer 596 000 x 2592 -> 128 with its pooling, among others, 458 -> 452).
#define MP_RULES 1024
struct PoolDivisor { // x / chunks = (x * magic >> 32) >> shift, x < 2^31 (magic 0: divided)
  unsigned magic;
  int shift;
};
template <int VEC, int PS>
__global__ void __launch_bounds__(256)
    k_maxpool(const float *__restrict__ in, float *__restrict__ out,
              const int *__restrict__ rules, long long bound, int ps,
              int C, int chunks, PoolDivisor div, int *__restrict__ choice,
              const float *__restrict__ spare, const long long *dRows, uint2 *__restrict__ out16) {
  __shared__ int sRules[PS ? MP_RULES : 1];
  if (PS)
    ps = PS;
  const long long nOutSites = live_rows(bound, dRows), all = nOutSites * chunks;
  const unsigned tiles = (unsigned)((all + 255) / 256);
  if (blockIdx.x >= tiles)
    return;
  const long long tile = xcd_eighth(blockIdx.x, tiles);
  const long long idx = tile * 256 + threadIdx.x;
  long long r, r0; // this lane's row, the workgroup's first
  if (div.magic) { // uniform
    r = __umulhi((unsigned)idx << 1, div.magic) >> div.shift;
    r0 = __umulhi((unsigned)(tile * 256) << 1, div.magic) >> div.shift;
  } else {
    r = idx / chunks;
    r0 = tile * 256 / chunks;
  }
  if (PS) {
    const long long last = tile * 256 + 255 < all ? tile * 256 + 255 : all - 1;
    const int n = ((int)((div.magic ? (long long)(__umulhi((unsigned)last << 1, div.magic) >> div.shift) : last / chunks) - r0) + 1) * PS;
    const int *const from = rules + r0 * PS;
    for (int i = threadIdx.x; i < n; i += 256)
      sRules[i] = from[i];
  }
  if (PS)
    __syncthreads();
  if (idx >= all)
    return;
  const int c0 = (int)(idx - r * chunks) * VEC;
  const int *const rr = PS ? sRules + (int)(r - r0) * PS : rules + r * ps;
  float best[VEC];
  int arg[VEC];
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    best[k] = 0.f;
    arg[k] = 0;
  }
  bool none = true;
  // Nine candidates at a time: their rules are requested together, then
  // their values (a skipped rule reads the context's spare row -- never `in`,
  // which may have no rows at all -- and is dropped below), so that a window
  // costs two trips to memory rather than two per candidate; they are
  // compared in rule order.
  constexpr int MP = PS && PS < 9 ? PS : 9;
  for (int p0 = 0; p0 < ps; p0 += MP) {
    int rule[MP];
#pragma unroll
    for (int u = 0; u < MP; ++u)
      rule[u] = rr[p0 + u < ps ? p0 + u : ps - 1];
    float v[MP][VEC];
#pragma unroll
    for (int u = 0; u < MP; ++u) {
      const float *src = rule[u] >= 0 ? in + (long long)rule[u] * C + c0
                                      : spare + (c0 & (SCN_ZERO_FLOATS - VEC));
      if (VEC == 4) {
        float4 t = *reinterpret_cast<const float4 *>(src);
        v[u][0] = t.x;
        v[u][1] = t.y;
        v[u][2] = t.z;
        v[u][3] = t.w;
      } else {
        v[u][0] = src[0];
      }
    }
#pragma unroll
    for (int u = 0; u < MP; ++u) {
      if (p0 + u >= ps || rule[u] < 0)
        continue;
      // 32-bit, as the reference's poolingChoices (the entry points refuse
      // inputs of 2^31 elements and more where they know the input's size)
      const int flat = (int)((unsigned)rule[u] * (unsigned)C + (unsigned)c0);
#pragma unroll
      for (int k = 0; k < VEC; ++k)
        if (none || best[k] < v[u][k]) {
          best[k] = v[u][k];
          arg[k] = flat + k;
        }
      none = false;
    }
  }
  long long o = r * C + c0;
  if (VEC == 4) {
    *reinterpret_cast<float4 *>(out + o) =
        make_float4(best[0], best[1], best[2], best[3]);
    *reinterpret_cast<int4 *>(choice + o) =
        make_int4(arg[0], arg[1], arg[2], arg[3]);
    if (out16) // uniform
      out16[o / 4] = make_uint2(pack_bf16x2(best[0], best[1]), pack_bf16x2(best[2], best[3]));
  } else {
    out[o] = best[0];
    choice[o] = arg[0];
  }
}

static int maxpool(scn_ctx *ctx, const float *d_in, float *d_out, const int32_t *d_rules, int64_t nOutSites, int ps,
                   int C, int32_t *d_choice, void *d_out16) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_maxpool: null context");
  SCN_REQUIRE(nOutSites >= 0 && ps >= 1 && C >= 1, SCN_ERR_ARG,
              "scn_maxpool: nOutSites %lld ps %d C %d", (long long)nOutSites,
              ps, C);
  if (nOutSites == 0)
    return SCN_OK;
  // (d_in may be null: an input without rows, every rule negative)
  SCN_REQUIRE(d_out && d_rules && d_choice, SCN_ERR_ARG,
              "scn_maxpool: null buffer");
  ProfScope prof(ctx, SCN_K_MAXPOOL);
  const long long *dRows = ctx->d_meta ? ctx->d_meta + META_SITES : nullptr;
  const bool wide = C % 4 == 0 && aligned16(d_in) && aligned16(d_out) && aligned16(d_choice);
  SCN_REQUIRE(!d_out16 || (wide && ((uintptr_t)d_out16 & 7) == 0), SCN_ERR_ARG,
              "scn_maxpool_rounded: %d features, or a buffer that does not start on 16 bytes", C);
  const int chunks = wide ? C / 4 : C;
  const long long total = nOutSites * chunks;
  PoolDivisor div = {0u, 0};
  if (total + 256 < (1ll << 31)) { // ceil(2^(31 + shift) / chunks), 2^shift >= chunks
    while ((1ll << div.shift) < chunks)
      ++div.shift;
    div.magic = (unsigned)(((1ull << (31 + div.shift)) + chunks - 1) / chunks);
  }
  // (rows that a workgroup's 256 lanes may touch)
  const bool fits = (256 / chunks + 2ll) * ps <= MP_RULES;
#define SCN_MP_GO(VEC, PS)                                                                                       \
  hipLaunchKernelGGL((k_maxpool<VEC, PS>), dim3(scn_ceil_div(total, 256)), dim3(256), 0, ctx->stream, d_in, d_out, \
                     d_rules, (long long)nOutSites, ps, C, chunks, div, d_choice, (const float *)ctx->d_zeros, dRows, (uint2 *)d_out16)
  if (!wide)
    SCN_MP_GO(1, 0);
  else if (fits && ps == 9)
    SCN_MP_GO(4, 9);
  else if (fits && ps == 8)
    SCN_MP_GO(4, 8);
  else if (fits && ps == 4)
    SCN_MP_GO(4, 4);
  else
    SCN_MP_GO(4, 0);
#undef SCN_MP_GO
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

extern "C" int scn_maxpool(scn_ctx *ctx, const float *d_in, float *d_out, const int32_t *d_rules, int64_t nOutSites,
                           int ps, int C, int32_t *d_choice) {
  return maxpool(ctx, d_in, d_out, d_rules, nOutSites, ps, C, d_choice, nullptr);
}

extern "C" int scn_maxpool_checked(scn_ctx *ctx, const float *d_in,
                                   int64_t nInRows, float *d_out,
                                   const int32_t *d_rules, int64_t nOutSites,
                                   int ps, int C, int32_t *d_choice) {
  return scn_maxpool_rounded(ctx, d_in, nInRows, d_out, nullptr, d_rules, nOutSites, ps, C, d_choice);
}
extern "C" int scn_maxpool_rounded(scn_ctx *ctx, const float *d_in, int64_t nInRows, float *d_out, void *d_out16,
                                   const int32_t *d_rules, int64_t nOutSites, int ps, int C, int32_t *d_choice) {
  SCN_REQUIRE(nInRows >= 0 && C >= 1, SCN_ERR_ARG,
              "scn_maxpool_checked: nInRows %lld C %d", (long long)nInRows, C);
  SCN_REQUIRE(nInRows * (int64_t)C <= 2147483647ll, SCN_ERR_CAPACITY,
              "scn_maxpool: %lld input rows of %d features are %lld elements; "
              "the 32-bit pooling choices index at most 2^31 - 1",
              (long long)nInRows, C, (long long)(nInRows * (int64_t)C));
  return maxpool(ctx, d_in, d_out, d_rules, nOutSites, ps, C, d_choice, d_out16);
}

// dTerminalPool (TerminalPoolingLayer.cu:22-34): sequential fp32 sum in rule
// order, then divide by the number of rows summed.
__global__ void k_terminal_pool(const float *__restrict__ in,
                                float *__restrict__ out,
                                const int *__restrict__ rules, long long count,
                                int S, int C, const float *__restrict__ spare,
                                const long long *meta) {
  if (meta) // (the width is a bound, the rows lie at the true one)
    S = meta[META_OVERFLOW] ? 0 : (int)(meta[META_WIDTH] < S ? meta[META_WIDTH] : S);
  long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= count * C)
    return;
  long long b = idx / C;
  int j = (int)(idx - b * C);
  const int *rr = rules + b * S;
  float t = 0.f;
  int p = 0;
  // four rows at a time: their rules requested together, then their values
  // (a rule past the sample's last reads the context's spare row, never `in`,
  // and ends the sum); added in rule order
  bool more = true;
  for (int p0 = 0; p0 < S && more; p0 += 4) {
    int rule[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      rule[u] = p0 + u < S ? rr[p0 + u] : -1;
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = rule[u] >= 0 ? in[(long long)rule[u] * C + j] : spare[j & (SCN_ZERO_FLOATS - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      more = more && rule[u] >= 0;
      if (more) {
        t += v[u];
        ++p;
      }
    }
  }
  out[idx] = t / (float)p;
}

extern "C" int scn_terminal_pool(scn_ctx *ctx, const float *d_in, float *d_out,
                                 const int32_t *d_rules, int64_t count, int S,
                                 int C) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_terminal_pool: null context");
  SCN_REQUIRE(count >= 0 && S >= 1 && C >= 1, SCN_ERR_ARG,
              "scn_terminal_pool: count %lld S %d C %d", (long long)count, S,
              C);
  if (count == 0)
    return SCN_OK;
  // (d_in may be null: an input without rows, every rule negative)
  SCN_REQUIRE(d_out && d_rules, SCN_ERR_ARG,
              "scn_terminal_pool: null buffer");
  ProfScope prof(ctx, SCN_K_TERMINAL);
  hipLaunchKernelGGL(k_terminal_pool, dim3(scn_ceil_div(count * C, 256)),
                     dim3(256), 0, ctx->stream, d_in, d_out, d_rules,
                     (long long)count, S, C, (const float *)ctx->d_zeros,
                     ctx->d_meta);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

// dSigmoidSoftmax (SigmoidLayer.cu:160-177): running maximum starts at -10000.
// One wavefront per row; lanes stride over the classes.
__global__ void __launch_bounds__(256)
    k_softmax(const float *in, float *out, long long M, int N) {
  const int lane = threadIdx.x & 63;
  long long row = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= M)
    return;
  const float *a = in + row * N;
  float *b = out + row * N;
  float mx = -10000.0f;
  for (int k = lane; k < N; k += 64)
    mx = fmaxf(mx, a[k]);
  for (int off = 32; off > 0; off >>= 1)
    mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  float acc = 0.f;
  for (int k = lane; k < N; k += 64) {
    float e = expf(a[k] - mx);
    b[k] = e;
    acc += e;
  }
  for (int off = 32; off > 0; off >>= 1)
    acc += __shfl_xor(acc, off, 64);
  for (int k = lane; k < N; k += 64)
    b[k] = b[k] / acc;
}

// dSigmoidTanh / dSigmoidLogistic (SigmoidLayer.cu:43-48, 80-85): in place,
// four elements per lane where the count allows
__global__ void __launch_bounds__(256)
    k_squash(float *x, long long n, int logistic) {
  const long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i + 4 <= n && ((uintptr_t)x & 15) == 0) {
    float4 v = *reinterpret_cast<float4 *>(x + i);
    if (logistic) {
      v.x = 1.0f / (1.0f + expf(-v.x)), v.y = 1.0f / (1.0f + expf(-v.y));
      v.z = 1.0f / (1.0f + expf(-v.z)), v.w = 1.0f / (1.0f + expf(-v.w));
    } else {
      v.x = tanhf(v.x), v.y = tanhf(v.y), v.z = tanhf(v.z), v.w = tanhf(v.w);
    }
    *reinterpret_cast<float4 *>(x + i) = v;
  } else {
    for (long long k = i; k < n && k < i + 4; ++k)
      x[k] = logistic ? 1.0f / (1.0f + expf(-x[k])) : tanhf(x[k]);
  }
}
int scn_squash_launch(scn_ctx *ctx, float *d_x, long long n, int logistic) {
  if (n <= 0)
    return SCN_OK;
  hipLaunchKernelGGL(k_squash, dim3((unsigned)scn_ceil_div(scn_ceil_div(n, 4), 256)),
                     dim3(256), 0, ctx->stream, d_x, n, logistic);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

int scn_softmax_launch(scn_ctx *ctx, const float *d_in, float *d_out,
                       long long M, int N) {
  hipLaunchKernelGGL(k_softmax, dim3(scn_ceil_div(M, 4)), dim3(256), 0,
                     ctx->stream, d_in, d_out, M, N);
  SCN_HIP_CHECK(hipGetLastError());
  return SCN_OK;
}

extern "C" int scn_softmax_rows(scn_ctx *ctx, const float *d_in, float *d_out,
                                int64_t M, int N) {
  SCN_REQUIRE(ctx, SCN_ERR_ARG, "scn_softmax_rows: null context");
  SCN_REQUIRE(M >= 0 && N >= 1, SCN_ERR_ARG, "scn_softmax_rows: M %lld N %d",
              (long long)M, N);
  if (M == 0)
    return SCN_OK;
  SCN_REQUIRE(d_in && d_out, SCN_ERR_ARG, "scn_softmax_rows: null buffer");
  ProfScope prof(ctx, SCN_K_SOFTMAX);
  return scn_softmax_launch(ctx, d_in, d_out, (long long)M, N);
}
