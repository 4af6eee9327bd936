// Internal declarations shared by the translation units of libscn_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <mutex>
#include <vector>
#include "scn_hip.h"

void scn_set_error(const char *fmt, ...);

#define SCN_HIP_CHECK(expr)                                                    \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess) {                                                    \
      scn_set_error("%s:%d: %s failed: %s", __FILE__, __LINE__, #expr,         \
                    hipGetErrorString(e_));                                    \
      return SCN_ERR_HIP;                                                      \
    }                                                                          \
  } while (0)

#define SCN_REQUIRE(cond, code, ...)                                           \
  do {                                                                         \
    if (!(cond)) {                                                             \
      scn_set_error(__VA_ARGS__);                                              \
      return (code);                                                           \
    }                                                                          \
  } while (0)

#define SCN_TRY(expr)                                                          \
  do {                                                                         \
    int rc_ = (expr);                                                          \
    if (rc_ != SCN_OK)                                                         \
      return rc_;                                                              \
  } while (0)

// words of a plan's counts on the device (scn_grids::meta)
enum { META_SITES = 0, META_ACTIVE = 1, META_OVERFLOW = 2, META_WIDTH = 3 };

struct ProfSpan {
  int family;
  int tag;
  hipEvent_t a, b;
};

#define SCN_ZERO_FLOATS 4096
#define SCN_IMAGE_BYTES (16u << 20)
#define SCN_MAX_PENDING 62 // plans per settle; 16 + 4 * 62 = 264 pinned words
#define SCN_PINNED_WORDS (16 + 4 * SCN_MAX_PENDING)
// images of weights to be made (weight_image, scn_image_dev.h)
struct ImageList {
  const float *W[SCN_IMAGES_MAX];
  unsigned char *image[SCN_IMAGES_MAX];
  unsigned firstBlock[SCN_IMAGES_MAX + 1];
  int K[SCN_IMAGES_MAX], N[SCN_IMAGES_MAX], fs[SCN_IMAGES_MAX], planes[SCN_IMAGES_MAX];
  int count;
};
struct scn_ctx {
  int device;
  hipStream_t stream;
  int numCU;
  // small pinned buffer for counts that must come back to the host
  int64_t *h_pinned; // SCN_PINNED_WORDS int64, host view
  int64_t *d_pinned; // the same memory as the device sees it
  int64_t *d_scalars; // 16 int64
  float *d_zeros;     // SCN_ZERO_FLOATS zeros: the row a negative rule stands for
  unsigned char *d_image; // SCN_IMAGE_BYTES or null: a layer's weights as its contraction reads them
  long long ticket;   // number of the last count readback (h_pinned[14] echoes it)
  // deferred counts (scn_ctx_defer_counts): plans whose counts are still on
  // their way; slot i of them reports into h_pinned[16 + 4 i ..]
  bool deferCounts;
  bool wstream; // NiN: W-streaming kernel allowed (SCN_NIN_WSTREAM=0 turns it off)
  std::vector<struct scn_grids *> pendingGrids;
  // scn_ctx_rows_from: where the feature kernels read their number of rows
  // (META_* words of the grids), the bound they were launched with, and the
  // pinned slot that holds the same once the stream is through
  const long long *d_meta;
  long long rowsBound, rowsHint; // (hint: what they are likely to be)
  int rowsSlot;
  // the kernels chosen meanwhile are those for above < rows <= upTo
  struct RowsChosen {
    int slot;
    long long above, upTo;
  };
  std::vector<RowsChosen> rowsChosen;
  bool rowsHeld;
  struct ChainState *chain; // recorded rule-book plans (scn_chain.hip)
  ImageList imagesLater; // scn_weight_images_later's, until a launch takes them along
  // profiling
  bool prof;
  int profTag;
  std::vector<ProfSpan> spans;
  std::vector<hipEvent_t> freeEvents;
  double profMs[SCN_K_COUNT];
  int64_t profCalls[SCN_K_COUNT];
};

// Records a start event on construction and a stop event on destruction when
// profiling is enabled.
struct ProfScope {
  scn_ctx *ctx;
  int idx;
  ProfScope(scn_ctx *ctx, int family);
  ~ProfScope();
};

// grow-only device buffer
template <typename T> struct DevBuf {
  T *p = nullptr;
  size_t cap = 0; // elements
  int reserve(size_t n) {
    if (n <= cap)
      return SCN_OK;
    size_t want = n + n / 4 + 64;
    T *q = nullptr;
    hipError_t e = hipMalloc((void **)&q, want * sizeof(T));
    if (e != hipSuccess) {
      scn_set_error("hipMalloc(%zu bytes) failed: %s", want * sizeof(T),
                    hipGetErrorString(e));
      return SCN_ERR_HIP;
    }
    if (p)
      (void)hipFree(p);
    p = q;
    cap = want;
    return SCN_OK;
  }
  void release() {
    if (p)
      (void)hipFree(p);
    p = nullptr;
    cap = 0;
  }
};

static inline int scn_ceil_div(int64_t a, int64_t b) {
  return (int)((a + b - 1) / b);
}

// address of the static scratch of scn_sgemm_ABt_static on `device` (scn_train.hip)
int scn_abt_static_setup(int device);
void scn_abt_static_forget(const scn_ctx *ctx);

// For a feature call that can not read its rows on the device: waits for the
// stream and replaces the bound M by the rows there are (per: rows of the call
// for each of the grids' rows).
int scn_rows_exact(scn_ctx *ctx, int64_t *M);
// The number of rows by which a call chooses its kernel ...
static inline long long scn_rows_hint(const scn_ctx *ctx, long long M) {
  return ctx->d_meta && ctx->rowsHint < M ? ctx->rowsHint : M;
}
// ... and the numbers for which another choice would have given other roundings:
// kept until the counts are settled.
static inline void scn_rows_chosen(scn_ctx *ctx, long long above, long long upTo) {
  if (ctx->d_meta)
    ctx->rowsChosen.push_back({ctx->rowsSlot, above, upTo});
}
// what a kernel does with the bound it was launched with
__device__ __forceinline__ long long live_rows(long long bound, const long long *d_rows) {
  if (!d_rows)
    return bound;
  const long long n = *d_rows;
  return n < bound ? n : bound;
}

// Workgroups are dealt to the 8 XCDs in turn, each with an L2 of its own: this
// gives XCD x the x-th eighth of n tiles, for a grid of at least n workgroups
// (those from n on have no tile).  Rows lie sample by sample in every layer, so
// an eighth of one layer's rows gathers from about the same eighth of the
// layer's below, and the column tiles of a row tile meet in one L2.  Microseconds
// with tiles dealt out in turn -> in eighths: dW of 28000 x 256 x 96 and its like
// 17.6 -> 14.5, of 139000 x 384 x 128 115.5 -> 106; contractions of bf16 rows
// through rules 50.2 -> 45.5, 53.8 -> 47.8; three planes 61.4 -> 57.4, 58.8 ->
// 57.3, 20.4 -> 19.9; max-pooling 6.2 -> 6.0; its gradient 76.6 -> 72.7.  Nothing
// for activation gradients (6.9 -> 7.2, rows in one range a workgroup) and for
// scatters through rules (14.8 -> 15.0), which stay as they were.
__device__ __forceinline__ unsigned xcd_eighth(unsigned b, unsigned n) {
  const unsigned x = b & 7, rem = n & 7;
  return x * (n >> 3) + (x < rem ? x : rem) + (b >> 3);
}

// Four words a store between the ends that are not on 16 bytes: the fills of the
// backward kernels of a middle layer (77 MB and less) 9.2 -> 7.0 us on average.
__device__ __forceinline__ void fill32(uint32_t *dst, uint32_t w, size_t n, size_t i, size_t step) {
  const size_t off = (16 - ((uintptr_t)dst & 15) & 15) / 4;
  const size_t head = off < n ? off : n, quads = (n - head) / 4, tail = head + 4 * quads;
  uint4 *const body = reinterpret_cast<uint4 *>(dst + head);
  for (size_t q = i; q < quads; q += step)
    body[q] = make_uint4(w, w, w, w);
  if (i < head)
    dst[i] = w;
  if (i < n - tail)
    dst[tail + i] = w;
}
// Several buffers in one launch (a launch of its own is 2 us and the gap before
// it): a workgroup finds its buffer from the running workgroup counts.
struct FillList {
  uint32_t *dst[SCN_FILL_MAX];
  size_t n[SCN_FILL_MAX];
  unsigned firstBlock[SCN_FILL_MAX + 1];
  int count;
};
__device__ __forceinline__ void fill32_list_block(const FillList &l, uint32_t w, unsigned block, unsigned tid) {
  int t = 0;
  while (t + 1 < l.count && block >= l.firstBlock[t + 1])
    ++t;
  const unsigned blocks = l.firstBlock[t + 1] - l.firstBlock[t];
  fill32(l.dst[t], w, l.n[t], (size_t)(block - l.firstBlock[t]) * 256 + tid, (size_t)blocks * 256);
}
int scn_fill_list(scn_ctx *c, void *const *d_dst, const size_t *nWords, int n, FillList *list, unsigned *blocksOf);

// What a backward pass begins with: buffers cleared, and Wt[(f N + n) nIn + c] = W[(f nIn
// + c) N + n], the weights of the convolutions that its inputs' gradients are, all
// layers', a tile of 32 x 32 to 256 lanes.
struct FilterList {
  const float *W[SCN_FILTERS_MAX];
  float *Wt[SCN_FILTERS_MAX];
  unsigned firstBlock[SCN_FILTERS_MAX + 1];
  int nIn[SCN_FILTERS_MAX], N[SCN_FILTERS_MAX];
  int count;
};
struct BeginList {
  FilterList filters;
  FillList fill;
  unsigned fillBlocks, blocks; // of 256 lanes; the fills' come first
};
// (called by 256 lanes for each block, and by all of a workgroup together: a block
// past the last one does nothing)
__device__ __forceinline__ void begin_list_block(const BeginList &b, unsigned block, unsigned tid, float (&tile)[32][33]) {
  const FilterList &l = b.filters;
  const bool filter = block >= b.fillBlocks && block < b.blocks;
  const int tx = tid & 31, ty = tid >> 5; // 32 x 8
  int nIn = 0, N = 0, n0 = 0, c0 = 0;
  float *Wt = nullptr;
  if (filter) {
    const unsigned at = block - b.fillBlocks;
    const int lane = tid & 63;
    const int t = __popcll(__ballot(lane < l.count && at >= l.firstBlock[lane < SCN_FILTERS_MAX ? lane : 0])) - 1;
    nIn = l.nIn[t], N = l.N[t];
    const int across = (N + 31) / 32, down = (nIn + 31) / 32;
    const unsigned x = at - l.firstBlock[t];
    const int f = (int)(x / (across * down));
    n0 = (int)(x % across) * 32, c0 = (int)(x / across % down) * 32;
    const float *const W = l.W[t] + (long long)f * nIn * N;
    Wt = l.Wt[t] + (long long)f * nIn * N;
    for (int i = ty; i < 32; i += 8)
      if (c0 + i < nIn && n0 + tx < N)
        tile[i][tx] = W[(long long)(c0 + i) * N + n0 + tx];
  } else if (block < b.fillBlocks) {
    fill32_list_block(b.fill, 0u, block, tid);
  }
  __syncthreads();
  if (filter)
    for (int i = ty; i < 32; i += 8)
      if (n0 + i < N && c0 + tx < nIn)
        Wt[(long long)(n0 + i) * nIn + c0 + tx] = tile[tx][i];
}
int scn_begin_list(scn_ctx *ctx, void *const *d_clear, const size_t *nWords, int nClear, const scn_filter_item *items,
                   int nItems, BeginList *list);

// Kernel attributes (the dynamic LDS limit) are set per device: fn runs once for
// every device a context of this process lives on, and again if it failed.
struct OncePerDevice {
  std::mutex m;
  unsigned long long done = 0;
  template <class F> int run(int device, F fn) {
    std::lock_guard<std::mutex> lock(m);
    if (device >= 0 && device < 64 && ((done >> device) & 1ull))
      return SCN_OK;
    const int rc = fn();
    if (rc == SCN_OK && device >= 0 && device < 64)
      done |= 1ull << device;
    return rc;
  }
};

// runs the recorded rule-book plans of the context, if any (scn_chain.hip)
int scn_chain_flush(scn_ctx *ctx);
void scn_chain_release(scn_ctx *ctx);

// exclusive prefix sum of n uint32 values; out has n + 1 elements (out[n] =
// total).  `tmp` must hold scn_scan_tmp_elems(n) uint32.
size_t scn_scan_tmp_elems(size_t n);
// What a scan of n elements wants zero in `tmp`.  The kernel that writes its
// input, with as many lanes at least, may clear it (`cleared`): a launch of its
// own takes 4 us.
struct ScanState {
  unsigned long long *state;
  size_t words;
  __device__ __forceinline__ void clear(size_t lane) const {
    if (lane < words)
      state[lane] = 0ull;
  }
};
ScanState scn_scan_state(size_t n, uint32_t *tmp);
int scn_scan_exclusive_u32(hipStream_t s, const uint32_t *in, uint32_t *out,
                           size_t n, uint32_t *tmp, bool cleared = false);
// same, over popcounts of 64-bit words
int scn_scan_exclusive_popc64(hipStream_t s, const uint64_t *words,
                              uint32_t *out, size_t n, uint32_t *tmp, bool cleared = false);
// two of these at once, their states cleared
int scn_scan_exclusive_popc64_pair(hipStream_t s, const uint64_t *wordsA, uint32_t *outA, size_t nA, uint32_t *tmpA,
                                   const uint64_t *wordsB, uint32_t *outB, size_t nB, uint32_t *tmpB);
