// Token selection over float32 logits rows for gfx950: arg-max, and temperature / top-k / top-p
// sampling with a counter-based random stream.
//
// Sampling order follows the reference (clockwork/engine/model_runner.py:147-164):
// logits / temperature -> top-k (ties at the k-th value survive) -> top-p (a token stays while
// the probability mass of the tokens strictly more likely than it is <= top_p) -> softmax -> draw.
// The draw is ours: u = Philox4x32-10(key = seed, counter = draw index) mapped to [0, 1), then
// the first index whose running sum of weights, taken in index order, exceeds u * total. A row's
// result depends on that row, its seed and its draw index only.
#include "common.h"
#include "sampling.h"

#include <mutex>


__device__ __forceinline__ uint32_t order_key(float x) {
  if (x != x) x = -INFINITY;
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// ---------------------------------------------------------------- arg-max, two stages
// The first index wins among equal maxima (torch.argmax semantics, model_runner.py:137).
__device__ __forceinline__ void argmax_merge(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
}

__global__ __launch_bounds__(256) void argmax_partial_kernel(const float* __restrict__ logits,
                                                             int64_t row_stride, int V, int chunks,
                                                             float* __restrict__ pv,
                                                             int* __restrict__ pi) {
  __shared__ float sv[4];
  __shared__ int si[4];
  const int row = blockIdx.y, chunk = blockIdx.x;
  const int per = (V + chunks - 1) / chunks;
  const int lo = chunk * per, hi = min(V, lo + per);
  const float* x = logits + (int64_t)row * row_stride;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = lo + threadIdx.x; i < hi; i += 256) {
    float v = x[i];
    if (v != v) v = -INFINITY;
    argmax_merge(bv, bi, v, i);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(bv, off, 64);
    const int oi = __shfl_xor(bi, off, 64);
    argmax_merge(bv, bi, ov, oi);
  }
  if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = bv; si[threadIdx.x >> 6] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) argmax_merge(bv, bi, sv[w], si[w]);
    pv[row * chunks + chunk] = bv;
    pi[row * chunks + chunk] = bi;
  }
}

__global__ void argmax_final_kernel(const float* __restrict__ pv, const int* __restrict__ pi,
                                    int chunks, int V, int* __restrict__ out) {
  const int row = blockIdx.x;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int c = threadIdx.x; c < chunks; c += 64) argmax_merge(bv, bi, pv[row * chunks + c], pi[row * chunks + c]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(bv, off, 64);
    const int oi = __shfl_xor(bi, off, 64);
    argmax_merge(bv, bi, ov, oi);
  }
  if (threadIdx.x == 0) out[row] = bi < V ? bi : 0;
}

#define ARGMAX_MAX_CHUNKS 64

// workspace: n * chunks floats followed by n * chunks ints; chunks = cw_argmax_chunks(V).
CW_EXPORT int cw_argmax_chunks(int V) {
  int c = (V + 4095) / 4096;
  return c < 1 ? 1 : (c > ARGMAX_MAX_CHUNKS ? ARGMAX_MAX_CHUNKS : c);
}

CW_EXPORT int cw_argmax(const float* logits, int64_t row_stride, int n, int V, int* out,
                        void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  if (n < 0 || V <= 0 || row_stride < V) return CW_ERR_ARG;
  if (n == 0) return CW_OK;
  if (n > 65535) return CW_ERR_SIZE;
  const int chunks = cw_argmax_chunks(V);
  if (workspace == nullptr || workspace_bytes < (int64_t)n * chunks * 8) return CW_ERR_ARG;
  float* pv = (float*)workspace;
  int* pi = (int*)(pv + (int64_t)n * chunks);
  hipLaunchKernelGGL(argmax_partial_kernel, dim3(chunks, n), dim3(256), 0, stream, logits, row_stride, V, chunks, pv, pi);
  hipLaunchKernelGGL(argmax_final_kernel, dim3(n), dim3(64), 0, stream, pv, pi, chunks, V, out);
  return cw_launch_status();
}

// ---------------------------------------------------------------- arg-max without a workspace
// For callers that cannot allocate (see sampling.h): the partial results live in this array, one
// copy on every GPU that loads the library. In host code its name is only a handle for
// hipGetSymbolAddress; the kernels get the address that call returned for the current GPU.
static __device__ __align__(256) unsigned char scratch[CW_ARGMAX_STATIC_BYTES];
static_assert(CW_ARGMAX_STATIC_BYTES == CW_ARGMAX_STATIC_MAX_ROWS * ARGMAX_MAX_CHUNKS * 8, "scratch holds a value and an index per row and chunk");

#define ARGMAX_STATIC_MAX_DEVICES 64
static void* scratch_of_device[ARGMAX_STATIC_MAX_DEVICES];
static std::mutex scratch_lock;

// The array's address on the current GPU, looked up at the first call on that GPU.
static int argmax_static_scratch(void** out) {
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess) return CW_ERR_LAUNCH;
  if (device < 0 || device >= ARGMAX_STATIC_MAX_DEVICES) return CW_ERR_SIZE;
  std::lock_guard<std::mutex> guard(scratch_lock);
  if (scratch_of_device[device] == nullptr) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) {
      (void)hipGetLastError();
      return CW_ERR_LAUNCH;
    }
    scratch_of_device[device] = ptr;
  }
  *out = scratch_of_device[device];
  return CW_OK;
}

CW_EXPORT int cw_argmax_static_init(void) {
  void* ptr = nullptr;
  return argmax_static_scratch(&ptr);
}

CW_EXPORT int cw_argmax_static(const float* logits, int64_t row_stride, int n, int V, int* out,
                               hipStream_t stream) {
  if (n < 0 || V <= 0 || row_stride < V || logits == nullptr || out == nullptr) return CW_ERR_ARG;
  if (n == 0) return CW_OK;
  if (n > CW_ARGMAX_STATIC_MAX_ROWS) return CW_ERR_SIZE;
  void* ptr = nullptr;
  const int status = argmax_static_scratch(&ptr);
  if (status != CW_OK) return status;
  const int chunks = cw_argmax_chunks(V);
  // values in the first half of the array, indices in the second, wherever n and chunks end
  float* pv = (float*)ptr;
  int* pi = (int*)((unsigned char*)ptr + CW_ARGMAX_STATIC_BYTES / 2);
  hipLaunchKernelGGL(argmax_partial_kernel, dim3(chunks, n), dim3(256), 0, stream, logits, row_stride, V, chunks, pv, pi);
  hipLaunchKernelGGL(argmax_final_kernel, dim3(n), dim3(64), 0, stream, pv, pi, chunks, V, out);
  return cw_launch_status();
}

// ---------------------------------------------------------------- Philox4x32-10
__device__ __forceinline__ uint32_t philox_first_word(uint64_t seed, uint64_t counter) {
  uint32_t c0 = (uint32_t)counter, c1 = (uint32_t)(counter >> 32), c2 = 0u, c3 = 0u;
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
  for (int round = 0; round < 10; ++round) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
    const uint32_t n1 = (uint32_t)p1;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
    const uint32_t n3 = (uint32_t)p0;
    c0 = n0; c1 = n1; c2 = n2; c3 = n3;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c0;
}

// ---------------------------------------------------------------- sampling
// A row is cut into chunks, and a pass over the logits is a kernel over (chunk, row): a row's work is spread over
// many compute units. What is then known about a whole row is worked out by a kernel of a workgroup a row. (The
// last of a row's workgroups to finish could do that without a launch, but what the others wrote has to be made
// visible to it: the fences that do so cost 170 us for 64 rows, the two launches 10.)
//
//   MAX      per chunk: the largest logit and its first index; and 64 logits of the row, one every V / 64;
//   HIST     per chunk, over 512 bins of logit / T: how many tokens fall into each (rows with top-k) and what they
//            weigh, the weights being exp(logit / T - mx) (rows with top-p), added to the row's bins; and what the chunk
//            weighs. Greedy rows end here;
//   COLLECT  per chunk: the bin that holds the k-th largest token, or the bin in which the weight from the top exceeds
//            top_p * total, from the row's bins, by every workgroup for itself; what the tokens above that bin weigh (all of
//            them stay), and a list of the tokens in it;
//   DRAW     per row: the k-th largest token of the list (radix selection over the order-preserving keys, 8 bits a
//            step; dividing by the temperature keeps the order, so the floor of what is kept is
//            (k-th largest) / temperature: ties at the k-th value survive, also ties that the division makes) and
//            the nucleus's last token (the largest key K with weight(keys >= K) > top_p * total: a token stays
//            while the tokens strictly more likely than it weigh <= top_p * total), then the draw. Rows without
//            either option come here from HIST. For a row with both options whose nucleus ends in a bin above the
//            k-th token's, COLLECT and DRAW run once more.
//
// A token's bin does not fall as its logit falls, and equal logits / T share a bin: what lies in bins of lower number
// is kept, what lies in bins of higher number is not.
// The bins: 3 segments of 170 equal bins, from the row's maximum to the 9th of its 64 sampled logits in descending
// order, from there to the 33rd, and from there on (sample_segments). However the row is spread, a segment holds about
// as many tokens as the samples say, so that a bin of a row of 151,936 tokens holds some hundreds and its list is short:
// rows of a spread of 0.02 to 60 (logits / T, normal) and rows that are mostly -inf take the same time. (Bins of one
// width for all rows, 1 / 16, held 4200 tokens at a spread of 0.8 and all but a few at 60. Top-p 0.9 in us, 8 rows,
// radix steps over whole rows / bins of one width / these: spread 3 57 / 47 / 47, spread 0.4 58 / 903 / 51; top-k 50 at a
// spread of 60 41 / 915 / 35.)
// A list does not fit where more than SAMPLE_LIST tokens share a bin all the same: thousands of equal logits, of which
// only their number matters (64 rows of one value: 245 / 625 / 95 us), or a cluster much narrower than the samples lie
// apart. DRAW then walks the row instead of the list, one workgroup a row (a third of the row within 3e-5, the nucleus's
// last token in it, 64 rows: 169 us by radix steps over whole rows, 563 so).
// The draw: u * total falls into a chunk, and in it on the first index whose running sum exceeds it.
// Weights are integers, exp(.) * 2^40 rounded down: their sums do not depend on the order of
// addition, so every comparison above gives the same answer however the row is cut and however
// the additions are scheduled (LDS atomics included), run after run.
// Bound by the passes over the logits, which come from the memory-side cache after the first, by the exponential, the quotient and
// the sums of every token and, in DRAW and for few rows, by a chain of trips, barriers and sums over a wave. 64 rows of 151,936
// logits, a quarter each greedy, temperature, top-k and top-p, us: 119 as twelve kernels (a radix step of 8 bits of the
// key each, over the whole rows), 63 as five, the row's bin by a kernel of its own from every chunk's bins, 50 as four with the
// chunks' bins added up by atomics (in a trace MAX 9.3, HIST 16.0, COLLECT 9.0, DRAW 12.2), 46 without the copy of the counts, 39 with
// quotients of five instructions, float64 sums and sums over a wave without shuffles (8.3, 14.2, 7.6, 10.3); 64 rows of
// temperature 33 -> 26, one row of top-p 30 -> 25.
// Tried: a token's first loads asked for before its row is known (no gain).
#define SAMPLE_THREADS 256
#define SAMPLE_WAVES (SAMPLE_THREADS / 64)
#define SAMPLE_MAX_CHUNKS 64
#define SAMPLE_BINS 512
#define SAMPLE_SEGMENT_BINS 170  // of each of three segments
#define SAMPLE_POINTS 64         // logits of a row that are sampled: a lane each
#define SAMPLE_LIST 4096         // tokens of a row's list
#define SAMPLE_BLOCK_LIST 1024   // tokens that one workgroup may add to it
#define SAMPLE_WEIGHT_SCALE 1099511627776.0f  // 2^40

typedef unsigned long long u64_t;

struct SampleRow {     // what is known about a row between two kernels
  u64_t limit;         // top_p * total (rows with top-p)
  uint32_t bin;        // the bin that COLLECT's second run collects
  uint32_t rank;       // rows with top-k: which of the bin's tokens, from the largest, is the k-th
  uint32_t collect;    // 2: COLLECT's second run has to run
  uint32_t listed[2];  // tokens that COLLECT's two runs found in the bin
  uint32_t unused;     // (a whole number of 8 bytes)
  float2 segments[3];  // see SampleBins
};

struct SampleArgs {
  const float* logits;
  int64_t row_stride;
  int n, V, chunks, per;  // per: a multiple of 4
  int vec;                // rows begin at 16-byte boundaries
  const float* temperature;
  const int* top_k;
  const float* top_p;
  const int64_t* seeds;
  const int64_t* draws;   // nullptr: they come with the launch (DrawCounts)
  int* out;
  // workspace
  u64_t* hist_w;      // [n][SAMPLE_BINS], zeroed by MAX as hist_n
  u64_t* sums;        // [n][chunks] weight of the chunk (of its bins above the collected one, after COLLECT)
  SampleRow* rows;    // [n], zeroed by MAX
  uint4* found;       // [n][chunks] smallest and largest key that COLLECT found in the bin, (~0, 0) for none, and how many
  uint32_t* hist_n;   // [n][SAMPLE_BINS]
  uint2* list;        // [n][SAMPLE_LIST] (key, index)
  float* pmax;        // [n][chunks]
  int* pmax_i;        // [n][chunks]
  float* points;      // [n][SAMPLE_POINTS]
};

// How many draws each of up to 64 rows has made, in the kernel's arguments: what changes from one step of a batch to the next is
// then no copy to the device (a launch of its own, and twice as long on the host as the kernels' four: 38 -> 21 us a call of few rows).
#define SAMPLE_COUNTED_ROWS 64
struct DrawCounts {
  uint32_t of_row[SAMPLE_COUNTED_ROWS];
};

// Chunks a row is cut into: at least 2048 tokens each; 64 for few rows, for many rows as few as still make two
// thousand workgroups (a row's bins take an addition from each).
// The most tokens of a chunk whose weights (2^40 at most) a thread may add up in float64: of 2^21 it takes 4 of every 1024, 2^13, and
// every sum of these is a whole number of at most 2^53, which float64 holds.
#define SAMPLE_FLOAT64_TOKENS (1 << 21)
static_assert(4ll * (SAMPLE_FLOAT64_TOKENS / (4 * SAMPLE_THREADS)) << 40 <= 1ll << 53, "a thread's sums are exact");
static int sample_chunks(int n, int V) {
  int c = (V + 2047) / 2048;
  const int most = n <= 32 ? SAMPLE_MAX_CHUNKS : n >= 512 ? 4 : 2048 / n;
  if (c > most) c = most;
  const int least = (int)(((int64_t)V + SAMPLE_FLOAT64_TOKENS - 1) / SAMPLE_FLOAT64_TOKENS);
  if (c < least) c = least < SAMPLE_MAX_CHUNKS ? least : SAMPLE_MAX_CHUNKS;
  return c < 1 ? 1 : c;
}

CW_EXPORT int64_t cw_sample_workspace_bytes(int n, int V) {
  const int64_t rc = (int64_t)n * sample_chunks(n, V);
  return rc * 32 + (int64_t)n * ((int64_t)sizeof(SampleRow) + SAMPLE_BINS * 12 + SAMPLE_LIST * 8 + SAMPLE_POINTS * 4) + 64;
}

__device__ __forceinline__ float key_to_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
__device__ __forceinline__ bool row_has_top_k(const SampleArgs& a, int row) {
  const int k = a.top_k[row];
  return k > 0 && k < a.V;
}
__device__ __forceinline__ bool row_has_top_p(const SampleArgs& a, int row) { return a.top_p[row] < 1.0f; }
__device__ __forceinline__ u64_t weight_of(float v, float mx) {
  const float e = expf(v - mx);  // NaN for inf - inf: no weight
  return e == e ? (u64_t)(e * SAMPLE_WEIGHT_SCALE) : 0;
}
// A row's temperature and what divides by it. ``of(a)`` is a / T, rounded once: a product with the reciprocal, then twice the remainder
// times the reciprocal, each remainder exact by a fused multiply-add; the first step leaves a quotient that is off by less than one
// unit of its last place, and of such a one the second makes the correctly rounded quotient (Markstein). Five instructions for the
// division's eleven, one of them at a quarter of the rate. The same bits as the division's where 1 / T is a normal number (T from 3e-39 to 8.5e37) and
// the remainders are exact (a from 2^-100 in size, or 0; -0 / T comes out as 0): of smaller a, and larger T, a quotient may be off by a unit of its last
// place, next to 0, where every weight is the same. Infinite quotients come out as NaN, which everything here takes for -inf (a row whose
// largest logit is +inf, or a T below 3e-39, leaves no weight at all, and its first maximum is taken, as with the division).
struct Quotient {
  float t, y;
  __device__ __forceinline__ explicit Quotient(float temp) : t(temp), y(1.0f / temp) {}
  __device__ __forceinline__ float of(float a) const {
    float q = a * y;
    q = fmaf(fmaf(-t, q, a), y, q);
    return fmaf(fmaf(-t, q, a), y, q);
  }
};
// The three segments of a row's bins: x is the largest logit / T of one, y how many bins go into a unit below that (0
// where the segment has no width: it is one bin then).
struct SampleBins {
  float2 s0, s1, s2;
};
__device__ __forceinline__ SampleBins sample_bins(const float2* p) { return SampleBins{p[0], p[1], p[2]}; }
// The bin of v = logit / T (-inf and NaN go last): the last segment whose top it lies below, or the first, and there
// the distance from the top in bins.
__device__ __forceinline__ uint32_t bin_of(const SampleBins& bins, float v) {
  const float2 s0 = bins.s0, s1 = bins.s1, s2 = bins.s2;
  const bool b1 = v < s1.x, b2 = v < s2.x;
  const float x = b2 ? s2.x : b1 ? s1.x : s0.x, y = b2 ? s2.y : b1 ? s1.y : s0.y;
  const float d = __builtin_amdgcn_fmed3f((x - v) * y, 0.0f, (float)(SAMPLE_SEGMENT_BINS - 1));  // (NaN for inf - inf: 0)
  const uint32_t first = b2 ? 2u * SAMPLE_SEGMENT_BINS : b1 ? (uint32_t)SAMPLE_SEGMENT_BINS : 0u;
  return v > -INFINITY ? first + (uint32_t)d : SAMPLE_BINS - 1;
}
__device__ __forceinline__ float bins_per_unit(float width) {
  const float y = (float)SAMPLE_SEGMENT_BINS / width;
  return y > 0.0f && y < INFINITY ? y : 0.0f;
}
// The segments of a row, by one wave: ``point`` is the lane's sample. The second and the third begin at the
// 9th and the 33rd sample in descending order, and the bins of a segment go down to where the next one begins; the third's
// twice as far down as the 62nd sample. Where the samples further down are masks (-inf, or as low as the type goes) a
// segment's bins go twice as far down as the last sample that is not. ``out`` (LDS): the second and the third segment, and
// ahead of them what the first one's bins go down to, and how many times as far.
__device__ __forceinline__ void sample_segments(float point, float temp, float2* out) {
  const int lane = threadIdx.x & 63;
  // the order of the samples; those that are all but equal by their lanes
  const uint32_t key = (order_key(point) & ~63u) | (uint32_t)lane;
  int rank = 0;
#pragma unroll
  for (int l = 0; l < SAMPLE_POINTS; ++l) rank += (uint32_t)__builtin_amdgcn_readlane((int)key, l) > key ? 1 : 0;
  const int last = SAMPLE_POINTS - 1 - __popcll(__ballot(!(point > -1e30f)));  // -1: all are masks
  // lanes 0 to 4 take a sample each: the tops of segments 1 and 2, and the ends of 0, 1 and 2
  const int ranks[5] = {8, 32, min(8, last), min(32, last), min(61, last)};
  int from = 0;
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int l = __ffsll((unsigned long long)__ballot(rank == max(ranks[i], 0))) - 1;
    from = lane == i ? l : from;
  }
  const float v = __shfl(point, from, 64) / temp;
  const float mine = v == v ? v : -INFINITY;
  const float top1 = __shfl(mine, 0, 64), top2 = __shfl(mine, 1, 64), end0 = __shfl(mine, 2, 64), end1 = __shfl(mine, 3, 64), end2 = __shfl(mine, 4, 64);
  if (lane == 0) {
    out[0] = make_float2(last < 0 ? -INFINITY : end0, last < 8 ? 2.0f : 1.0f);
    out[1] = make_float2(top1, bins_per_unit((last < 32 ? 2.0f : 1.0f) * (top1 - end1)));
    out[2] = make_float2(top2, bins_per_unit(2.0f * (top2 - end2)));
  }
}
__device__ __forceinline__ u64_t topp_limit(float p, u64_t total) { return (u64_t)((double)p * (double)total); }

// The row and the chunk of a workgroup of a pass: rows next to each other go to different XCDs and compute units, and a unit's
// workgroups are of rows that lie an odd number apart, so that rows that need more work (their options may repeat every few
// rows) are dealt evenly. (A quarter each greedy, temperature, top-k and top-p, in turn: with row = blockIdx.y a unit had rows of
// one kind, and HIST took 20.7 us, as long as for 64 rows of top-p.)
__device__ __forceinline__ void row_and_chunk(const SampleArgs& a, int& row, int& chunk) {
  const int id = blockIdx.y * gridDim.x + blockIdx.x;
  chunk = id / a.n;
  row = (id - chunk * a.n + chunk + chunk / 4) % a.n;
}

// Four neighbouring logits from token i on (i a multiple of 4); NaN from ``hi`` on.
__device__ __forceinline__ void sample_load4(const float* x, int i, int hi, int vec, float (&o)[4]) {
  if (vec && i + 4 <= hi) {
    const float4 v = *reinterpret_cast<const float4*>(x + i);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = i + e < hi ? x[i + e] : NAN;
  }
}
// f(index, logit) for the tokens of [lo, hi) (lo a multiple of 4), by THREADS neighbouring threads (all of the workgroup, or
// a wave), 4 U loads in flight a thread. Up to three tokens past hi come as NaN, which everything here takes for -inf: a
// test for each token by itself would cost as much as what most tokens need.
template <int U, int THREADS = SAMPLE_THREADS>
__device__ __forceinline__ void sample_batch(const float* x, int i0, int hi, int vec, float (&t)[U][4]) {
#pragma unroll
  for (int u = 0; u < U; ++u) sample_load4(x, min(i0 + u * 4 * THREADS, (int)((unsigned)(hi - 1) & ~3u)), hi, vec, t[u]);
}
template <int U, int THREADS = SAMPLE_THREADS, typename F>
__device__ __forceinline__ void sample_take(const float (&t)[U][4], int i0, int hi, F f) {
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (i0 + u * 4 * THREADS < hi)
#pragma unroll
      for (int e = 0; e < 4; ++e) f(i0 + u * 4 * THREADS + e, t[u][e]);
}
template <int U = 2, int THREADS = SAMPLE_THREADS, typename F>
__device__ __forceinline__ void sample_walk(const float* x, int lo, int hi, int vec, F f) {
  for (int i0 = lo + (int)(threadIdx.x & (THREADS - 1)) * 4; i0 < hi; i0 += U * 4 * THREADS) {
    float t[U][4];
    sample_batch<U, THREADS>(x, i0, hi, vec, t);
    sample_take<U, THREADS>(t, i0, hi, f);
  }
}

// Sums over a wave, every lane ending with the total, and running sums (of a lane and those before it), by data-parallel operands:
// a shuffle through the LDS unit takes ten times as long, and a sum has six of them one after the other.
template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ uint32_t sample_dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, true);
}
template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ u64_t sample_dpp(u64_t v) {
  return ((u64_t)sample_dpp<CTRL, ROWS>((uint32_t)(v >> 32)) << 32) | sample_dpp<CTRL, ROWS>((uint32_t)v);
}
template <typename T> __device__ __forceinline__ T wave_running_sum(T v) {
  v += sample_dpp<0x111>(v);       // the lane before, of the same row of 16
  v += sample_dpp<0x112>(v);       // two before
  v += sample_dpp<0x114>(v);
  v += sample_dpp<0x118>(v);
  v += sample_dpp<0x142, 0xa>(v);  // the last lane of rows 0 and 2 to rows 1 and 3
  v += sample_dpp<0x143, 0xc>(v);  // lane 31 to rows 2 and 3
  return v;
}
__device__ __forceinline__ uint32_t last_lane(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 63); }
__device__ __forceinline__ u64_t last_lane(u64_t v) { return ((u64_t)last_lane((uint32_t)(v >> 32)) << 32) | last_lane((uint32_t)v); }
__device__ __forceinline__ u64_t wave_sum(u64_t v) { return last_lane(wave_running_sum(v)); }
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x111, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x112, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x114, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x118, 0xf, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x142, 0xa, 0xf, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x143, 0xc, 0xf, false));
  return last_lane(v);
}

// Sum over the workgroup; every thread gets it.
__device__ __forceinline__ u64_t block_sum(u64_t v) {
  __shared__ u64_t part[SAMPLE_WAVES];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  u64_t t = 0;
#pragma unroll
  for (int w = 0; w < SAMPLE_WAVES; ++w) t += part[w];
  __syncthreads();
  return t;
}
// Sum of the values of this thread and of those before it.
template <typename T>
__device__ __forceinline__ T block_running_sum(T v) {
  __shared__ T part[SAMPLE_WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_running_sum(v);
  if (lane == 63) part[wave] = v;
  __syncthreads();
  for (int w = 0; w < wave; ++w) v += part[w];
  __syncthreads();
  return v;
}

// The largest value of a wave and the least index that goes with it.
__device__ __forceinline__ void wave_argmax(float& v, int& i) {
  const float best = cw_wave_max(v);
  i = (int)wave_min(v == best ? (uint32_t)i : 0x7fffffffu);
  v = best;
}

// The row's largest logit (NaN counts as -inf) and its first index, from the chunk maxima: the
// first wave takes a chunk a lane (there are at most 64), every thread gets the result.
__device__ __forceinline__ void row_max(const SampleArgs& a, int row, float& bv, int& bi) {
  __shared__ float best_v;
  __shared__ int best_i;
  if (threadIdx.x < 64) {
    float v = -INFINITY;
    int i = 0x7fffffff;
    if ((int)threadIdx.x < a.chunks) {
      v = a.pmax[row * a.chunks + threadIdx.x];
      i = a.pmax_i[row * a.chunks + threadIdx.x];
    }
    wave_argmax(v, i);
    if (threadIdx.x == 0) { best_v = v; best_i = i; }
  }
  __syncthreads();
  bv = best_v;
  bi = best_i;
  __syncthreads();
}

// MAX
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_max_kernel(SampleArgs a) {
  __shared__ float sv[SAMPLE_WAVES];
  __shared__ int si[SAMPLE_WAVES];
  int row, chunk;
  row_and_chunk(a, row, chunk);
  if (chunk == 0 && threadIdx.x < sizeof(SampleRow) / 4) reinterpret_cast<uint32_t*>(a.rows + row)[threadIdx.x] = 0u;
  for (int b = chunk * SAMPLE_THREADS + (int)threadIdx.x; b < SAMPLE_BINS; b += a.chunks * SAMPLE_THREADS) {
    a.hist_w[(int64_t)row * SAMPLE_BINS + b] = 0;
    a.hist_n[(int64_t)row * SAMPLE_BINS + b] = 0u;
  }
  const int lo = chunk * a.per, hi = min(a.V, lo + a.per);
  const float* x = a.logits + (int64_t)row * a.row_stride;
  if (threadIdx.x < SAMPLE_POINTS) {
    const int at = (int)((2 * (int64_t)threadIdx.x + 1) * a.V / (2 * SAMPLE_POINTS));
    if (at >= lo && at < hi) a.points[(int64_t)row * SAMPLE_POINTS + threadIdx.x] = x[at];
  }
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  sample_walk(x, lo, hi, a.vec, [&](int i, float v) __attribute__((always_inline)) {
    if (v != v) v = -INFINITY;
    argmax_merge(bv, bi, v, i);
  });
  wave_argmax(bv, bi);
  if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = bv; si[threadIdx.x >> 6] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < SAMPLE_WAVES; ++w) argmax_merge(bv, bi, sv[w], si[w]);
    a.pmax[row * a.chunks + chunk] = bv;
    a.pmax_i[row * a.chunks + chunk] = bi;
  }
}

// Draws the row's token among those whose scaled key is floor_key or more; ``chunk_w`` (LDS): what each chunk's
// such tokens weigh. All threads of one workgroup.
__device__ __forceinline__ void sample_locate(const SampleArgs& a, int row, float temp, float mx, int mi, uint32_t floor_key,
                                              const u64_t* chunk_w, const DrawCounts& counts) {
  __shared__ int sel_chunk, sel_run, found;
  __shared__ u64_t sel_base, sel_total;
  if (threadIdx.x == 0) sel_chunk = sel_run = 0, found = -1, sel_base = 0;
  __syncthreads();
  const uint32_t r = philox_first_word((uint64_t)a.seeds[row], a.draws ? (uint64_t)a.draws[row] : (uint64_t)counts.of_row[row]);
  if (threadIdx.x < 64) {  // the chunk the target falls into: a running sum over the chunks
    const u64_t v = (int)threadIdx.x < a.chunks ? chunk_w[threadIdx.x] : 0;
    const u64_t incl = wave_running_sum(v);
    const u64_t total = last_lane(incl);
    // u = (r >> 8) / 2^24; the drawn token is the first whose running weight exceeds u * total
    u64_t target = (u64_t)((double)(r >> 8) * (1.0 / 16777216.0) * (double)total);
    if (total > 0 && target >= total) target = total - 1;  // (total >= 2^40: the largest logit weighs that much)
    if (v > 0 && incl - v <= target && target < incl) {
      sel_chunk = threadIdx.x;
      sel_base = target - (incl - v);  // the target inside the chunk
    }
    if (threadIdx.x == 0) sel_total = total;
  }
  __syncthreads();
  if (sel_total == 0) {  // no token has any weight (every logit -inf or NaN): the first maximum, as greedy
    if (threadIdx.x == 0) a.out[row] = mi < a.V ? mi : 0;
    return;
  }
  const float* x = a.logits + (int64_t)row * a.row_stride;
  const Quotient over_t(temp);
  auto weight = [&](float raw) __attribute__((always_inline)) -> u64_t {
    const float v = over_t.of(raw);
    return v == v && order_key(v) >= floor_key ? weight_of(v, mx) : 0;
  };
  // in the chunk: thread t weighs a run of consecutive tokens; then a lane of the first wave takes a token of
  // the run that the target falls into
  const int lo = sel_chunk * a.per, hi = min(a.V, lo + a.per);
  const u64_t target = sel_base;
  const int run = ((hi - lo + SAMPLE_THREADS - 1) / SAMPLE_THREADS + 3) / 4 * 4;
  const int my_lo = min(hi, lo + (int)threadIdx.x * run), my_hi = min(hi, my_lo + run);
  u64_t w = 0;
  for (int i = my_lo; i < my_hi; i += 20) {  // (all of a thread's loads of 64 rows' chunks in flight at once)
    float t[5][4];
    sample_batch<5, 1>(x, i, my_hi, a.vec, t);
    sample_take<5, 1>(t, i, my_hi, [&](int, float raw) __attribute__((always_inline)) { w += weight(raw); });
  }
  const u64_t incl = block_running_sum(w);
  if (w > 0 && incl - w <= target && target < incl) {
    sel_run = threadIdx.x;
    sel_base = incl - w;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    u64_t before = sel_base;
    const int run_lo = min(hi, lo + sel_run * run), run_hi = min(hi, run_lo + run);
    for (int i0 = run_lo; i0 < run_hi; i0 += 64) {
      const int i = i0 + (int)threadIdx.x;
      const u64_t q = i < run_hi ? weight(x[i]) : 0;
      const u64_t upto = before + wave_running_sum(q);
      if (q > 0 && upto - q <= target && target < upto) found = i;
      before = last_lane(upto);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) a.out[row] = found >= 0 ? found : (mi < a.V ? mi : 0);
}

// HIST
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_hist_kernel(SampleArgs a) {
  __shared__ u64_t bins_w[SAMPLE_BINS];
  __shared__ uint32_t bins_n[SAMPLE_BINS];
  __shared__ float2 segments[3];
  int row, chunk;
  row_and_chunk(a, row, chunk);
  const float temp = a.temperature[row];
  const int lo = chunk * a.per, hi = min(a.V, lo + a.per);
  const float* x = a.logits + (int64_t)row * a.row_stride;
  const bool with_k = row_has_top_k(a, row), with_p = row_has_top_p(a, row);
  // the second wave works the segments out while the first looks for the maximum
  const float point = a.points[(int64_t)row * SAMPLE_POINTS + (threadIdx.x & 63)];
  if (temp > 0.0f && (with_k || with_p) && threadIdx.x >> 6 == 1) sample_segments(point, temp, segments);
  float mraw;
  int mi;
  row_max(a, row, mraw, mi);
  if (!(temp > 0.0f)) {  // greedy row inside a sampled batch
    if (chunk == 0 && threadIdx.x == 0) a.out[row] = mi < a.V ? mi : 0;
    return;
  }
  const float mx = mraw / temp;
  SampleBins bins = {};
  if (with_k || with_p) {
    bins = sample_bins(segments);  // (behind row_max's barriers)
    // (without a sample that is no mask: bins of 1 / 16)
    bins.s0 = make_float2(mx, bins.s0.x == -INFINITY ? 16.0f : bins_per_unit(bins.s0.y * (mx - bins.s0.x)));
    for (int b = threadIdx.x; b < SAMPLE_BINS; b += SAMPLE_THREADS) {
      bins_w[b] = 0;
      bins_n[b] = 0u;
    }
    __syncthreads();
    if (chunk == 0 && threadIdx.x == 0) {
      SampleRow& known = a.rows[row];
      known.segments[0] = bins.s0;
      known.segments[1] = bins.s1;
      known.segments[2] = bins.s2;
    }
  }
  const Quotient over_t(temp);
  if (!with_k && !with_p) {
    // a thread's sum of whole numbers as float64, exact: one conversion a token instead of a 64-bit integer's six instructions. (Of
    // more than 64 chunks' tokens, 2^27 logits, a chunk has more than such a sum may: those are added up as integers.)
    u64_t mine = 0;
    if (a.per <= SAMPLE_FLOAT64_TOKENS) {
      double sum = 0.0;
      sample_walk(x, lo, hi, a.vec, [&](int, float raw) __attribute__((always_inline)) {
        const float e = expf(over_t.of(raw) - mx);  // NaN: no weight
        sum += e == e ? (double)truncf(e * SAMPLE_WEIGHT_SCALE) : 0.0;
      });
      mine = (u64_t)sum;
    } else {
      sample_walk(x, lo, hi, a.vec, [&](int, float raw) __attribute__((always_inline)) { mine += weight_of(over_t.of(raw), mx); });
    }
    const u64_t total = block_sum(mine);
    if (threadIdx.x == 0) a.sums[(int64_t)row * a.chunks + chunk] = total;
    return;
  }
  // (COLLECT weighs what it leaves above the bin)
  if (!with_p) {
    sample_walk(x, lo, hi, a.vec, [&](int, float raw) __attribute__((always_inline)) { atomicAdd(&bins_n[bin_of(bins, over_t.of(raw))], 1u); });
  } else {
    sample_walk(x, lo, hi, a.vec, [&](int, float raw) __attribute__((always_inline)) {
      const float v = over_t.of(raw);
      const uint32_t bin = bin_of(bins, v);
      if (with_k) atomicAdd(&bins_n[bin], 1u);
      const u64_t w = v == v ? weight_of(v, mx) : 0;
      if (w) atomicAdd(&bins_w[bin], w);
    });
  }
  __syncthreads();
  // the row's bins: integers, so the order in which its chunks come does not matter
  for (int b = threadIdx.x; b < SAMPLE_BINS; b += SAMPLE_THREADS) {
    if (with_k && bins_n[b]) atomicAdd(a.hist_n + (int64_t)row * SAMPLE_BINS + b, bins_n[b]);
    if (with_p && bins_w[b]) atomicAdd(a.hist_w + (int64_t)row * SAMPLE_BINS + b, bins_w[b]);
  }
}

// The weights of bins 2 t and 2 t + 1 of the whole row, for thread t.
__device__ __forceinline__ void row_bins(const SampleArgs& a, int row, u64_t& w0, u64_t& w1) {
  const ulonglong2 h = *reinterpret_cast<const ulonglong2*>(a.hist_w + (int64_t)row * SAMPLE_BINS + 2 * threadIdx.x);
  w0 = h.x;
  w1 = h.y;
}

// The bin to collect and, with top-k, which of its tokens is the k-th, with top-p what the tokens more likely than the nucleus's
// last weigh at most: by every workgroup of a row for itself.
__device__ __forceinline__ void sample_pick(const SampleArgs& a, int row, bool with_k, uint32_t& bin, uint32_t& rank, u64_t& limit) {
  __shared__ uint32_t picked_bin, picked_rank;
  __shared__ u64_t all;
  // thread t: bins 2 t and 2 t + 1 of the whole row
  if (threadIdx.x == 0) picked_bin = 0u, picked_rank = 1u;
  limit = 0;
  if (with_k) {
    const uint2 h = *reinterpret_cast<const uint2*>(a.hist_n + (int64_t)row * SAMPLE_BINS + 2 * threadIdx.x);
    const uint32_t upto = block_running_sum(h.x + h.y), k = (uint32_t)a.top_k[row];
    const uint32_t before = upto - h.x - h.y;
    if (before < k && k <= upto) {
      picked_bin = 2 * threadIdx.x + (before + h.x < k ? 1 : 0);
      picked_rank = k - (before + h.x < k ? before + h.x : before);
    }
  } else {
    u64_t w0, w1;
    row_bins(a, row, w0, w1);
    const u64_t upto = block_running_sum(w0 + w1);
    if (threadIdx.x == SAMPLE_THREADS - 1) all = upto;
    __syncthreads();
    limit = topp_limit(a.top_p[row], all);
    const u64_t before = upto - w0 - w1;
    if (before <= limit && limit < upto) picked_bin = 2 * threadIdx.x + (before + w0 <= limit ? 1 : 0);
  }
  __syncthreads();
  bin = picked_bin;
  rank = picked_rank;
}

// COLLECT; ``again``: its second run
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_collect_kernel(SampleArgs a, int again) {
  __shared__ uint2 mine[SAMPLE_BLOCK_LIST];
  __shared__ uint32_t n_mine, at_list, ends[2];
  int row, chunk;
  row_and_chunk(a, row, chunk);
  SampleRow& known = a.rows[row];
  const float temp = a.temperature[row];
  if (!(temp > 0.0f)) return;
  uint32_t bin = 0u;
  const bool with_k = row_has_top_k(a, row);
  if (again ? known.collect != 2u : !with_k && !row_has_top_p(a, row)) return;
  const int lo = chunk * a.per, hi = min(a.V, lo + a.per);
  const float* x = a.logits + (int64_t)row * a.row_stride;
  if (again) {
    bin = known.bin;
  } else {
    uint32_t rank;
    u64_t limit;
    sample_pick(a, row, with_k, bin, rank, limit);
    if (chunk == 0 && threadIdx.x == 0) {
      known.rank = rank;
      known.limit = limit;
    }
  }
  if (threadIdx.x == 0) n_mine = ends[1] = 0u, ends[0] = 0xffffffffu;
  const SampleBins bins = sample_bins(known.segments);
  float mraw;
  int mi;
  row_max(a, row, mraw, mi);  // (and barriers behind the above)
  const float mx = mraw / temp;
  u64_t sum = 0;
  uint32_t least = 0xffffffffu, most = 0u;  // of the bin's keys
  // most tokens lie below the bin, and a comparison says so (the threshold is a little lower than the bin's end,
  // by more than the divisions and products round; NaN, which compares with nothing, goes the long way)
  const float2 s0 = bins.s0, s1 = bins.s1, s2 = bins.s2;
  const uint32_t segment = min(bin / SAMPLE_SEGMENT_BINS, 2u), j = bin - segment * SAMPLE_SEGMENT_BINS;
  const float seg_top = segment == 0 ? s0.x : segment == 1 ? s1.x : s2.x, seg_y = segment == 0 ? s0.y : segment == 1 ? s1.y : s2.y;
  float end = segment == 0 ? s1.x : segment == 1 ? s2.x : -INFINITY;
  if (j < SAMPLE_SEGMENT_BINS - 1 && seg_y > 0.0f) end = fmaxf(end, seg_top - (float)(j + 1) / seg_y);
  const float surely_below = (end - 1e-5f * (fabsf(end) + fabsf(seg_top)) - 1e-30f) * temp;
  const Quotient over_t(temp);
  auto look = [&](int i, float raw) __attribute__((always_inline)) {
    if (raw < surely_below) return;
    const float v = over_t.of(raw);
    const uint32_t b = bin_of(bins, v);
    if (b < bin) {
      sum += weight_of(v, mx);
    } else if (b == bin) {
      const uint32_t key = order_key(raw), at = atomicAdd(&n_mine, 1u);
      most = max(most, key);
      least = min(least, key);
      if (at < SAMPLE_BLOCK_LIST) mine[at] = make_uint2(key, (uint32_t)i);
    }
  };
  sample_walk(x, lo, hi, a.vec, look);
  if (__ballot(most >= least)) {
    least = wave_min(least);
    most = ~wave_min(~most);
    if ((threadIdx.x & 63) == 0) {
      atomicMin(&ends[0], least);
      atomicMax(&ends[1], most);
    }
  }
  sum = block_sum(sum);  // (and a barrier behind the list)
  // a workgroup whose tokens do not fit its own list makes the row's look too long for everybody
  const uint32_t n_here = n_mine;
  if (threadIdx.x == 0) {
    a.sums[(int64_t)row * a.chunks + chunk] = sum;
    a.found[(int64_t)row * a.chunks + chunk] = make_uint4(ends[0], ends[1], n_here, 0u);
    if (n_here) at_list = atomicAdd(&known.listed[again], n_here <= SAMPLE_BLOCK_LIST ? n_here : SAMPLE_LIST + 1u);
  }
  __syncthreads();
  if (n_here <= SAMPLE_BLOCK_LIST)
    for (uint32_t i = threadIdx.x; i < n_here; i += SAMPLE_THREADS)
      if (at_list + i < SAMPLE_LIST) a.list[(int64_t)row * SAMPLE_LIST + at_list + i] = mine[i];
}

// DRAW; ``again``: behind COLLECT's second run
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_draw_kernel(SampleArgs a, int again, DrawCounts counts) {
  __shared__ u64_t chunk_w[SAMPLE_MAX_CHUNKS];
  __shared__ u64_t bins_w[256];
  __shared__ uint32_t bins_n[256];
  __shared__ uint2 list[SAMPLE_LIST];
  __shared__ u64_t picked_above;
  __shared__ uint32_t picked, picked_rank, ends[2], chunk_n[SAMPLE_MAX_CHUNKS];
  const int row = blockIdx.x;
  SampleRow& known = a.rows[row];
  const float temp = a.temperature[row];
  if (!(temp > 0.0f) || (again && known.collect != 2u)) return;
  const bool with_k = row_has_top_k(a, row), with_p = row_has_top_p(a, row);
  // (a token of the list a thread before the list's length is known: what lies past it is not looked at)
  const uint2 first_listed = a.list[(int64_t)row * SAMPLE_LIST + threadIdx.x];
  float mraw;
  int mi;
  row_max(a, row, mraw, mi);
  const float mx = mraw / temp;
  if ((int)threadIdx.x < a.chunks) chunk_w[threadIdx.x] = a.sums[(int64_t)row * a.chunks + threadIdx.x];
  __syncthreads();
  if (!with_k && !with_p) {
    sample_locate(a, row, temp, mx, mi, 0u, chunk_w, counts);
    return;
  }
  const uint32_t listed = known.listed[again];
  const float* x = a.logits + (int64_t)row * a.row_stride;
  const bool fits = listed <= SAMPLE_LIST;
  if (fits)
    for (uint32_t i = threadIdx.x; i < listed; i += SAMPLE_THREADS)
      list[i] = i < SAMPLE_THREADS ? first_listed : a.list[(int64_t)row * SAMPLE_LIST + i];
  if (threadIdx.x < 64) {  // a chunk a lane (there are at most 64)
    uint4 e = make_uint4(0xffffffffu, 0u, 0u, 0u);
    if ((int)threadIdx.x < a.chunks) e = a.found[(int64_t)row * a.chunks + threadIdx.x];
    chunk_n[threadIdx.x] = e.z;
    e.x = wave_min(e.x);
    e.y = ~wave_min(~e.y);
    if (threadIdx.x == 0) ends[0] = e.x, ends[1] = e.y;
  }
  __syncthreads();
  // the bin's tokens are those with keys from least to most
  const uint32_t least = ends[0], most = ends[1];
  // f(key, index) for the tokens of the bin; a row that is walked waits for its loads, 32 of them a thread at a time
  auto candidates = [&](auto f) __attribute__((always_inline)) {
    if (fits) {
      for (uint32_t i = threadIdx.x; i < listed; i += SAMPLE_THREADS) f(list[i].x, (int)list[i].y);
    } else {
      sample_walk<8>(x, 0, a.V, a.vec, [&](int i, float raw) __attribute__((always_inline)) {
        const uint32_t key = order_key(raw);
        if (key >= least && key <= most) f(key, i);
      });
    }
  };
  // the keys of a bin have most of their bits in common: the selections below begin at the highest in which they differ
  const int differing = least < most ? 32 - __clz(least ^ most) : 0;  // low bits that are not the same in all
  const uint32_t common = differing == 32 ? 0u : (most >> differing) << differing;
  // (a NaN's key is that of -inf: neither weighs anything)
  const Quotient over_t(temp);
  auto scaled = [&](uint32_t key) __attribute__((always_inline)) -> float { return over_t.of(key_to_float(key)); };
  const u64_t above = block_sum((int)threadIdx.x < a.chunks ? chunk_w[threadIdx.x] : 0);
  uint32_t floor_key = 0u;
  // a bin whose largest token has no weight (masked tokens; at low temperatures most of a row): whichever of its
  // tokens stay, none is drawn, and nothing below it
  const bool weightless = listed == 0u || weight_of(scaled(most), mx) == 0;
  // equal logits, however many: all of them stay (the k-th largest is one of them, or the nucleus ends with them)
  const u64_t equal_weight = least == most ? weight_of(scaled(most), mx) : 0;
  if (with_k && !again && !weightless) {
    // the rank-th largest key of the bin
    uint32_t prefix = common, rank = known.rank;
    for (int left = differing; left > 0;) {
      const int width = min(left, 8), shift = left - width;
      bins_n[threadIdx.x] = 0u;
      if (threadIdx.x == 0) picked = 0u, picked_rank = rank;
      __syncthreads();
      candidates([&](uint32_t key, int) __attribute__((always_inline)) {
        if (left == 32 || (key >> left) == (prefix >> left)) atomicAdd(&bins_n[(key >> shift) & ((1u << width) - 1u)], 1u);
      });
      __syncthreads();
      const uint32_t b = 255u - threadIdx.x, n_b = bins_n[b];  // from the largest down
      const uint32_t upto = block_running_sum(n_b);
      if (upto >= rank && upto - n_b < rank) {
        picked = b;
        picked_rank = rank - (upto - n_b);
      }
      __syncthreads();
      prefix |= picked << shift;
      rank = picked_rank;
      left = shift;
      __syncthreads();
    }
    floor_key = order_key(scaled(prefix));
  }
  if (with_p) {
    u64_t limit = known.limit;
    if (with_k && !again) {
      u64_t kept = 0;
      if (equal_weight > 0) {
        if ((int)threadIdx.x < a.chunks) kept = chunk_n[threadIdx.x] * equal_weight;
      } else if (!weightless) {
        candidates([&](uint32_t key, int) __attribute__((always_inline)) {
          const float v = scaled(key);
          if (order_key(v) >= floor_key) kept += weight_of(v, mx);
        });
      }
      const u64_t total = above + block_sum(kept);
      limit = topp_limit(a.top_p[row], total);
      if (total == 0) {
        if (threadIdx.x == 0) a.out[row] = mi < a.V ? mi : 0;
        return;
      }
      if (above > limit) {
        // the nucleus ends in a bin above this one, all of whose tokens are among the k
        u64_t w0, w1;
        row_bins(a, row, w0, w1);
        const u64_t upto = block_running_sum(w0 + w1);
        const u64_t before = upto - w0 - w1;
        if (before <= limit && limit < upto) {
          known.bin = 2 * threadIdx.x + (before + w0 <= limit ? 1 : 0);
          known.limit = limit;
          known.collect = 2u;
        }
        return;
      }
    }
    // the largest key K of the bin with above + weight(kept keys >= K) > limit
    uint32_t prefix = common;
    u64_t over = above;
    for (int left = differing; left > 0;) {
      const int width = min(left, 8), shift = left - width;
      bins_w[threadIdx.x] = 0;
      if (threadIdx.x == 0) picked = 0u, picked_above = over;
      __syncthreads();
      candidates([&](uint32_t key, int) __attribute__((always_inline)) {
        if (left < 32 && (key >> left) != (prefix >> left)) return;
        const float v = scaled(key);
        if (order_key(v) >= floor_key) atomicAdd(&bins_w[(key >> shift) & ((1u << width) - 1u)], weight_of(v, mx));
      });
      __syncthreads();
      const uint32_t b = 255u - threadIdx.x;
      const u64_t w_b = bins_w[b];
      const u64_t upto = over + block_running_sum(w_b);
      if (upto > limit && !(upto - w_b > limit)) {
        picked = b;
        picked_above = upto - w_b;
      }
      __syncthreads();
      prefix |= picked << shift;
      over = picked_above;
      left = shift;
      __syncthreads();
    }
    const uint32_t floor_p = order_key(scaled(prefix));
    if (floor_p > floor_key) floor_key = floor_p;
  }
  // what is kept of the bin joins its chunks; of a row that is walked a wave takes whole chunks, and adds up by itself
  if (weightless) {
  } else if (equal_weight > 0) {
    if ((int)threadIdx.x < a.chunks) chunk_w[threadIdx.x] += chunk_n[threadIdx.x] * equal_weight;
  } else if (fits) {
    for (uint32_t i = threadIdx.x; i < listed; i += SAMPLE_THREADS) {
      const float v = scaled(list[i].x);
      const u64_t w = order_key(v) >= floor_key ? weight_of(v, mx) : 0;
      if (w) atomicAdd(&chunk_w[list[i].y / a.per], w);
    }
  } else {
    for (int c = threadIdx.x >> 6; c < a.chunks; c += SAMPLE_WAVES) {
      const int lo = c * a.per, hi = min(a.V, lo + a.per);
      u64_t sum = 0;
      sample_walk<8, 64>(x, lo, hi, a.vec, [&](int, float raw) __attribute__((always_inline)) {
        const uint32_t key = order_key(raw);
        if (key < least || key > most) return;
        const float v = over_t.of(raw);
        if (order_key(v) >= floor_key) sum += weight_of(v, mx);
      });
      sum = wave_sum(sum);
      if ((threadIdx.x & 63) == 0) chunk_w[c] += sum;
    }
  }
  __syncthreads();
  sample_locate(a, row, temp, mx, mi, floor_key, chunk_w, counts);
}

// flags: bit 0 some row may have top-k, bit 1 some row may have top-p (3 when unknown), bit 2 no row has both: the steps
// no row needs are not launched. workspace: cw_sample_workspace_bytes(n, V) bytes, 16-byte
// aligned.
static int launch_sample(const float* logits, int64_t row_stride, int n, int V,
                         const float* temperature, const int* top_k, const float* top_p,
                         const int64_t* seeds, const int64_t* draws, const DrawCounts& counts, int* out, void* workspace,
                         int64_t workspace_bytes, int flags, hipStream_t stream) {
  if (n < 0 || V <= 0 || row_stride < V) return CW_ERR_ARG;
  if (n == 0) return CW_OK;
  if (n > 65535) return CW_ERR_SIZE;
  if (workspace == nullptr || ((uintptr_t)workspace & 15) || workspace_bytes < cw_sample_workspace_bytes(n, V))
    return CW_ERR_ARG;
  SampleArgs a;
  a.logits = logits; a.row_stride = row_stride; a.n = n; a.V = V;
  a.chunks = sample_chunks(n, V);
  a.per = ((V + a.chunks - 1) / a.chunks + 3) / 4 * 4;
  a.vec = !(row_stride & 3) && !((uintptr_t)logits & 15);
  a.temperature = temperature; a.top_k = top_k; a.top_p = top_p; a.seeds = seeds; a.draws = draws; a.out = out;
  const int64_t rc = (int64_t)n * a.chunks;
  // 16-byte items first
  u64_t* p8 = (u64_t*)workspace;
  a.hist_w = p8; p8 += (int64_t)n * SAMPLE_BINS;
  a.list = (uint2*)p8; p8 += (int64_t)n * SAMPLE_LIST;
  a.hist_n = (uint32_t*)p8; p8 += (int64_t)n * SAMPLE_BINS / 2;
  a.found = (uint4*)p8; p8 += 2 * rc;
  a.sums = p8; p8 += rc;
  a.rows = (SampleRow*)p8; p8 += (int64_t)n * sizeof(SampleRow) / 8;
  a.pmax = (float*)p8;
  a.pmax_i = (int*)(a.pmax + rc);
  a.points = (float*)(a.pmax_i + rc);
  if ((char*)(a.points + (int64_t)n * SAMPLE_POINTS) > (char*)workspace + workspace_bytes) return CW_ERR_ARG;
  const dim3 grid(a.chunks, n), block(SAMPLE_THREADS);
  hipLaunchKernelGGL(sample_max_kernel, grid, block, 0, stream, a);
  hipLaunchKernelGGL(sample_hist_kernel, grid, block, 0, stream, a);
  if (flags & 3) hipLaunchKernelGGL(sample_collect_kernel, grid, block, 0, stream, a, 0);
  hipLaunchKernelGGL(sample_draw_kernel, dim3(n), block, 0, stream, a, 0, counts);
  if ((flags & 7) == 3) {
    hipLaunchKernelGGL(sample_collect_kernel, grid, block, 0, stream, a, 1);
    hipLaunchKernelGGL(sample_draw_kernel, dim3(n), block, 0, stream, a, 1, counts);
  }
  return cw_launch_status();
}
CW_EXPORT int cw_sample(const float* logits, int64_t row_stride, int n, int V,
                        const float* temperature, const int* top_k, const float* top_p,
                        const int64_t* seeds, const int64_t* draws, int* out, void* workspace,
                        int64_t workspace_bytes, int flags, hipStream_t stream) {
  if (n > 0 && !draws) return CW_ERR_ARG;
  return launch_sample(logits, row_stride, n, V, temperature, top_k, top_p, seeds, draws, DrawCounts{}, out, workspace, workspace_bytes, flags,
                       stream);
}
// The same for up to 64 rows whose draw counts [n] (0 to 2^32 - 1) lie in host memory and are read before the call returns.
CW_EXPORT int cw_sample_counted(const float* logits, int64_t row_stride, int n, int V,
                                const float* temperature, const int* top_k, const float* top_p,
                                const int64_t* seeds, const int64_t* host_draws, int* out, void* workspace,
                                int64_t workspace_bytes, int flags, hipStream_t stream) {
  if (n > SAMPLE_COUNTED_ROWS) return CW_ERR_SIZE;
  if (n > 0 && !host_draws) return CW_ERR_ARG;
  DrawCounts counts{};
  for (int i = 0; i < n; ++i) {
    if (host_draws[i] < 0 || host_draws[i] > (int64_t)UINT32_MAX) return CW_ERR_ARG;
    counts.of_row[i] = (uint32_t)host_draws[i];
  }
  return launch_sample(logits, row_stride, n, V, temperature, top_k, top_p, seeds, nullptr, counts, out, workspace, workspace_bytes, flags, stream);
}
static_assert(sizeof(SampleRow) % 8 == 0 && sizeof(SampleRow) / 4 <= SAMPLE_THREADS, "MAX zeroes a row's record, a word a thread");
