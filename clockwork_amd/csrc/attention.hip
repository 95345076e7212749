// Causal attention over a paged key/value cache for gfx950, one head size per build
// (compile with -DCW_HD=<head_dim>, a multiple of 16 from 16 to 256).
//
// The first kernel serves portions of prompts and single decoded tokens of any type: a work item is a run of
// consecutive query tokens of one request; a workgroup takes rows of one item, one key/value head and
// all (or a chunk of) the query heads of that head's group, so a key/value tile is fetched once
// for the whole group. The key range of an item can be cut into splits that run in parallel
// and are merged by a second kernel (decode with few requests and long contexts).
//
// Scores, softmax and the output accumulation are float32 whatever the cache type is.
// A token at position p reads keys j <= p, and j > p - window when a window is set. Pages are
// found through the request's block table; positions outside an item's key range are never
// dereferenced (their table entries may be stale or -1).
#include "common.h"

#include <limits.h>
#include <type_traits>
#include <utility>

#ifndef CW_HD
#error "compile with -DCW_HD=<head_dim>"
#endif
static_assert(CW_HD % 16 == 0 && CW_HD >= 16 && CW_HD <= 256, "head_dim: multiples of 16 up to 256");

struct AttnParams {
  const void* q;          // [tokens, q_stride] query heads at column head * HD
  int64_t q_stride;
  void* out;              // [tokens, out_stride]
  int64_t out_stride;
  const void* k_cache;    // [slots, nkv, HD]
  const void* v_cache;
  const int* block_tables;  // [requests, table_stride]
  int table_stride;
  const int* ctx_lens;    // [requests] keys of the request after this step
  const int* cu_q;        // [requests + 1] offsets of each request's tokens in the batch
  const int* items;       // [n_items, 4]: request, first token (relative), tokens, part | parts << 8 (prefill kernel)
  int nh, nkv, block_size;
  int bs_shift;           // log2(block_size) when it is a power of two, else -1
  int gh;                 // query heads of a group handled by one workgroup
  int n_chunks;           // ceil(group / gh)
  int n_splits;
  int window;             // 0: none
  float scale;
  float softcap;          // > 0: score <- softcap * tanh(scale * q . k / softcap) (the matrix-core kernels)
  float* part_o;          // [n_items, nkv * n_chunks, n_splits, ROWS, HD] unnormalised outputs
  float* part_ml;         // [n_items, nkv * n_chunks, n_splits, ROWS, 2] running max, sum
  const void* zeros;      // at least HD zero elements: what a masked key or value row is loaded from
  const void* gate;       // bfloat16 rows, or null: head h's output is multiplied by logistic(gate[token, gate_off + h])
  int64_t gate_stride;    //   (the matrix-core kernels)
  int gate_off;
  // decode kernel only
  int identity;           // 1: item i is request i and its one token is row i of the batch (items, cu_q unread)
  int split_keys;         // > 0: split s takes keys [s * split_keys, (s + 1) * split_keys), a multiple of 32
  int decode_pages;       // -1: a split's pages do not fit LDS, they are looked up in memory
};

// the factor of a head's output of the token in row ``token`` of the batch
__device__ __forceinline__ float attn_head_gate(const AttnParams& p, int64_t token, int head) {
  return p.gate ? cw_logistic(cw_to_float(((const bf16_t*)p.gate)[token * p.gate_stride + p.gate_off + head])) : 1.0f;
}

// page of a position and the offset inside it; POW2: the page size is a power of two (shift given)
template <bool POW2> __device__ __forceinline__ int cw_page_index(int pos, int bs, int shift) {
  return POW2 ? pos >> shift : pos / bs;
}
template <bool POW2> __device__ __forceinline__ int cw_page_offset(int pos, int bs, int shift) {
  return POW2 ? pos & (bs - 1) : pos % bs;
}
static inline int cw_log2_or_minus1(int v) {
  for (int s = 0; s < 31; ++s) if ((1 << s) == v) return s;
  return -1;
}

// Four neighbouring elements of a cache or query row as float32, and VW of them (1, 2 or 4).
typedef __attribute__((ext_vector_type(4))) float attn_f32x4_t;
template <int VW> __device__ __forceinline__ void attn_load(const float* p, float (&o)[VW]) {
  if (VW == 4) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    o[0] = v.x; o[1 % VW] = v.y; o[2 % VW] = v.z; o[3 % VW] = v.w;
  } else if (VW == 2) {
    const float2 v = *reinterpret_cast<const float2*>(p);
    o[0] = v.x; o[1 % VW] = v.y;
  } else {
    o[0] = p[0];
  }
}
template <int VW> __device__ __forceinline__ void attn_load(const bf16_t* p, float (&o)[VW]) {
  if (VW == 1) {
    o[0] = cw_to_float(p[0]);
  } else {
    uint32_t w[VW / 2 + (VW == 1)];
    __builtin_memcpy(w, __builtin_assume_aligned(p, VW * 2), VW * 2);
#pragma unroll
    for (int i = 0; i < VW / 2; ++i) {
      o[(2 * i) % VW] = __uint_as_float(w[i] << 16);
      o[(2 * i + 1) % VW] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
}

// Float32 scores, softmax and sums for any cache type, all products on the matrix cores
// (v_mfma_f32_16x16x4_f32: float32 operands, products and sums).
//
// A workgroup takes RB blocks of 16 rows (token, head of the group) of one item, one key/value head and one
// split of the keys; its waves take tiles of 16 keys in turn and meet in LDS at the end. Lane (c, s) = (l % 16, l / 16):
//   S^T[key, row] = K * Q^T    lane holds four neighbouring elements, from 4 s on, of key c / of row c: the j-th of four
//                              products takes element j of every lane, which is the same k-value in both operands;
//   softmax                    the lane comes out with keys 4 s .. 4 s + 3 of row c: a row is four lanes;
//   O^T[d, row] += V^T * P^T   the j-th product takes key 4 s + j: P^T is what the lane holds, and V's elements come in
//                              runs of VW along a row, tile e of a run's VW tiles taking element e.
// Nothing passes through LDS in the loop, and the next tile's keys are on their way over this one's products.
// What bounds it is the trip to memory of a wave's first tiles with short ranges (so 16 rows a workgroup while that
// leaves compute units idle) and the matrix cores' float32 rate with long ones (32 rows: a key is read for twice the rows).
// Measured: see launch_attention.
template <typename T, int HD, int RB, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void attn_f32_kernel(AttnParams p, int rows, int subs) {
  constexpr int VW = HD % 64 == 0 ? 4 : HD % 32 == 0 ? 2 : 1;  // elements of a value row that a lane loads at once
  constexpr int KB = HD / 16, VG = HD / (16 * VW), OS = HD + 4;
  extern __shared__ __align__(16) float smem[];  // [WAVES][16][OS] sums, then [WAVES][16][2] maxima and sums of weights
  float* const o_s = smem;
  float* const ml_s = smem + WAVES * 16 * OS;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, s = lane >> 4;
  const int turn = gridDim.x - 1 - blockIdx.x;  // a portion's last tokens have the longest key ranges: they begin first
  const int item = turn / subs, row0 = (turn % subs) * (16 * RB);
  const int kvh = blockIdx.y / p.n_chunks, chunk = blockIdx.y % p.n_chunks;
  const int split = blockIdx.z;
  const int req = p.items[4 * item], tok0 = p.items[4 * item + 1];
  const int ctx = p.ctx_lens[req];
  const int q_begin = p.cu_q[req];
  const int qlen = p.cu_q[req + 1] - q_begin;
  // an item may reach past the request's tokens (work items laid out for a longer portion than
  // the step brings): what lies past them is not computed
  const int ntok = min(p.items[4 * item + 2], qlen - tok0);
  const int group = p.nh / p.nkv;
  const int gh = p.gh;
  const int tok_first = row0 / gh;                              // tokens of this workgroup's rows
  const int tok_end = min(ntok, (row0 + 16 * RB - 1) / gh + 1);
  if (tok_first >= tok_end) return;
  const int pos0 = ctx - qlen + tok0;  // absolute position of the item's first token
  const int kv_end = pos0 + tok_end;
  const int kv_lo = p.window > 0 ? max(0, pos0 + tok_first - p.window + 1) : 0;
  const int tile0 = kv_lo / 16, n_tiles = (kv_end + 15) / 16 - tile0;
  const int tps = (n_tiles + p.n_splits - 1) / p.n_splits;
  const int t_begin = tile0 + split * tps, t_end = min(tile0 + n_tiles, t_begin + tps);
  const T* const qp = (const T*)p.q;
  const T* const kc = (const T*)p.k_cache + (int64_t)kvh * HD;
  const T* const vc = (const T*)p.v_cache + (int64_t)kvh * HD;
  const int64_t row_stride = (int64_t)p.nkv * HD;
  const int* const table = p.block_tables + (int64_t)req * p.table_stride;

  // this lane's row of every block: its query, its last and first key
  float qf[RB][KB][4];
  int last_key[RB], first_key[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = row0 + rb * 16 + c, tok = r / gh, hig = chunk * gh + (r - tok * gh);
    const bool ok = r < rows && tok < ntok && hig < group;
    last_key[rb] = ok ? pos0 + tok : -1;
    first_key[rb] = p.window > 0 ? pos0 + tok - p.window + 1 : 0;
    const T* q = qp + (int64_t)(q_begin + tok0 + (ok ? tok : tok_first)) * p.q_stride + (kvh * group + (ok ? hig : 0)) * HD + 4 * s;
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      // a row's start is not always a multiple of 16 bytes: the caller's stride decides
#pragma unroll
      for (int j = 0; j < 4; ++j) qf[rb][b][j] = ok ? cw_to_float(q[16 * b + j]) : 0.0f;
    }
  }

  // A tile's places in the cache: key c's and keys 4 s .. 4 s + 3's rows, -1 where the table names no page. Positions
  // outside the range are moved to its edge: their scores are masked, and what is read lies in the request's own
  // pages. Pages of a multiple of 16 keys hold a tile whole: one page for the wave then, by a scalar load.
  const bool whole = !(p.block_size & 15);
  auto places = [&](int t, int64_t (&at)[5]) __attribute__((always_inline)) {
    int page = 0, page_first = 0;
    if (whole) {
      const int first = __builtin_amdgcn_readfirstlane(16 * t);
      const int n = p.bs_shift >= 0 ? first >> p.bs_shift : first / p.block_size;
      page = table[n];
      page_first = n * p.block_size;
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const int pos = min(max(16 * t + (i == 0 ? c : 4 * s + i - 1), kv_lo), kv_end - 1);
      int pg = page, off = pos - page_first;
      if (!whole) {
        pg = table[p.bs_shift >= 0 ? pos >> p.bs_shift : pos / p.block_size];
        off = p.bs_shift >= 0 ? pos & (p.block_size - 1) : pos % p.block_size;
      }
      at[i] = pg >= 0 ? (int64_t)pg * p.block_size + off : -1;
    }
  };
  auto load = [&](const int64_t (&at)[5], float (&k)[KB][4], float (&v)[4][VG][VW]) __attribute__((always_inline)) {
    const T* row = kc + max(at[0], (int64_t)0) * row_stride + 4 * s;
#pragma unroll
    for (int b = 0; b < KB; ++b) attn_load<4>(row + 16 * b, k[b]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const T* vrow = vc + max(at[1 + j], (int64_t)0) * row_stride + VW * c;
#pragma unroll
      for (int g = 0; g < VG; ++g) attn_load<VW>(vrow + 16 * VW * g, v[j][g]);
    }
  };

  attn_f32x4_t acc[RB][VG * VW];
  float m[RB], l[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    m[rb] = -INFINITY;
    l[rb] = 0.0f;
#pragma unroll
    for (int e = 0; e < VG * VW; ++e) acc[rb][e] = (attn_f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
  }

  // one tile: ``at`` where it lay, ``k`` and ``v`` what lay there
  auto compute = [&](int t, const int64_t (&at)[5], float (&k)[KB][4], float (&v)[4][VG][VW]) __attribute__((always_inline)) {
    const int kv0 = 16 * t;
    // no page: zeros; and zeros for values outside the range (what lies there is another key's, and a weight of
    // zero times an infinite value is no zero)
    if (kv0 < kv_lo || kv0 + 16 > kv_end ||
        __builtin_amdgcn_ballot_w64(at[0] < 0 || at[1] < 0 || at[2] < 0 || at[3] < 0 || at[4] < 0)) {
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j) k[b][j] = at[0] >= 0 ? k[b][j] : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int pos = kv0 + 4 * s + j;
        const bool there = at[1 + j] >= 0 && pos >= kv_lo && pos < kv_end;
#pragma unroll
        for (int g = 0; g < VG; ++g)
#pragma unroll
          for (int e = 0; e < VW; ++e) v[j][g][e] = there ? v[j][g][e] : 0.0f;
      }
    }
    attn_f32x4_t sc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) sc[rb] = (attn_f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) sc[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[b][j], qf[rb][b][j], sc[rb], 0, 0, 0);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float top = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int pos = kv0 + 4 * s + i;
        sc[rb][i] = pos <= last_key[rb] && pos >= first_key[rb] ? sc[rb][i] * p.scale : -INFINITY;
        top = fmaxf(top, sc[rb][i]);
      }
      const float m_new = fmaxf(m[rb], cw_quad_max(top));
      const float ref = m_new == -INFINITY ? 0.0f : m_new;  // no key of the row yet: every weight is exp(-inf)
      const float alpha = expf(m[rb] - ref);
      m[rb] = m_new;
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[rb][i] = expf(sc[rb][i] - ref);
        sum += sc[rb][i];
      }
      l[rb] = fmaf(l[rb], alpha, sum);  // of this lane's keys; the four lanes of a row are added at the end
#pragma unroll
      for (int e = 0; e < VG * VW; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rb][e][i] *= alpha;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int g = 0; g < VG; ++g)
#pragma unroll
        for (int e = 0; e < VW; ++e)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
            acc[rb][g * VW + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j][g][e], sc[rb][j], acc[rb][g * VW + e], 0, 0, 0);
  };
  // Two tiles take turns: one is on its way while the other is multiplied, and the places of the one after are
  // looked up meanwhile. Past the last tile the last one is asked for again: no load hangs on a condition.
  const int t_first = t_begin + wave;
  if constexpr (HD > 192) {  // two tiles do not fit the registers
    float ka[KB][4], va[4][VG][VW];
    int64_t at[5], next[5];
    if (t_first < t_end) places(t_first, at);
    for (int t = t_first; t < t_end; t += WAVES) {
      load(at, ka, va);
      places(t + WAVES < t_end ? t + WAVES : t, next);
      compute(t, at, ka, va);
#pragma unroll
      for (int i = 0; i < 5; ++i) at[i] = next[i];
    }
  } else if (t_first < t_end) {
    const int t_last = t_first + (t_end - 1 - t_first) / WAVES * WAVES;
    float ka[KB][4], va[4][VG][VW], kb[KB][4], vb[4][VG][VW];
    int64_t at_a[5], at_b[5];
    places(t_first, at_a);
    load(at_a, ka, va);
    places(min(t_first + WAVES, t_last), at_b);
    for (int t = t_first; t < t_end; t += 2 * WAVES) {
      load(at_b, kb, vb);
      int64_t next[5];
      places(min(t + 2 * WAVES, t_last), next);
      compute(t, at_a, ka, va);
#pragma unroll
      for (int i = 0; i < 5; ++i) at_a[i] = next[i];
      if (t + WAVES >= t_end) break;
      load(at_a, ka, va);
      places(min(t + 3 * WAVES, t_last), next);
      compute(t + WAVES, at_b, kb, vb);
#pragma unroll
      for (int i = 0; i < 5; ++i) at_b[i] = next[i];
    }
  }

  // ---- the waves' results meet, one block of rows after the other: final rows when there is one split, partial sums
  // otherwise
  const int64_t base = ((int64_t)item * gridDim.y + blockIdx.y) * p.n_splits + split;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    if (rb > 0) __syncthreads();
    const float total = cw_quad_sum(l[rb]);
    float* mine = o_s + (wave * 16 + c) * OS + 4 * VW * s;
    // lane (c, s) holds, of row c, elements 16 VW g + VW (4 s + i) + e
#pragma unroll
    for (int g = 0; g < VG; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < VW; ++e) mine[16 * VW * g + VW * i + e] = acc[rb][g * VW + e][i];
    if (s == 0) {
      ml_s[(wave * 16 + c) * 2] = m[rb];
      ml_s[(wave * 16 + c) * 2 + 1] = total;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < 16 * HD; idx += WAVES * 64) {
      const int rr = idx / HD, d = idx - rr * HD;
      const int r = row0 + rb * 16 + rr, tok = r / gh, hig = chunk * gh + (r - tok * gh);
      if (r >= rows || tok >= ntok || hig >= group) continue;
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) M = fmaxf(M, ml_s[(w * 16 + rr) * 2]);
      float L = 0.0f, O = 0.0f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const float mw = ml_s[(w * 16 + rr) * 2];
        const float f = mw == -INFINITY ? 0.0f : expf(mw - M);
        L = fmaf(ml_s[(w * 16 + rr) * 2 + 1], f, L);
        O = fmaf(o_s[(w * 16 + rr) * OS + d], f, O);
      }
      if (p.n_splits == 1) {
        ((T*)p.out)[(int64_t)(q_begin + tok0 + tok) * p.out_stride + (kvh * group + hig) * HD + d] = cw_from_float<T>(O * (1.0f / L));
      } else {
        p.part_o[(base * rows + r) * HD + d] = O;
        if (d == 0) {
          p.part_ml[(base * rows + r) * 2] = M;
          p.part_ml[(base * rows + r) * 2 + 1] = L;
        }
      }
    }
  }
}

// Merge the splits of every (item, head) row: out = sum_s e^(m_s - M) o_s / sum_s e^(m_s - M) l_s,
// splits taken in ascending order.
template <typename T, int HD, int ROWS>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnParams p) {
  const int item = blockIdx.x;
  const int kvh = blockIdx.y / p.n_chunks;
  const int chunk = blockIdx.y % p.n_chunks;
  const int req = p.items[4 * item], tok0 = p.items[4 * item + 1];
  const int q_begin = p.cu_q[req];
  // as in the kernel above: an item may reach past the request's tokens, and those rows are nobody's
  const int ntok = min(p.items[4 * item + 2], p.cu_q[req + 1] - q_begin - tok0);
  const int group = p.nh / p.nkv;
  const int gh = p.gh;
  const int64_t base = ((int64_t)item * gridDim.y + blockIdx.y) * p.n_splits;
  T* op = (T*)p.out;
  // a thread has one element, and its splits' numbers are asked for side by side
  const int idx = blockIdx.z * 256 + threadIdx.x;
  if (idx < ROWS * HD) {
    const int r = idx / HD, d = idx - r * HD;
    const int tok = r / gh, hig = chunk * gh + (r - tok * gh);
    if (tok >= ntok || hig >= group) return;
    float M = -INFINITY;
#pragma unroll 4
    for (int s = 0; s < p.n_splits; ++s) M = fmaxf(M, p.part_ml[((base + s) * ROWS + r) * 2]);
    float L = 0.0f, O = 0.0f;
#pragma unroll 4
    for (int s = 0; s < p.n_splits; ++s) {
      const float m = p.part_ml[((base + s) * ROWS + r) * 2];
      if (m == -INFINITY) continue;
      const float w = expf(m - M);
      L = fmaf(p.part_ml[((base + s) * ROWS + r) * 2 + 1], w, L);
      O = fmaf(p.part_o[((base + s) * ROWS + r) * HD + d], w, O);
    }
    op[(int64_t)(q_begin + tok0 + tok) * p.out_stride + (kvh * group + hig) * HD + d] =
        cw_from_float<T>(O / L);
  }
}

template <typename T, int RB, int WAVES>
static int launch_attention_rows(const AttnParams& p, int rows, int n_items, hipStream_t stream) {
  constexpr int HD = CW_HD;
  constexpr size_t smem = sizeof(float) * WAVES * 16 * (HD + 4 + 2);
  static bool raised = false;
  if (smem > 65536 && !raised) {
    if (hipFuncSetAttribute((const void*)attn_f32_kernel<T, HD, RB, WAVES>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)smem) != hipSuccess)
      return CW_ERR_LAUNCH;
    raised = true;
  }
  const int subs = rows / (16 * RB);
  if ((int64_t)n_items * subs > 0x7fffffff) return CW_ERR_SIZE;
  const dim3 grid(n_items * subs, p.nkv * p.n_chunks, p.n_splits);
  hipLaunchKernelGGL((attn_f32_kernel<T, HD, RB, WAVES>), grid, dim3(WAVES * 64), smem, stream, p, rows, subs);
  return cw_launch_status();
}

// 32 rows a workgroup (four waves) where that still gives every compute unit two workgroups, else 16 rows (eight waves).
// Measured on an MI355X, float32, us a call, before (vector-unit tiles of 64 rows and 64 keys in LDS) and now: heads of
// 64, 14 on 2: 17 tokens 24 -> 8.8, 300 97 -> 17.5, 1000 298 -> 58; heads of 128, 12 on 2: 300 tokens 174 -> 23, 2048
// 1571 -> 229 (16 rows: 283); one token behind 300 keys 33 -> 10.3, 8 behind 2048 (8 parts) 62 -> 22.5.
template <typename T, int ROWS>
static int launch_attention(const AttnParams& p, int n_items, hipStream_t stream) {
  constexpr int HD = CW_HD;
  int rc;
  if constexpr (HD > 128) {  // registers for four waves of 16 rows only
    rc = launch_attention_rows<T, 1, 4>(p, ROWS, n_items, stream);
  } else if constexpr (ROWS == 64) {
    const int64_t pairs = (int64_t)n_items * p.nkv * p.n_chunks * p.n_splits * 2;  // workgroups of 32 rows
    rc = pairs >= 512 ? launch_attention_rows<T, 2, 4>(p, ROWS, n_items, stream) : launch_attention_rows<T, 1, 8>(p, ROWS, n_items, stream);
  } else {
    rc = launch_attention_rows<T, 1, 8>(p, ROWS, n_items, stream);
  }
  if (rc != CW_OK) return rc;
  if (p.n_splits > 1) {
    dim3 mgrid(n_items, p.nkv * p.n_chunks, (ROWS * HD + 255) / 256);
    hipLaunchKernelGGL((attn_merge_kernel<T, HD, ROWS>), mgrid, dim3(256), 0, stream, p);
  }
  return cw_launch_status();
}

CW_EXPORT int cw_attention_head_dim() { return CW_HD; }

// Floats of workspace a launch with these sizes needs (0 when n_splits == 1).
CW_EXPORT int64_t cw_attention_workspace_floats(int rows, int n_items, int nkv, int n_chunks, int n_splits) {
  if (n_splits <= 1) return 0;
  return (int64_t)n_items * nkv * n_chunks * n_splits * rows * (CW_HD + 2);
}

// rows of an item: 64 (portions of prompts) or 16 (single tokens, few tokens). gh * tokens-per-item <= rows.
CW_EXPORT int cw_attention(int rows, int dtype, const void* q, int64_t q_stride, void* out,
                           int64_t out_stride, const void* k_cache, const void* v_cache,
                           const int* block_tables, int table_stride, const int* ctx_lens,
                           const int* cu_q, const int* items, int n_items, int nh, int nkv,
                           int block_size, int gh, int n_splits, int window, float scale,
                           float* workspace, int64_t workspace_floats, hipStream_t stream) {
  if (n_items < 0 || nh <= 0 || nkv <= 0 || nh % nkv != 0 || block_size <= 0 || table_stride <= 0)
    return CW_ERR_ARG;
  if (rows != 64 && rows != 16) return CW_ERR_ARG;
  const int group = nh / nkv;
  if (gh < 1 || gh > group || gh > rows || n_splits < 1 || n_splits > 65535 || window < 0) return CW_ERR_ARG;
  if (n_items == 0) return CW_OK;
  AttnParams p{};
  p.q = q; p.q_stride = q_stride; p.out = out; p.out_stride = out_stride;
  p.k_cache = k_cache; p.v_cache = v_cache; p.block_tables = block_tables;
  p.table_stride = table_stride; p.ctx_lens = ctx_lens; p.cu_q = cu_q; p.items = items;
  p.nh = nh; p.nkv = nkv; p.block_size = block_size; p.bs_shift = cw_log2_or_minus1(block_size); p.gh = gh;
  p.n_chunks = (group + gh - 1) / gh; p.n_splits = n_splits; p.window = window; p.scale = scale; p.softcap = 0.0f;
  if ((int64_t)nkv * p.n_chunks > 65535) return CW_ERR_SIZE;
  const int64_t need = cw_attention_workspace_floats(rows, n_items, nkv, p.n_chunks, n_splits);
  if (need > 0 && (workspace == nullptr || workspace_floats < need)) return CW_ERR_ARG;
  const int64_t n_o = need / (CW_HD + 2) * CW_HD;
  p.part_o = workspace;
  p.part_ml = workspace ? workspace + n_o : nullptr;
  p.zeros = nullptr;
  if (dtype == CW_F32) {
    return rows == 64 ? launch_attention<float, 64>(p, n_items, stream) : launch_attention<float, 16>(p, n_items, stream);
  } else if (dtype == CW_BF16) {
    return rows == 64 ? launch_attention<bf16_t, 64>(p, n_items, stream) : launch_attention<bf16_t, 16>(p, n_items, stream);
  }
  return CW_ERR_DTYPE;
}

// =====================================================================================
// What the bfloat16 kernels below share: tiles of keys and values in LDS, as blocks of 16 keys x 32 elements (1 KB: what one
// load of a wave with the LDS target brings), a key's four 16-byte granules permuted.
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;
typedef __attribute__((address_space(3))) void lds_raw_t;

// Where granule g of key k (0 to 15) lies in a block. K: eight neighbouring lanes of a ds_read_b128 take one
// granule of eight keys, 64 bytes apart, and with these permutations every bank once; V: 16 lanes of a transposing read
// take 32 bytes of four keys.
__device__ __forceinline__ int k_granule(int k, int g) { return g ^ ((((k >> 1) ^ (k >> 3)) & 1) | (((k >> 2) & 1) << 1)); }
__device__ __forceinline__ int v_granule(int k, int g) { return g ^ ((((k >> 1) ^ (k >> 2)) & 1) << 1); }

// 16 bytes a lane from memory to LDS, to 1 KB at ``to`` (the same for all lanes), lane by lane; from an address a lane, or
// from one address for all and an offset a lane. Written out, because behind the builtin the compiler puts a wait for all
// such loads before the next transposing read, of whatever tile: what the kernel waits for and where is its own to say.
// (No vector register is written; m0, where the instruction finds the address in LDS, is.)
__device__ __forceinline__ void load_to_lds(const void* from, void* to) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               : : "v"(from), "s"((uint32_t)(uintptr_t)(lds_raw_t*)to) : "memory", "m0");
}
// (``OFFSET`` bytes further on at both ends: the instruction's own offset counts for the address in LDS as well)
template <int OFFSET>
__device__ __forceinline__ void load_to_lds(const void* from, void* to) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off offset:%2"
               : : "v"(from), "s"((uint32_t)(uintptr_t)(lds_raw_t*)to), "n"(OFFSET) : "memory", "m0");
}
// The blocks of 32 elements of 16 rows, 64 bytes apart in memory and 1 KB in LDS.
template <int... J>
__device__ __forceinline__ void row_to_lds(const void* from, unsigned char* to, std::integer_sequence<int, J...>) {
  (load_to_lds<J * 64>(from, to + J * (1024 - 64)), ...);
}
// Two of them at once of 8 rows: 128 bytes apart in memory, 2 KB in LDS; lines that nobody reads again, for the caches not to keep.
template <int OFFSET>
__device__ __forceinline__ void load_lines_to_lds(const void* from, void* to) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off offset:%2 nt"
               : : "v"(from), "s"((uint32_t)(uintptr_t)(lds_raw_t*)to), "n"(OFFSET) : "memory", "m0");
}
template <int... J>
__device__ __forceinline__ void lines_to_lds(const void* from, unsigned char* to, std::integer_sequence<int, J...>) {
  (load_lines_to_lds<J * 128>(from, to + J * (2048 - 128)), ...);
}
__device__ __forceinline__ void load_to_lds(const void* base, uint32_t offset, void* to) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               : : "v"(offset), "s"(base), "s"((uint32_t)(uintptr_t)(lds_raw_t*)to) : "memory", "m0");
}

// =====================================================================================
// bfloat16 decode attention: one query token per work item, keys and values streamed at memory
// speed, all products on the matrix cores.
//
// A workgroup (4 or 8 waves) takes one (request, key/value head, split of the key range); its waves
// take turns on tiles of 32 keys. Per tile:
//   S^T[key, head] = K * Q^T        v_mfma_f32_16x16x32_bf16; the up to 16 heads of the group are
//                                   the columns, so every key is fetched once for the whole group;
//   softmax per head in float32: a lane holds 8 keys of one head, two swaps of lanes across the wave's rows finish a head;
//   O^T[d, head] += V^T * P^T       P^T is the softmax output as it lies in the registers.
// A wave's tile comes from the pages straight into LDS of its own, four neighbouring lanes 64 bytes of a key, and its operands
// from there: K fragments by 16-byte reads, V^T fragments by the transposing read (see the kernel for portions). Once a tile's
// operands are in registers the next one is asked for (room for two tiles of heads of 64 gained nothing). Through registers,
// with a lane exchange of every fragment into operand layout and V^T by products with 0/1 selector matrices, a tile of 32
// keys of 128 elements cost a wave some 700 instructions, 1.8 us. Waves are merged through LDS at the end; splits are merged
// by a second, small kernel. Bound by the chain from the context's length over the table to the keys, for many requests by memory.
// Measured on an MI355X (with the merge; us, that way -> this): one request of 120 keys, 14 heads of 64 on 2, 4.7 -> 3.9, of 400
// keys 6.4 -> 5.2; 12 heads of 128 on 2, one request of 2048 10.3 -> 8.7, 8 of 2048 12.8 -> 10.9, 32 of 2048 21.6 -> 20.3, 64 of
// 2048 34.1 -> 32.3; 8 of 2048, 16 heads of 256 on 4, 26.5 -> 21.2. A decode step of 8 requests (1.5B shape) 1445 -> 1414 us.
template <int HD> struct DecodeTile {
  static constexpr int BYTES = 32 * HD * 4;  // 32 keys and values: a wave's LDS; its 16 heads' outputs lie over it at the end
};

// LINES (heads of 128): a load takes 128 bytes of 8 keys, whole lines that the caches need not keep, and a tile lies in LDS as blocks of
// 16 keys x 64 elements, a key's eight granules permuted so that 16 lanes' operands (K: a granule of 16 keys; V: 32 bytes of four) take every
// bank once. It costs a second table entry and address a key and pays where keys and values come at memory's speed and nobody else reads them. Where
// another request has the same pages (a prefix, a fork), whole lines past the caches come from memory each time: such a split, which looks
// for one at its first page, loads half lines as a kernel without LINES. Same bits either way. us, half lines only / whole lines only / this, heads of 128,
// nothing shared: 12 on 2, 64 requests of 2048 keys 31.7 / 29.3 / 29.9, 32 of 2048 20.4 / 19.3 / 19.7, 32 of 1000 14.4 / 13.8 / 14.1; 28 on 4, 64 of
// 1500 42.4 / 36.3 / 36.6. The first 1024 keys of 32 of 64 requests of 2048 the same 26.9 / 28.8 / 25.6, of all 22.6 / 25.3 / 22.0, the first
// 1900 16.7 / 21.9 / 17.3; 28 on 4, 1024 of 32 of 64 of 1500 33.2 / 33.5 / 29.4, of all 64 of 1200 17.6 / 22.0 / 17.9. 8 of 2048, in 256 workgroups of 160 keys,
// 10.7 / 10.0 alone and 1309 / 1324 a step; with few workgroups, whose time is trips to memory, 8 of 300 7.1 / 8.3, one of 2048 9.2 / 9.8: half lines. So,
// too, where a group's heads are cut into several workgroups, which read the same keys (66 heads on 1, 64 of 1000: 25.1 / 31.8), and heads of
// 64, whose keys are one line each (14 on 2, 64 of 2048: 19.5 / 20.5).
template <int HD, bool POW2, int WAVES, bool CAP, bool LINES = false>
__device__ __forceinline__ void attn_decode_of(const AttnParams& p, const int item, const int y, const int split) {
  constexpr int NF = HD / 32;  // 32-element steps over the head dimension
  constexpr int ND = HD / 16;  // 16-wide blocks of the head dimension
  using Tile = DecodeTile<HD>;
  extern __shared__ __align__(1024) unsigned char dec_smem[];  // [waves][a tile], then this split's pages if they fit
  const bool in_lds = p.decode_pages >= 0;
  int* const tbl = reinterpret_cast<int*>(dec_smem + WAVES * Tile::BYTES);
  __shared__ float M_s[WAVES][16];
  __shared__ float L_s[WAVES][16];
  __shared__ int shared_s;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, s = lane >> 4;
  const int kvh = y / p.n_chunks, chunk = y % p.n_chunks;
  // Every trip to memory that depends on an earlier one costs about a microsecond, which is what
  // a short context takes in all: with ``identity`` and fixed key ranges per split, the context
  // length, the table entries and the query are fetched side by side, then keys and values.
  const bool ident = p.identity != 0;
  const int req = ident ? item : p.items[4 * item];
  const int tok0 = ident ? 0 : p.items[4 * item + 1];
  const int ctx = p.ctx_lens[req];
  const int q_begin = ident ? item : p.cu_q[req];
  const int qlen = ident ? 1 : p.cu_q[req + 1] - q_begin;
  const int group = p.nh / p.nkv;
  const int gh = p.gh;
  const bf16_t* kc = (const bf16_t*)p.k_cache;
  const bf16_t* vc = (const bf16_t*)p.v_cache;
  const bf16_t* zrow = (const bf16_t*)p.zeros;
  const int bs = p.block_size, sh = p.bs_shift;
  const int* table = p.block_tables + (int64_t)req * p.table_stride;
  int page0 = 0;
  if (p.split_keys > 0) {
    // the pages of this split's key range -> LDS, whatever the context length turns out to be
    const int k_first = split * p.split_keys;
    const int k_last = min(k_first + p.split_keys, p.table_stride * bs) - 1;
    page0 = cw_page_index<POW2>(k_first, bs, sh);
    const int n_pages = k_last >= k_first ? cw_page_index<POW2>(k_last, bs, sh) - page0 + 1 : 0;
    if (in_lds)
      for (int i = threadIdx.x; i < n_pages; i += WAVES * 64) tbl[i] = table[page0 + i];
    // LINES (item i is request i): does one of the 64 requests after this one have the same page where this split begins? Asked for beside
    // the entries above. (A row of the batch without a request may hold anything: its context ends inside its first page.)
    if (LINES && wave == WAVES - 1) {
      const int n = (int)gridDim.x, other = req + 1 + lane - (req + 1 + lane < n ? 0 : n);
      bool same = lane + 1 < n && n_pages > 0;  // (so other is one of n)
      if (same) {
        const int mine = table[page0];
        same = p.block_tables[(int64_t)other * p.table_stride + page0] == mine && mine >= 0 && p.ctx_lens[other] > k_first + bs;
      }
      const bool any = __any(same);
      if (lane == 0) shared_s = any;
    }
  }
  const int pos = ctx - qlen + tok0;
  const int lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  const int tile0 = lo / 32;
  const int n_tiles = pos / 32 + 1 - tile0;
  int t_begin, t_end;
  if (p.split_keys > 0) {
    t_begin = max(tile0, split * (p.split_keys / 32));
    t_end = min(tile0 + n_tiles, (split + 1) * (p.split_keys / 32));
  } else {
    const int tps = (n_tiles + p.n_splits - 1) / p.n_splits;
    t_begin = tile0 + split * tps;
    t_end = min(tile0 + n_tiles, t_begin + tps);
    // the pages of this split's keys -> LDS, so that no tile waits for a table entry from memory
    page0 = cw_page_index<POW2>(t_begin * 32, bs, sh);
    const int last_key = min(pos, t_end * 32 - 1);
    const int n_pages = t_end > t_begin ? cw_page_index<POW2>(last_key, bs, sh) - page0 + 1 : 0;
    if (in_lds)
      for (int i = threadIdx.x; i < n_pages; i += WAVES * 64) tbl[i] = table[page0 + i];
  }
  __syncthreads();

  // query fragments (B operand): lane (c, s) holds head c, elements (j * 4 + s) * 8 .. + 7
  bf16x8_t qf[NF];
  const int hig = chunk * gh + c;
  const bool head_ok = c < gh && hig < group;
  {
    const bf16_t* qrow = head_ok ? (const bf16_t*)p.q + (int64_t)(q_begin + tok0) * p.q_stride + (kvh * group + hig) * HD : zrow;
#pragma unroll
    for (int j = 0; j < NF; ++j) qf[j] = *reinterpret_cast<const bf16x8_t*>(qrow + (j * 4 + s) * 8);
  }
  // tile t into the wave's LDS; a masked key is read from a row of zeros
  unsigned char* const region = dec_smem + wave * Tile::BYTES;
  // lines: granule g of key k lies in slot g ^ (k >> 1 & 7) of its 128 bytes, of a value pair g / 2 of granules in pair g / 2 ^ (k >> 1 & 3)
  const bool lines = LINES && __builtin_amdgcn_readfirstlane(shared_s) == 0;
  const int f_key = lane >> 2;
  const int k_piece = (lines ? (lane & 7) ^ (lane >> 4) : k_granule(f_key, lane & 3)) * 8;
  const int v_piece = (lines ? ((((lane >> 1) ^ (lane >> 4)) & 3) << 1 | (lane & 1)) : v_granule(f_key, lane & 3)) * 8;
  auto bring_by = [&](auto whole, int t) __attribute__((always_inline)) {
    constexpr bool WHOLE = decltype(whole)::value;
#pragma unroll
    for (int part = 0; part < (WHOLE ? 4 : 2); ++part) {  // of 8 keys or 16
      const int kb = WHOLE ? part >> 1 : part, h = WHOLE ? part & 1 : 0;
      const int kp = t * 32 + (WHOLE ? part * 8 + (lane >> 3) : part * 16 + f_key);
      const bool ok = kp >= lo && kp <= pos;
      const int at = ok ? cw_page_index<POW2>(kp, bs, sh) - page0 : 0;
      const int page = in_lds ? tbl[at] : ok ? table[page0 + at] : -1;
      const bool have = ok && page >= 0;
      const int64_t off = (((int64_t)page * bs + cw_page_offset<POW2>(kp, bs, sh)) * p.nkv + kvh) * HD;
      const bf16_t* kr = (have ? kc + off : zrow) + (WHOLE ? k_piece ^ (h * 32) : k_piece);
      const bf16_t* vr = (have ? vc + off : zrow) + v_piece;
      unsigned char* const to = region + kb * NF * 1024 + h * 1024;
      if constexpr (WHOLE) {
        lines_to_lds(kr, to, std::make_integer_sequence<int, NF / 2>{});
        lines_to_lds(vr, to + Tile::BYTES / 2, std::make_integer_sequence<int, NF / 2>{});
      } else {
        row_to_lds(kr, to, std::make_integer_sequence<int, NF>{});
        row_to_lds(vr, to + Tile::BYTES / 2, std::make_integer_sequence<int, NF>{});
      }
    }
  };
  auto bring = [&](int t) __attribute__((always_inline)) {
    if constexpr (LINES)
      if (lines) return bring_by(std::true_type{}, t);
    bring_by(std::false_type{}, t);
  };
  // where a lane finds its operands: of two steps of the head, or of four blocks of 16 elements, 2 KB each
  const int v_key = 4 * s + (c >> 2);
  const int k0 = lines ? c * 128 + (s ^ (c >> 1)) * 16 : c * 64 + k_granule(c, s) * 16, k1 = lines ? k0 ^ 64 : k0 + 1024;
  const int v_base = (lines ? v_key * 128 + ((v_key >> 1) & 3) * 32 : v_key * 64 + v_granule(v_key, 0) * 16) + (c & 3) * 8;
  const int v_at[4] = {v_base, v_base ^ 32, lines ? v_base ^ 64 : v_base + 1024, lines ? v_base ^ 96 : (v_base ^ 32) + 1024};
  auto k_in = [&](int j) __attribute__((always_inline)) { return (j >> 1) * 2048 + (j & 1 ? k1 : k0); };  // step j of the head
  auto v_in = [&](int db) __attribute__((always_inline)) { return (db >> 2) * 2048 + v_at[db & 3]; };

  f32x4_t o[ND];
#pragma unroll
  for (int db = 0; db < ND; ++db) o[db] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -INFINITY, l_run = 0.0f;  // of head c, the same in all four lane groups
  if (t_begin + wave < t_end) bring(t_begin + wave);
  // the query is home, too: a wait for it inside the loop would be one for the tile on its way
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  for (int t = t_begin + wave; t < t_end; t += WAVES) {
    const int kv0 = t * 32;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the wave's own loads: its tile is in LDS
    asm volatile("" ::: "memory");
    bf16x8_t kf[2][NF], vt[ND];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int j = 0; j < NF; ++j) kf[kb][j] = *reinterpret_cast<const bf16x8_t*>(region + kb * NF * 1024 + k_in(j));
#pragma unroll
    for (int db = 0; db < ND; ++db) {
      unsigned char* vp = region + Tile::BYTES / 2 + v_in(db);
      const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)vp);
      const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vp + NF * 1024));
      vt[db] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    if (t + WAVES < t_end) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the tile has been read
      asm volatile("" ::: "memory");
      bring(t + WAVES);
    }
    // ---- S^T = K Q^T, keys 4s..4s+3 of each 16-key block for head c
    float sv[8];
    float tmax = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x4_t sc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < NF; ++j) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][j], qf[j], sc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kp = kv0 + kb * 16 + 4 * s + i;
        float v = sc[i] * p.scale;
        if (CAP) v = p.softcap * tanhf(v / p.softcap);
        v = (kp >= lo && kp <= pos) ? v : -INFINITY;
        sv[kb * 4 + i] = v;
        tmax = fmaxf(tmax, v);
      }
    }
    tmax = cw_quad_max(tmax);
    const float m_new = fmaxf(m_run, tmax);
    float alpha = 1.0f, psum = 0.0f;
    bf16x8_t pf;
#pragma unroll
    for (int e = 0; e < 8; ++e) pf[e] = (__bf16)0.0f;
    if (m_new != -INFINITY) {
      alpha = __expf(m_run - m_new);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float pe = __expf(sv[e] - m_new);
        psum += pe;
        pf[e] = (__bf16)pe;
      }
    }
    psum = cw_quad_sum(psum);
    l_run = l_run * alpha + psum;
    m_run = m_new;
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int db = 0; db < ND; ++db) o[db] *= alpha;
    }
    // ---- O^T += V^T P^T
#pragma unroll
    for (int db = 0; db < ND; ++db) o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt[db], pf, o[db], 0, 0, 0);
  }

  // a context beyond the fixed key ranges (the caller promised there is none) must not pass for a result
  if (p.split_keys > 0 && pos >= p.n_splits * p.split_keys) l_run = NAN;
  // ---- merge the waves: [head c][d] over the wave's tiles, lane (c, s) holds d = db * 16 + 4s .. + 3
  if (s == 0) { M_s[wave][c] = m_run; L_s[wave][c] = l_run; }
  float* const mine = reinterpret_cast<float*>(region);
#pragma unroll
  for (int db = 0; db < ND; ++db) *reinterpret_cast<f32x4_t*>(&mine[c * HD + db * 16 + 4 * s]) = o[db];
  __syncthreads();
  const int64_t base = ((int64_t)item * (p.nkv * p.n_chunks) + y) * p.n_splits + split;
  for (int idx = threadIdx.x; idx < gh * (HD / 4); idx += WAVES * 64) {
    const int g = idx / (HD / 4), d = (idx - g * (HD / 4)) * 4;
    const int hg = chunk * gh + g;
    if (hg >= group) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) M = fmaxf(M, M_s[w][g]);
    float L = 0.0f;
    f32x4_t O = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float mw = M_s[w][g];
      const float wgt = mw == -INFINITY ? 0.0f : __expf(mw - M);
      L = fmaf(L_s[w][g], wgt, L);
      O += *reinterpret_cast<const f32x4_t*>(dec_smem + w * Tile::BYTES + (g * HD + d) * 4) * wgt;
    }
    if (p.n_splits == 1) {
      const float scale = attn_head_gate(p, q_begin + tok0, kvh * group + hg) / L;
      bf16_t* const out = (bf16_t*)p.out + (int64_t)(q_begin + tok0) * p.out_stride + (kvh * group + hg) * HD + d;
      if (((uintptr_t)p.out & 7) == 0 && (p.out_stride & 3) == 0) {
        *reinterpret_cast<uint2*>(out) = make_uint2((uint32_t)cw_float_to_bf16_bits(O[0] * scale) | ((uint32_t)cw_float_to_bf16_bits(O[1] * scale) << 16),
                                                    (uint32_t)cw_float_to_bf16_bits(O[2] * scale) | ((uint32_t)cw_float_to_bf16_bits(O[3] * scale) << 16));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = cw_from_float<bf16_t>(O[e] * scale);
      }
    } else {
      float* const out = p.part_o + (base * gh + g) * HD + d;  // (8 bytes aligned)
      *reinterpret_cast<float2*>(out) = make_float2(O[0], O[1]);
      *reinterpret_cast<float2*>(out + 2) = make_float2(O[2], O[3]);
      if (d == 0) {
        p.part_ml[(base * gh + g) * 2] = M;
        p.part_ml[(base * gh + g) * 2 + 1] = L;
      }
    }
  }
}

template <int HD, bool POW2, int WAVES, bool CAP, bool LINES>
__global__ __launch_bounds__(WAVES * 64) void attn_decode_bf16_kernel(AttnParams p) {
  attn_decode_of<HD, POW2, WAVES, CAP, LINES>(p, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Merge of the decode kernel's splits: one wave per (item, head, EL elements of the head). EL / 4 lanes take a split's
// output, four elements each, so a wave reads 64 / (EL / 4) splits at a time, eight times on their way: whole heads where
// that is all splits, else 32 elements, of which 64 splits come at once. Lane l holds the statistics of splits l, l + 64, ...
// (STATS of them). The kernel is bound by its one trip to memory (outputs and statistics are asked for together), by the
// exchange between lanes and by its own code: no LDS, no barrier, no loop over single splits. Decode steps on an MI355X, before
// (threads of a head element each, statistics through LDS) -> now: 8 requests of the 1.5B shape 1465 -> 1445 us, 64 requests
// 2379 -> 2359, 8 of the 7B shape 3410 -> 3392.
#define DEC_MAX_SPLITS 256
typedef float dec_f32x4_t __attribute__((ext_vector_type(4), aligned(8)));  // the workspace is a multiple of 8 bytes away

template <int HD, int EL, int STATS>
__global__ __launch_bounds__(64) void attn_decode_merge_kernel(AttnParams p) {
  constexpr int LPS = EL / 4, SPP = 64 / LPS;
  const int lane = threadIdx.x, sub = lane / LPS, read = min(sub, SPP - 1), d = blockIdx.z % (HD / EL) * EL + (lane - sub * LPS) * 4;
  const int gh = p.gh, n = p.n_splits;
  const int item = blockIdx.x, y = blockIdx.y, g = blockIdx.z / (HD / EL);
  int kvh = y, group = gh, hg = g;
  if (p.n_chunks > 1) {
    kvh = y / p.n_chunks;
    group = p.nh / p.nkv;
    hg = (y - kvh * p.n_chunks) * gh + g;
    if (hg >= group) return;
  }
  const int64_t first = (((int64_t)item * gridDim.y + y) * n) * gh + g;  // split 0; the next ones lie gh rows further each
  const float* const po = p.part_o + first * HD + (read * (gh * HD) + d);
  const float* const pm = p.part_ml + first * 2;
  dec_f32x4_t part[8];
  auto load_parts = [&](int sp0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int at = sp0 + u * SPP;  // lanes past the last split read one that is there, and drop it
      if (at < n) part[u] = *reinterpret_cast<const dec_f32x4_t*>(po + (int64_t)(at + read < n ? at : at - read) * (gh * HD));
    }
  };
  load_parts(0);
  float w[STATS], l[STATS], M = -INFINITY;
#pragma unroll
  for (int k = 0; k < STATS; ++k) {
    const int sp = k * 64 + lane;
    w[k] = -INFINITY;
    l[k] = 0.0f;
    if (sp < n) {
      const float2 ml = *reinterpret_cast<const float2*>(pm + sp * (2 * gh));
      w[k] = ml.x;
      l[k] = ml.y;
    }
  }
  const int64_t token = p.identity != 0 ? item : p.cu_q[p.items[4 * item]] + p.items[4 * item + 1];
  const float gate = attn_head_gate(p, token, kvh * group + hg);
#pragma unroll
  for (int k = 0; k < STATS; ++k) M = fmaxf(M, w[k]);
  M = cw_wave_max(M);
  float L = 0.0f;
#pragma unroll
  for (int k = 0; k < STATS; ++k) {
    w[k] = w[k] == -INFINITY ? 0.0f : __expf(w[k] - M);
    L = fmaf(l[k], w[k], L);
  }
  L = cw_wave_sum(L);
  dec_f32x4_t O = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int sp0 = 0; sp0 < n; sp0 += 8 * SPP) {
    if (STATS > 1 && sp0 > 0) load_parts(sp0);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int at = sp0 + u * SPP;
      if (at < n) {
        float held = w[0];
#pragma unroll
        for (int k = 1; k < STATS; ++k) held = at >> 6 == k ? w[k] : held;
        const float weight = __shfl(held, (at + sub) & 63);
        if (sub < SPP && at + sub < n) O += part[u] * weight;
      }
    }
  }
  dec_f32x4_t total = O;
#pragma unroll
  for (int z = 1; z < SPP; ++z)
#pragma unroll
    for (int e = 0; e < 4; ++e) total[e] += __shfl(O[e], (lane + z * LPS) & 63);
  if (sub > 0) return;
  const float scale = gate / L;
  bf16_t* const out = (bf16_t*)p.out + token * p.out_stride + (kvh * group + hg) * HD + d;
  if (((uintptr_t)p.out & 7) == 0 && (p.out_stride & 3) == 0) {
    *reinterpret_cast<uint2*>(out) = make_uint2((uint32_t)cw_float_to_bf16_bits(total[0] * scale) | ((uint32_t)cw_float_to_bf16_bits(total[1] * scale) << 16),
                                                (uint32_t)cw_float_to_bf16_bits(total[2] * scale) | ((uint32_t)cw_float_to_bf16_bits(total[3] * scale) << 16));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = cw_from_float<bf16_t>(total[e] * scale);
  }
}

#if CW_HD % 32 == 0
#define CW_HAS_DECODE 1
#else
#define CW_HAS_DECODE 0
#endif

// 1 when this head size has the bfloat16 decode kernel (multiples of 32).
CW_EXPORT int cw_attention_decode_supported() { return CW_HAS_DECODE; }

// The most splits cw_attention_decode_bf16 takes.
CW_EXPORT int cw_attention_decode_max_splits() { return DEC_MAX_SPLITS; }

// Heads of a group one workgroup of the decode kernel takes, for a group of this size.
CW_EXPORT int cw_attention_decode_gh(int group) { return group < 16 ? group : 16; }

CW_EXPORT int64_t cw_attention_decode_workspace_floats(int n_items, int nh, int nkv, int n_splits) {
  if (n_splits <= 1) return 0;
  const int group = nh / nkv;
  const int gh = cw_attention_decode_gh(group);
  const int n_chunks = (group + gh - 1) / gh;
  return (int64_t)n_items * nkv * n_chunks * n_splits * gh * (CW_HD + 2);
}

#if CW_HAS_DECODE
// The most pages of a split that are taken by this many waves: 160 KB less 16 rows of float32 a wave. (Pages beyond
// what LDS holds beside the tiles are looked up in memory, so the kernel itself would take any number; four waves' bound is
// what the entries refuse beyond, eight waves' where four take over.)
static constexpr int64_t decode_pages_most(int waves) { return (160 * 1024 - (int64_t)sizeof(float) * waves * 16 * CW_HD) / (int64_t)sizeof(int); }
static bool decode_pages_ok(int waves, int64_t pages) { return pages <= decode_pages_most(waves); }

// Dynamic LDS of a workgroup of single tokens at most: 160 KB less the waves' statistics.
#define DEC_MOST_LDS (158 * 1024)

// Pages of a split that lie in LDS beside ``tiles`` bytes: all of them, or -1.
static int decode_pages_in_lds(size_t tiles, int64_t pages) {
  return tiles + sizeof(int) * (size_t)pages <= DEC_MOST_LDS ? (int)pages : -1;
}

static void launch_decode_merge(const AttnParams& p, int n_items, hipStream_t stream) {
  constexpr int HD = CW_HD;
  if (p.n_splits > 1) {
    const dim3 heads(n_items, p.nkv * p.n_chunks, p.gh), pieces(heads.x, heads.y, heads.z * (HD / 32));
    if (p.n_splits <= 8 * (256 / HD))  // whole heads while all splits come in one go
      hipLaunchKernelGGL((attn_decode_merge_kernel<HD, HD, 1>), heads, dim3(64), 0, stream, p);
    else if (p.n_splits <= 64)
      hipLaunchKernelGGL((attn_decode_merge_kernel<HD, 32, 1>), pieces, dim3(64), 0, stream, p);
    else
      hipLaunchKernelGGL((attn_decode_merge_kernel<HD, 32, DEC_MAX_SPLITS / 64>), pieces, dim3(64), 0, stream, p);
  }
}

template <bool POW2, int WAVES, bool CAP>
static int launch_decode_of(AttnParams& p, int n_items, hipStream_t stream) {
  constexpr int HD = CW_HD;
  // keys of a split: at most ceil(tiles / splits) tiles of 32; their pages go to LDS
  const int64_t max_tiles = ((int64_t)p.table_stride * p.block_size + 31) / 32;
  const int64_t tiles_per_split = p.split_keys > 0 ? p.split_keys / 32 : (max_tiles + p.n_splits - 1) / p.n_splits;
  const int64_t pages = (tiles_per_split * 32 + p.block_size - 1) / p.block_size + 2;
  if (!decode_pages_ok(WAVES, pages)) return CW_ERR_SIZE;
  constexpr size_t tiles = (size_t)WAVES * DecodeTile<HD>::BYTES;
  static_assert(tiles <= DEC_MOST_LDS, "the waves' tiles fit LDS");
  p.decode_pages = decode_pages_in_lds(tiles, pages);
  const size_t smem = tiles + (p.decode_pages > 0 ? sizeof(int) * (size_t)p.decode_pages : 0);
  dim3 grid(n_items, p.nkv * p.n_chunks, p.n_splits), block(WAVES * 64);
  auto launch = [&](auto kernel, std::atomic<bool>& allowed) -> int {
    if (cw_allow_lds(allowed, (const void*)kernel, DEC_MOST_LDS) != CW_OK) return CW_ERR_LAUNCH;
    hipLaunchKernelGGL(kernel, grid, block, smem, stream, p);
    return CW_OK;
  };
  static std::atomic<bool> allowed[2];
  // whole lines where the card is as good as full of workgroups of 256 keys and more each, at places that they know before the context's
  // length (the look for the same page elsewhere costs no trip of its own then): see attn_decode_of
  int status = CW_OK;
  if constexpr (HD == 128 && WAVES == 8) {
    const bool lines = p.identity && p.split_keys >= 256 && p.n_chunks == 1 && (int64_t)n_items * p.nkv * p.n_splits >= 192;
    status = lines ? launch(attn_decode_bf16_kernel<HD, POW2, WAVES, CAP, true>, allowed[1]) : launch(attn_decode_bf16_kernel<HD, POW2, WAVES, CAP, false>, allowed[0]);
  } else {
    status = launch(attn_decode_bf16_kernel<HD, POW2, WAVES, CAP, false>, allowed[0]);
  }
  if (status != CW_OK) return status;
  launch_decode_merge(p, n_items, stream);
  return cw_launch_status();
}

template <int WAVES>
static int launch_decode(AttnParams& p, int n_items, hipStream_t stream) {
  if (p.softcap > 0.0f) return p.bs_shift >= 0 ? launch_decode_of<true, WAVES, true>(p, n_items, stream) : launch_decode_of<false, WAVES, true>(p, n_items, stream);
  return p.bs_shift >= 0 ? launch_decode_of<true, WAVES, false>(p, n_items, stream) : launch_decode_of<false, WAVES, false>(p, n_items, stream);
}
#endif

#if CW_HAS_DECODE
// The decode kernel's parameters from its entry points' arguments, checked.
static int decode_params(AttnParams& p, const void* q, int64_t q_stride, void* out, int64_t out_stride,
                                       const void* k_cache, const void* v_cache, const int* block_tables,
                                       int table_stride, const int* ctx_lens, const int* cu_q,
                                       const int* items, int n_items, int nh, int nkv, int block_size,
                                       int n_splits, int window, float scale, float* workspace,
                                       int64_t workspace_floats, const void* zeros, int identity,
                                       int split_keys, int max_ctx, float softcap, const void* gate, int64_t gate_stride,
                                       int gate_off) {
  if (n_items < 0 || nh <= 0 || nkv <= 0 || nh % nkv != 0 || block_size <= 0 || table_stride <= 0)
    return CW_ERR_ARG;
  if (n_splits < 1 || n_splits > DEC_MAX_SPLITS || window < 0) return CW_ERR_ARG;
  if (((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15) || (q_stride & 7))
    return CW_ERR_ARG;
  if (zeros == nullptr || ((uintptr_t)zeros & 15)) return CW_ERR_ARG;
  // fixed key ranges must cover the longest context the caller will run
  if (split_keys < 0 || (split_keys & 31) || max_ctx < 0) return CW_ERR_ARG;
  if (split_keys > 0 && (int64_t)split_keys * n_splits < max_ctx) return CW_ERR_ARG;
  const int group = nh / nkv;
  p.q = q; p.q_stride = q_stride; p.out = out; p.out_stride = out_stride;
  p.k_cache = k_cache; p.v_cache = v_cache; p.block_tables = block_tables;
  p.table_stride = table_stride; p.ctx_lens = ctx_lens; p.cu_q = cu_q; p.items = items;
  p.nh = nh; p.nkv = nkv; p.block_size = block_size; p.bs_shift = cw_log2_or_minus1(block_size);
  p.identity = identity ? 1 : 0; p.split_keys = split_keys;
  if (gate && (gate_off < 0 || gate_off + nh > gate_stride)) return CW_ERR_ARG;
  p.gate = gate; p.gate_stride = gate_stride; p.gate_off = gate_off;
  p.gh = cw_attention_decode_gh(group);
  p.n_chunks = (group + p.gh - 1) / p.gh; p.n_splits = n_splits; p.window = window; p.scale = scale; p.softcap = softcap;
  if ((int64_t)nkv * p.n_chunks * p.gh > 65535) return CW_ERR_SIZE;
  const int64_t need = cw_attention_decode_workspace_floats(n_items, nh, nkv, n_splits);
  if (need > 0 && (workspace == nullptr || workspace_floats < need)) return CW_ERR_ARG;
  if ((uintptr_t)workspace & 7) return CW_ERR_ARG;
  p.part_o = workspace;
  p.part_ml = workspace ? workspace + need / (CW_HD + 2) * CW_HD : nullptr;
  p.zeros = zeros;
  return CW_OK;
}
#endif

// Single-token items (every item: one token), bfloat16. Same arguments as cw_attention;
// ``zeros``: at least CW_HD zero elements (16-byte aligned) that masked rows are read from.
// ``identity``: item i is request i and its token is row i (a batch of single tokens only): items
// and cu_q are not read. ``split_keys`` > 0 (a multiple of 32): split s takes keys
// [s * split_keys, (s + 1) * split_keys) instead of a share of each request's own length, and
// ``max_ctx``, the longest context among the requests, must not exceed n_splits * split_keys.
CW_EXPORT int cw_attention_decode_bf16(const void* q, int64_t q_stride, void* out, int64_t out_stride,
                                       const void* k_cache, const void* v_cache, const int* block_tables,
                                       int table_stride, const int* ctx_lens, const int* cu_q,
                                       const int* items, int n_items, int nh, int nkv, int block_size,
                                       int n_splits, int window, float scale, float* workspace,
                                       int64_t workspace_floats, const void* zeros, int identity,
                                       int split_keys, int max_ctx, float softcap, const void* gate, int64_t gate_stride,
                                       int gate_off, hipStream_t stream) {
#if CW_HAS_DECODE
  AttnParams p{};
  const int status = decode_params(p, q, q_stride, out, out_stride, k_cache, v_cache, block_tables, table_stride, ctx_lens, cu_q, items, n_items, nh, nkv, block_size, n_splits, window, scale, workspace, workspace_floats, zeros, identity, split_keys, max_ctx, softcap, gate, gate_stride, gate_off);
  if (status != CW_OK || n_items == 0) return status;
  // what a split's keys are shared among: the most keys a split may have, by the caller's fixed places or by its table
  const int64_t keys = split_keys > 0 ? split_keys : ((int64_t)table_stride * block_size + n_splits - 1) / n_splits;
  // more than four waves can have on their way at once: eight (larger heads' tiles have no room for them)
  if constexpr (CW_HD <= 128)
    if (keys > 128 && decode_pages_ok(8, (keys + 63) / block_size + 3)) return launch_decode<8>(p, n_items, stream);
  return launch_decode<4>(p, n_items, stream);
#else
  return CW_ERR_ARG;
#endif
}

// =====================================================================================
// bfloat16 attention for portions of prompts on the matrix cores.
//
// A workgroup takes a run of query tokens of one request and one key/value head. A wave owns 32 query
// rows (row = token * gh + head of the group, so the group shares every key and value); NH sets of waves
// own the same rows and each set takes its share of a stage's keys. The sets' running states are
// put together through LDS at the end.
//   S^T[key, row] = K * Q^T     v_mfma_f32_16x16x32_bf16; K fragments come from LDS in operand
//                               layout (lane = key l%16, 8 consecutive head elements at slot l/16),
//                               Q fragments are loaded once from global memory the same way;
//   softmax per row in float32: a lane holds 8 or 16 keys of one row; the running maximum is shared by
//                               the row's 4 lanes every stage, the running sum only at the end;
//                               stages that no row masks skip the position tests;
//   O^T[d, row] += V^T * P^T    P^T is already in operand layout (the lane's keys of its row).
//                               V^T fragments come from the row-major V tile through the LDS
//                               transposing read (ds_read_b64_tr_b16): in a group of 16 lanes, lane
//                               i receives element i%4 of what lanes i/4, 4 + i/4, 8 + i/4 and
//                               12 + i/4 addressed, so four lanes that point at one key's 16 head
//                               elements hand every lane its column of 4 keys.
// The element order inside an MFMA's k dimension is free as long as both operands agree; that
// is what lets every fragment be filled by plain 8- and 16-byte reads.
//
// What bounds it: a SIMD's vector unit (an exponential, a fused multiply-add, an addition, a maximum and half a conversion a
// score, some 450 cycles a wave and 32 x 32 scores) beside its matrix instructions (512 cycles); 128 bytes a cycle out of LDS
// feed one such product, so operands of 32 rows a wave ask for as much as LDS gives. Hence: loads go straight into
// LDS with addresses made by the scalar unit (addresses a lane, stores and page look-ups cost as much vector time as
// half the softmax), the row's reference point is looked up in other lanes only when it moves, operand reads run
// ahead of the products in a written order, and the two waves of a SIMD are half an interval apart. Measured on an MI355X, before
// (tiles through registers, all waves in step) -> now: 2048 tokens of 12 heads of 128 on 2 behind 6144, 164 -> 117 us
// (0.77 PFLOP/s on 196 compute units); of 28 on 4, 319 -> 222 (0.95; 233 with every wave's rows in whole tokens, 28 of 32 for
// groups of 7); 2048 tokens without a prefix 43 -> 31; 137 tokens 11.7 -> 9.0; 1000 tokens of 14 heads of 64 behind 7000, 69 -> 50;
// of 16 of 256 on 4 behind 4000, 218 -> 143.
// RB: row blocks (waves that own 32 query rows each) of a workgroup, 4 or 2. With 2 the same eight
// waves cut a stage's keys four ways instead of two: half the rows per workgroup and half the
// time per stage, for launches whose portions would otherwise leave compute units without work
// and wait for the workgroups with the longest key ranges.
template <int HD, int RB>
struct PrefillTile {
  static_assert(RB == 4 || (RB == 2 && HD <= 128), "two row blocks only with the eight-wave workgroup");
  static constexpr int NH = HD <= 128 ? 8 / RB : 1;     // sets of waves: they share a row block and split its keys
  static constexpr int KW = HD <= 128 && RB == 4 ? 64 : 32;  // keys a wave takes from a stage
  static constexpr int KT = KW * NH;                    // keys of one stage
  static constexpr int WAVES = RB * NH;
  static constexpr int NT = 64 * WAVES;                 // threads of a workgroup
  // A K or V tile lies in LDS as blocks of 16 keys x 32 elements (1 KB: what one load of a wave with the
  // LDS target brings), [16-key group][32 elements]. Inside a block a key's four 16-byte granules are
  // permuted (k_granule, v_granule) so that no bank is hit twice when operands are read.
  static constexpr int TILE = KT * HD * 2;              // bytes of a tile
  static constexpr size_t TILES = 4 * (size_t)TILE;     // two of K, two of V
  // what the sets of waves exchange at the end: accumulators of all sets, then maxima and sums
  static constexpr size_t XO_BYTES = NH > 1 ? (size_t)NH * RB * 2 * (HD / 16) * 64 * 16 : 0;
  static constexpr size_t XCHG_BYTES = XO_BYTES + (NH > 1 ? (size_t)NH * RB * 2 * 2 * 64 * 4 : 0);
  static constexpr size_t BYTES = TILES > XCHG_BYTES ? TILES : XCHG_BYTES;
};

// PAGES16: a page holds 2^n keys, 16 or more, so that 16 keys of a stage lie in one page
template <int HD, bool PAGES16, int RB, bool CAP>
__device__ __forceinline__ void attn_prefill_of(const AttnParams& p, const int item, const int y) {
  using Tile = PrefillTile<HD, RB>;
  constexpr int NF = HD / 32;     // k-steps of the score product, blocks of 32 elements of a row
  constexpr int ND = HD / 16;     // 16-wide blocks of the head dimension
  constexpr int NH = Tile::NH, KW = Tile::KW, KT = Tile::KT;
  constexpr int NKB = KW / 16;    // 16-key blocks of a wave's keys
  extern __shared__ __align__(1024) unsigned char smem_raw[];  // K tiles 0 and 1, V tiles 0 and 1

  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wid % RB;  // the wave's row block
  const int half = wid / RB;  // its share of a stage's keys
  const int c = lane & 15, s = lane >> 4;
  const int kvh = y / p.n_chunks, chunk = y % p.n_chunks;
  const int req = p.items[4 * item], tok0 = p.items[4 * item + 1];
  const int gh = p.gh;
  const int ctx = p.ctx_lens[req];
  const int q_begin = p.cu_q[req];
  const int qlen = p.cu_q[req + 1] - q_begin;
  // an item may reach past the request's tokens (work items laid out for a longer portion than
  // the step brings): what lies past them is not computed
  const int ntok = min(p.items[4 * item + 2], qlen - tok0);
  if (ntok <= 0) return;
  const int group = p.nh / p.nkv;
  const int pos0 = ctx - qlen + tok0;
  const int wg_last = pos0 + ntok - 1;
  const int wg_lo = p.window > 0 ? max(0, pos0 - p.window + 1) : 0;
  const int bs = p.block_size, sh = p.bs_shift;
  // the stages of keys this workgroup walks: all that its rows see, or one of ``parts`` runs of
  // them when the item's key range is shared among workgroups (the merge kernel puts the parts'
  // results together); a part may be empty
  int t_first = wg_lo / KT, t_last = wg_last / KT;
  const int packed = p.items[4 * item + 3];
  const int parts = p.part_o != nullptr ? max(1, (packed >> 8) & 0xff) : 1;  // no workspace: every part is the whole
  const int part = packed & 0xff;
  if (parts > 1) {
    const int per = (t_last - t_first + parts) / parts;
    t_first += part * per;
    t_last = min(t_last, t_first + per - 1);
  }

  // ---- tile traffic. A wave brings 16 keys of a stage (all of their blocks, or every other one where the stage has
  // fewer groups of keys than waves): lane l takes granule l % 4 of key l / 4, four lanes 64 bytes of one row.
  // (constant memory for the kernel: a page's number that all lanes want comes by the scalar unit)
  const __attribute__((address_space(4))) int* const table =
      (const __attribute__((address_space(4))) int*)(p.block_tables + (int64_t)req * p.table_stride);
  constexpr int KG = KT / 16, SHARE = Tile::WAVES / KG;  // groups of 16 keys of a stage, waves that share one
  static_assert(Tile::WAVES % KG == 0, "a whole number of waves a group of keys");
  const int kg = wid % KG, sub = wid / KG;
  const int f_key = kg * 16 + (lane >> 2);
  const int row_elems = p.nkv * HD;
  const bf16_t* const kc = (const bf16_t*)p.k_cache + kvh * HD;
  const bf16_t* const vc = (const bf16_t*)p.v_cache + kvh * HD;
  const bf16_t* const zrow = (const bf16_t*)p.zeros;
  const int k_piece = k_granule(lane >> 2, lane & 3) * 8, v_piece = v_granule(lane >> 2, lane & 3) * 8;
  // A key that no row sees (past the last token, or before the window's first key) is brought as its neighbour that
  // some row sees: it is masked by its position. With whole pages a wave's 16 keys have one page and one address, and a
  // lane an offset; else every lane has an address of its own. No page: zeros; and zeros for the values of a key that no
  // row sees (a weight of zero times a neighbour's infinite value would be no zero).
  auto group_of = [&](int t) __attribute__((always_inline)) { return min(max(t * KT + kg * 16, wg_lo & ~15), wg_last & ~15); };
  auto key_of = [&](int t) __attribute__((always_inline)) { return min(max(t * KT + f_key, wg_lo), wg_last); };
  auto page_of = [&](int t) __attribute__((always_inline)) {
    return PAGES16 ? table[group_of(t) >> sh] : table[cw_page_index<false>(key_of(t), bs, sh)];
  };
  int64_t at_row = 0;   // in elements from the head's first: PAGES16 the row of the group's first key, else of the lane's key
  int at_key = 0;       // PAGES16: the lane's row in the group, in elements
  bool at_page = false;
  int at_first = 0;     // the group's first key, whoever sees it
  auto aim = [&](int t, int page) __attribute__((always_inline)) {
    at_page = page >= 0;
    at_first = t * KT + kg * 16;
    if constexpr (PAGES16) {
      const int g = group_of(t);
      at_row = (int64_t)(((uint64_t)(uint32_t)page * (uint32_t)bs + (uint32_t)(g & (bs - 1))) * (uint32_t)row_elems);
      at_key = min(max(lane >> 2, wg_lo - g), wg_last - g) * (at_page ? row_elems : 0);
    } else {
      const uint32_t slot = (uint32_t)page * (uint32_t)bs + (uint32_t)cw_page_offset<false>(key_of(t), bs, sh);
      at_row = (int64_t)((uint64_t)slot * (uint32_t)row_elems);
    }
  };
  auto bring = [&](const bf16_t* head, int piece, int tile, auto values) __attribute__((always_inline)) {  // the wave's blocks of a tile
    auto blocks = [&](auto&& load) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < (NF + SHARE - 1) / SHARE; ++j) {
        const int blk = j * SHARE + sub;
        if (NF % SHARE == 0 || blk < NF) load(blk * 32, smem_raw + tile * Tile::TILE + (kg * NF + blk) * 1024);
      }
    };
    const int key = at_first + (lane >> 2);
    const bool seen = !decltype(values)::value || (key >= wg_lo && key <= wg_last);
    if (!PAGES16 || (decltype(values)::value && (at_first < wg_lo || at_first + 15 > wg_last))) {
      const bf16_t* const from = (at_page && seen ? head + at_row + (PAGES16 ? at_key : 0) : zrow) + piece;
      blocks([&](int at, unsigned char* to) { load_to_lds(from + at, to); });
    } else {
      const bf16_t* const from = at_page ? head + at_row : zrow;
      blocks([&](int at, unsigned char* to) { load_to_lds(from + at, (uint32_t)(at_key + piece) * 2, to); });
    }
  };

  // ---- the wave's rows: block b, column c -> row wave * 32 + b * 16 + c of the workgroup, token row / gh, head row % gh
  const bool wave_on = wave * 32 < ntok * gh;
  const int p_first = pos0 + wave * 32 / gh;
  const int p_last = pos0 + min(ntok - 1, (wave * 32 + 31) / gh);
  const int lo = p.window > 0 ? max(0, p_first - p.window + 1) : 0;
  int row_pos[2];  // position of the row's token, far below zero for an unused row
  bf16x8_t qf[2][NF];
  int page_a = 0, page_b = 0;
  if (t_first <= t_last) {
    page_a = page_of(t_first);
    page_b = page_of(t_first + 1);
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int row = wave * 32 + b * 16 + c;
    const int tokw = row / gh, hig = chunk * gh + row - tokw * gh;
    const bool ok = tokw < ntok && hig < group;
    row_pos[b] = ok ? pos0 + tokw : INT_MIN / 2;
    const bf16_t* qrow = ok ? (const bf16_t*)p.q + (int64_t)(q_begin + tok0 + tokw) * p.q_stride + (kvh * group + hig) * HD : zrow;
#pragma unroll
    for (int j = 0; j < NF; ++j) qf[b][j] = *reinterpret_cast<const bf16x8_t*>(qrow + (j * 4 + s) * 8);
  }

  f32x4_t o[2][ND];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int db = 0; db < ND; ++db) o[b][db] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
  // The running maximum in units of the raw score (the scale is positive) and the lane's share of the sum; the
  // exponentials' reference point (the maximum times the scale, 0 while no key has been seen); and the score beyond which it moves
  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.0f, 0.0f}, ref[2] = {0.0f, 0.0f}, limit[2] = {-INFINITY, -INFINITY};
  const float sl2 = p.scale * 1.4426950408889634f;  // exp(x * scale) = exp2(x * sl2)
  const float rescale_step = 8.0f / sl2;            // 8 in the exponent, in units of the raw score

  // where a lane's operands lie in a block: of K granule s of key c; of V 8 bytes of key 4 s + c / 4, in the
  // first or the second 16 elements
  const int k_at = c * 64 + k_granule(c, s) * 16;
  const int v_key = 4 * s + (c >> 2);
  const int v_at0 = v_key * 64 + v_granule(v_key, 0) * 16 + (c & 3) * 8, v_at1 = v_at0 ^ 32;

  // the stages in which the wave has rows that see keys of its share
  const int own = half * KW;  // the share's first key in a stage
  const int on_first = max(t_first, (max(0, lo - own - (KW - 1)) + KT - 1) / KT);
  const int on_last = wave_on && p_last >= own ? min(t_last, (p_last - own) / KT) : -1;
  const int all_see = p_first - own - KW + 1;                                         // a stage that begins up to here and
  const int all_hold = p.window > 0 ? max(wg_lo, p_last - p.window + 1) - own : -KT;  // from here on has no masked pair
  const unsigned reach = p.window > 0 ? p.window : 0x7fffffff;                       // a row sees this many keys, its own the last
  f32x4_t sc[NKB][2];
  bf16x8_t pf[2][NKB / 2];
  // The matrix products of an interval: O^T += V^T P^T of stage t - 1, then S^T = K Q^T of stage t, four products at a
  // time, whose two operands from LDS are read DEPTH times four products ahead. The order is the one written here: left to
  // itself the compiler reads two operands, waits for them, multiplies, and so on.
  constexpr int DEPTH = 4;
  auto products = [&](int t, auto with_outputs, auto with_scores) __attribute__((always_inline)) {
    constexpr int OUT = decltype(with_outputs)::value ? NKB / 2 * (ND / 2) : 0;
    constexpr int ALL = OUT + (decltype(with_scores)::value ? NKB / 2 * NF : 0);
    unsigned char* const vs = smem_raw + (2 + ((t - 1 - t_first) & 1)) * Tile::TILE + half * (NKB * NF * 1024);
    const unsigned char* const ks = smem_raw + ((t - t_first) & 1) * Tile::TILE + half * (NKB * NF * 1024) + k_at;
    bf16x8_t f[DEPTH + 1][2];
    auto read = [&](int i) __attribute__((always_inline)) {
      bf16x8_t(&to)[2] = f[i % (DEPTH + 1)];
      if (i < OUT) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {  // 16-wide blocks 2 d and 2 d + 1 of the head dimension
          unsigned char* vp = vs + (u ? v_at1 : v_at0) + (i / (ND / 2) * 2 * NF + i % (ND / 2)) * 1024;
          const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)vp);
          const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vp + NF * 1024));
          to[u] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
        }
      } else {
#pragma unroll
        for (int u = 0; u < 2; ++u)  // 16-key blocks 2 k and 2 k + 1
          to[u] = *reinterpret_cast<const bf16x8_t*>(ks + (((i - OUT) / NF * 2 + u) * NF + (i - OUT) % NF) * 1024);
      }
    };
#pragma unroll
    for (int i = 0; i < (DEPTH < ALL ? DEPTH : ALL); ++i) read(i);
#pragma unroll
    for (int i = 0; i < ALL; ++i) {
      if (i + DEPTH < ALL) read(i + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const bf16x8_t x = f[i % (DEPTH + 1)][u];
          if (i < OUT) {
            f32x4_t& to = o[b][i % (ND / 2) * 2 + u];
            to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, pf[b][i / (ND / 2)], to, 0, 0, 0);
          } else {
            const int j = (i - OUT) % NF;
            f32x4_t& to = sc[(i - OUT) / NF * 2 + u][b];
            to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, qf[b][j], j ? to : (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
          }
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // ---- softmax per row; P^T packed as the B operand of the output product
  auto softmax = [&](int t) __attribute__((always_inline)) {
    if (CAP) {
      // capped scores, kept in units of the raw score: s <- (cap / scale) * tanh(s * scale / cap)
      const float up = p.softcap / p.scale, down = p.scale / p.softcap;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[kb][b][i] = up * tanhf(sc[kb][b][i] * down);
    }
    // a stage needs the position tests only if some row of the wave masks some key of it
    if (t * KT > all_see || t * KT < all_hold) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int behind = row_pos[b] - (t * KT + own + 4 * s);  // the row's distance from the lane's first key
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if ((unsigned)(behind - (kb * 16 + i)) >= reach) sc[kb][b][i] = -INFINITY;
          __builtin_amdgcn_sched_barrier(0);  // (the compiler would make all comparisons first, and spill them)
        }
      }
    }
    // The reference point of the exponentials moves only when the maximum has grown by more
    // than 2^8 in the exponent (or is the row's first): probabilities then reach 256 at most,
    // which float32 sums and bfloat16 products take without loss, and the accumulators are
    // rescaled a few times per row instead of in most stages. The result is the same quotient.
    // (fmed3 with infinity is the maximum without fmaxf's care for signalling NaNs, an instruction a score)
    float most[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      most[b] = sc[0][b][0];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (kb + i > 0) most[b] = __builtin_amdgcn_fmed3f(most[b], sc[kb][b][i], INFINITY);
    }
    if (__any(most[0] > limit[0] || most[1] > limit[1])) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const float top = cw_quad_max(most[b]);
        const bool moves = top > limit[b];
        const float to = moves ? top * sl2 : ref[b];
        // (a row that has seen no key yet has nothing to rescale)
        const float a = !moves || m_run[b] == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(ref[b] - to);
        ref[b] = to;
        m_run[b] = moves ? top : m_run[b];
        limit[b] = moves ? top + rescale_step : limit[b];
        l_run[b] *= a;
#pragma unroll
        for (int db = 0; db < ND; ++db) o[b][db] *= a;
      }
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float psum = 0.0f;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pe = __builtin_amdgcn_exp2f(fmaf(sc[kb][b][i], sl2, -ref[b]));
          psum += pe;
          pf[b][kb / 2][(kb & 1) * 4 + i] = (__bf16)pe;
        }
      l_run[b] += psum;
    }
  };

  // ---- the walk. An interval between two barriers makes the output product of stage t - 1 and the scores and softmax
  // of stage t, while K of stage t + 1 and V of stage t come into the tiles that the interval before has read last.
  // The two waves of a SIMD (sets h and h + NH / 2) would walk through it in step, both in the products, then both in the
  // softmax, each waiting for the unit that the other holds. So the later sets pass the barrier between
  // products and softmax instead of behind the softmax, and one's products run beside the other's softmax.
  const bool late = NH > 1 && half >= NH / 2;
  auto next_interval = [&](int t, int page) __attribute__((always_inline)) {  // the one of stage t begins; the page of stage t + 1
    // vmcnt(0), lgkmcnt(0): this wave's share of K of stage t and of V of stage t - 1 is in LDS, and its reads are back
    __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();        // everyone's is, and the tiles that stage t + 1 comes into have been read
    asm volatile("" ::: "memory");
    if (t > t_last) return;
    if (t > t_first) bring(vc, v_piece, 2 + ((t - t_first) & 1), std::true_type{});
    aim(t + 1, page);  // (behind the last stage: a tile that nobody reads)
    bring(kc, k_piece, (t + 1 - t_first) & 1, std::false_type{});
  };
  if (t_first <= t_last) {
    aim(t_first, page_a);
    bring(kc, k_piece, 0, std::false_type{});
    bring(vc, v_piece, 2, std::true_type{});  // (later V comes one interval after K)
    const bool active = on_first <= on_last;
    const int until = active ? on_first : t_last + 1;
    next_interval(t_first, page_b);
    for (int t = t_first + 1; t <= until; ++t) next_interval(t, page_of(t + 1));
    if (active) {
      products(on_first, std::false_type{}, std::true_type{});
      int page = page_of(on_first + 2);
      for (int t = on_first; t <= on_last; ++t) {
        if (late) next_interval(t + 1, page);
        page = page_of(t + (late ? 3 : 2));  // (here no read of LDS is on its way: with one the wait for either is for both)
        softmax(t);
        if (!late) next_interval(t + 1, page);
        products(t + 1, std::true_type{}, std::true_type{});  // (the last scores go nowhere: one copy of the products keeps
      }                                                        // the accumulators in their registers)
      for (int t = on_last + 2; t <= t_last + 1; ++t) next_interval(t, page_of(t + 1));
    }
  }

  // ---- the sets of waves put their rows' states together through LDS: everyone's accumulators, maxima and sums go
  // there, and each set finishes its share of the head dimension
  constexpr int DB = (ND + NH - 1) / NH;  // 16-wide blocks of the head dimension that a set finishes
  const int db0 = NH > 1 ? half * DB : 0;
  if constexpr (NH > 1) {
    f32x4_t* xo = reinterpret_cast<f32x4_t*>(smem_raw);
    float* xml = reinterpret_cast<float*>(smem_raw + Tile::XO_BYTES);
    cw_lds_barrier();  // the tiles are dead
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int db = 0; db < ND; ++db) xo[(((half * RB + wave) * 2 + b) * ND + db) * 64 + lane] = o[b][db];
      xml[((half * RB + wave) * 2 + b) * 128 + lane] = m_run[b];
      xml[((half * RB + wave) * 2 + b) * 128 + 64 + lane] = l_run[b];
    }
    cw_lds_barrier();
    if (db0 >= ND) return;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float mh[NH], m = -INFINITY, l = 0.0f;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        mh[h] = xml[((h * RB + wave) * 2 + b) * 128 + lane];
        m = fmaxf(m, mh[h]);
      }
      const float msc = m == -INFINITY ? 0.0f : m * sl2;
#pragma unroll
      for (int d = 0; d < DB; ++d) o[b][d] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const float a = __builtin_amdgcn_exp2f(mh[h] * sl2 - msc);
        l += xml[((h * RB + wave) * 2 + b) * 128 + 64 + lane] * a;
#pragma unroll
        for (int d = 0; d < DB; ++d) o[b][d] += xo[(((h * RB + wave) * 2 + b) * ND + db0 + d) * 64 + lane] * a;
      }
      m_run[b] = m;
      l_run[b] = l;
    }
  }
  constexpr int DF = NH > 1 ? DB : ND;  // blocks of the head dimension in o

  // ---- a part of the key range: unnormalised sums, maximum and sum of every row of the workgroup
  // (unused rows too: zeros) for the merge kernel
  if (parts > 1) {
    const int64_t slot = ((int64_t)item * (p.nkv * p.n_chunks) + y) * (RB * 32);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const float l = cw_quad_sum(l_run[b]);
      const int64_t row = slot + wave * 32 + b * 16 + c;
#pragma unroll
      for (int d = 0; d < DF; ++d) *reinterpret_cast<f32x4_t*>(p.part_o + row * HD + (db0 + d) * 16 + 4 * s) = o[b][d];
      if (s == 0 && half == 0) {
        p.part_ml[row * 2] = m_run[b];
        p.part_ml[row * 2 + 1] = l;
      }
    }
    return;
  }

  // ---- out[row][d]: lane (c, s) holds d = db * 16 + 4s .. + 3 of row (b, c)
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float l = l_run[b];
    l = cw_quad_sum(l);
    if (row_pos[b] < 0) continue;
    const int head = kvh * group + chunk * gh + (wave * 32 + b * 16 + c) % gh;
    const int64_t token = q_begin + (row_pos[b] - (ctx - qlen));
    const float inv = attn_head_gate(p, token, head) / l;
    bf16_t* orow = (bf16_t*)p.out + token * p.out_stride + head * HD;
#pragma unroll
    for (int d = 0; d < DF; ++d) {
      uint2 packed;
      packed.x = (uint32_t)cw_float_to_bf16_bits(o[b][d][0] * inv) | ((uint32_t)cw_float_to_bf16_bits(o[b][d][1] * inv) << 16);
      packed.y = (uint32_t)cw_float_to_bf16_bits(o[b][d][2] * inv) | ((uint32_t)cw_float_to_bf16_bits(o[b][d][3] * inv) << 16);
      *reinterpret_cast<uint2*>(orow + (db0 + d) * 16 + 4 * s) = packed;
    }
  }
}

template <int HD, bool PAGES16, int RB, bool CAP>
__global__ __launch_bounds__((PrefillTile<HD, RB>::NT), (HD <= 128 ? 2 : 1)) void attn_prefill_bf16_kernel(AttnParams p) {
  attn_prefill_of<HD, PAGES16, RB, CAP>(p, blockIdx.x, blockIdx.y);
}

#if CW_HD % 32 == 0 && CW_HD <= 128
// A step's portions and its single tokens in one launch: the first workgroups take the portions' items, the others the single
// tokens' splits, eight waves each. One workgroup fits a compute unit, and each launch by itself is bound by its longest
// workgroup's chain of trips to memory: 320 tokens beside 16 requests of 1500 (12 heads of 128 on 2) are 64 workgroups
// and then 256 of some 10 us each; together, 64 and 192, they take little longer than the longer ones (28 layers: 3.30 -> 3.04 ms).
struct AttnBoth {
  AttnParams portions, singles;
  int n_portions, n_singles;  // items of each
};
template <int HD, bool PAGES16, int RB>
__global__ __launch_bounds__((PrefillTile<HD, RB>::NT), 2) void attn_together_bf16_kernel(AttnBoth a) {
  static_assert(PrefillTile<HD, RB>::NT == 512, "both kinds of workgroups have eight waves");
  const int first = a.n_portions * a.portions.nkv * a.portions.n_chunks;
  int b = blockIdx.x;
  if (b < first) {
    attn_prefill_of<HD, PAGES16, RB, false>(a.portions, b % a.n_portions, b / a.n_portions);
  } else {
    b -= first;
    const int of = b / a.n_singles, heads = a.singles.nkv * a.singles.n_chunks;
    attn_decode_of<HD, PAGES16, 8, false>(a.singles, b - of * a.n_singles, of % heads, of / heads);
  }
}
#endif

// Puts together the parts of items whose key range was shared among workgroups. Four workgroups per (item, key/value
// head) of the kernel above (with one a thread had eight rounds of loads: 1000 tokens behind 7000, 14 -> 6 us). The
// workgroups of an item's parts share its rows, each reading its rows of every part. With few rows a workgroup its threads
// also share the parts: thread (row, 4 elements, slice) sums the parts slice, slice + S, ..., and the slices meet in LDS
// in a fixed order.
#define PREFILL_MAX_PARTS 255

template <int HD, int RB>
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(AttnParams p) {
  constexpr int ROWS = RB * 32;
  constexpr int VEC = HD / 4;  // 16-byte pieces of a row
  __shared__ float ms[ROWS + PREFILL_MAX_PARTS + 1], ls[ROWS + PREFILL_MAX_PARTS + 1];
  __shared__ __align__(16) float red[256 * 4];
  const int packed = p.items[4 * blockIdx.x + 3];
  const int parts = (packed >> 8) & 0xff, part = packed & 0xff;
  if (parts <= 1) return;
  const int item = blockIdx.x - part;  // the item's part 0
  const int kvh = blockIdx.y / p.n_chunks, chunk = blockIdx.y % p.n_chunks;
  const int req = p.items[4 * item], tok0 = p.items[4 * item + 1];
  const int gh = p.gh, group = p.nh / p.nkv;
  const int q_begin = p.cu_q[req];
  const int ntok = min(p.items[4 * item + 2], p.cu_q[req + 1] - q_begin - tok0);
  const float sl2 = p.scale * 1.4426950408889634f;
  const int shares = parts * gridDim.z;
  const int rpb = (ROWS + shares - 1) / shares;  // rows of this workgroup
  const int row0 = (part * gridDim.z + blockIdx.z) * rpb;
  if (row0 >= ROWS) return;
  auto slot = [&](int z, int row) { return ((int64_t)(item + z) * gridDim.y + blockIdx.y) * ROWS + row; };
  for (int i = threadIdx.x; i < rpb * parts; i += 256) {
    const int r = i / parts, z = i - r * parts;
    const bool in = row0 + r < ROWS;
    ms[i] = in ? p.part_ml[slot(z, row0 + r) * 2] : -INFINITY;
    ls[i] = in ? p.part_ml[slot(z, row0 + r) * 2 + 1] : 0.0f;
  }
  __syncthreads();
  const int n_pairs = rpb * VEC;                      // (row, 4 elements) pairs of this workgroup
  const int slices = n_pairs >= 256 ? 1 : 256 / n_pairs;
  for (int u0 = 0; u0 < n_pairs * slices; u0 += 256) {  // one round when the parts are shared
    const int u = u0 + threadIdx.x;
    const bool has = u < n_pairs * slices;
    const int pair = has ? u % n_pairs : 0, slice = has ? u / n_pairs : 0;
    const int r = pair / VEC, d = (pair - r * VEC) * 4;
    const int row = row0 + r;
    const int tokw = row / gh, hig = chunk * gh + row - tokw * gh;
    const bool valid = has && row < ROWS && tokw < ntok && hig < group;
    float m = -INFINITY, l = 0.0f;
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    if (valid) {
      for (int z = 0; z < parts; ++z) m = fmaxf(m, ms[r * parts + z]);
      for (int z = 0; z < parts; ++z) {
        const float mz = ms[r * parts + z];
        l = fmaf(ls[r * parts + z], mz == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((mz - m) * sl2), l);
      }
      for (int z = slice; z < parts; z += slices) {
        const float mz = ms[r * parts + z];
        if (mz == -INFINITY) continue;
        acc += *reinterpret_cast<const f32x4_t*>(p.part_o + slot(z, row) * HD + d) * __builtin_amdgcn_exp2f((mz - m) * sl2);
      }
    }
    if (slices > 1) {
      *reinterpret_cast<f32x4_t*>(&red[threadIdx.x * 4]) = acc;
      __syncthreads();
      if (slice == 0)
        for (int sl = 1; sl < slices; ++sl) acc += *reinterpret_cast<const f32x4_t*>(&red[(sl * n_pairs + pair) * 4]);
    }
    if (valid && slice == 0) {
      const float inv = attn_head_gate(p, q_begin + tok0 + tokw, kvh * group + hig) / l;
      bf16_t* orow = (bf16_t*)p.out + (int64_t)(q_begin + tok0 + tokw) * p.out_stride + (int64_t)(kvh * group + hig) * HD;
      uint2 two;
      two.x = (uint32_t)cw_float_to_bf16_bits(acc[0] * inv) | ((uint32_t)cw_float_to_bf16_bits(acc[1] * inv) << 16);
      two.y = (uint32_t)cw_float_to_bf16_bits(acc[2] * inv) | ((uint32_t)cw_float_to_bf16_bits(acc[3] * inv) << 16);
      *reinterpret_cast<uint2*>(orow + d) = two;
    }
  }
}

#if CW_HD % 32 == 0
#define CW_HAS_PREFILL 1
#else
#define CW_HAS_PREFILL 0
#endif

// 1 when this head size has the bfloat16 matrix-core kernel for portions (multiples of 32).
CW_EXPORT int cw_attention_prefill_supported() { return CW_HAS_PREFILL; }

#if CW_HAS_PREFILL
template <bool PAGES16, int RB, bool CAP>
static int launch_prefill(const AttnParams& p, int n_items, hipStream_t stream) {
  using Tile = PrefillTile<CW_HD, RB>;
  dim3 grid(n_items, p.nkv * p.n_chunks), block(Tile::NT);
  constexpr size_t smem = Tile::BYTES;
  static_assert(smem <= 160 * 1024, "the tiles of two stages fit a compute unit's LDS");
  static bool raised = false;
  if (!raised && smem > 48 * 1024) {
    if (hipFuncSetAttribute((const void*)attn_prefill_bf16_kernel<CW_HD, PAGES16, RB, CAP>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      return CW_ERR_LAUNCH;
    raised = true;
  }
  hipLaunchKernelGGL((attn_prefill_bf16_kernel<CW_HD, PAGES16, RB, CAP>), grid, block, smem, stream, p);
  if (p.part_o != nullptr)
    hipLaunchKernelGGL((attn_prefill_merge_kernel<CW_HD, RB>), dim3(grid.x, grid.y, 4), dim3(256), 0, stream, p);
  return cw_launch_status();
}
#endif

// Floats of workspace cw_attention_prefill_bf16 needs when some items are parts of a key range.
CW_EXPORT int64_t cw_attention_prefill_workspace_floats(int n_items, int nh, int nkv, int row_blocks) {
  if (n_items <= 0 || nh <= 0 || nkv <= 0) return 0;
  const int group = nh / nkv;
  const int gh = group < 32 ? group : 32;
  const int n_chunks = (group + gh - 1) / gh;
  return (int64_t)n_items * nkv * n_chunks * row_blocks * 32 * (CW_HD + 2);
}

// 1 if the kernel for portions can run with this many row blocks a workgroup (4, and 2 for head
// sizes up to 128).
CW_EXPORT int cw_attention_prefill_row_blocks_ok(int row_blocks) {
  return CW_HAS_PREFILL && (row_blocks == 4 || (row_blocks == 2 && CW_HD <= 128)) ? 1 : 0;
}

#if CW_HAS_PREFILL
// The parameters of the kernel for portions from its entry points' arguments, checked.
static int prefill_params(AttnParams& p, const void* q, int64_t q_stride, void* out, int64_t out_stride,
                                        const void* k_cache, const void* v_cache, const int* block_tables,
                                        int table_stride, const int* ctx_lens, const int* cu_q,
                                        const int* items, int n_items, int nh, int nkv, int block_size,
                                        int window, float scale, const void* zeros, int row_blocks,
                                        int with_parts, float* workspace, int64_t workspace_floats,
                                        float softcap, const void* gate, int64_t gate_stride, int gate_off) {
  if (zeros == nullptr || ((uintptr_t)zeros & 15)) return CW_ERR_ARG;
  if (n_items < 0 || nh <= 0 || nkv <= 0 || nh % nkv != 0 || block_size <= 0 || table_stride <= 0 || window < 0)
    return CW_ERR_ARG;
  if (!cw_attention_prefill_row_blocks_ok(row_blocks)) return CW_ERR_ARG;
  if (((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15) || ((uintptr_t)out & 7) ||
      (q_stride & 7) || (out_stride & 3))
    return CW_ERR_ARG;
  const int group = nh / nkv;
  p.q = q; p.q_stride = q_stride; p.out = out; p.out_stride = out_stride;
  p.k_cache = k_cache; p.v_cache = v_cache; p.block_tables = block_tables;
  p.table_stride = table_stride; p.ctx_lens = ctx_lens; p.cu_q = cu_q; p.items = items;
  p.nh = nh; p.nkv = nkv; p.block_size = block_size; p.bs_shift = cw_log2_or_minus1(block_size); p.gh = group < 32 ? group : 32;
  p.n_chunks = (group + p.gh - 1) / p.gh; p.n_splits = 1; p.window = window; p.scale = scale; p.softcap = softcap;
  p.part_o = nullptr; p.part_ml = nullptr; p.zeros = zeros;
  if (gate && (gate_off < 0 || gate_off + nh > gate_stride)) return CW_ERR_ARG;
  p.gate = gate; p.gate_stride = gate_stride; p.gate_off = gate_off;
  if ((int64_t)nkv * p.n_chunks > 65535) return CW_ERR_SIZE;
  if (with_parts) {
    const int64_t need = cw_attention_prefill_workspace_floats(n_items, nh, nkv, row_blocks);
    if (workspace == nullptr || workspace_floats < need || ((uintptr_t)workspace & 15)) return CW_ERR_ARG;
    p.part_o = workspace;
    p.part_ml = workspace + need / (CW_HD + 2) * CW_HD;
  }
  return CW_OK;
}
#endif

// Portions of prompts, bfloat16. items: (request, first token, tokens, part | parts << 8) with
// tokens <= row_blocks * 32 / gh, gh = min(group, 32) heads of a group per workgroup; tokens of
// an item beyond that are not computed. row_blocks: 4, or 2 (see PrefillTile). An item with
// parts > 1 stands ``parts`` times in the list, one after the other, as part 0, 1, ...: each takes
// a share of the keys that its tokens see, and a second kernel puts the shares together. Any item
// of that kind (``with_parts``) needs a float32 workspace of
// cw_attention_prefill_workspace_floats(n_items, ...) elements; parts at most 255.
CW_EXPORT int cw_attention_prefill_bf16(const void* q, int64_t q_stride, void* out, int64_t out_stride,
                                        const void* k_cache, const void* v_cache, const int* block_tables,
                                        int table_stride, const int* ctx_lens, const int* cu_q,
                                        const int* items, int n_items, int nh, int nkv, int block_size,
                                        int window, float scale, const void* zeros, int row_blocks,
                                        int with_parts, float* workspace, int64_t workspace_floats,
                                        float softcap, const void* gate, int64_t gate_stride, int gate_off,
                                        hipStream_t stream) {
#if CW_HAS_PREFILL
  AttnParams p{};
  const int status = prefill_params(p, q, q_stride, out, out_stride, k_cache, v_cache, block_tables, table_stride, ctx_lens, cu_q, items, n_items, nh, nkv, block_size, window, scale, zeros, row_blocks, with_parts, workspace, workspace_floats, softcap, gate, gate_stride, gate_off);
  if (status != CW_OK || n_items == 0) return status;
  const bool cap = softcap > 0.0f;
  auto launch = [&](auto rb) {
    constexpr int RB = decltype(rb)::value;
    if (p.bs_shift >= 4) return cap ? launch_prefill<true, RB, true>(p, n_items, stream) : launch_prefill<true, RB, false>(p, n_items, stream);
    return cap ? launch_prefill<false, RB, true>(p, n_items, stream) : launch_prefill<false, RB, false>(p, n_items, stream);
  };
#if CW_HD <= 128
  if (row_blocks == 2) return launch(std::integral_constant<int, 2>{});
#endif
  return launch(std::integral_constant<int, 4>{});
#else
  return CW_ERR_ARG;
#endif
}

// 1 if portions and single tokens of one step can run as one launch (see attn_together_bf16_kernel).
CW_EXPORT int cw_attention_together_supported() { return CW_HAS_PREFILL && CW_HD <= 128 ? 1 : 0; }

// The most keys that a split of cw_attention_together_bf16 takes with pages of this size, a multiple of 32 (0: there is no
// such launch): what cw_attention_decode_bf16 takes, whose splits may be shorter.
CW_EXPORT int cw_attention_together_split_keys(int block_size) {
#if CW_HAS_PREFILL && CW_HD <= 128
  if (block_size <= 0) return 0;
  const int64_t keys = (decode_pages_most(4) - 2) * (int64_t)block_size;
  return (int)((keys < INT_MAX ? keys : INT_MAX) & ~31);
#else
  return 0;
#endif
}

// cw_attention_prefill_bf16 of ``portions`` (whole items, no parts) and cw_attention_decode_bf16 of ``singles`` in one
// launch, then the merge of the single tokens' splits; the arguments are theirs.
CW_EXPORT int cw_attention_together_bf16(const void* q, int64_t q_stride, void* out, int64_t out_stride, const void* k_cache,
                                         const void* v_cache, const int* block_tables, int table_stride, const int* ctx_lens,
                                         const int* cu_q, const int* portions, int n_portions, int row_blocks, const int* singles,
                                         int n_singles, int n_splits, int split_keys, int max_ctx, int nh, int nkv,
                                         int block_size, int window, float scale, float* workspace, int64_t workspace_floats,
                                         const void* zeros, hipStream_t stream) {
#if CW_HAS_PREFILL && CW_HD <= 128
  AttnBoth a{};
  int status = prefill_params(a.portions, q, q_stride, out, out_stride, k_cache, v_cache, block_tables, table_stride, ctx_lens, cu_q,
                              portions, n_portions, nh, nkv, block_size, window, scale, zeros, row_blocks, 0, nullptr, 0, 0.0f,
                              nullptr, 0, 0);
  if (status != CW_OK) return status;
  status = decode_params(a.singles, q, q_stride, out, out_stride, k_cache, v_cache, block_tables, table_stride, ctx_lens, cu_q,
                         singles, n_singles, nh, nkv, block_size, n_splits, window, scale, workspace, workspace_floats, zeros, 0,
                         split_keys, max_ctx, 0.0f, nullptr, 0, 0);
  if (status != CW_OK) return status;
  if (n_portions == 0 || n_singles == 0) return CW_ERR_ARG;
  a.n_portions = n_portions; a.n_singles = n_singles;
  const int64_t groups = (int64_t)n_portions * nkv * a.portions.n_chunks + (int64_t)n_singles * nkv * a.singles.n_chunks * n_splits;
  if (groups > 0x7fffffff) return CW_ERR_SIZE;
  // LDS: the portions' tiles, or the single tokens' outputs and the pages of a split
  const int64_t max_tiles = ((int64_t)table_stride * block_size + 31) / 32;
  const int64_t tiles_per_split = split_keys > 0 ? split_keys / 32 : (max_tiles + n_splits - 1) / n_splits;
  const int64_t pages = (tiles_per_split * 32 + block_size - 1) / block_size + 2;
  if (!decode_pages_ok(4, pages)) return CW_ERR_SIZE;  // (eight waves here, but as many pages as the launch alone takes)
  constexpr size_t tiles = 8 * (size_t)DecodeTile<CW_HD>::BYTES;
  a.singles.decode_pages = decode_pages_in_lds(tiles, pages);
  const size_t for_singles = tiles + (a.singles.decode_pages > 0 ? sizeof(int) * (size_t)a.singles.decode_pages : 0);
  auto launch = [&](auto rb, auto pages16) {
    constexpr int RB = decltype(rb)::value;
    constexpr bool P16 = decltype(pages16)::value;
    const size_t smem = for_singles > PrefillTile<CW_HD, RB>::BYTES ? for_singles : PrefillTile<CW_HD, RB>::BYTES;
    static_assert(PrefillTile<CW_HD, RB>::BYTES <= DEC_MOST_LDS, "tiles and the single tokens' statistics fit LDS");
    static std::atomic<bool> allowed{false};
    if (cw_allow_lds(allowed, (const void*)attn_together_bf16_kernel<CW_HD, P16, RB>, DEC_MOST_LDS) != CW_OK) return CW_ERR_LAUNCH;
    hipLaunchKernelGGL((attn_together_bf16_kernel<CW_HD, P16, RB>), dim3((unsigned)groups), dim3(512), smem, stream, a);
    launch_decode_merge(a.singles, n_singles, stream);
    return cw_launch_status();
  };
  using Two = std::integral_constant<int, 2>;
  using Four = std::integral_constant<int, 4>;
  if (a.portions.bs_shift >= 4)
    return row_blocks == 2 ? launch(Two{}, std::true_type{}) : launch(Four{}, std::true_type{});
  return row_blocks == 2 ? launch(Two{}, std::false_type{}) : launch(Four{}, std::false_type{});
#else
  return CW_ERR_ARG;
#endif
}
