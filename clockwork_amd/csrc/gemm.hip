// Matrix products y = x * W^T (+ bias) for gfx950, W stored [N, K] row-major as checkpoints
// hold it.
//  * cw_gemm_f32: true float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32 operands, products
//    and sums). The order in which the products of one output element are summed depends on N and K
//    alone, never on M, so a row's result does not depend on what else is in the batch.
#include <climits>
#include <type_traits>

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// How these kernels load operands of few rows. An MFMA operand wants lane l to hold row l % 16 of a tile and
// the 8 k-values of slot l / 16: loaded that way every lane asks for 16 bytes of a row of its own,
// 64 requests an instruction to a compute unit's load path, which takes in about 30 GB/s of such.
// So a lane loads row l / 4, slot l % 4 instead (four neighbouring lanes cover 64 bytes of one row:
// 16 requests an instruction), and the lanes swap what they hold afterwards, lane (r, s) taking
// from lane 4 r + s (ds_bpermute: through the LDS unit's crossbar, no memory). Measured on the
// 1.5B shape's gate/up product: 12.8 -> 11.7 us with 8 rows of x, 19.8 -> 17.5 us with 64.
typedef __attribute__((ext_vector_type(4))) int cw_i32x4_t;
__device__ __forceinline__ cw_i32x4_t cw_swap_to_operand(const cw_i32x4_t& q, int lane) {
  const int r = lane & 15, s = lane >> 4;
  const int from = (r * 4 + s) * 4;  // byte address of the lane that loaded what lane (r, s) multiplies
  cw_i32x4_t t;
#pragma unroll
  for (int d = 0; d < 4; ++d) t[d] = __builtin_amdgcn_ds_bpermute(from, q[d]);
  return t;
}
__device__ __forceinline__ bf16x8_t cw_to_operand_layout(const bf16x8_t& v, int lane) {
  return __builtin_bit_cast(bf16x8_t, cw_swap_to_operand(__builtin_bit_cast(cw_i32x4_t, v), lane));
}

// Two steps of K at once: lane l loads slot l % 8 of the 128 bytes that hold both, of row 2 (l / 8) into a and of the row after it
// into b, so that a load asks for whole lines. Then lanes 4 to 7 of eight hold the second step: they change places with the
// other row's first, and a and b are the two steps as a load of one each would have left them.
__device__ __forceinline__ void cw_lines_to_steps(bf16x8_t& a, bf16x8_t& b) {
  cw_i32x4_t p = __builtin_bit_cast(cw_i32x4_t, a), q = __builtin_bit_cast(cw_i32x4_t, b);
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int first = p[d], second = q[d];
    p[d] = __builtin_amdgcn_update_dpp(first, second, 0x114, 0xf, 0xa, false);   // row_shr:4 into lanes 4 .. 7 and 12 .. 15 of 16
    q[d] = __builtin_amdgcn_update_dpp(second, first, 0x104, 0xf, 0x5, false);   // row_shl:4 into the others
  }
  a = __builtin_bit_cast(bf16x8_t, p), b = __builtin_bit_cast(bf16x8_t, q);
}

// =====================================================================================
// float32. What a product of one output element is, whichever kernel makes it: K is cut into parts
// (gemm_f32_plan), a part into blocks of 16 k-values. Lane (row, s) of an operand holds k-values
// 4 s .. 4 s + 3 of a block; the four MFMAs of a block, the j-th with element j of every lane, sum it
// from zero; the blocks' sums are added up in order, then the parts' in order, then the bias. (A sum of
// 16 on its own before it joins the total: a long K, 8960 in a feed-forward, rounds about
// sqrt(16) + sqrt(K / 16) times instead of sqrt(K).)
__device__ __forceinline__ f32x4_t gemm_f32_block(const f32x4_t& w, const f32x4_t& x) {
  f32x4_t t = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < 4; ++j) t = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], t, 0, 0, 0);
  return t;
}

// Four k-values of a row from k on; zeros from k_end on. VEC: rows of 16-byte multiples (k and k_end are
// multiples of 4 then), loaded from a clamped address so that the load does not hang on a condition.
template <bool VEC>
__device__ __forceinline__ f32x4_t gemm_f32_load4(const float* __restrict__ row, int k, int k_end) {
  f32x4_t v;
  if (VEC) {
    const bool ok = k < k_end;
    v = *reinterpret_cast<const f32x4_t*>(row + (ok ? k : 0));
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = ok ? v[j] : 0.0f;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = k + j < k_end ? row[k + j] : 0.0f;
  }
  return v;
}

// Up to 16 rows of x (single tokens): W is streamed once, straight into the operands' registers. A wave
// owns 16 rows of W and a run of the parts of K; ``part_waves`` waves share a tile's parts and the block
// holds blockDim / 64 / part_waves tiles. What bounds it is the stream of W (and, for the small
// projections, one trip to memory): eight blocks of 16 k-values are on their way while eight are multiplied.
// With plane_stride > 0 a part's sum is written out as plane z of C (whoever reads y next adds the planes
// in order); else the parts meet in LDS.
// For rows of whole blocks there is a faster kernel below; this one serves other K, the widest outputs and long K
// whose parts meet in LDS.
template <bool VEC>
__global__ __launch_bounds__(512) void gemm_f32_rows_kernel(const float* __restrict__ A, int64_t lda,
                                                            const float* __restrict__ W,
                                                            const float* __restrict__ bias,
                                                            float* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                            int parts, int k_per_part, int part_waves,
                                                            int64_t plane_stride) {
  extern __shared__ __align__(16) float red[];  // [tile of the block][part][token][row of W]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, s = lane >> 4, lr = lane >> 2, ls = lane & 3;
  const int tiles_here = (blockDim.x >> 6) / part_waves;
  const int tile_here = wave / part_waves;
  const int64_t n0 = ((int64_t)blockIdx.x * tiles_here + tile_here) * 16;
  const float* wrow = W + min(n0 + lr, (int64_t)N - 1) * K;
  const float* xrow = A + (int64_t)min(r, M - 1) * lda;
  constexpr int U = 8;
  const int z_step = part_waves * gridDim.y;
  for (int z = blockIdx.y * part_waves + wave % part_waves; z < parts; z += z_step) {
    const int k_begin = z * k_per_part, k_end = min(K, k_begin + k_per_part);
    const int blocks = (k_end - k_begin + 15) / 16;
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4_t wa[U], xa[U], wb[U], xb[U];
    auto load = [&](f32x4_t (&w)[U], f32x4_t (&x)[U], int b0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k_begin + (b0 + u) * 16;
        w[u] = gemm_f32_load4<VEC>(wrow, k + 4 * ls, k_end);
        x[u] = gemm_f32_load4<VEC>(xrow, k + 4 * s, k_end);
      }
    };
    auto multiply = [&](const f32x4_t (&w)[U], const f32x4_t (&x)[U], int b0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (b0 + u >= blocks) break;
        acc += gemm_f32_block(__builtin_bit_cast(f32x4_t, cw_swap_to_operand(__builtin_bit_cast(cw_i32x4_t, w[u]), lane)), x[u]);
      }
    };
    load(wa, xa, 0);
    for (int b0 = 0; b0 < blocks; b0 += 2 * U) {
      if (b0 + U < blocks) load(wb, xb, b0 + U);
      multiply(wa, xa, b0);
      if (b0 + U >= blocks) break;
      if (b0 + 2 * U < blocks) load(wa, xa, b0 + 2 * U);
      multiply(wb, xb, b0 + U);
    }
    // lane (r, s) holds rows 4 s .. 4 s + 3 of W for token r
    if (plane_stride > 0) {
      float* out = C + (int64_t)z * plane_stride + (int64_t)r * ldc + n0 + 4 * s;
      if (r < M)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n0 + 4 * s + i < N) out[i] = acc[i];
    } else {
      *reinterpret_cast<f32x4_t*>(&red[(tile_here * parts + z) * 256 + r * 16 + 4 * s]) = acc;
    }
  }
  if (plane_stride > 0) return;
  __syncthreads();
  for (int idx = threadIdx.x; idx < tiles_here * 256; idx += blockDim.x) {
    const int m = (idx >> 4) & 15, t = idx >> 8;
    const int64_t n = ((int64_t)blockIdx.x * tiles_here + t) * 16 + (idx & 15);
    const float* p = red + t * parts * 256 + (idx & 255);
    float total = p[0];
    for (int z = 1; z < parts; ++z) total += p[z * 256];
    if (m < M && n < N) C[(int64_t)m * ldc + n] = total + (bias ? bias[n] : 0.0f);
  }
}

// The same sums for rows of whole blocks (K a multiple of 16): the waves of a workgroup share the blocks of 16 k-values of
// its parts of a tile of 16 rows of W, not the parts, so a workgroup's whole share of W is asked for at once; the blocks'
// sums meet in LDS, [block][token][row of W], and are added in their order there. What bounds it is one trip to memory
// and, for the large matrices, the stream of W. Measured on an MI355X with one row of x against the kernel above (whose waves
// make a part each, eight blocks at a time, and which is twice the code): 1152 x 896 8.0 -> 5.0 us, 9728 x 896 14.4 -> 12.0,
// 2048 x 1536 9.9 -> 8.3; the sums are the same bit for bit.
#define GT_BLOCK_WAVES 8
#define GT_BLOCKS 120   // blocks a workgroup takes: 1 KB of LDS each with 16 rows of x
// and of the parts that they make, of 256 k-values at least, where those meet in LDS as well
#define GT_BLOCKS_LDS ((GT_BLOCKS + GT_BLOCKS / 16) * 1024)
// GLU: W = [gate; up], a tile is 8 gate rows and the 8 up rows that belong to them, C the gated product [M, N / 2].
// PAIRS: W = [queries; keys; values] of ``to``, a tile of a query or key head is 8 rows of its first half and the 8 of its second
// that they are rotated with; C the rotated queries, keys and values go to their cache rows. The
// rotation as a kernel of its own is a launch that moves a few KB: 3.7 us of a layer's decode step of the 0.5B shape.
#define GT_PLAIN 0
#define GT_GLU 1
#define GT_PAIRS 2
struct F32PairsOut {
  const int* positions;
  const int* slots;
  const float* inv_freq;
  float* k_cache;
  float* v_cache;
  int64_t cache_rows;
  int nh, nkv, hd;
};
template <int KIND>
__global__ __launch_bounds__(GT_BLOCK_WAVES * 64) void gemm_f32_blocks_kernel(const float* __restrict__ A, int64_t lda,
                                                                              const float* __restrict__ W,
                                                                              const float* __restrict__ bias, float* __restrict__ C,
                                                                              int64_t ldc, int M, int N, int K, int parts, int part_blocks,
                                                                              int parts_here, int64_t plane_stride, float act, F32PairsOut to) {
  constexpr bool GLU = KIND == GT_GLU, PAIRS = KIND == GT_PAIRS;
  extern __shared__ __align__(16) float red[];
  constexpr int U = 8;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, s = lane >> 4;
  const int n0 = blockIdx.x * (GLU ? 8 : 16), cols = GLU ? N / 2 : N;
  const int z0 = blockIdx.y * parts_here, z1 = min(parts, z0 + parts_here);
  const int b0 = z0 * part_blocks, b1 = min(K / 16, z1 * part_blocks);
  const int tile_row = lane >> 2;
  int row = GLU ? min(n0 + (tile_row & 7), cols - 1) + (tile_row >> 3) * cols : min(n0 + tile_row, N - 1);
  // what a thread's output takes besides its sum is asked for beside the weights
  int head = 0, first = 0, pos = 0;
  int64_t slot = -1;
  float inv = 0.0f, bias_a = 0.0f, bias_b = 0.0f;
  bool rotated = false;
  if constexpr (PAIRS) {
    head = n0 / to.hd;
    rotated = head < to.nh + to.nkv;
    const int half = to.hd / 2;
    first = rotated ? (n0 - head * to.hd) / 2 : n0 - head * to.hd;
    if (rotated) row = head * to.hd + first + (tile_row & 7) + (tile_row >> 3) * half;
    const int at = threadIdx.x, m = rotated ? at >> 3 : at >> 4, d = first + (at & (rotated ? 7 : 15));
    if (m < M) {
      slot = to.slots[m];
      if (bias) bias_a = bias[head * to.hd + d];
      if (rotated) {
        pos = to.positions[m];
        inv = to.inv_freq[d];
        if (bias) bias_b = bias[head * to.hd + d + half];
      }
    }
  }
  const float* const w = W + (int64_t)row * K + 4 * (lane & 3);
  const float* const x = A + (int64_t)min(r, M - 1) * lda + 4 * s;
  for (int b = b0 + wave; b < b1; b += U * GT_BLOCK_WAVES) {
    f32x4_t wv[U], xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (b + u * GT_BLOCK_WAVES < b1) {
        wv[u] = *reinterpret_cast<const f32x4_t*>(w + (b + u * GT_BLOCK_WAVES) * 16);
        xv[u] = *reinterpret_cast<const f32x4_t*>(x + (b + u * GT_BLOCK_WAVES) * 16);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (b + u * GT_BLOCK_WAVES < b1) {
        // lane (r, s) holds rows 4 s .. 4 s + 3 of W for token r
        const f32x4_t t = gemm_f32_block(__builtin_bit_cast(f32x4_t, cw_swap_to_operand(__builtin_bit_cast(cw_i32x4_t, wv[u]), lane)), xv[u]);
        if (r < M) *reinterpret_cast<f32x4_t*>(&red[((b + u * GT_BLOCK_WAVES - b0) * M + r) * 16 + 4 * s]) = t;
      }
  }
  cw_lds_barrier();
  // a thread takes one output of one part; without planes the parts' sums meet in LDS again, behind the blocks'
  float* const sums = red + (b1 - b0) * M * 16;
  const int outputs = M * 16;
  for (int i = threadIdx.x; i < outputs * (z1 - z0); i += GT_BLOCK_WAVES * 64) {
    const int z = i / outputs, at = i - z * outputs;
    const int from = z * part_blocks, to = min(b1 - b0, from + part_blocks);
    float total = red[from * outputs + at];
#pragma unroll 8
    for (int b = from + 1; b < to; ++b) total += red[b * outputs + at];
    const int n = n0 + (at & 15);
    if (plane_stride > 0) {
      if (n < N) C[(z0 + z) * plane_stride + (int64_t)(at >> 4) * ldc + n] = total;
    } else if (parts == 1 && KIND == GT_PLAIN) {
      if (n < N) C[(int64_t)(at >> 4) * ldc + n] = total + (bias ? bias[n] : 0.0f);
    } else {
      sums[i] = total;
    }
  }
  if (plane_stride > 0 || (parts == 1 && KIND == GT_PLAIN)) return;
  cw_lds_barrier();
  if constexpr (GLU) {
    for (int i = threadIdx.x; i < M * 8; i += GT_BLOCK_WAVES * 64) {
      const int at = (i >> 3) * 16 + (i & 7), n = n0 + (i & 7);
      float gate = sums[at], up = sums[at + 8];
      for (int z = 1; z < parts; ++z) {
        gate += sums[z * outputs + at];
        up += sums[z * outputs + at + 8];
      }
      if (n < cols) C[(int64_t)(i >> 3) * ldc + n] = cw_gated(gate, up, act);
    }
    return;
  }
  if constexpr (PAIRS) {
    const int at = threadIdx.x, m = rotated ? at >> 3 : at >> 4, d = first + (at & (rotated ? 7 : 15)), half = to.hd / 2;
    if (m >= M) return;  // up to 16 rows: an output or a pair of them a thread
    auto summed = [&](int column) __attribute__((always_inline)) {
      float total = sums[m * 16 + column];
      for (int z = 1; z < parts; ++z) total += sums[z * outputs + m * 16 + column];
      return total;
    };
    const bool kept = slot >= 0 && slot < to.cache_rows;
    if (!rotated) {
      if (kept) to.v_cache[(slot * to.nkv + (head - to.nh - to.nkv)) * to.hd + d] = summed(at & 15) + bias_a;
      return;
    }
    const float a = summed(at & 7) + bias_a, b = summed((at & 7) + 8) + bias_b;
    float sn, cs;
    sincosf((float)pos * inv, &sn, &cs);
    float* const out = head < to.nh ? C + (int64_t)m * ldc + head * to.hd : to.k_cache + (slot * to.nkv + (head - to.nh)) * to.hd;
    if (head < to.nh || kept) {
      out[d] = a * cs - b * sn;
      out[d + half] = b * cs + a * sn;
    }
    return;
  }
  for (int at = threadIdx.x; at < outputs; at += GT_BLOCK_WAVES * 64) {
    const int n = n0 + (at & 15);
    float total = sums[at];
    for (int z = 1; z < parts; ++z) total += sums[z * outputs + at];
    if (n < N) C[(int64_t)(at >> 4) * ldc + n] = total + (bias ? bias[n] : 0.0f);
  }
}

// A wave's sums to C, TN x TM tiles from row m0 of x and row n0 of W: lane (r, s) holds rows 4 s .. 4 s + 3 of
// W for token r of each.
template <int TN, int TM>
__device__ __forceinline__ void gemm_f32_store_tile(const f32x4_t (&total)[TN][TM], float* __restrict__ C,
                                                    const float* __restrict__ bias, int plane, int64_t plane_stride,
                                                    int64_t ldc, int m0, int n0, int M, int N, int r, int s) {
  const bool planes = plane_stride > 0;
  float* out = C + (int64_t)plane * plane_stride;
  const bool vec_store = !(ldc & 3) && !((uintptr_t)out & 15);
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int m = m0 + 16 * j + r, n = n0 + 16 * i + 4 * s;
      if (m >= M) continue;
      f32x4_t v = total[i][j];
      if (bias && !planes)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += n + e < N ? bias[n + e] : 0.0f;
      float* p = out + (int64_t)m * ldc + n;
      if (vec_store && n + 4 <= N) {
        *reinterpret_cast<f32x4_t*>(p) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) p[e] = v[e];
      }
    }
}

// More rows, of any length: tiles of 64 rows of x by 64 rows of W, 256 threads, the K loop through registers
// and LDS in steps of 32 (two buffers, the next step's loads on their way over the products of this one). Wave
// (i, j) of the 2 x 2 owns 32 rows of W and 32 of x. A row of a step takes 36 floats in LDS: the 16 rows that a
// quarter of a wave reads 16 bytes of then begin in 16 different groups of four banks.
// gridDim.z > 1: block z makes part z alone, into plane z of C; else a block adds its parts up itself.
// For rows that gemm_f32_ring_kernel does not take (K no multiple of 16).
template <bool VEC, bool ONE_PART>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const float* __restrict__ A, int64_t lda,
                                                            const float* __restrict__ W,
                                                            const float* __restrict__ bias,
                                                            float* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                            int parts, int k_per_part, int64_t plane_stride) {
  constexpr int BM = 64, BN = 64, BK = 32, LD = BK + 4, TM = BM / 32, XL = BM / 32;
  __shared__ __align__(16) float Ws[2][BN * LD];
  __shared__ __align__(16) float Xs[2][BM * LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, s = lane >> 4;
  const int wn = (wave & 1) * 32, wm = (wave >> 1) * (BM / 2);
  const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM;
  const int z_first = ONE_PART ? blockIdx.z : 0, z_last = ONE_PART ? blockIdx.z : parts - 1;

  // what this thread brings in: 16 bytes of rows tid / 8 and tid / 8 + 32 of a step
  const int lrow = tid >> 3, lk = (tid & 7) * 4;
  const float* wrow[2];
  const float* xrow[XL];
#pragma unroll
  for (int i = 0; i < 2; ++i) wrow[i] = W + (int64_t)min(n0 + lrow + 32 * i, N - 1) * K;
#pragma unroll
  for (int i = 0; i < XL; ++i) xrow[i] = A + (int64_t)min(m0 + lrow + 32 * i, M - 1) * lda;
  f32x4_t wreg[2], xreg[XL];
  auto load = [&](int k0, int k_end) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) wreg[i] = gemm_f32_load4<VEC>(wrow[i], k0 + lk, k_end);
#pragma unroll
    for (int i = 0; i < XL; ++i) xreg[i] = gemm_f32_load4<VEC>(xrow[i], k0 + lk, k_end);
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4_t*>(&Ws[buf][(lrow + 32 * i) * LD + lk]) = wreg[i];
#pragma unroll
    for (int i = 0; i < XL; ++i) *reinterpret_cast<f32x4_t*>(&Xs[buf][(lrow + 32 * i) * LD + lk]) = xreg[i];
  };

  f32x4_t acc[2][TM], total[2][TM];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = total[i][j] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};

  int z = z_first, k0 = z * k_per_part, k_end = min(K, k0 + k_per_part), buf = 0;
  load(k0, k_end);
  store(0);
  __syncthreads();
  while (true) {
    // the step after this one: of the same part, or the first of the next
    int next_z = z, next_k0 = k0 + BK, next_end = k_end;
    const bool last_of_part = next_k0 >= k_end;
    if (last_of_part) {
      next_z = z + 1;
      next_k0 = next_z * k_per_part;
      next_end = min(K, next_k0 + k_per_part);
    }
    const bool more = next_z <= z_last;
    if (more) load(next_k0, next_end);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (b == 1 && k0 + 16 >= k_end) break;  // a part is a whole number of blocks, not of steps
      f32x4_t wf[2], xf[TM];
#pragma unroll
      for (int i = 0; i < 2; ++i) wf[i] = *reinterpret_cast<const f32x4_t*>(&Ws[buf][(wn + 16 * i + r) * LD + b * 16 + 4 * s]);
#pragma unroll
      for (int j = 0; j < TM; ++j) xf[j] = *reinterpret_cast<const f32x4_t*>(&Xs[buf][(wm + 16 * j + r) * LD + b * 16 + 4 * s]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] += gemm_f32_block(wf[i], xf[j]);
    }
    if (last_of_part) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          total[i][j] = (ONE_PART || z == z_first) ? acc[i][j] : total[i][j] + acc[i][j];
          acc[i][j] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    if (!more) break;
    buf ^= 1;
    store(buf);
    __syncthreads();
    z = next_z;
    k0 = next_k0;
    k_end = next_end;
  }

  gemm_f32_store_tile(total, C, bias, blockIdx.z, plane_stride, ldc, m0 + wm, n0 + wn, M, N, r, s);
}

// The same product, rows of whole blocks of 16 k-values: tiles of BM rows of x by 64 rows of W, K in stages of
// 32 values that go from global memory straight into LDS (buffer loads with the LDS target), a ring of four.
// What bounds it is the trip to memory of a tile's stages: a compute unit has one to three tiles at a time, and
// with one stage under way over another's products (0.2 to 0.4 us against a trip of 1 us and more) it waited
// most of the time; three are under way here. A load instruction brings eight rows of 128 bytes; the eight 16-byte
// granules of row R change places by (R >> 1) & 7, so that the 16 lanes that read one granule of 16 rows touch
// every bank once. The descriptors end with the matrices: rows past the end read as zeros. What a stage holds past
// the end of its part is not multiplied. BM is 32 where 64 would leave compute units without a tile.
// The operands of a block are read from LDS beside the products of the block before it, across the stages' barriers, and the
// loop's two blocks have sums of their own: read at the head of a stage, and with the sums moved to other registers, the matrix cores
// waited for a tenth of the time. The matrix cores bound it now where there are tiles enough: 124 TFLOP/s for 2048 rows of 4096 x
// 4096 (114 before), and tiles of 128 x 128, which load half as much, reach the same. Measured on an MI355X, us, before and now:
// 336 rows of 9728 x 896 78 and 68, 896 x 4864 45 and 40, 1152 x 896 16.4 and 16.1 (108 tiles); 1000 rows of 17920 x 1536 555 and
// 497; 40 rows of 1536 x 8960 25.5 and 23.0. (The four products of a layer of the 0.5B shape with 384 rows, 919 us on 64 x 64
// tiles of the vector units.)
typedef __attribute__((address_space(3))) void lds_void_t;
// s_waitcnt for "at most n vector-memory operations in flight" and nothing else
#define GF_WAIT_LOADS(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14))
// a barrier without a fence (a fence would wait for every load in flight)
#define GF_BARRIER()               \
  do {                             \
    asm volatile("" ::: "memory"); \
    __builtin_amdgcn_s_barrier();  \
    asm volatile("" ::: "memory"); \
  } while (0)

template <int BM, bool ONE_PART>
__global__ __launch_bounds__(256, 2) void gemm_f32_ring_kernel(const float* __restrict__ A, int64_t lda,
                                                            const float* __restrict__ W,
                                                            const float* __restrict__ bias,
                                                            float* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                            int parts, int k_per_part, int64_t plane_stride) {
  constexpr int BN = 64, BK = 32, SLOTS = 4, TM = BM / 32, TN = 2;
  constexpr int XB = BM / 8, WB = BN / 8, LOADS = (XB + WB) / 4;  // 1 KB blocks of a stage; loads of a wave
  constexpr int STAGE = (XB + WB) * 1024;
  extern __shared__ __align__(1024) unsigned char ring[];  // SLOTS * STAGE bytes
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, s = lane >> 4;
  const int wn = (wave & 1) * 32, wm = (wave >> 1) * (BM / 2);
  // Workgroups are dealt to the 8 XCDs in turn. Each XCD takes a run of neighbouring tiles, those of the same rows
  // of W next to each other: W then comes from memory once, into one L2.
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int run = gridDim.x >> 3, rest = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int tile = xcd * run + min(xcd, rest) + (blockIdx.x >> 3);
  const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m % tiles_n * BN;
  const int plane = tile / (tiles_m * tiles_n);
  const int z_first = ONE_PART ? plane : 0, z_last = ONE_PART ? plane : parts - 1;

  __amdgpu_buffer_rsrc_t xr, wr;
  xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A + (int64_t)m0 * lda), 0, (int)(uint32_t)(((int64_t)(M - m0 - 1) * lda + K) * 4), 0x00020000);
  wr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(W + (int64_t)n0 * K), 0, (int)(uint32_t)(((int64_t)(N - n0 - 1) * K + K) * 4), 0x00020000);
  // load i of a wave: block wave * LOADS + i of a stage, the x blocks first
  uint32_t at[4];  // (of a size that hangs on no template parameter, as the buffer is: the host pass drops the kernel otherwise)
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int block = wave * LOADS + i, row = (block < XB ? block : block - XB) * 8 + (lane >> 3);
    const int granule = (lane & 7) ^ ((row >> 1) & 7);
    at[i] = (uint32_t)(((int64_t)row * (block < XB ? lda : K) + granule * 4) * 4);
  }
  auto fetch = [&](int k0, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int block = wave * LOADS + i;
      unsigned char* to = ring + (slot * STAGE + block * 1024);
      if (block < XB) __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void_t*)to, 16, at[i], k0 * 4, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void_t*)to, 16, at[i], k0 * 4, 0, 0);
    }
  };
  // the stage that is asked for next; past the last one it is asked for again (nobody reads it, but the
  // number of loads in flight stays what the waits count on)
  int fz = z_first, fk = z_first * k_per_part;
  auto fetch_next = [&](int slot) __attribute__((always_inline)) {
    fetch(fk, slot);
    const int end = min(K, (fz + 1) * k_per_part);
    if (fk + BK < end) fk += BK;
    else if (fz < z_last) fk = ++fz * k_per_part;
  };
  // even, odd: the sums of the last block of 16 with an even and with an odd number in its stage. A block's sums join
  // the part's beside the products of the next one: added at once they would wait for the last product, with the matrix
  // core idle, and so they did when they were moved to other registers first.
  f32x4_t acc[TN][TM], total[TN][TM], even[TN][TM], odd[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = total[i][j] = odd[i][j] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
  const unsigned char* mine = ring + r * 128;
  const int turn = (r >> 1) & 7;
  auto read = [&](f32x4_t (&wf)[TN], f32x4_t (&xf)[TM], int slot, int b) __attribute__((always_inline)) {
    const unsigned char* from = mine + slot * STAGE + ((b * 4 + s) ^ turn) * 16;
#pragma unroll
    for (int i = 0; i < TN; ++i) wf[i] = *reinterpret_cast<const f32x4_t*>(from + XB * 1024 + wn * 128 + i * 2048);
#pragma unroll
    for (int j = 0; j < TM; ++j) xf[j] = *reinterpret_cast<const f32x4_t*>(from + wm * 128 + j * 2048);
  };
  // gemm_f32_block for each pair, the pairs' products taking turns, and the sums of the block before to the part's
  auto multiply = [&](const f32x4_t (&wf)[TN], const f32x4_t (&xf)[TM], f32x4_t (&sums)[TN][TM], const f32x4_t (&before)[TN][TM])
      __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
          sums[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][q], xf[j][q], q == 0 ? (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f} : sums[i][j], 0, 0, 0);
      if (q == 1) {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j) acc[i][j] += before[i][j];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int i = 0; i < SLOTS - 1; ++i) fetch_next(i);
  GF_WAIT_LOADS((SLOTS - 2) * LOADS);
  GF_BARRIER();
  f32x4_t w0[TN], x0[TM], w1[TN], x1[TM];
  read(w0, x0, 0, 0);
  for (int z = z_first, slot = 0; z <= z_last; ++z) {
    const int k_end = min(K, (z + 1) * k_per_part);
    for (int k0 = z * k_per_part; k0 < k_end; k0 += BK) {
      read(w1, x1, slot, 1);
      multiply(w0, x0, even, odd);
      // this wave's loads of the next stage are in; behind the barrier every wave's are, and every wave has read all
      // of the stage before this one, whose slot the next loads take
      GF_WAIT_LOADS((SLOTS - 3) * LOADS);
      GF_BARRIER();
      fetch_next((slot + SLOTS - 1) % SLOTS);
      slot = (slot + 1) % SLOTS;
      read(w0, x0, slot, 0);
      if (k0 + 16 < k_end) {
        multiply(w1, x1, odd, even);
      } else {  // a part is a whole number of blocks, not of stages
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j) odd[i][j] = even[i][j];
      }
    }
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        acc[i][j] += odd[i][j];
        total[i][j] = (ONE_PART || z == z_first) ? acc[i][j] : total[i][j] + acc[i][j];
        acc[i][j] = odd[i][j] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
      }
  }
  GF_WAIT_LOADS(0);  // no load may reach LDS after the workgroup has gone
  gemm_f32_store_tile(total, C, bias, plane, plane_stride, ldc, m0 + wm, n0 + wn, M, N, r, s);
}

// C[m, n] = ((p_0 + p_1) + ... + p_{splits-1}) + bias[n] over the partial sums p_z[m, n] (rows of N
// floats, part_stride floats between two splits): always in the order of the splits.
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(const float* __restrict__ parts, int splits,
                                                           int64_t part_stride, const float* __restrict__ bias,
                                                           float* __restrict__ C, int64_t ldc, int rows, int N) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)rows * N) return;
  const int m = (int)(idx / N), n = (int)(idx - (int64_t)m * N);
  float total = parts[idx];
  for (int z = 1; z < splits; ++z) total += parts[z * part_stride + idx];
  C[(int64_t)m * ldc + n] = total + (bias ? bias[n] : 0.0f);
}

// Up to this many rows of x the parts of K are made by blocks of their own (beyond, there are mostly
// blocks enough without, and a block sums its parts itself).
#define GT_SPLIT_ROWS 256
#define GT_ROWS_MAX 16    // gemm_f32_rows_kernel's rows
#define GT_LDS_PARTS 48   // parts that may meet in that kernel's LDS (1 KB each)
#define GT_MAX_PLANES 64  // planes that the residual-add + norm kernel adds

// How the float32 product cuts K for an [N, K] weight matrix: a narrow output (24 blocks of 64
// columns for a width of 1536) with few rows of x would leave most compute units without work and
// stream the matrix through the few that have some, so K is cut until there are about 512 blocks
// per 64 rows, with at least 256 values of K each. A function of N and K alone: the order of the
// sums must not depend on how many rows the step has.
static void gemm_f32_plan(int N, int K, int* splits, int* k_per_split) {
  const int col_blocks = (N + 63) / 64;
  int s = (512 + col_blocks / 2) / col_blocks;
  if (s > K / 256) s = K / 256;
  if (s < 1) s = 1;
  const int per = ((K + s - 1) / s + 15) / 16 * 16;
  *k_per_split = per;
  *splits = (K + per - 1) / per;
}

// Are the parts of K made apart, as planes of partial sums, for this many rows? Up to GT_SPLIT_ROWS rows
// always (but not where the parts of few rows meet in LDS); beyond, where tiles of 64 x 64 would leave
// compute units idle and K is long enough to pay for writing and reading the planes (300 rows of the 0.5B
// shape's down product, 70 tiles of 4864 k-values: 65 us for the products of one tile, 46 us as 19 planes).
static bool gemm_f32_planes(int M, int N, int K, int splits) {
  if (splits <= 1) return false;
  if (M <= GT_ROWS_MAX) return splits > GT_LDS_PARTS;
  if (M <= GT_SPLIT_ROWS) return true;
  return K >= 2048 && (int64_t)((M + 63) / 64) * ((N + 63) / 64) < 96;
}

// Floats of workspace cw_gemm_f32 needs for this product (0: none).
CW_EXPORT int64_t cw_gemm_f32_workspace_floats(int M, int N, int K) {
  int splits, per;
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  gemm_f32_plan(N, K, &splits, &per);
  return gemm_f32_planes(M, N, K, splits) ? (int64_t)splits * M * N : 0;
}

// Planes of partial sums that cw_gemm_f32_partial writes for this product, 0 where it should not be
// asked: one part, blocks enough without, or more planes than the norm kernel adds.
CW_EXPORT int cw_gemm_f32_partial_planes(int M, int N, int K) {
  int splits, per;
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  gemm_f32_plan(N, K, &splits, &per);
  if (splits <= 1 || splits > GT_MAX_PLANES) return 0;
  return M <= GT_ROWS_MAX || gemm_f32_planes(M, N, K, splits) ? splits : 0;
}

// C: y [M, N] with row stride ldc, or with planes float32 [splits, M, N].
static int launch_gemm_f32(const float* A, int64_t lda, const float* W, const float* bias, float* C, int64_t ldc, int M,
                           int N, int K, int splits, int per, bool planes, hipStream_t stream) {
  const bool vec = !(K & 3) && !(lda & 3);
  const int64_t stride = planes ? (int64_t)M * N : 0;
  // Whole blocks of 16: the kernel whose waves share blocks. Without planes a workgroup takes all parts, with planes
  // as many as make GT_BLOCKS blocks at most and leave a workgroup for every compute unit. (Not for outputs as wide as a
  // vocabulary, which stream either way: 151936 x 896 with 16 rows 152 us the other way, 158 this.)
  if (M <= GT_ROWS_MAX && !(K & 15) && !(lda & 3) && N <= 65536) {
    const int part_blocks = per / 16, tiles = (N + 15) / 16;
    int here = splits;
    if (planes) {
      const int most = GT_BLOCKS / part_blocks, spread = (int)((int64_t)splits * tiles / 256);
      here = spread < most ? spread : most;
      if (here < 1) here = 1;
      if (here > splits) here = splits;
    }
    const int blocks = here * part_blocks < K / 16 ? here * part_blocks : K / 16;
    if (blocks <= GT_BLOCKS) {
      const size_t lds = (size_t)(blocks + (planes || splits == 1 ? 0 : splits)) * M * 16 * sizeof(float);
      const dim3 grid(tiles, (splits + here - 1) / here);
      static std::atomic<bool> allowed{false};
      if (cw_allow_lds(allowed, (const void*)gemm_f32_blocks_kernel<GT_PLAIN>, GT_BLOCKS_LDS) != CW_OK) return CW_ERR_LAUNCH;
      hipLaunchKernelGGL(gemm_f32_blocks_kernel<GT_PLAIN>, grid, dim3(GT_BLOCK_WAVES * 64), lds, stream, A, lda, W, bias, C, ldc, M, N, K,
                         splits, part_blocks, here, stride, 0.0f, F32PairsOut{});
      return cw_launch_status();
    }
  }
  if (M <= GT_ROWS_MAX) {
    // as planes: four parts a block, each wave its own. Else all of a tile's parts in one block of up to
    // eight waves, and as many tiles as make it four waves or more.
    const int part_waves = planes ? (splits < 4 ? splits : 4) : (splits + (splits + 7) / 8 - 1) / ((splits + 7) / 8);
    const int tiles_here = planes || part_waves >= 4 ? 1 : 4 / part_waves;
    const int tiles = (N + 15) / 16;
    const dim3 grid((tiles + tiles_here - 1) / tiles_here, planes ? (splits + part_waves - 1) / part_waves : 1);
    const dim3 block(64 * part_waves * tiles_here);
    const size_t lds = planes ? 0 : (size_t)tiles_here * splits * 256 * sizeof(float);
    if (vec) hipLaunchKernelGGL(gemm_f32_rows_kernel<true>, grid, block, lds, stream, A, lda, W, bias, C, ldc, M, N, K, splits, per, part_waves, stride);
    else hipLaunchKernelGGL(gemm_f32_rows_kernel<false>, grid, block, lds, stream, A, lda, W, bias, C, ldc, M, N, K, splits, per, part_waves, stride);
    return cw_launch_status();
  }
  const int z = planes ? splits : 1;
  const int col_tiles = (N + 63) / 64;
  const bool one = planes || splits == 1;
  const dim3 block(256);
  if ((M + 63) / 64 > 65535) return CW_ERR_SIZE;
  // whole blocks of 16, and offsets that a 32-bit buffer descriptor reaches
  if (!(K & 15) && !(lda & 3) && ((int64_t)M * lda + K) * 4 < (int64_t)UINT32_MAX && (int64_t)N * K * 4 < (int64_t)UINT32_MAX) {
    const bool small = M <= 32 || (int64_t)((M + 63) / 64) * col_tiles * z < 256;
    const int64_t tiles = (int64_t)col_tiles * (small ? (M + 31) / 32 : (M + 63) / 64) * z;
    if (tiles > 0x7fffffff) return CW_ERR_SIZE;
    const dim3 grid((unsigned)tiles);
#define CW_RING_F32(BM_, ONE_)                                                                                     \
  hipLaunchKernelGGL((gemm_f32_ring_kernel<BM_, ONE_>), grid, block, 4 * (BM_ + 64) * 128, stream, A, lda, W, bias, C, ldc, M, N, K, \
                     splits, per, stride)
    if (small) { if (one) CW_RING_F32(32, true); else CW_RING_F32(32, false); }
    else { if (one) CW_RING_F32(64, true); else CW_RING_F32(64, false); }
#undef CW_RING_F32
    return cw_launch_status();
  }
  const dim3 grid(col_tiles, (M + 63) / 64, z);
#define CW_TILE_F32(VEC_, ONE_)                                                                                     \
  hipLaunchKernelGGL((gemm_f32_tile_kernel<VEC_, ONE_>), grid, block, 0, stream, A, lda, W, bias, C, ldc, M, N, K, \
                     splits, per, stride)
  if (vec) { if (one) CW_TILE_F32(true, true); else CW_TILE_F32(true, false); }
  else { if (one) CW_TILE_F32(false, true); else CW_TILE_F32(false, false); }
#undef CW_TILE_F32
  return cw_launch_status();
}

CW_EXPORT int cw_gemm_f32(const float* A, int64_t lda, const float* W, const float* bias, float* C,
                          int64_t ldc, int M, int N, int K, float* workspace, int64_t workspace_floats,
                          hipStream_t stream) {
  if (M < 0 || N <= 0 || K <= 0 || lda < K || ldc < N) return CW_ERR_ARG;
  if (M == 0) return CW_OK;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  int splits, per;
  gemm_f32_plan(N, K, &splits, &per);
  if (!gemm_f32_planes(M, N, K, splits))
    return launch_gemm_f32(A, lda, W, bias, C, ldc, M, N, K, splits, per, false, stream);
  const int64_t part_stride = (int64_t)M * N;
  if (workspace == nullptr || workspace_floats < splits * part_stride) return CW_ERR_ARG;
  const int rc = launch_gemm_f32(A, lda, W, nullptr, workspace, (int64_t)N, M, N, K, splits, per, true, stream);
  if (rc != CW_OK) return rc;
  hipLaunchKernelGGL(gemm_f32_sum_kernel, dim3((unsigned)((part_stride + 255) / 256)), dim3(256), 0, stream, workspace,
                     splits, part_stride, bias, C, ldc, M, N);
  return cw_launch_status();
}

// Does cw_gemm_f32_swiglu take this product (few rows, whole blocks of K that one workgroup takes)?
CW_EXPORT int cw_gemm_f32_swiglu_ok(int M, int N, int K, int64_t lda) {
  return M > 0 && M <= GT_ROWS_MAX && N > 0 && !(N & 1) && N <= 65536 && K > 0 && !(K & 15) && !(lda & 3) && lda >= K && K / 16 <= GT_BLOCKS ? 1 : 0;
}

// The gated product of W = [gate; up] [N, K] as float32 [M, N / 2]: what cw_gemm_f32 and the gate kernel give, bit for bit,
// without the [M, N] between them (``act`` as for the bfloat16 products).
CW_EXPORT int cw_gemm_f32_swiglu(const float* A, int64_t lda, const float* W, float* C, int64_t ldc, int M, int N, int K, float act,
                                 hipStream_t stream) {
  if (M == 0) return CW_OK;
  if (!cw_gemm_f32_swiglu_ok(M, N, K, lda) || ldc < N / 2 || !C || ((uintptr_t)A & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  int splits, per;
  gemm_f32_plan(N, K, &splits, &per);
  const size_t lds = (size_t)(K / 16 + splits) * M * 16 * sizeof(float);
  static std::atomic<bool> allowed{false};
  if (cw_allow_lds(allowed, (const void*)gemm_f32_blocks_kernel<GT_GLU>, GT_BLOCKS_LDS) != CW_OK) return CW_ERR_LAUNCH;
  hipLaunchKernelGGL(gemm_f32_blocks_kernel<GT_GLU>, dim3((N / 2 + 7) / 8), dim3(GT_BLOCK_WAVES * 64), lds, stream, A, lda, W, nullptr, C, ldc,
                     M, N, K, splits, per / 16, splits, 0, act, F32PairsOut{});
  return cw_launch_status();
}

// Does cw_gemm_f32_pairs take queries, keys and values of these heads (rotated whole) of few rows, whole blocks of K?
CW_EXPORT int cw_gemm_f32_pairs_ok(int M, int K, int nh, int nkv, int hd) {
  return nh > 0 && nkv > 0 && hd > 0 && !(hd & 15) && hd <= 1024 && nh + 2 * nkv <= 65536 / hd && M > 0 && M <= GT_ROWS_MAX && K > 0 && !(K & 15) &&
                 K / 16 <= GT_BLOCKS
             ? 1
             : 0;
}

// A [M, K] W^T + bias for W [(nh + 2 nkv) hd, K]: rotated queries to Q [M, nh hd], rotated keys and the values to rows ``slots`` of
// the caches (negative, or past cache_rows: none). What cw_gemm_f32 and cw_rope_kv_write give, in one kernel; bias or nullptr.
CW_EXPORT int cw_gemm_f32_pairs(const float* A, const float* W, const float* bias, const int* positions, const int* slots,
                                const float* inv_freq, float* Q, float* k_cache, float* v_cache, int64_t cache_rows, int M, int K,
                                int nh, int nkv, int hd, hipStream_t stream) {
  if (M == 0) return CW_OK;
  if (!cw_gemm_f32_pairs_ok(M, K, nh, nkv, hd)) return CW_ERR_SIZE;
  if (!A || !W || !positions || !slots || !inv_freq || !Q || !k_cache || !v_cache || ((uintptr_t)A & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  const int N = (nh + 2 * nkv) * hd;
  int splits, per;
  gemm_f32_plan(N, K, &splits, &per);
  const size_t lds = (size_t)(K / 16 + splits) * M * 16 * sizeof(float);
  static std::atomic<bool> allowed{false};
  if (cw_allow_lds(allowed, (const void*)gemm_f32_blocks_kernel<GT_PAIRS>, GT_BLOCKS_LDS) != CW_OK) return CW_ERR_LAUNCH;
  hipLaunchKernelGGL(gemm_f32_blocks_kernel<GT_PAIRS>, dim3(N / 16), dim3(GT_BLOCK_WAVES * 64), lds, stream, A, (int64_t)K, W, bias, Q,
                     (int64_t)nh * hd, M, N, K, splits, per / 16, splits, 0, 0.0f,
                     F32PairsOut{positions, slots, inv_freq, k_cache, v_cache, cache_rows, nh, nkv, hd});
  return cw_launch_status();
}

// The parts of the product as they are, float32 [cw_gemm_f32_partial_planes(M, N, K), M, N]: added in order
// they are what cw_gemm_f32 gives (without a bias), bit for bit. For a result that the residual-add + norm
// kernel reads next, which adds them itself.
CW_EXPORT int cw_gemm_f32_partial(const float* A, int64_t lda, const float* W, float* planes, int M, int N, int K,
                                  hipStream_t stream) {
  if (M < 0 || N <= 0 || K <= 0 || lda < K || !planes) return CW_ERR_ARG;
  if (M == 0) return CW_OK;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  int splits, per;
  gemm_f32_plan(N, K, &splits, &per);
  if (cw_gemm_f32_partial_planes(M, N, K) != splits) return CW_ERR_SIZE;
  return launch_gemm_f32(A, lda, W, nullptr, planes, (int64_t)N, M, N, K, splits, per, true, stream);
}

// =====================================================================================
// bfloat16 products with few rows of x (decode: 1 to 64 tokens): the weight matrix is streamed
// once at memory speed. A workgroup of WAVES waves owns RT * 16 weight rows; its waves split the K
// loop and are summed through LDS at the end, in a fixed order (no atomics: the result does not
// depend on timing). Few weight rows (a narrow output) get more waves each, so that enough loads
// are in flight on every compute unit that has work.
// Each wave feeds 16 weight rows x 32 k-values to one MFMA (v_mfma_f32_16x16x32_bf16) as the A
// operand, loaded from global memory directly in operand layout (lane = row l%16, 8 consecutive
// k at slot l/16), and 16 tokens x the same k-values as the B operand.
//
// MODE 0: y bfloat16 [M, N]; MODE 4: the same with the erf GELU (``act`` > 0: its tanh form) applied
// to the float32 sums before they are rounded; MODE 5: with max(z, 0)^2 applied to them; MODE 1: y float32 [M, N] (logits); MODE 2: W is [2I, K] with gate
// rows first, y[m, i] = silu(gate_i) * up_i as bfloat16 [M, I] (``act`` > 0: the clipped gated
// activation with that limit instead; -1: max(gate, 0) * up, -2: gelu_tanh(gate) * up): a row tile holds 8 gate rows and the 8 up rows that belong to them. MODE 3: K is also split over gridDim.y workgroups, each
// writing its float32 partial product [split, M, N]; whoever reads y next sums the partials in
// order (the residual-add + norm kernel does): a narrow output with a long K (96 row tiles for
// 27 MB of weights) then streams on all compute units instead of 96.
__device__ __forceinline__ float cw_gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752440f)); }
__device__ __forceinline__ float cw_relu_squared(float z) { const float r = fmaxf(z, 0.0f); return r * r; }

// A norm that the product before has begun (gemm_join_bf16_kernel): x holds the rows times the norm's weights, ``squares``
// [M, parts] the sums of squares of each row's pieces (parts: a multiple of 4, at most 256). A row's factor 1 / sqrt(mean + eps)
// multiplies the finished sums instead of the elements, so no product waits for it: the pieces are asked for ahead of the
// weights, and a wave adds up those of its rows (wave, wave + WAVES, ...) while or after the weights come in.
struct RowFactors {
  const float* squares;
  int parts;
  float of_width, eps;  // 1 / elements of a row
};
template <int WAVES> struct RowPieces {
  static constexpr int ROWS = 16 / WAVES;
  float4 v[ROWS];
  __device__ __forceinline__ void load(const RowFactors& in, int M) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int m = wave + i * WAVES;
      v[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (m < M && lane * 4 < in.parts) v[i] = *reinterpret_cast<const float4*>(in.squares + m * in.parts + lane * 4);
    }
  }
  // visible behind the next barrier
  __device__ __forceinline__ void factors(const RowFactors& in, float* to) const {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const float total = cw_wave_sum((v[i].x + v[i].y) + (v[i].z + v[i].w));
      if ((threadIdx.x & 63) == 0) to[(threadIdx.x >> 6) + i * WAVES] = __builtin_amdgcn_rsqf(fmaf(total, in.of_width, in.eps));
    }
  }
};

// ROWS (16, 8 or 4) is the number of weight rows a tile really holds: a narrow output with a long K
// is cut into more, smaller tiles so that every compute unit streams a share of the matrix (the
// unused rows of the MFMA tile are zeros). MODE 2 needs ROWS == 16.
template <int MT, int RT, int MODE, int WAVES, int ROWS, bool BEGUN = false>
__device__ __forceinline__ void skinny_tiles(const bf16_t* __restrict__ X, int64_t ldx, const bf16_t* __restrict__ W,
                                             void* __restrict__ C, int64_t ldc, int M, int N, int K, float act, const int block,
                                             const RowFactors& begun = RowFactors{}) {
  static_assert(!BEGUN || (MT == 1 && MODE == 2), "begun norms are gate/up products' of up to 16 rows");
  __shared__ float red[WAVES][RT * MT * 256];
  __shared__ float factors[16];
  [[maybe_unused]] RowPieces<WAVES> pieces;
  if constexpr (BEGUN) pieces.load(begun, M);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, s = lane >> 4;
  const int lr = lane >> 2, ls = lane & 3;  // the row of a tile and the slot of a k-step that this lane loads
  const int I = N / 2;  // MODE 2 only

  // weight rows that this lane loads, one per row tile
  const bf16_t* wrow[RT];
  bool wok[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    int64_t n;
    if (MODE == 2) {
      const int64_t i = ((int64_t)block * RT + rt) * 8 + (lr & 7);
      n = (lr < 8) ? i : I + i;
      wok[rt] = i < I;
    } else {
      n = ((int64_t)block * RT + rt) * ROWS + lr;
      wok[rt] = lr < ROWS && n < N;
    }
    wrow[rt] = W + (wok[rt] ? n : 0) * K;
  }
  // x: one tile of tokens is few bytes beside the weights and is loaded in operand layout as it is
  // (a swap would only add to the wait before the first product); several tiles are loaded like the weights
  constexpr bool X_SWAP = MT > 1;
  const int xr = X_SWAP ? lr : r, xs = X_SWAP ? ls : s;
  const bf16_t* xrow[MT];
  bool xok[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + xr;
    xok[mt] = m < M;
    xrow[mt] = X + (int64_t)(xok[mt] ? m : 0) * ldx;
  }

  f32x4_t acc[RT][MT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};

  bf16x8_t zero;
#pragma unroll
  for (int e = 0; e < 8; ++e) zero[e] = (__bf16)0.0f;

  const int k_steps = (K + 31) / 32;
  constexpr int U = 4;  // k-steps in flight per wave
  const int n_ksplit = MODE == 3 ? gridDim.y : 1;
  int ks0 = ((MODE == 3 ? blockIdx.y : 0) * WAVES + wave) * U;
  [[maybe_unused]] bool first = true;
  // (BEGUN: also a wave without a step adds up its rows' pieces)
  for (; BEGUN && first || ks0 < k_steps; ks0 += n_ksplit * WAVES * U) {
    bf16x8_t wf[U][RT], xf[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (ks0 + u) * 32 + ls * 8;
      const bool kok = (ks0 + u) < k_steps && k + 8 <= K;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        wf[u][rt] = (kok && wok[rt]) ? *reinterpret_cast<const bf16x8_t*>(wrow[rt] + k) : zero;
      const int kx = (ks0 + u) * 32 + xs * 8;
      const bool kxok = (ks0 + u) < k_steps && kx + 8 <= K;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        xf[u][mt] = (kxok && xok[mt]) ? *reinterpret_cast<const bf16x8_t*>(xrow[mt] + kx) : zero;
    }
    if constexpr (BEGUN) {
      if (first) pieces.factors(begun, factors);
      first = false;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      bf16x8_t xo[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xo[mt] = X_SWAP ? cw_to_operand_layout(xf[u][mt], lane) : xf[u][mt];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const bf16x8_t wo = cw_to_operand_layout(wf[u][rt], lane);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wo, xo[mt], acc[rt][mt], 0, 0, 0);
      }
    }
  }

  // D tile of (rt, mt): lane (r, s) holds weight rows 4s..4s+3 of token r -> red[wave][tile][row][token]
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][(rt * MT + mt) * 256 + (4 * s + i) * 16 + r] = acc[rt][mt][i];
  __syncthreads();
  for (int idx = threadIdx.x; idx < RT * MT * 256; idx += WAVES * 64) {
    float sum = red[0][idx];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += red[w][idx];
    red[0][idx] = sum;
  }
  __syncthreads();

  if (MODE == 2) {
    // outputs: 8 per row tile and token; idx -> (token, rt, j) with j fastest
    for (int idx = threadIdx.x; idx < RT * MT * 128; idx += WAVES * 64) {
      const int j = idx & 7, rt = (idx >> 3) % RT, m = idx / (8 * RT);
      const int mt = m >> 4, tok = m & 15;
      const int64_t i = ((int64_t)block * RT + rt) * 8 + j;
      if (m >= M || i >= I) continue;
      const float factor = BEGUN ? factors[m] : 1.0f;
      const float g = red[0][(rt * MT + mt) * 256 + j * 16 + tok] * factor;
      const float u = red[0][(rt * MT + mt) * 256 + (j + 8) * 16 + tok] * factor;
      ((bf16_t*)C)[(int64_t)m * ldc + i] = __float2bfloat16(act > 0.0f ? cw_clipped_glu(g, u, act) : act < 0.0f ? cw_gated_below(g, u, act) : g / (1.0f + __expf(-g)) * u);
    }
  } else {
    for (int idx = threadIdx.x; idx < RT * MT * 256; idx += WAVES * 64) {
      const int j = idx & 15, rt = (idx >> 4) % RT, m = idx / (16 * RT);
      const int mt = m >> 4, tok = m & 15;
      const int64_t n = ((int64_t)block * RT + rt) * ROWS + j;
      if (m >= M || n >= N || j >= ROWS) continue;
      const float v = red[0][(rt * MT + mt) * 256 + j * 16 + tok];
      if (MODE == 3) ((float*)C)[((int64_t)blockIdx.y * M + m) * ldc + n] = v;
      else if (MODE == 1) ((float*)C)[(int64_t)m * ldc + n] = v;
      else if (MODE == 4) ((bf16_t*)C)[(int64_t)m * ldc + n] = __float2bfloat16(act > 0.0f ? cw_gelu_tanh(v) : cw_gelu_erf(v));
      else if (MODE == 5) ((bf16_t*)C)[(int64_t)m * ldc + n] = __float2bfloat16(cw_relu_squared(v));
      else ((bf16_t*)C)[(int64_t)m * ldc + n] = __float2bfloat16(v);
    }
  }
}

template <int MT, int RT, int MODE, int WAVES, int ROWS>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_bf16_kernel(const bf16_t* __restrict__ X, int64_t ldx,
                                                               const bf16_t* __restrict__ W,
                                                               void* __restrict__ C, int64_t ldc,
                                                               int M, int N, int K, float act) {
  skinny_tiles<MT, RT, MODE, WAVES, ROWS>(X, ldx, W, C, ldc, M, N, K, act, blockIdx.x);
}

template <int RT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_begun_bf16_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                                            bf16_t* __restrict__ C, int64_t ldc, int M, int N, int K,
                                                                            float act, RowFactors begun) {
  skinny_tiles<1, RT, 2, WAVES, 16, true>(X, K, W, C, ldc, M, N, K, act, blockIdx.x, begun);
}

// Several products of the same rows and the same K as one launch, each with an x, a matrix and an output of its own: a layer that
// multiplies one input by three matrices of 2 to 5 thousand rows, or two inputs by a matrix each. By itself such a product streams
// 1 to 2.5 TB/s, for its 100 to 300 row tiles leave compute units idle and every launch pays its ramp of 2 to 3 us. Measured on an
// MI355X, a width of 1536, apart and together (us): 8 rows, outputs of 2048, 4640 and 3072 16.6 and 7.6, two of 1536 9.2 and 5.1;
// one row 13.7 and 7.5, 7.6 and 4.4; a width of 896, three outputs of 2048, 2000 and 1024, 8 rows 9.7 and 3.7.
#define GROUP_MAX 4
struct ProductGroup {
  const bf16_t* x[GROUP_MAX];
  const bf16_t* w[GROUP_MAX];
  bf16_t* c[GROUP_MAX];
  int n[GROUP_MAX];
  int first[GROUP_MAX + 1];  // tiles of 16 rows of W before each product's, INT_MAX past the last
};
// the product that row tile ``tile`` belongs to (the same for a whole workgroup)
__device__ __forceinline__ int group_of(const ProductGroup& group, int tile) {
  int g = 0;
#pragma unroll
  for (int i = 1; i < GROUP_MAX; ++i) g += tile >= group.first[i];
  return g;
}

template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_group_bf16_kernel(ProductGroup group, int M, int K) {
  const int g = group_of(group, blockIdx.x);
  skinny_tiles<1, 1, 0, WAVES, 16>(group.x[g], K, group.w[g], group.c[g], group.n[g], M, group.n[g], K, 0.0f, (int)blockIdx.x - group.first[g]);
}

// The same product with the x fragments of a wave's whole share of the K loop (up to 24 steps of
// 32, as many as its registers hold beside MT tiles of 16 tokens) kept in registers for good, so
// that only weights move.
// A workgroup walks over row tiles blockIdx.x, blockIdx.x + gridDim.x, ...; the weights of its
// next tile are on their way while the current one is reduced through LDS (one barrier per tile
// while the reduction buffer can be doubled, two for MT = 4). Loads are never conditional: a row
// or k-step outside the matrix reads a valid address instead and meets zeros in x or is not
// stored, which lets the compiler wait for exactly the loads a product needs. Wave w of k-split
// blockIdx.y owns k-steps [(blockIdx.y * WAVES + w) * SPW, + SPW). Modes and layouts as in
// gemm_skinny_bf16_kernel.
// NORM (MT = 1, no k-split): x is not read but made here, x = rmsnorm(resid + delta) * weight over
// the K elements of a row, with the rounding steps of the stand-alone norm kernel; every
// workgroup does so for itself (the rows are few and come from L2), nothing is written back.
static __device__ uint4 cw_zeros[1];  // 8 elements (never written; not const, or loads from it or a matrix would be flat ones)

struct StreamNormIn {
  const float* resid;    // [M, K] float32
  const bf16_t* delta;   // [M, K] bfloat16
  const void* weight;    // [K] bfloat16 or float32
  int weight_f32;
  float eps;
};

// Weight fragments of a tile are fetched CH steps at a time (two sets in flight), while the x
// fragments of all SPW steps stay in registers: a long K costs registers for x only.
constexpr int cw_stream_chunk(int spw) { return spw <= 8 ? spw : (spw <= 12 ? spw / 2 : spw / 4); }

// GROUP (MODE 0): row tiles of several products of the same x, ``in`` a ProductGroup (W, C, ldc and N are not used).
// BEGUN (MODE 2, MT = 1): x comes with its norm begun, ``in`` a RowFactors.
// LINES: whole lines a load, which the caches need not keep: a stream of 110 MB comes in at 5.8 TB/s so and at 5.2 otherwise (half lines a
// load that the caches need not keep: each comes twice), and what the step reads beside it has the caches for itself. us, without / with: [gate;
// up] of 37888 x 3584 with 1, 8, 16 rows 48.8 / 43.0, 49.3 / 43.3, 51.0 / 44.5; 152064 x 3584 184 / 163, 190 / 170, 202 / 178; 151936 x 1536 with 1, 16, 64
// rows 79 / 73, 89 / 80, 107 / 97; 17920 x 1536 12.0 / 11.9 to 14.3 / 13.8 (32 rows). In a wave's one pair (K up to 1024) of more than 16 rows
// nothing is left of that (151936 x 896 with 32, 64 rows 60.2 / 60.7, 69.9 / 70.3), nor in partial sums of fewer than 64 MB (MODE 3; 1536 x 8960 6.7
// to 10.8 / 7.6 to 10.1, the first row's wait for memory is the longer one; 3584 x 18944 with 1, 8, 16, 32 rows 25.0 / 24.3, 26.9 / 25.8, 28.3 / 28.3, 29.5 / 29.1;
// 5120 x 13824 25.8 / 24.0, 27.5 / 24.6, 28.4 / 25.7, 29.3 / 27.3). A step of one request, us: 0.5B shape 714 / 703, 7B shape 3212 / 3085.
template <int MODE, int WAVES, int SPW, int MT, bool NORM = false, bool GROUP = false, bool BEGUN = false, bool LINES = MODE != 3 && (MT == 1 || SPW > 2)>
__global__ __launch_bounds__(WAVES * 64) void gemm_stream_bf16_kernel(const bf16_t* __restrict__ X, int64_t ldx,
                                                               const bf16_t* __restrict__ W,
                                                               void* __restrict__ C, int64_t ldc,
                                                               int M, int N, int K, int n_tiles, float act,
                                                               std::conditional_t<GROUP, ProductGroup, std::conditional_t<BEGUN, RowFactors, StreamNormIn>> in) {
  static_assert(!BEGUN || (MODE == 2 && MT == 1 && !NORM), "begun norms are gate/up products' of up to 16 rows");
  static_assert(!GROUP || (MODE == 0 && !NORM), "grouped products are plain ones");
  constexpr int NBUF = MT <= 2 ? 2 : 1;
  constexpr int CH = cw_stream_chunk(SPW), NC = SPW / CH;
  static_assert(SPW % CH == 0, "the steps of a wave are whole chunks");
  __shared__ __align__(16) float red[NBUF][WAVES][MT * 256];
  const int lane = threadIdx.x & 63, wave = LINES ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
  const int r = lane & 15, s = lane >> 4;
  const int I = N / 2;  // MODE 2 only
  __shared__ float factors[16];
  [[maybe_unused]] RowPieces<WAVES> pieces;
  if constexpr (BEGUN) pieces.load(in, M);

  // Loads as cw_to_operand_layout describes: this lane loads row lr of a tile, slot ls of a k-step.
  const int lr = lane >> 2, ls = lane & 3;
  auto to_operand = [&](const bf16x8_t& v) __attribute__((always_inline)) -> bf16x8_t {
    return cw_to_operand_layout(v, lane);
  };
  // LINES: weights come in two steps of K a pair of loads (cw_lines_to_steps), which begin at even steps; of an odd number of steps the
  // wave's first or last is left over and loaded alone, as x is.
  constexpr int PAIRED = LINES ? CH & ~1 : 0;  // fragments of a set that come in pairs
  const int step0 = (blockIdx.y * WAVES + wave) * SPW;
  auto step_of = [&](int u) __attribute__((always_inline)) -> int {  // that set of fragments u of the wave holds
    const int begin = step0 + u / CH * CH, i = u % CH;
    if (!LINES || (CH & 1) == 0) return begin + i;
    const int late = begin & 1;
    return i < CH - 1 ? begin + late + i : begin + (late ? 0 : CH - 1);
  };
  // Where the loading lane finds its 8 k-values of a step or, with 8 slots, of a pair. What lies outside of K meets zeros in x; it reads zeros, so
  // that an infinite weight stays one, or in the products with a long K, whose loads the choice of address would slow by 4 %, k = 0;
  // there a pair outside of K as a whole reads the row's last one, which is on its way, and becomes zeros (k = 0, not kept by the caches, came from
  // memory each time: 18944 columns of 3584 rows, where a wave in thirteen lies outside, 26.8 -> 24.3 us with 1 row, 27.7 -> 25.8 with 8).
  constexpr bool ZEROS = MODE != 3 && NC == 1;
  int koff[SPW];  // one load at a time
#pragma unroll
  for (int u = 0; u < SPW; ++u) {
    const int k = (step0 + u) * 32 + ls * 8;
    koff[u] = k + 8 <= K ? k : ZEROS ? -1 : 0;
  }
  auto at = [&](const bf16_t* row, int u, int slot, bool pair) __attribute__((always_inline)) -> const bf16x8_t* {
    const int begin = step_of(u) * 32, k = (!ZEROS && pair && begin >= K ? max(K - 64, 0) : begin) + slot * 8;
    return reinterpret_cast<const bf16x8_t*>(k + 8 <= K ? row + k : ZEROS ? reinterpret_cast<const bf16_t*>(cw_zeros) : row);
  };
  auto wrow = [&](int tile, int tile_row) __attribute__((always_inline)) -> const bf16_t* {
    int64_t n;
    if constexpr (GROUP) {
      const int g = group_of(in, tile);
      return in.w[g] + (int64_t)min((tile - in.first[g]) * 16 + tile_row, in.n[g] - 1) * K;
    }
    if (MODE == 2) {  // gate and up rows alternate, so that a pair lies side by side in the tile
      const int64_t i = min((int64_t)tile * 8 + (tile_row >> 1), (int64_t)I - 1);
      n = (tile_row & 1) ? I + i : i;
    } else {
      n = min((int64_t)tile * 16 + tile_row, (int64_t)N - 1);
    }
    return W + n * K;
  };
  struct Rows {
    const bf16_t *even, *odd, *alone;
  };
  auto rows_of = [&](int tile) __attribute__((always_inline)) -> Rows {
    const int first = (lane >> 3) * 2;
    return {PAIRED ? wrow(tile, first) : nullptr, PAIRED ? wrow(tile, first + 1) : nullptr, PAIRED < CH ? wrow(tile, lr) : nullptr};
  };
  // (whole lines that nobody reads again: they leave the caches to the others)
  auto weights = [&](bf16x8_t (&dst)[CH], const Rows& rows, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PAIRED; u += 2) {
      dst[u] = __builtin_nontemporal_load(at(rows.even, c * CH + u, lane & 7, true));
      dst[u + 1] = __builtin_nontemporal_load(at(rows.odd, c * CH + u, lane & 7, true));
    }
#pragma unroll
    for (int u = PAIRED; u < CH; ++u) dst[u] = LINES ? *at(rows.alone, c * CH + u, ls, false) : *reinterpret_cast<const bf16x8_t*>(!ZEROS || koff[c * CH + u] >= 0 ? rows.alone + koff[c * CH + u] : reinterpret_cast<const bf16_t*>(cw_zeros));
  };
  auto products = [&](bf16x8_t (&w)[CH], const auto& x, int c, f32x4_t (&acc)[MT]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (u % 2 == 0 && u < PAIRED) {
        if (!ZEROS && step_of(c * CH + u) * 32 >= K) w[u] = w[u + 1] = bf16x8_t{};
        cw_lines_to_steps(w[u], w[u + 1]);
      }
      const bf16x8_t wu = to_operand(w[u]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wu, x[c * CH + u][mt], acc[mt], 0, 0, 0);
    }
  };
  // the first tile's weights are requested before anything else: x, and with NORM the norm's
  // statistics, are fetched in their shadow
  int tile = blockIdx.x;
  bf16x8_t cur[CH], nxt[CH];
  Rows w_tile = rows_of(tile);
  weights(cur, w_tile, 0);

  bf16x8_t xf[SPW][MT];
  if constexpr (NORM) {
    static_assert(MT == 1 && SPW <= 4, "the fused norm serves one tile of tokens and rows of up to 2048 elements");
    __shared__ float ssq[WAVES][16];
    float v[SPW][8], wv[SPW][8];  // resid + delta and the norm weight at the lane's elements
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < SPW; ++u) {
      const int k = step_of(u) * 32 + s * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[u][e] = wv[u][e] = 0.0f;
      if (k + 8 <= K && r < M) {
        const float4 a = *reinterpret_cast<const float4*>(in.resid + (int64_t)r * K + k);
        const float4 b = *reinterpret_cast<const float4*>(in.resid + (int64_t)r * K + k + 4);
        const bf16x8_t d = *reinterpret_cast<const bf16x8_t*>(in.delta + (int64_t)r * K + k);
        v[u][0] = a.x + (float)d[0]; v[u][1] = a.y + (float)d[1]; v[u][2] = a.z + (float)d[2]; v[u][3] = a.w + (float)d[3];
        v[u][4] = b.x + (float)d[4]; v[u][5] = b.y + (float)d[5]; v[u][6] = b.z + (float)d[6]; v[u][7] = b.w + (float)d[7];
        if (in.weight_f32) {
          const float4 w0 = *reinterpret_cast<const float4*>((const float*)in.weight + k);
          const float4 w1 = *reinterpret_cast<const float4*>((const float*)in.weight + k + 4);
          wv[u][0] = w0.x; wv[u][1] = w0.y; wv[u][2] = w0.z; wv[u][3] = w0.w;
          wv[u][4] = w1.x; wv[u][5] = w1.y; wv[u][6] = w1.z; wv[u][7] = w1.w;
        } else {
          const bf16x8_t w8 = *reinterpret_cast<const bf16x8_t*>((const bf16_t*)in.weight + k);
#pragma unroll
          for (int e = 0; e < 8; ++e) wv[u][e] = (float)w8[e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += v[u][e] * v[u][e];
      }
    }
    ss = cw_quad_sum(ss);
    if (s == 0) ssq[wave][r] = ss;
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) total += ssq[w][r];
    const float inv = 1.0f / sqrtf(total / (float)K + in.eps);
#pragma unroll
    for (int u = 0; u < SPW; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) xf[u][0][e] = (__bf16)(wv[u][e] * (float)(__bf16)(v[u][e] * inv));
  } else {
    // Every workgroup pulls all of x from L2 (with 64 rows that is as many bytes as its weights),
    // loaded like the weights, four lanes to a row's step, and swapped into operand layout. The
    // loads are unconditional, from clamped addresses; what lies past M or K is zeroed first.
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = mt * 16 + lr;
      const bf16_t* xrow = X + (int64_t)min(m, M - 1) * ldx;
#pragma unroll
      for (int u = 0; u < SPW; ++u) {
        const int k = LINES ? step_of(u) * 32 + ls * 8 : koff[u];
        const bool ok = step_of(u) * 32 + ls * 8 + 8 <= K && m < M;
        bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(xrow + (LINES ? (k + 8 <= K ? k : 0) : ZEROS ? max(k, 0) : k));
        if (!ok) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (__bf16)0.0f;
        }
        xf[u][mt] = to_operand(v);
      }
    }
  }
  if constexpr (BEGUN) pieces.factors(in, factors);
  // what the waves' partial tiles of ``tile`` (in red[buf]) become: summed over the waves, then
  // stored as the mode says. One barrier before; a second after, when the buffer is not doubled.
  auto finish_tile = [&](const f32x4_t (&acc)[MT], int tile, int buf) __attribute__((always_inline)) {
    // lane (r, s) holds weight rows 4s..4s+3 of token r of tile mt -> red[buf][wave][mt][token][row]:
    // one 16-byte store a lane, the lanes of a wave side by side (no bank is hit twice)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      *reinterpret_cast<f32x4_t*>(&red[buf][wave][mt * 256 + r * 16 + 4 * s]) = acc[mt];
    cw_lds_barrier();  // not __syncthreads(): the next tile's weights stay in flight across it
    if (MODE == 2) {
      if (threadIdx.x < MT * 128) {  // (token, j): the gate and the up value of output j are neighbours
        const int j = threadIdx.x & 7, m = threadIdx.x >> 3;
        float g = 0.0f, up = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
          const float2 gu = *reinterpret_cast<const float2*>(&red[buf][w][m * 16 + 2 * j]);
          g += gu.x;
          up += gu.y;
        }
        if constexpr (BEGUN) {
          g *= factors[m];
          up *= factors[m];
        }
        const int64_t i = (int64_t)tile * 8 + j;
        if (m < M && i < I) ((bf16_t*)C)[(int64_t)m * ldc + i] =
              __float2bfloat16(act > 0.0f ? cw_clipped_glu(g, up, act) : act < 0.0f ? cw_gated_below(g, up, act) : g / (1.0f + __expf(-g)) * up);
      }
    } else {
      for (int idx = threadIdx.x; idx < MT * 256; idx += WAVES * 64) {  // (token, j): 16 outputs side by side
        const int j = idx & 15, m = idx >> 4;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) v += red[buf][w][idx];
        if constexpr (GROUP) {
          const int g = group_of(in, tile), n = (tile - in.first[g]) * 16 + j;
          if (m < M && n < in.n[g]) in.c[g][(int64_t)m * in.n[g] + n] = __float2bfloat16(v);
          continue;
        }
        const int64_t n = (int64_t)tile * 16 + j;
        if (m < M && n < N) {
          if (MODE == 3) ((float*)C)[((int64_t)blockIdx.y * M + m) * ldc + n] = v;
          else if (MODE == 1) ((float*)C)[(int64_t)m * ldc + n] = v;
          else if (MODE == 4) ((bf16_t*)C)[(int64_t)m * ldc + n] = __float2bfloat16(act > 0.0f ? cw_gelu_tanh(v) : cw_gelu_erf(v));
          else if (MODE == 5) ((bf16_t*)C)[(int64_t)m * ldc + n] = __float2bfloat16(cw_relu_squared(v));
          else ((bf16_t*)C)[(int64_t)m * ldc + n] = __float2bfloat16(v);
        }
      }
    }
    if (NBUF == 1) cw_lds_barrier();
  };
  int buf = 0;
  if constexpr (NC == 1) {
    // A wave's whole share of a tile is one set of fragments. Two sets take turns, without a
    // copy between them (a copy has to wait for the loads it copies): the loads of the tile
    // after this one are issued before this tile's products and are waited for only when their
    // own products begin, so they are in flight during the whole of this tile's products,
    // reduction and stores. Past the last tile a valid address is read and dropped.
    auto load_set = [&](bf16x8_t (&dst)[CH], int t) __attribute__((always_inline)) { weights(dst, rows_of(min(t, n_tiles - 1)), 0); };
    auto zero = [&](f32x4_t (&acc)[MT]) __attribute__((always_inline)) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
    };
    const int stride = (int)gridDim.x;
    while (tile < n_tiles) {
      f32x4_t acc[MT];
      load_set(nxt, tile + stride);
      __builtin_amdgcn_sched_barrier(0);  // the loads stay in front of the products
      zero(acc);
      products(cur, xf, 0, acc);
      finish_tile(acc, tile, buf);
      buf = (buf + 1) % NBUF;
      tile += stride;
      if (tile >= n_tiles) break;
      load_set(cur, tile + stride);
      __builtin_amdgcn_sched_barrier(0);
      zero(acc);
      products(nxt, xf, 0, acc);
      finish_tile(acc, tile, buf);
      buf = (buf + 1) % NBUF;
      tile += stride;
    }
  } else {
    for (; tile < n_tiles; tile += gridDim.x) {
      const Rows w_next = rows_of(min(tile + (int)gridDim.x, n_tiles - 1));
      f32x4_t acc[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        // the chunk after this one: of this tile, or the first of the workgroup's next tile
        if (c + 1 < NC) weights(nxt, w_tile, c + 1);
        else weights(nxt, w_next, 0);
        products(cur, xf, c, acc);
#pragma unroll
        for (int u = 0; u < CH; ++u) cur[u] = nxt[u];
      }
      w_tile = w_next;
      finish_tile(acc, tile, buf);
      buf = (buf + 1) % NBUF;
    }
  }
}

static int cw_num_compute_units() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 256;
    cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  }
  return cus;
}

// Do a wave's x fragments, two sets of weight fragments and the accumulators fit its registers?
constexpr bool cw_stream_fits(int waves, int spw, int mt) {
  return spw * mt * 4 + cw_stream_chunk(spw) * 8 + mt * 4 <= (waves == 16 ? 100 : 220);
}

// Steps per wave the kernel is built for: every count up to 8, then even counts, then multiples of 4.
constexpr int cw_stream_round_spw(int spw) {
  return spw <= 8 ? spw : (spw <= 12 ? (spw + 1) / 2 * 2 : (spw + 3) / 4 * 4);
}

template <int MODE, int WAVES, int SPW, int MT>
static int launch_stream_one(dim3 grid, const bf16_t* X, int64_t ldx, const bf16_t* W, void* C, int64_t ldc,
                             int M, int N, int K, int n_tiles, float act, hipStream_t stream) {
  if constexpr (cw_stream_fits(WAVES, SPW, MT)) {
    if constexpr (MODE == 3 && SPW >= 4) {
      if ((int64_t)N * K >= (1 << 25)) {
        hipLaunchKernelGGL((gemm_stream_bf16_kernel<MODE, WAVES, SPW, MT, false, false, false, true>), grid, dim3(WAVES * 64), 0, stream, X, ldx,
                           W, C, ldc, M, N, K, n_tiles, act, StreamNormIn{});
        return cw_launch_status();
      }
    }
    hipLaunchKernelGGL((gemm_stream_bf16_kernel<MODE, WAVES, SPW, MT>), grid, dim3(WAVES * 64), 0, stream, X, ldx,
                       W, C, ldc, M, N, K, n_tiles, act, StreamNormIn{});
    return cw_launch_status();
  } else {
    return CW_ERR_SIZE;
  }
}

template <int MODE, int WAVES, int MT>
static int launch_stream(int spw, dim3 grid, const bf16_t* X, int64_t ldx, const bf16_t* W, void* C, int64_t ldc,
                         int M, int N, int K, int n_tiles, float act, hipStream_t stream) {
#define CW_STREAM(SPW_) \
  case SPW_: return launch_stream_one<MODE, WAVES, SPW_, MT>(grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream)
  switch (spw) {
    CW_STREAM(1); CW_STREAM(2); CW_STREAM(3); CW_STREAM(4); CW_STREAM(5); CW_STREAM(6); CW_STREAM(7); CW_STREAM(8);
    CW_STREAM(10); CW_STREAM(12); CW_STREAM(16); CW_STREAM(20); CW_STREAM(24);
    default: return CW_ERR_SIZE;
  }
#undef CW_STREAM
}

template <int MODE, int WAVES>
static int launch_stream_mt(int mt, int spw, dim3 grid, const bf16_t* X, int64_t ldx, const bf16_t* W, void* C,
                            int64_t ldc, int M, int N, int K, int n_tiles, float act, hipStream_t stream) {
  if (mt == 1) return launch_stream<MODE, WAVES, 1>(spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
  if (mt == 2) return launch_stream<MODE, WAVES, 2>(spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
  return launch_stream<MODE, WAVES, 4>(spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
}

// Shape of the streaming kernel's launch for this product, or false if it does not apply: a
// wave's share of K must be short enough for its registers and there must be enough row tiles.
static bool plan_stream(int mode, int M, int N, int K, int k_splits, int* mt, int* spw, dim3* grid, int* n_tiles) {
  const int k_steps = (K + 31) / 32;
  *n_tiles = mode == 2 ? (N / 2 + 7) / 8 : (N + 15) / 16;
  const int waves = mode == 3 ? 8 : 16;
  *mt = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
  *spw = cw_stream_round_spw((k_steps + k_splits * waves - 1) / (k_splits * waves));
  // A K of less than two steps a wave leaves waves idle and still is the faster way from 16 steps on beyond 16 rows, where the other
  // way is a library product, and from 24 on for fewer, where it is a workgroup a tile or four (us, that way / this one: [gate;
  // up] of 9728 x 896 with 1, 8, 16 rows 6.0 / 6.0, 6.7 / 5.9, 7.7 / 5.9, with 17, 32, 64 14.1 / 6.7, 14.2 / 6.7, 14.7 / 9.4; 151936 x 896 53.5 / 49.1,
  // 61.5 / 55.9, 65.9 / 58.0, 71.3 / 59.7, 74.9 / 62.9, 85.9 / 71.9; [gate; up] of 6144 x 768 3.8 / 3.7 to 4.3 / 4.3, 9.9 / 4.8 to 10.3 / 6.9; 16384 x 512
  // with 1 and 8 rows 5.5 / 6.1, 5.9 / 5.8, with 17 to 64 12.5 / 6.6 to 12.7 / 9.8, its head of 151936 31.7 / 40.4, 35.4 / 41.1, 66.6 / 43.4, 66.0 / 59.2).
  const int least_steps = M > 16 ? waves : waves + waves / 2;
  if (M > 64 || *spw > 24 || !cw_stream_fits(waves, *spw, *mt) || (mode != 3 && k_steps < least_steps)) return false;
  // tiles per workgroup: one workgroup on every compute unit (a second round of these large
  // workgroups costs more than it brings), each with the same share
  // (up to 16 rows the one-tile kernels are as fast below two rounds; beyond, the alternative
  // is a library product that is slower as soon as every compute unit has a tile)
  const int slots = cw_num_compute_units();
  // (partial sums of 17 rows and more go by cw_gemm_bf16_skinny_planes, down to a sixteenth of the units)
  if ((int64_t)*n_tiles * k_splits < (M <= 16 ? 2 * slots : mode == 3 ? slots / 16 : slots)) return false;
  const int per = (*n_tiles * k_splits + slots - 1) / slots;
  *grid = dim3((*n_tiles + per - 1) / per, k_splits);
  return true;
}

static int try_stream(int mode, const bf16_t* X, int64_t ldx, const bf16_t* W, void* C, int64_t ldc,
                      int M, int N, int K, int k_splits, float act, hipStream_t stream) {
  int mt, spw, n_tiles;
  dim3 grid;
  if (!plan_stream(mode, M, N, K, k_splits, &mt, &spw, &grid, &n_tiles)) return CW_ERR_SIZE;
  switch (mode) {
    case 0: return launch_stream_mt<0, 16>(mt, spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
    case 1: return launch_stream_mt<1, 16>(mt, spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
    case 2: return launch_stream_mt<2, 16>(mt, spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
    case 4: return launch_stream_mt<4, 16>(mt, spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
    case 5: return launch_stream_mt<5, 16>(mt, spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
    default: return launch_stream_mt<3, 8>(mt, spw, grid, X, ldx, W, C, ldc, M, N, K, n_tiles, act, stream);
  }
}

#define CW_SKINNY_MAX_M 64

template <int MT, int RT, int WAVES, int ROWS = 16>
static int launch_skinny(int mode, const bf16_t* X, int64_t ldx, const bf16_t* W, void* C, int64_t ldc,
                         int M, int N, int K, int k_splits, float act, hipStream_t stream) {
  const int rows_per_group = (mode == 2 ? 8 : ROWS) * RT;
  const int rows = mode == 2 ? N / 2 : N;
  dim3 grid((rows + rows_per_group - 1) / rows_per_group, mode == 3 ? k_splits : 1), block(WAVES * 64);
  if (mode == 0) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MT, RT, 0, WAVES, ROWS>), grid, block, 0, stream, X, ldx, W, C, ldc, M, N, K, act);
  else if (mode == 1) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MT, RT, 1, WAVES, ROWS>), grid, block, 0, stream, X, ldx, W, C, ldc, M, N, K, act);
  else if (mode == 3) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MT, RT, 3, WAVES, ROWS>), grid, block, 0, stream, X, ldx, W, C, ldc, M, N, K, act);
  else if (mode == 4) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MT, RT, 4, WAVES, ROWS>), grid, block, 0, stream, X, ldx, W, C, ldc, M, N, K, act);
  else if (mode == 5) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MT, RT, 5, WAVES, ROWS>), grid, block, 0, stream, X, ldx, W, C, ldc, M, N, K, act);
  else if (ROWS == 16) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MT, RT, 2, WAVES, 16>), grid, block, 0, stream, X, ldx, W, C, ldc, M, N, K, act);
  else return CW_ERR_ARG;
  return cw_launch_status();
}

// How many ways cw_gemm_bf16_skinny would split K for a partial-sum product of this shape
// (1: not worth it). The caller allocates [splits, M, N] float32 and passes mode 3.
CW_EXPORT int cw_gemm_bf16_skinny_ksplits(int M, int N, int K) {
  const int tiles = (N + 15) / 16;
  const int k_steps = (K + 31) / 32;
  if (M > 64 || tiles > 512) return 1;
  if (M > 16) {
    // Only the streaming kernel takes partial sums of more than 16 rows, and the alternative is a
    // library product that leaves most compute units idle on so narrow an output. Split K far
    // enough that every compute unit gets a tile (two for a long K) and that a wave's share of x
    // fits its registers, down to 8 steps of 32 per split.
    // (an output wide enough for half the compute units is split only if K is much longer still)
    if (tiles > 128 && K < 2 * N) return 1;
    const int mt = M <= 32 ? 2 : 4;
    int s = (cw_num_compute_units() + tiles - 1) / tiles;
    if (K >= 4096 && s < 512 / tiles) s = 512 / tiles;
    if (s > 8) s = 8;
    while (s < 16 && !cw_stream_fits(8, cw_stream_round_spw((k_steps + s * 8 - 1) / (s * 8)), mt)) ++s;
    while (s > 1 && K / s < 256) --s;
    int mt_, spw, n_tiles;
    dim3 grid;
    if (s <= 1 || tiles * s < cw_num_compute_units() || !plan_stream(3, M, N, K, s, &mt_, &spw, &grid, &n_tiles)) return 1;
    return s;
  }
  // up to 16 rows: a long K; or an output so wide that its norm does not run inside the next product (that kernel
  // takes a whole sum, and rows of up to 2048 elements)
  if (K < 4096 && !(K > 2048 && N > 2048)) return 1;
  // Among the counts that the streaming kernel takes: a wave's steps times the tiles of its workgroup are its time
  // (steps as the kernel is built for; 16 of them come in fours, too few on their way: 15 % more), a part costs its
  // way to memory and back. With the norm behind it, the count before and now (us, 8 rows): 7B shape's down product 38.4
  // (5 parts) and 33.4 (8), output product 14.3 and 12.1; 14B shape's down 38.9 and 35.2; 32B shape's down 64.4 and 59.9.
  // A count whose shares come to more workgroups than there are units has a second round for the few beyond (4096 x
  // 14336: 8 parts in 256 workgroups 28.9, 7 in 259 37.5; 72B shape's down: 8 in 256 105, 5 in 260 124).
  int best = 0;
  float least = 0.0f;
  for (int s = 2; s <= 12 && K / s >= 1024; ++s) {
    int mt, spw, n_tiles;
    dim3 grid;
    if (!plan_stream(3, M, N, K, s, &mt, &spw, &grid, &n_tiles) || (int)(grid.x * grid.y) > cw_num_compute_units()) continue;
    const int per = (n_tiles + (int)grid.x - 1) / (int)grid.x;
    const float t = (float)(per * spw) * (spw == 16 ? 1.15f : 1.0f) + 0.6f * (float)s * (float)N / 3584.0f;
    if (best == 0 || t < least) {
      least = t;
      best = s;
    }
  }
  if (best) return best;
  if (K < 4096) return 1;
  int s = 512 / tiles;  // about two workgroups per compute unit,
  if (s > 8) s = 8;
  const int for_registers = (k_steps + 8 * 16 - 1) / (8 * 16);  // and at most 16 steps for each of 8 waves
  if (s < for_registers) s = for_registers;
  if (s > 16) s = 16;
  while (s > 1 && K / s < 1024) --s;
  if (s < 1) s = 1;
  return s;
}

// The same for 17 to 64 rows and a reader that adds the planes inside its own kernel (the residual-add + norm kernel does): from 2
// planes on, 1 where none of these counts is taken. A workgroup's time is its row tiles of W times its steps, its x (every
// workgroup takes in all rows of its part), a reduction a tile, and the planes' way to memory and back; a count that comes to more
// workgroups than units has a second round for the few beyond. Without planes a narrow output's tiles leave units idle, and the
// alternative is a library product that does the same. Product and the norm behind it, us, before (the library's, or as many
// parts as fill the units) and by this rule, with 17 / 64 rows: 896 x 896 9.5 / 13.4, now 5.7 / 6.5; 1536 x 1536 6.5 / 8.0, now 6.2 / 7.3;
// 2560 x 2560 12.8 / 17.0, now 8.2 / 10.8; 3584 x 3584 15.4 / 17.6, now 11.6 / 14.4; 4096 x 14336 48.7 / 51.8, now 29.0 / 33.6; 5120 x
// 13824 43.4 / 45.7, now 36.9 / 41.3; 1536 x 8960 as before. (Over 30 shapes and 17, 32, 33 and 64 rows within 2 % of the best
// count's time in the mean, 21 % at worst.)
CW_EXPORT int cw_gemm_bf16_skinny_planes(int M, int N, int K) {
  if (M <= 16 || M > 64 || N <= 0 || (N + 15) / 16 > 512) return 1;
  int best = 1;
  float least = 0.0f;
  for (int s = 2; s <= 16 && K / s >= 256; ++s) {
    int mt, spw, n_tiles;
    dim3 grid;
    if (!plan_stream(3, M, N, K, s, &mt, &spw, &grid, &n_tiles) || (int)(grid.x * grid.y) > cw_num_compute_units()) continue;
    const int per = (n_tiles + (int)grid.x - 1) / (int)grid.x;
    const float t = 0.22f * (float)(per * spw) + 0.11f * (float)(spw * mt) + 0.55f * (float)per + 2e-6f * (float)s * (float)M * (float)N;
    if (best == 1 || t < least) {
      least = t;
      best = s;
    }
  }
  return best;
}

// 1 if cw_gemm_bf16_skinny streams the weights once for this shape at full speed: every shape
// with M <= 16, and the shapes with 16 < M <= 64 that the streaming kernel takes (other shapes of
// that range run, but a library product is faster). mode 3 is answered by ..._ksplits() > 1.
CW_EXPORT int cw_gemm_bf16_skinny_fast(int mode, int M, int N, int K) {
  if (M <= 16) return 1;
  if (mode < 0 || (mode > 2 && mode != 4 && mode != 5)) return 0;
  int mt, spw, n_tiles;
  dim3 grid;
  return plan_stream(mode, M, N, K, 1, &mt, &spw, &grid, &n_tiles) ? 1 : 0;
}

// 1 if cw_gemm_bf16_swiglu_normed takes this shape (the streaming kernel with one tile of tokens).
CW_EXPORT int cw_gemm_bf16_swiglu_normed_ok(int M, int N, int K) {
  int mt, spw, n_tiles;
  dim3 grid;
  // rows of up to 2048 elements: a lane holds its share of a row in registers over the statistics
  return M >= 1 && M <= 16 && K >= 1024 && !(N & 1) && !(K & 7) && plan_stream(2, M, N, K, 1, &mt, &spw, &grid, &n_tiles) &&
                 spw <= 4
             ? 1
             : 0;
}

// y[m, i] = silu(gate_i . x_m) * (up_i . x_m) with x = rmsnorm(resid + delta) * norm_weight made
// inside the product kernel: resid float32 [M, K], delta bfloat16 [M, K], norm_weight [K]
// bfloat16 (norm_weight_f32 = 0) or float32, W [N = 2 I, K] with the gate rows first, y bfloat16
// [M, I] with row stride ldc. resid is not changed: whoever adds delta to it must still do so.
CW_EXPORT int cw_gemm_bf16_swiglu_normed(const float* resid, const void* delta, const void* norm_weight,
                                         int norm_weight_f32, float eps, const void* W, void* C, int64_t ldc,
                                         int M, int N, int K, hipStream_t stream) {
  if (!cw_gemm_bf16_swiglu_normed_ok(M, N, K)) return CW_ERR_SIZE;
  if (!resid || !delta || !norm_weight || !W || !C || ldc < N / 2) return CW_ERR_ARG;
  if (((uintptr_t)resid & 15) || ((uintptr_t)delta & 15) || ((uintptr_t)norm_weight & 15) || ((uintptr_t)W & 15))
    return CW_ERR_ARG;
  int mt, spw, n_tiles;
  dim3 grid;
  plan_stream(2, M, N, K, 1, &mt, &spw, &grid, &n_tiles);
  const StreamNormIn nin{resid, (const bf16_t*)delta, norm_weight, norm_weight_f32, eps};
#define CW_NORMED(SPW_)                                                                                        \
  case SPW_:                                                                                                   \
    if constexpr (cw_stream_fits(16, SPW_, 1))                                                                 \
      hipLaunchKernelGGL((gemm_stream_bf16_kernel<2, 16, SPW_, 1, true>), grid, dim3(16 * 64), 0, stream,      \
                         (const bf16_t*)nullptr, (int64_t)K, (const bf16_t*)W, C, ldc, M, N, K, n_tiles, 0.0f, nin); \
    break
  switch (spw) {
    CW_NORMED(1); CW_NORMED(2); CW_NORMED(3); CW_NORMED(4);
    default: return CW_ERR_SIZE;
  }
#undef CW_NORMED
  return cw_launch_status();
}

// y = x W^T for M <= 64 rows of bfloat16 x [M, K] (row stride ldx) and bfloat16 W [N, K].
// mode 0: y bfloat16 [M, N] (4: gelu(y), the erf form, with ``act`` > 0 the tanh form; 5: max(y, 0)^2);
// 1: y float32 [M, N]; 2: y = silu(gate) * up, with ``act`` > 0 the clipped gated activation of that limit, -1 max(gate, 0) * up, -2 gelu_tanh(gate) * up, bfloat16 [M, N / 2];
// 3: float32 partial products [splits, M, N], splits = ``k_splits`` if that is positive (up to 16
// rows of x; what a caller has measured to be the best for the shape), else
// cw_gemm_bf16_skinny_ksplits(M, N, K). K must be a multiple of 8 (16-byte rows).
CW_EXPORT int cw_gemm_bf16_skinny(int mode, const void* X, int64_t ldx, const void* W, void* C,
                                  int64_t ldc, int M, int N, int K, int k_splits, float act, hipStream_t stream) {
  if (M < 0 || N <= 0 || K <= 0 || mode < 0 || mode > 5 || !(act >= 0.0f || mode == 2)) return CW_ERR_ARG;
  if (M > CW_SKINNY_MAX_M) return CW_ERR_SIZE;
  if ((K & 7) || (ldx & 7) || ((uintptr_t)X & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  if (mode == 2 && (N & 1)) return CW_ERR_ARG;
  if (ldx < K || ldc < (mode == 2 ? N / 2 : N)) return CW_ERR_ARG;
  if (M == 0) return CW_OK;
  const bf16_t* x = (const bf16_t*)X;
  const bf16_t* w = (const bf16_t*)W;
  const int rows = mode == 2 ? N / 2 : N;
  const int tiles = (rows + (mode == 2 ? 7 : 15)) / (mode == 2 ? 8 : 16);
  if (mode == 3) {
    const int ks = k_splits > 0 ? k_splits : cw_gemm_bf16_skinny_ksplits(M, N, K);
    if (ks > 16 || K / ks < 32) return CW_ERR_ARG;
    const int rc = try_stream(3, x, ldx, w, C, ldc, M, N, K, ks, act, stream);
    if (rc != CW_ERR_SIZE) return rc;
    if (M > 16) return CW_ERR_SIZE;
    return launch_skinny<1, 1, 8>(3, x, ldx, w, C, ldc, M, N, K, ks, act, stream);
  }
  {
    const int rc = try_stream(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
    if (rc != CW_ERR_SIZE) return rc;
  }
  if (M <= 16) {
    // few tiles: many waves on each tile keep enough loads in flight
    if (tiles <= 256 && K >= 1024) return launch_skinny<1, 1, 16>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
    // very many tiles: several per workgroup, so that x is fetched from L2 less often
    if (tiles >= 4096) return launch_skinny<1, 4, 4>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
    if (tiles <= 1024 && K >= 512) return launch_skinny<1, 1, 8>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
    return launch_skinny<1, 1, 4>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
  }
  if (M <= 32) {
    if (tiles <= 256 && K >= 1024) return launch_skinny<2, 1, 16>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
    return rows >= 4096 ? launch_skinny<2, 2, 4>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream)
                        : launch_skinny<2, 1, 4>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
  }
  if (tiles <= 256 && K >= 1024) return launch_skinny<4, 1, 8>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
  return rows >= 4096 ? launch_skinny<4, 2, 4>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream)
                      : launch_skinny<4, 1, 4>(mode, x, ldx, w, C, ldc, M, N, K, 1, act, stream);
}

// Are these products of ``M`` rows and K columns taken as one launch (``tiles``: their tiles of 16 rows of W)? Up to 16 rows
// always; beyond, and up to 64, where all have the same x of 768 columns and more and the streaming kernel takes them (apart, those of
// fewer than 256 tiles are products of the library or of 64-row tiles). 17 / 64 rows of 896, outputs of 1152, 3600 and 1792, us apart and
// together: 26.7 and 5.4, 30.9 and 6.9; of 768, outputs of 2304, 3072 and 4096: 22.7 and 6.6, 24.4 and 8.7.
CW_EXPORT int cw_gemm_bf16_group_ok(int count, int same_x, int M, int64_t tiles, int K) {
  if (count < 2 || count > GROUP_MAX || M < 1 || M > CW_SKINNY_MAX_M || K < 8 || (K & 7) || tiles < count || tiles > (1 << 20)) return 0;
  if (M <= 16) return 1;
  int mt, spw, n_tiles;
  dim3 grid;
  return same_x && K >= 768 && plan_stream(0, M, (int)tiles * 16, K, 1, &mt, &spw, &grid, &n_tiles) && spw <= 8 ? 1 : 0;
}

// C[i] [M, N[i]] = X[i] W[i]^T for ``count`` products, all bfloat16, rows without gaps: X[i] [M, K], W[i] [N[i], K].
CW_EXPORT int cw_gemm_bf16_group(int count, const void* const* X, const void* const* W, void* const* C, const int* N, int M, int K,
                                 hipStream_t stream) {
  if (count < 2 || count > GROUP_MAX || M < 0 || !X || !W || !C || !N) return CW_ERR_ARG;
  ProductGroup group{};
  int64_t tiles = 0;
  bool same_x = true;
  for (int i = 0; i < GROUP_MAX; ++i) {
    group.first[i] = i < count ? (int)tiles : INT_MAX;
    if (i >= count) continue;
    if (N[i] <= 0 || N[i] > (1 << 24) || !X[i] || !W[i] || !C[i] || ((uintptr_t)X[i] & 15) || ((uintptr_t)W[i] & 15)) return CW_ERR_ARG;
    group.x[i] = (const bf16_t*)X[i];
    group.w[i] = (const bf16_t*)W[i];
    group.c[i] = (bf16_t*)C[i];
    group.n[i] = N[i];
    tiles += (N[i] + 15) / 16;
    same_x = same_x && X[i] == X[0];
  }
  group.first[GROUP_MAX] = INT_MAX;
  if (M == 0) return CW_OK;
  if (!cw_gemm_bf16_group_ok(count, same_x, M, tiles, K)) return CW_ERR_SIZE;
  int mt, spw, n_tiles;
  dim3 grid;
  if (same_x && plan_stream(0, M, (int)tiles * 16, K, 1, &mt, &spw, &grid, &n_tiles) && spw <= 8) {
#define CW_GROUP(SPW_, MT_)                                                                                                  \
  if constexpr (cw_stream_fits(16, SPW_, MT_))                                                                               \
    hipLaunchKernelGGL((gemm_stream_bf16_kernel<0, 16, SPW_, MT_, false, true>), grid, dim3(16 * 64), 0, stream, group.x[0], \
                       (int64_t)K, (const bf16_t*)nullptr, (void*)nullptr, (int64_t)0, M, 0, K, n_tiles, 0.0f, group)
#define CW_GROUP_STEPS(SPW_)             \
  case SPW_:                             \
    if (mt == 1) { CW_GROUP(SPW_, 1); }  \
    else if (mt == 2) { CW_GROUP(SPW_, 2); } \
    else { CW_GROUP(SPW_, 4); }          \
    break
    switch (spw) {
      CW_GROUP_STEPS(1); CW_GROUP_STEPS(2); CW_GROUP_STEPS(3); CW_GROUP_STEPS(4); CW_GROUP_STEPS(5); CW_GROUP_STEPS(6);
      CW_GROUP_STEPS(7); CW_GROUP_STEPS(8);
      default: return CW_ERR_SIZE;
    }
#undef CW_GROUP_STEPS
#undef CW_GROUP
    return cw_launch_status();
  }
  // waves a tile as for one product of as many tiles
  const dim3 blocks((unsigned)tiles);
  if (tiles <= 256 && K >= 1024) hipLaunchKernelGGL(gemm_skinny_group_bf16_kernel<16>, blocks, dim3(16 * 64), 0, stream, group, M, K);
  else if (K >= 512) hipLaunchKernelGGL(gemm_skinny_group_bf16_kernel<8>, blocks, dim3(8 * 64), 0, stream, group, M, K);
  else hipLaunchKernelGGL(gemm_skinny_group_bf16_kernel<4>, blocks, dim3(4 * 64), 0, stream, group, M, K);
  return cw_launch_status();
}

// =====================================================================================
// Fused q/k/v product + bias + rotary encoding + cache write for few rows of x (decode).
// The weight-streaming product above with another row order and epilogue: a tile of a q or k
// head holds rows (i .. i+7) and (i + hd/2 .. i + hd/2 + 7) of that head, so both elements of
// every rotary pair (half-split pairing, full rotary dimension) end up in one workgroup. The
// epilogue adds the bias, rotates by float32(pos) * inv_freq[i] and writes q to ``q_out``
// [M, nh * hd], rotated k and plain v to their cache rows ``slots[m]`` ([rows, nkv, hd]).
// blockIdx.y takes MT tiles of 16 tokens.
// BEGUN (MT = 1, at most 16 rows): x comes with its norm begun.
template <int WAVES, int MT, bool BEGUN = false>
__global__ __launch_bounds__(WAVES * 64) void gemm_qkv_rope_bf16_kernel(
    const bf16_t* __restrict__ X, int64_t ldx, const bf16_t* __restrict__ W, const void* __restrict__ bias,
    int bias_f32, const int* __restrict__ positions, const int* __restrict__ slots,
    const float* __restrict__ inv_freq, bf16_t* __restrict__ q_out, bf16_t* __restrict__ k_cache,
    bf16_t* __restrict__ v_cache, int64_t cache_rows, int M, int K, int nh, int nkv, int hd, RowFactors begun) {
  static_assert(!BEGUN || MT == 1, "begun norms are products' of up to 16 rows");
  __shared__ __align__(16) float red[WAVES][MT * 256];  // [wave][token tile][token][tile row]
  __shared__ float factors[16];
  [[maybe_unused]] RowPieces<WAVES> pieces;
  if constexpr (BEGUN) pieces.load(begun, M);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, s = lane >> 4;
  const int half = hd / 2;
  const int tiles_per_head = hd / 16;
  const int m0 = blockIdx.y * (MT * 16);          // the workgroup's first token
  M = min(M - m0, MT * 16);
  X += m0 * ldx;
  positions += m0;
  slots += m0;
  q_out += (int64_t)m0 * nh * hd;
  const int head = blockIdx.x / tiles_per_head;   // 0 .. nh + 2 nkv - 1
  const int tile = blockIdx.x % tiles_per_head;
  const bool is_v = head >= nh + nkv;
  // the weight row inside the head that this lane loads: row lr of the tile (see cw_to_operand_layout)
  const int lr = lane >> 2, ls = lane & 3;
  const int row_in_head = is_v ? tile * 16 + lr : (lr < 8 ? tile * 8 + lr : half + tile * 8 + (lr - 8));
  const bf16_t* wrow = W + ((int64_t)head * hd + row_in_head) * K;
  constexpr bool X_SWAP = MT > 1;  // one tile of tokens is loaded in operand layout as it is (see gemm_skinny_bf16_kernel)
  const int xr = X_SWAP ? lr : r, xs = X_SWAP ? ls : s;
  bool xok[MT];
  const bf16_t* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    xok[mt] = mt * 16 + xr < M;
    xrow[mt] = X + (int64_t)(xok[mt] ? mt * 16 + xr : 0) * ldx;
  }

  auto bias_at = [&](int col) -> float {
    if (bias == nullptr) return 0.0f;
    return bias_f32 ? ((const float*)bias)[col] : __bfloat162float(((const bf16_t*)bias)[col]);
  };
  // MT == 1: what this thread's part of the epilogue needs (position, slot, frequency, bias) is
  // requested here, beside the weights, and not after the product, where it would be one more
  // trip to memory with nothing else to do meanwhile
  int e_pos = 0;
  int64_t e_slot = -1;
  float e_inv = 0.0f, e_ba = 0.0f, e_bb = 0.0f;
  if constexpr (MT == 1) {
    if (is_v) {
      const int j = threadIdx.x & 15, m = threadIdx.x >> 4;
      if (m < 16 && m < M) {
        e_slot = slots[m];
        e_ba = bias_at(head * hd + tile * 16 + j);
      }
    } else {
      const int p = threadIdx.x & 7, m = threadIdx.x >> 3;
      if (m < 16 && m < M) {
        const int i = tile * 8 + p;
        e_pos = positions[m];
        e_slot = slots[m];
        e_inv = inv_freq[i];
        e_ba = bias_at(head * hd + i);
        e_bb = bias_at(head * hd + half + i);
      }
    }
  }

  f32x4_t acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8_t zero;
#pragma unroll
  for (int e = 0; e < 8; ++e) zero[e] = (__bf16)0.0f;
  const int k_steps = (K + 31) / 32;
  constexpr int U = 4;  // k-steps in flight a wave
  [[maybe_unused]] bool first = true;
  // (BEGUN: also a wave without a step adds up its rows' pieces)
  for (int ks0 = wave * U; BEGUN && first || ks0 < k_steps; ks0 += WAVES * U) {
    bf16x8_t wf[U], xf[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (ks0 + u) * 32 + ls * 8;
      const bool kok = (ks0 + u) < k_steps && k + 8 <= K;
      wf[u] = kok ? *reinterpret_cast<const bf16x8_t*>(wrow + k) : zero;
      const int kx = (ks0 + u) * 32 + xs * 8;
      const bool kxok = (ks0 + u) < k_steps && kx + 8 <= K;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        xf[u][mt] = (kxok && xok[mt]) ? *reinterpret_cast<const bf16x8_t*>(xrow[mt] + kx) : zero;
    }
    if constexpr (BEGUN) {
      if (first) pieces.factors(begun, factors);
      first = false;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bf16x8_t wo = cw_to_operand_layout(wf[u], lane);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wo, X_SWAP ? cw_to_operand_layout(xf[u][mt], lane) : xf[u][mt],
                                                          acc[mt], 0, 0, 0);
    }
  }
  // lane (r, s) holds tile rows 4s..4s+3 of token r: one 16-byte store, no bank hit twice
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<f32x4_t*>(&red[wave][mt * 256 + r * 16 + 4 * s]) = acc[mt];
  __syncthreads();
  // MT * 256 values [token tile][token][tile row]; each is summed over the waves by one thread
  for (int idx = threadIdx.x; idx < MT * 256; idx += WAVES * 64) {
    float sum = red[0][idx];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sum += red[w][idx];
    red[0][idx] = sum;
  }
  __syncthreads();
  auto summed = [&](int row, int m) -> float { return BEGUN ? red[0][m * 16 + row] * factors[m] : red[0][m * 16 + row]; };
  if constexpr (MT == 1) {
    // every thread has at most one output (v: 256 of them, q and k: 128 pairs)
    if (is_v) {
      const int j = threadIdx.x & 15, m = threadIdx.x >> 4;
      if (m < 16 && m < M && e_slot >= 0 && e_slot < cache_rows) {
        const int d = tile * 16 + j;
        v_cache[(e_slot * nkv + (head - nh - nkv)) * hd + d] = __float2bfloat16(summed(j, m) + e_ba);
      }
    } else {
      const int p = threadIdx.x & 7, m = threadIdx.x >> 3;
      if (m < 16 && m < M) {
        const int i = tile * 8 + p;
        const float a = summed(p, m) + e_ba;
        const float b = summed(p + 8, m) + e_bb;
        float sn, cs;
        sincosf((float)e_pos * e_inv, &sn, &cs);
        const bf16_t oa = __float2bfloat16(a * cs - b * sn), ob = __float2bfloat16(b * cs + a * sn);
        if (head < nh) {
          bf16_t* q = q_out + (int64_t)m * nh * hd + head * hd;
          q[i] = oa;
          q[i + half] = ob;
        } else if (e_slot >= 0 && e_slot < cache_rows) {
          bf16_t* kd = k_cache + (e_slot * nkv + (head - nh)) * hd;
          kd[i] = oa;
          kd[i + half] = ob;
        }
      }
    }
    return;
  }
  if (is_v) {
    // idx -> (token m, row j), j fastest: 16 consecutive elements of a cache row
    for (int idx = threadIdx.x; idx < MT * 256; idx += WAVES * 64) {
      const int j = idx & 15, m = idx >> 4;
      if (m >= M) continue;
      const int64_t slot = slots[m];
      if (slot < 0 || slot >= cache_rows) continue;
      const int d = tile * 16 + j;
      const float v = summed(j, m) + bias_at(head * hd + d);
      v_cache[(slot * nkv + (head - nh - nkv)) * hd + d] = __float2bfloat16(v);
    }
  } else {
    // idx -> (token m, pair p): elements i = tile * 8 + p and i + half
    for (int idx = threadIdx.x; idx < MT * 128; idx += WAVES * 64) {
      const int p = idx & 7, m = idx >> 3;
      if (m >= M) continue;
      const int i = tile * 8 + p;
      const float a = summed(p, m) + bias_at(head * hd + i);
      const float b = summed(p + 8, m) + bias_at(head * hd + half + i);
      float sn, cs;
      sincosf((float)positions[m] * inv_freq[i], &sn, &cs);
      const bf16_t oa = __float2bfloat16(a * cs - b * sn), ob = __float2bfloat16(b * cs + a * sn);
      if (head < nh) {
        bf16_t* q = q_out + (int64_t)m * nh * hd + head * hd;
        q[i] = oa;
        q[i + half] = ob;
      } else {
        const int64_t slot = slots[m];
        if (slot < 0 || slot >= cache_rows) continue;
        bf16_t* kd = k_cache + (slot * nkv + (head - nh)) * hd;
        kd[i] = oa;
        kd[i + half] = ob;
      }
    }
  }
}

// x [M <= 64, K] bfloat16, W [(nh + 2 nkv) * hd, K] bfloat16 (q heads, k heads, v heads), hd a
// multiple of 16, rotary dimension == hd. bias: nullptr, bfloat16 or float32 [(nh + 2 nkv) * hd].
CW_EXPORT int cw_gemm_qkv_rope_bf16(const void* X, int64_t ldx, const void* W, const void* bias,
                                    int bias_f32, const int* positions, const int* slots,
                                    const float* inv_freq, void* q_out, void* k_cache, void* v_cache,
                                    int64_t cache_rows, int M, int K, int nh, int nkv, int hd,
                                    hipStream_t stream) {
  if (M < 0 || M > 64 || K <= 0 || nh <= 0 || nkv <= 0 || hd <= 0 || (hd & 15)) return CW_ERR_ARG;
  if ((K & 7) || (ldx & 7) || ldx < K || ((uintptr_t)X & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  if (!positions || !slots || !inv_freq || !q_out || !k_cache || !v_cache) return CW_ERR_ARG;
  if (M == 0) return CW_OK;
  const int tiles = (nh + 2 * nkv) * (hd / 16);
  dim3 grid(tiles);
  const bf16_t* x = (const bf16_t*)X;
  const bf16_t* w = (const bf16_t*)W;
#define CW_QKV(WAVES_, MT_)                                                                              \
  hipLaunchKernelGGL((gemm_qkv_rope_bf16_kernel<WAVES_, MT_>), grid, dim3(WAVES_ * 64), 0, stream, x, ldx, \
                     w, bias, bias_f32, positions, slots, inv_freq, (bf16_t*)q_out, (bf16_t*)k_cache,    \
                     (bf16_t*)v_cache, cache_rows, M, K, nh, nkv, hd, RowFactors{})
  if (M <= 16) {
    if (tiles <= 256 && K >= 1024) CW_QKV(16, 1);
    else if (K >= 512) CW_QKV(8, 1);
    else CW_QKV(4, 1);
  } else {
    // One tile of tokens a workgroup while there are few of them, else two: a workgroup takes in its rows of x beside its
    // rows of W (four tiles: 196 KB beside 49 KB at a width of 1536), at some 30 GB/s. (us, four or two tiles and
    // one workgroup a tile of W / one tile / two, widths of 1536 and 128 tiles of W: 17 rows 5.80 / 4.78 / 5.80, 32 rows 6.35 /
    // 5.06 / 6.14, 48 rows 7.56 / 6.73 / 6.11, 64 rows 7.90 / 6.95 / 6.39; of 896 and 72 tiles, 64 rows 6.20 / 5.02 / 5.19; of
    // 2048 and 160 tiles, 17 rows 8.11 / 7.32 / 7.59, 64 rows 11.7 / 11.2 / 10.6.)
    const int groups = (M + 15) / 16;
    if (tiles * groups <= 320) {
      grid.y = groups;
      if (K >= 512) CW_QKV(8, 1);
      else CW_QKV(4, 1);
    } else {
      grid.y = (groups + 1) / 2;
      if (K >= 512) CW_QKV(8, 2);
      else CW_QKV(4, 2);
    }
  }
#undef CW_QKV
  return cw_launch_status();
}

// The same for at most 16 rows that come with their norm begun: X [M, K] and squares [M, parts] as cw_gemm_bf16_join writes them.
CW_EXPORT int cw_gemm_qkv_rope_begun_bf16(const void* X, const float* squares, int parts, float eps, const void* W, const void* bias,
                                          int bias_f32, const int* positions, const int* slots, const float* inv_freq, void* q_out,
                                          void* k_cache, void* v_cache, int64_t cache_rows, int M, int K, int nh, int nkv, int hd,
                                          hipStream_t stream) {
  if (M < 1 || M > 16 || K <= 0 || nh <= 0 || nkv <= 0 || hd <= 0 || (hd & 15) || parts < 4 || parts > 256 || (parts & 3) || ((uintptr_t)squares & 15)) return CW_ERR_ARG;
  if ((K & 7) || ((uintptr_t)X & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  if (!X || !squares || !W || !positions || !slots || !inv_freq || !q_out || !k_cache || !v_cache) return CW_ERR_ARG;
  const RowFactors begun{squares, parts, 1.0f / (float)K, eps};
  const int tiles = (nh + 2 * nkv) * (hd / 16);
#define CW_QKV(WAVES_)                                                                                                             \
  hipLaunchKernelGGL((gemm_qkv_rope_bf16_kernel<WAVES_, 1, true>), dim3(tiles), dim3(WAVES_ * 64), 0, stream, (const bf16_t*)X,      \
                     (int64_t)K, (const bf16_t*)W, bias, bias_f32, positions, slots, inv_freq, (bf16_t*)q_out, (bf16_t*)k_cache,    \
                     (bf16_t*)v_cache, cache_rows, M, K, nh, nkv, hd, begun)
  if (tiles <= 256 && K >= 1024) CW_QKV(16);
  else if (K >= 512) CW_QKV(8);
  else CW_QKV(4);
#undef CW_QKV
  return cw_launch_status();
}

// =====================================================================================
// A product of few rows that joins the residual stream and begins the norm behind it (decode: 1 to 16 tokens):
//   resid += x W^T;  y = resid * norm_weight (bfloat16);  squares[m, tile] = sum of resid[m, n]^2 over a tile's columns.
// The product that reads y multiplies its finished sums by 1 / sqrt(mean + eps) (RowFactors), so the residual add and the norm
// are no launch of their own.
// A workgroup owns up to R outputs (``rows`` of them) and all of K: the 16 rows of its matrix operand are R rows of W times 16 / R
// neighbouring pieces of 32 k-values, each multiplied with its own piece of x into sums of its own, of which the other pieces' rows are
// dropped. So a narrow output (N of 896 to 3584) makes enough workgroups for the card without planes of partial sums.
// Bound by the launch and its first trip to memory, then by what a workgroup takes in: its rows of W and all of x. Product and norm as two
// launches -> this one, us in a graph over 24 to 28 layers' matrices, 1 / 4 / 8 / 16 rows: 896 x 896 4.7 / 5.0 / 5.2 / 5.4 -> 3.1 / 3.2 / 3.2 /
// 3.5; 896 x 4864 6.4 / 6.7 / 6.7 / 7.1 -> 4.3 / 4.9 / 5.6 / 7.2; 1536 x 1536 5.2 / 5.6 / 5.8 / 6.3 -> 3.4 / 3.5 / 3.7 / 4.2; 1536 x 8960 9.6 / 9.8 /
// 10.0 / 10.4 -> 8.7 / 8.7 / 9.8 / 13.2; 3584 x 3584 9.9 / 10.0 / 10.0 / 10.3 -> 7.2 / 7.5 / 7.7 / 8.9; 3584 x 18944 28.7 / 29.5 / 30.8 / 32.1 -> 27.6 /
// 30.5 / 33.1 / 41.2. (Two sets of operands a wave in turns, rows of x swapped into operand layout: slower, both are more code.)
template <int WAVES, int R>
__global__ __launch_bounds__(WAVES * 64) void gemm_join_bf16_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                                    float* __restrict__ resid, const void* __restrict__ norm_weight,
                                                                    bf16_t* __restrict__ Y, float* __restrict__ squares, int M, int N,
                                                                    int K, int rows, int norm_weight_f32) {
  constexpr int P = 16 / R;                       // pieces of K side by side in an operand
  constexpr int U = P == 4 ? 3 : P == 2 ? 5 : 8;  // operands of W on their way a wave
  __shared__ __align__(16) float red[WAVES][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, s = lane >> 4;
  const int lr = lane >> 2, ls = lane & 3;
  const int n0 = blockIdx.x * rows;
  const bool w_ok = lr % R < rows && n0 + lr % R < N;  // a row that is not there counts as zeros
  const int w_k = (lr / R) * 32 + ls * 8;
  const bf16_t* const wrow = W + (int64_t)(w_ok ? n0 + lr % R : 0) * K + w_k;
  const bool x_ok = r < M;
  const bf16_t* const xrow = X + (int64_t)(x_ok ? r : 0) * K + s * 8;
  // what the last threads need of the stream and of the norm, asked for beside the weights
  const int e_m = threadIdx.x >> 4, e_j = threadIdx.x & 15;
  const bool e_ok = threadIdx.x < 256 && e_m < M && e_j < rows && n0 + e_j < N;
  const int64_t e_at = (int64_t)e_m * N + n0 + e_j;
  float e_resid = 0.0f, e_weight = 0.0f;
  if (e_ok) {
    e_resid = resid[e_at];
    e_weight = norm_weight_f32 ? ((const float*)norm_weight)[n0 + e_j] : __bfloat162float(((const bf16_t*)norm_weight)[n0 + e_j]);
  }
  bf16x8_t zero;
#pragma unroll
  for (int e = 0; e < 8; ++e) zero[e] = (__bf16)0.0f;
  f32x4_t acc[P];
#pragma unroll
  for (int p = 0; p < P; ++p) acc[p] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
  const int steps = (K + 32 * P - 1) / (32 * P);
  for (int at = wave; at < steps; at += WAVES * U) {
    bf16x8_t wf[U], xf[U][P];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int step = at + u * WAVES, k = step * (32 * P);
      const bool on = step < steps;
      wf[u] = on && w_ok && k + w_k + 8 <= K ? *reinterpret_cast<const bf16x8_t*>(wrow + k) : zero;
#pragma unroll
      for (int p = 0; p < P; ++p)
        xf[u][p] = on && x_ok && k + p * 32 + s * 8 + 8 <= K ? *reinterpret_cast<const bf16x8_t*>(xrow + k + p * 32) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bf16x8_t wo = cw_to_operand_layout(wf[u], lane);
#pragma unroll
      for (int p = 0; p < P; ++p) acc[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wo, xf[u][p], acc[p], 0, 0, 0);
    }
  }
  // lane (r, s) holds operand rows 4s..4s+3 of token r, which are rows of piece 4s / R: of that piece's sums
  f32x4_t mine = acc[0];
#pragma unroll
  for (int p = 1; p < P; ++p)
    if (s / (R / 4) == p) mine = acc[p];
  *reinterpret_cast<f32x4_t*>(&red[wave][r * 16 + 4 * s]) = mine;
  cw_lds_barrier();
  if (threadIdx.x >= 256) return;
  float v = 0.0f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) v += red[w][threadIdx.x];
  if constexpr (R == 4) v += cw_dpp<0x124>(v);  // rotated by 4 of a row's 16 lanes: the pieces of an output lie R lanes apart
  if constexpr (R <= 8) v += cw_dpp<0x128>(v);  // by 8
  v += e_resid;
  if (e_ok) {
    resid[e_at] = v;
    Y[e_at] = __float2bfloat16(v * e_weight);
  }
  float q = e_ok ? v * v : 0.0f;  // of the token's R neighbours, in pairs
  q += cw_dpp<0xB1>(q);
  q += cw_dpp<0x4E>(q);
  if constexpr (R >= 8) q += cw_dpp<0x141>(q);
  if constexpr (R >= 16) q += cw_dpp<0x140>(q);
  const int parts = ((int)gridDim.x + 3) & ~3;
  if (e_m < M && e_j == 0) squares[e_m * parts + blockIdx.x] = q;
  // (a row of pieces ends on a multiple of four: zeros)
  if (blockIdx.x == gridDim.x - 1 && e_m < M && e_j > 0 && (int)blockIdx.x + e_j < parts) squares[e_m * parts + blockIdx.x + e_j] = 0.0f;
}

// How cw_gemm_bf16_join cuts a product on a card of ``units`` compute units: outputs a workgroup, of ``*slots`` that its kernel has
// room for, and waves. 0: it does not take the product. Few rows of x beside the weights only, up to 72 K elements: every workgroup takes in
// all of x. Up to 16 outputs a compute unit in one round, so that all units stream; a K of up to 2048 is one trip to memory for eight waves, whose
// workgroup has room for 8 outputs: on a card of fewer units, where more come to one, it has sixteen.
static int join_plan(int M, int N, int K, int units, int* slots, int* waves) {
  if (M < 1 || M > 16 || N < 64 || N > 16 * units || K < 256 || (K & 7) || (int64_t)M * K > 72 * 1024) return 0;
  const int rows = (N + units - 1) / units;
  *waves = N <= 2048 && K <= 2048 && rows <= 8 ? 8 : 16;
  *slots = rows > 8 ? 16 : rows > 4 || *waves == 8 ? 8 : 4;
  const int taken = *waves == 8 ? *slots : rows;
  return (N + taken - 1) / taken <= 256 ? taken : 0;  // pieces of a row that its reader takes
}
// The same as one number for a check of the rule: outputs + 256 slots + 65536 waves.
CW_EXPORT int cw_gemm_bf16_join_rule(int M, int N, int K, int units) {
  int slots = 0, waves = 0;
  const int rows = units > 0 ? join_plan(M, N, K, units, &slots, &waves) : 0;
  return rows ? rows | slots << 8 | waves << 16 : 0;
}

// Is that also the faster way for a layer, against planes (of whole lines from 64 MB on) and the norm that adds them? Up to 64 K elements of x; where a
// workgroup has more than 8 outputs and its K is more than the one trip of 16 waves with 8 operands each, up to 16 K. Decode steps, us, a feed-forward's output
// as planes / joined (its mixer's joined), rows: 896 x 4864 1 712 / 673, 8 758 / 733; 1536 x 8960 1 1182 / 1180, 2 1191 / 1185, 4 1210 / 1205, 8 1244 /
// 1257; 2048 x 11008 1 1826 / 1808, 2 1845 / 1826, 4 1866 / 1856; 2560 x 9728 1 2234 / 2223, 2 2247 / 2244, 4 2278 / 2297; 4096 x 14336 1 1720 / 1711, 2 1732 /
// 1731, 4 1758 / 1777; 3584 x 18944 1 2892 / 2907, 2 2919 / 2961. A mixer's, whose norm would be made inside the gate/up product: 1536 x 1536 8
// 1377 / 1244, 3584 x 3584 1 2963 / 2892, 8 3096 / 3025, 16 3265 / 3244, 4096 x 4096 16 1951 / 1939.
CW_EXPORT int cw_gemm_bf16_join_pays(int M, int N, int K) {
  int slots, waves;
  if (!join_plan(M, N, K, cw_num_compute_units(), &slots, &waves)) return 0;
  const int64_t x = (int64_t)M * K;
  return x <= 64 * 1024 && (slots <= 8 || K <= 4096 || x <= 16 * 1024) ? 1 : 0;
}

// The number of sums of squares that cw_gemm_bf16_join leaves of a row (zeros up to a multiple of 4 at the end), 0 where it does not take these sizes.
CW_EXPORT int cw_gemm_bf16_join_parts(int M, int N, int K) {
  int slots, waves;
  const int rows = join_plan(M, N, K, cw_num_compute_units(), &slots, &waves);
  return rows ? ((N + rows - 1) / rows + 3) & ~3 : 0;
}

// resid [M, N] float32 += x W^T; Y [M, N] bfloat16 = resid * norm_weight [N]; squares [M, parts] float32. x [M, K] and W [N, K]
// bfloat16, rows without gaps.
CW_EXPORT int cw_gemm_bf16_join(const void* X, const void* W, float* resid, const void* norm_weight, int norm_weight_f32, void* Y,
                                float* squares, int M, int N, int K, hipStream_t stream) {
  int slots, waves;
  const int rows = join_plan(M, N, K, cw_num_compute_units(), &slots, &waves);
  if (!rows || rows > slots) return CW_ERR_SIZE;
  if (!X || !W || !resid || !norm_weight || !Y || !squares || ((uintptr_t)X & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  const dim3 grid((N + rows - 1) / rows);
#define CW_JOIN(WAVES_, R_)                                                                                                  \
  hipLaunchKernelGGL((gemm_join_bf16_kernel<WAVES_, R_>), grid, dim3(WAVES_ * 64), 0, stream, (const bf16_t*)X, (const bf16_t*)W, \
                     resid, norm_weight, (bf16_t*)Y, squares, M, N, K, rows, norm_weight_f32)
  if (waves == 8) CW_JOIN(8, 8);
  else if (slots == 4) CW_JOIN(16, 4);
  else if (slots == 8) CW_JOIN(16, 8);
  else CW_JOIN(16, 16);
#undef CW_JOIN
  return cw_launch_status();
}

// y[m, i] = silu(gate_i . x_m) * (up_i . x_m) as cw_gemm_bf16_skinny's mode 2, for rows that come with their norm begun: X [M, K]
// and squares [M, parts] as cw_gemm_bf16_join writes them.
CW_EXPORT int cw_gemm_bf16_swiglu_begun(const void* X, const float* squares, int parts, float eps, const void* W, void* C, int64_t ldc,
                                        int M, int N, int K, hipStream_t stream) {
  if (M < 1 || M > 16 || N < 2 || (N & 1) || K < 8 || (K & 7) || parts < 4 || parts > 256 || (parts & 3)) return CW_ERR_SIZE;
  if (!X || !squares || ((uintptr_t)squares & 15) || !W || !C || ldc < N / 2 || ((uintptr_t)X & 15) || ((uintptr_t)W & 15)) return CW_ERR_ARG;
  const RowFactors begun{squares, parts, 1.0f / (float)K, eps};
  const bf16_t *x = (const bf16_t*)X, *w = (const bf16_t*)W;
  int mt, spw, n_tiles;
  dim3 grid;
  if (plan_stream(2, M, N, K, 1, &mt, &spw, &grid, &n_tiles)) {
#define CW_BEGUN(SPW_)                                                                                                               \
  case SPW_:                                                                                                                         \
    if constexpr (cw_stream_fits(16, SPW_, 1)) {                                                                                     \
      hipLaunchKernelGGL((gemm_stream_bf16_kernel<2, 16, SPW_, 1, false, false, true>), grid, dim3(16 * 64), 0, stream, x, (int64_t)K, \
                         w, C, ldc, M, N, K, n_tiles, 0.0f, begun);                                                                  \
      return cw_launch_status();                                                                                                     \
    }                                                                                                                                \
    break
    switch (spw) {
      CW_BEGUN(1); CW_BEGUN(2); CW_BEGUN(3); CW_BEGUN(4); CW_BEGUN(5); CW_BEGUN(6); CW_BEGUN(7); CW_BEGUN(8);
      CW_BEGUN(10); CW_BEGUN(12); CW_BEGUN(16); CW_BEGUN(20); CW_BEGUN(24);
      default: break;
    }
#undef CW_BEGUN
    return CW_ERR_SIZE;
  }
  // waves and tiles as cw_gemm_bf16_skinny takes them
  const int tiles = (N / 2 + 7) / 8;
#define CW_SKINNY_BEGUN(RT_, WAVES_)                                                                                                \
  hipLaunchKernelGGL((gemm_skinny_begun_bf16_kernel<RT_, WAVES_>), dim3((tiles + RT_ - 1) / RT_), dim3(WAVES_ * 64), 0, stream, x, w, \
                     (bf16_t*)C, ldc, M, N, K, 0.0f, begun)
  if (tiles <= 256 && K >= 1024) CW_SKINNY_BEGUN(1, 16);
  else if (tiles >= 4096) CW_SKINNY_BEGUN(4, 4);
  else if (tiles <= 1024 && K >= 512) CW_SKINNY_BEGUN(1, 8);
  else CW_SKINNY_BEGUN(1, 4);
#undef CW_SKINNY_BEGUN
  return cw_launch_status();
}
