// bfloat16 matrix product y = x * W^T for many rows of x (portions of prompts) on the gfx950
// matrix cores, LDS tiled: x [M, K] row-major, W [N, K] row-major as checkpoints hold it.
//
// A workgroup of 4 waves owns a 128 x 128 tile of y and walks K in steps of 64. The x and W tiles
// of a step (128 rows x 64 elements each) go from global memory through registers into LDS, double
// buffered: the loads of step t + 1 are in flight while step t is multiplied, and one barrier per
// step separates writing a buffer from reading it. A wave owns a 64 x 64 quarter: per 32 elements
// of K it reads 4 + 4 fragments of 16 rows from LDS (16-byte reads; rows are padded by 16 bytes so
// that 16 lanes reading 16 different rows hit different banks) and issues 16
// v_mfma_f32_16x16x32_bf16. W is the first operand, so a lane ends up with 4 consecutive columns
// of one row of y, which it stores as 8 bytes. With quarters of this size the LDS reads (1 KB per
// 4 matrix instructions) hold the matrix cores to about a fifth of their peak: half of what the
// library's 256 x 256 tiles reach on the same shapes, so the engine takes this kernel only when it
// is asked to (``hip_products``) and the library product otherwise.
//
// What is fused in is chosen by MODE:
//   0  y bfloat16 [M, N], + bias [N] (bfloat16 or float32) when given;
//   2  W = [gate; up] stacked ([2 I, K]), y[m, i] = silu(gate_i . x_m) * (up_i . x_m), bfloat16
//      [M, I]: the tile holds 64 gate rows and the 64 up rows that belong to them, arranged so
//      that a lane holds both values of an output;
// Accumulation is float32; the K loop of an output runs in the same order whatever else is in
// the batch.
//
// The second kernel of this file, gemm_wide_bf16_kernel, is the one the engine takes by itself for most products of
// many rows: tiles of 96 x 96 to 256 x 288, K in stages of 64 that go from global memory
// straight into LDS (buffer loads with the LDS target, no registers between), a ring of stages that fills the LDS,
// and workgroups that stay and walk over their share of the tiles. It is described where
// it stands.
#include "common.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

#define GT_BM 128
#define GT_BN 128
#define GT_BK 64
#define GT_ROW (GT_BK + 8)  // LDS row in elements

struct TileArgs {
  const bf16_t* X;
  int64_t ldx;
  const bf16_t* W;
  const void* bias;   // nullptr, or [N]
  int bias_f32;
  void* C;
  int64_t ldc;
  int M, N, K;
  float act;          // MODE 2: > 0: the clipped gated activation with this limit, -1: max(gate, 0) * up, -2: gelu_tanh(gate) * up
};

// Row of W that row ``rb`` (0..127) of the workgroup's W tile ``tn`` is. MODE 2: a wave's 64 tile
// rows are 32 gate rows followed by the 32 up rows with the same indices.
template <int MODE>
__device__ __forceinline__ int64_t gt_w_row(int tn, int rb, int N, bool* ok) {
  if (MODE == 2) {
    const int I = N / 2;
    const int wn = rb >> 6, q = rb & 63;
    const int64_t i = (int64_t)tn * 64 + wn * 32 + (q & 31);
    *ok = i < I;
    return (q < 32 ? i : I + i);
  }
  const int64_t n = (int64_t)tn * GT_BN + rb;
  *ok = n < N;
  return n;
}

template <int MODE>
__global__ __launch_bounds__(256, 2) void gemm_tile_bf16_kernel(TileArgs a) {
  extern __shared__ __align__(16) unsigned char gt_smem[];
  bf16_t* As = reinterpret_cast<bf16_t*>(gt_smem);        // [2][128][GT_ROW]
  bf16_t* Bs = As + 2 * GT_BM * GT_ROW;                    // [2][128][GT_ROW]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int c = lane & 15, s = lane >> 4;
  const int tn = blockIdx.x, tm = blockIdx.y;
  const int M = a.M, N = a.N, K = a.K;

  // ---- global -> registers -> LDS: thread -> 16-byte chunk (tid & 7) of rows (tid >> 3) + 32 i
  const int chunk = tid & 7, row0 = tid >> 3;
  const bf16_t* xp[4];
  const bf16_t* wp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = min((int64_t)tm * GT_BM + row0 + 32 * i, (int64_t)M - 1);  // a row past the end repeats the last one
    xp[i] = a.X + m * a.ldx;
    bool ok;
    int64_t n = gt_w_row<MODE>(tn, row0 + 32 * i, N, &ok);
    if (!ok) n = 0;  // never stored
    wp[i] = a.W + n * K;
  }
  u32x4_t gx[4], gw[4];
  const int k_tiles = (K + GT_BK - 1) / GT_BK;
  auto fetch = [&](int kt) __attribute__((always_inline)) {
    const int k = kt * GT_BK + chunk * 8;
    const bool ok = k + 8 <= K;        // K is a multiple of 8: a chunk is inside or outside
    const int at = ok ? k : 0;         // a chunk outside reads the row's first one (inside the tensor) and is zeroed
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      gx[i] = *reinterpret_cast<const u32x4_t*>(xp[i] + at);
      gw[i] = *reinterpret_cast<const u32x4_t*>(wp[i] + at);
      if (!ok) {
        gx[i] = (u32x4_t){0u, 0u, 0u, 0u};
        gw[i] = (u32x4_t){0u, 0u, 0u, 0u};
      }
    }
  };
  auto stash = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<u32x4_t*>(As + (stage * GT_BM + row0 + 32 * i) * GT_ROW + chunk * 8) = gx[i];
      *reinterpret_cast<u32x4_t*>(Bs + (stage * GT_BN + row0 + 32 * i) * GT_ROW + chunk * 8) = gw[i];
    }
  };

  f32x4_t acc[4][4];  // [block of 16 rows of x][block of 16 rows of W]
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};

  auto multiply = [&](int stage) __attribute__((always_inline)) {
    const bf16_t* as = As + (stage * GT_BM + wm * 64 + c) * GT_ROW + s * 8;
    const bf16_t* bs = Bs + (stage * GT_BN + wn * 64 + c) * GT_ROW + s * 8;
#pragma unroll
    for (int kk = 0; kk < GT_BK / 32; ++kk) {
      bf16x8_t xf[4], wf[4];
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) xf[mi] = *reinterpret_cast<const bf16x8_t*>(as + mi * 16 * GT_ROW + kk * 32);
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) wf[ni] = *reinterpret_cast<const bf16x8_t*>(bs + ni * 16 * GT_ROW + kk * 32);
#pragma unroll
      for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
          acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ni], xf[mi], acc[mi][ni], 0, 0, 0);
    }
  };
  fetch(0);
  stash(0);
  __syncthreads();
  for (int kt = 0; kt < k_tiles; ++kt) {
    if (kt + 1 < k_tiles) fetch(kt + 1);  // in flight while this step is multiplied
    multiply(kt & 1);
    if (kt + 1 < k_tiles) stash((kt + 1) & 1);
    __syncthreads();
  }

  // ---- lane (c, s) holds y[m = .. + mi * 16 + c][4 s + e of W block ni], e = 0..3
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    const int64_t m = (int64_t)tm * GT_BM + wm * 64 + mi * 16 + c;
    if (m >= M) continue;
    if (MODE == 2) {
      const int I = N / 2;
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        const int64_t i0 = (int64_t)tn * 64 + wn * 32 + ni * 16 + 4 * s;
        if (i0 >= I) continue;
        uint16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = acc[mi][ni][e], up = acc[mi][ni + 2][e];
          o[e] = cw_float_to_bf16_bits(a.act > 0.0f ? cw_clipped_glu(g, up, a.act) : a.act < 0.0f ? cw_gated_below(g, up, a.act) : g / (1.0f + __expf(-g)) * up);
        }
        bf16_t* dst = (bf16_t*)a.C + m * a.ldc + i0;
        if (i0 + 4 <= I && !(a.ldc & 3)) {
          uint2 pk;
          pk.x = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
          pk.y = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
          *reinterpret_cast<uint2*>(dst) = pk;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (i0 + e < I) reinterpret_cast<uint16_t*>(dst)[e] = o[e];
        }
      }
    } else {
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        const int64_t n0 = (int64_t)tn * GT_BN + wn * 64 + ni * 16 + 4 * s;
        if (n0 >= N) continue;
        uint16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v = acc[mi][ni][e];
          if (a.bias != nullptr && n0 + e < N)
            v += a.bias_f32 ? ((const float*)a.bias)[n0 + e] : __bfloat162float(((const bf16_t*)a.bias)[n0 + e]);
          o[e] = cw_float_to_bf16_bits(v);
        }
        bf16_t* dst = (bf16_t*)a.C + m * a.ldc + n0;
        if (n0 + 4 <= N && !(a.ldc & 3)) {
          uint2 pk;
          pk.x = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
          pk.y = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
          *reinterpret_cast<uint2*>(dst) = pk;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n0 + e < N) reinterpret_cast<uint16_t*>(dst)[e] = o[e];
        }
      }
    }
  }
}

static const size_t GT_SMEM = (size_t)2 * (GT_BM + GT_BN) * GT_ROW * sizeof(bf16_t);

template <int MODE>
static int gt_launch(const TileArgs& a, hipStream_t stream) {
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_tile_bf16_kernel<MODE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)GT_SMEM) != hipSuccess)
      return CW_ERR_LAUNCH;
    raised = true;
  }
  const int out_cols = MODE == 2 ? a.N / 2 : a.N;
  const int per_tile = MODE == 2 ? 64 : GT_BN;
  dim3 grid((out_cols + per_tile - 1) / per_tile, (a.M + GT_BM - 1) / GT_BM);
  if (grid.y > 65535) return CW_ERR_SIZE;
  hipLaunchKernelGGL((gemm_tile_bf16_kernel<MODE>), grid, dim3(256), GT_SMEM, stream, a);
  return cw_launch_status();
}

// y = x W^T (+ bias) for bfloat16 x [M, K] (row stride ldx) and W [N, K]; K a multiple of 8.
// mode 0: y bfloat16 [M, N] (row stride ldc), bias nullptr or [N] bfloat16 / float32 (bias_f32);
// mode 2: y = silu(gate) * up, bfloat16 [M, N / 2], W = [gate; up], no bias.
CW_EXPORT int cw_gemm_bf16_tiled(int mode, const void* X, int64_t ldx, const void* W, const void* bias,
                                 int bias_f32, void* C, int64_t ldc, int M, int N, int K, float act, hipStream_t stream) {
  if (M < 0 || N <= 0 || K <= 0 || (mode != 0 && mode != 2) || !(act >= 0.0f || mode == 2)) return CW_ERR_ARG;
  if ((K & 7) || (ldx & 7) || ldx < K || ((uintptr_t)X & 15) || ((uintptr_t)W & 15) || ((uintptr_t)C & 7))
    return CW_ERR_ARG;
  if (mode == 2 && ((N & 1) || bias != nullptr)) return CW_ERR_ARG;
  if (ldc < (mode == 2 ? N / 2 : N)) return CW_ERR_ARG;
  if (M == 0) return CW_OK;
  TileArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, bias, bias_f32, C, ldc, M, N, K, act};
  return mode == 2 ? gt_launch<2>(a, stream) : gt_launch<0>(a, stream);
}


// ------------------------------------------------------------------------------------------------
// Wide tiles. One workgroup of 4 waves, or of 8 of which four load (APART below), per compute unit owns 32 MB rows of x by 32 NB rows of W; a
// wave owns a quarter of it in MB x NB accumulators of 16 x 16 (up to 288 registers; with 512
// registers a wave a SIMD holds this one wave, so everything that has a latency is overlapped by hand).
//
// K goes in stages of 64 elements: blocks of 8 rows x 128 bytes, whole lines of memory (half lines, as
// stages of 32 need them, take a fifth to a third longer). A block comes in by ONE buffer load with
// the LDS target (buffer_load_dwordx4 ... lds): lane l writes its 16 bytes at block + 16 l, no
// register and no LDS store instruction between. The eight granules of row r change places by
// (r >> 1) & 7, so that the 16 lanes that later read one granule column of 16 rows with ds_read_b128
// touch every bank once. The descriptors end with the matrices, so rows past the end read as zeros.
//
// SLOTS stages are in LDS. A stage is two phases of 32 elements of K: a phase multiplies one register
// set of fragments, reads the next phase's from LDS into the other set and, of 4 waves, takes part in the loads, all in
// the order written (sched_barrier). There is one wait and one barrier a stage, between its
// phases: there every wave has read the whole stage, whose slot the loads of SLOTS stages on then take, and
// stage t + 1 has landed, with SLOTS - 2 stages left in flight; the waits and barriers are bare
// instructions, since a fence would wait for every load in flight. The lower half of the x fragments
// has one register set: a row block's is read again when its products are issued.
//
// What bounds it. Inside a tile: with every load taken out the 1.5B shape's gate/up product of 2048
// rows takes 0.85 of its time, of 160 rows 0.6. A compute unit was seen to take in 43 GB/s from memory and 80 from
// L2 however deep the ring is, and x and W take the sum of what each takes alone (a queue of about 64 KB in the order of issue would do that), so a tile's
// loads go with (MB + NB) K, and its matrix instructions with MB NB K. Around it: a tile's first
// loads, its gate and its stores, 5 us a
// tile of 256 x 288, which only the next tile's first loads overlap. So few large tiles beat many small ones, in whole
// rounds over the units. Gate/up of the 1.5B shape, us by 256 x 192 tiles in stages of 32 -> here (tiles): 2048 rows
// 110 -> 99 (256 x 288, 504 in two rounds: 1.14 PFLOP/s), 1000 rows 70 -> 50 (256 x 288, 252 in one), 512 rows 37.3 -> 36.5
// (256 x 192, 188), 336 rows 35.6 -> 24.4 (192 x 160, 224), 160 rows 26.9 (64 x 128 below) -> 20.2 (160 x 96, 187). Two workgroups a unit of
// half the LDS each, to overlap one's gate with the other's products, gain nothing (2048 rows: 110).
//
// The workgroups of a launch are dealt to the 8 XCDs in turn; each XCD takes a run of consecutive
// tiles (8 row tiles by 4 W tiles at a time), each workgroup every
// 32nd tile of the run. Before a workgroup stores a tile it asks for the first stages of its
// next one, which arrive while the results go out.
//
// The rows of W are dealt to the 16 rows of a wave's blocks so that a lane ends up with neighbouring columns
// (wide_col). MODE 2: a block is 8 gate rows and the 8 up rows with the same indices, whose values a
// v_permlane32_swap of two blocks brings into one lane; four blocks give a lane 8 neighbouring outputs.
//
// MODE as above (2 with ``act`` > 0: the clipped gated activation of that limit, -1: max(gate, 0) * up, -2: gelu_tanh(gate) * up), and 5: MODE 0 with
// max(y, 0)^2, with ``act`` > 0 the tanh form of GELU, applied to the float32 sums (after the bias);
// K a multiple of 64, at least 256; both matrices below 4 GiB. MODE 3: the product
// of a narrow output with a long K (too few tiles to fill the card) summed in k_splits runs of K,
// each run of every tile a work item of its own; the items write float32 planes of partial sums
// [k_splits, M, N] that the next norm kernel adds up in their order.
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(2))) unsigned int w_u32x2_t;
typedef __attribute__((address_space(3))) void lds_void_t;

#define W_BM 256                           // the tile of the grouped products and of cw_gemm_bf16_wide_tiles
#define W_BN 192
#define W_BLOCK 1024                       // bytes of a block: 8 rows x 64 elements
#define W_GROUP_M 8                        // row tiles that run side by side

__device__ __forceinline__ uint32_t w_pack_bf16(float lo, float hi) {
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));  // v_cvt_pk_bf16_f32
}

struct WideArgs {
  const bf16_t* X;
  int64_t ldx;
  const bf16_t* W;
  const void* bias;
  int bias_f32;
  void* C;
  int64_t ldc;
  int M, N, K;
  int tiles_m, tiles_n;
  int k_splits;  // MODE 3: K is cut into this many runs, each a tile of its own with a float32 plane of partial sums
  // GROUPED: every row tile of x multiplies a matrix of its own (rows sorted by expert)
  const int* tile_group;    // [row tiles] which of the stacked matrices a row tile takes
  const int* n_row_tiles;   // [1] how many row tiles there are in this launch (on the device)
  const int* row_target;    // nullptr: row m of the result is row m of C; else its row there, < 0: not stored
  const float* row_factor;  // nullptr, or a factor for the results that go to row row_target[m]: row_factor[row_target[m]]
  int64_t w_group_stride;   // elements from one stacked matrix to the next
  float act;                // MODE 2 and 5: which activation (see above)
  // MODE 6 (of gemm_mid_bf16_kernel): heads of queries, keys and values, rotated and stored where they belong
  const float* angles;      // [rows][2][hd / 2] cosines and sines of a row's position
  const int* slots;         // [rows] the row of the caches, beyond them: none
  bf16_t* k_cache;          // [cache_rows][nkv][hd]
  bf16_t* v_cache;
  int64_t cache_rows;
  int nh, nkv, hd;
};

// MODE 6: a column of the result is a pair of a head, elements d and d + hd / 2; the row of W of its first element.
__device__ __forceinline__ int64_t pair_row(int pair, int hd) { return (int64_t)(pair / (hd / 2)) * hd + pair % (hd / 2); }

// Where the pairs of head ``head`` of row m go: a query to its row of C, a key or value to its slot; nullptr: nowhere.
__device__ __forceinline__ bf16_t* pair_target(const WideArgs& a, int64_t m, int head, int64_t slot) {
  if (head < a.nh) return (bf16_t*)a.C + m * a.ldc + (int64_t)head * a.hd;
  if (slot < 0 || slot >= a.cache_rows) return nullptr;
  return (head < a.nh + a.nkv ? a.k_cache + (slot * a.nkv + head - a.nh) * a.hd : a.v_cache + (slot * a.nkv + head - a.nh - a.nkv) * a.hd);
}

// The column of a wave's part of the tile (MODE 2: the output) that row r of its W block ni belongs to. The
// accumulator of a block holds rows 4 s .. 4 s + 3 in lane (c, s). Two blocks: 8 neighbouring columns a lane. MODE 2,
// where s of 0 and 1 hold gates and s of 2 and 3 the ups to them: after the swap of two blocks lane s has 4 outputs, of four
// blocks 8; what is left over keeps its order.
template <int MODE, int NB>
__host__ __device__ __forceinline__ int wide_col(int ni, int r) {
  const int s = r >> 2, e = r & 3;
  if (MODE == 2) {
    const int s1 = s & 1;
    if (ni < (NB & ~3)) return (ni >> 2) * 32 + ((ni & 1) * 2 + s1) * 8 + ((ni >> 1) & 1) * 4 + e;
    if ((NB & 2) && ni < (NB & ~1)) return (NB & ~3) * 8 + ((ni & 1) * 2 + s1) * 4 + e;
    return (NB - 1) * 8 + s1 * 4 + e;
  }
  return ni < (NB & ~1) ? (ni >> 1) * 32 + s * 8 + (ni & 1) * 4 + e : ni * 16 + r;
}

// cw_gated from the bare exp2 and reciprocal instructions (by expf and a division, as the smaller tiles do it, the bfloat16 results
// are as far from 64 bits to seven digits; 5 to 11 in a million are others). A build of the kernel for each: asked for at every value the activation
// took a fifth of 1600 rows' time with relu, asked for once a tile it took a copy of the tile's end for each, whose addresses
// went to scratch in the widest tile. 17920 x 1536 with silu / relu / GELU / clipped, us: 2048 rows 92.5 / 99.7 / 106.5 / 107.7 with
// three copies, 92.5 / 92.2 / 94.1 / 95.3 now; 1000 rows 49.4 / 52.0 / 56.2 / 56.6, now 49.3 / 48.2 / 49.6 / 50.0; 160 rows 22 throughout.
#define W_GATE_SILU 0
#define W_GATE_CLIPPED 1
#define W_GATE_RELU 2
#define W_GATE_GELU 3
static int w_gate(float act) {
  return act > 0.0f ? W_GATE_CLIPPED : act < -1.5f ? W_GATE_GELU : act < 0.0f ? W_GATE_RELU : W_GATE_SILU;
}
template <int GATE>
__device__ __forceinline__ float w_gated(float g, float up, float act) {
  if (GATE == W_GATE_CLIPPED) {
    const float gl = fminf(g, act), ul = fminf(fmaxf(up, -act), act);
    return gl * __builtin_amdgcn_rcpf(1.0f + __expf(-1.702f * gl)) * (ul + 1.0f);
  }
  if (GATE == W_GATE_RELU) return fmaxf(g, 0.0f) * up;
  if (GATE == W_GATE_GELU) return g * __builtin_amdgcn_rcpf(1.0f + __expf(-1.5957691216057308f * (g + 0.044715f * g * g * g))) * up;
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * up;
}

// s_waitcnt for "at most n vector-memory operations in flight" and nothing else
#define W_WAIT_LOADS(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14))
#define W_WAIT_LDS() __builtin_amdgcn_s_waitcnt(0xC07F)  // every LDS read of this wave is back
// a barrier without a fence: what it orders is said at each use
#define W_BARRIER()                 \
  do {                              \
    asm volatile("" ::: "memory"); \
    __builtin_amdgcn_s_barrier();   \
    asm volatile("" ::: "memory"); \
  } while (0)

// APART: four waves of their own load a tile, where its products leave them registers (256 a thread beside the four that multiply; 192 x
// 192 spilled 18). A wave that loads and multiplies stands still at each load that the load path does not take in yet, and its
// products with it: loads alone took 20.8 of 21.9 us of 160 rows of 17920 x 1536 (x alone 8.1, W alone 13.8: they add up, one queue of about 64 KB a
// compute unit in the order of issue; rings of their own, W eight stages deep, changed nothing). us, then / now: 160 and 352 rows of
// that 22.0 / 21.3, 26.1 / 25.3, 1000 of it by 192 x 160 62.5 / 54.9; 2048 rows of 1536 x 1536 13.9 / 13.1, of 2048 x 1536 17.0 / 16.0; 160 and 352 rows of 1536 x 8960 in
// planes 14.5 / 14.1, 19.7 / 19.2; over 26 shapes and the tiles in question 5 % in the mean.
static constexpr bool w_loads_apart(int mb, int nb) { return mb * nb <= 32; }

template <int MODE, int MB, int NB, int SLOTS, bool ANY_ROWS = true, bool GROUPED = false, int GATE = W_GATE_SILU, bool APART = w_loads_apart(MB, NB)>
__global__ __launch_bounds__(APART ? 512 : 256) void gemm_wide_bf16_kernel(WideArgs a) {
  extern __shared__ __align__(1024) unsigned char w_smem[];
  constexpr bool GATED = MODE == 2;
  constexpr int BM = 32 * MB, BN = 32 * NB, PER = GATED ? BN / 2 : BN;  // PER: columns of the result
  constexpr int LOADS = MB + NB;                                            // of a wave and stage: MB of x, NB of W
  constexpr int STAGE = 4 * LOADS * W_BLOCK;
  static_assert(SLOTS >= 2 && SLOTS * STAGE <= 160 * 1024 && SLOTS * LOADS <= 63 && SLOTS <= 6, "the ring is the LDS of a compute unit");
  const int tid = threadIdx.x, lane = tid & 63, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3;
  const int wm = wave >> 1, wn = wave & 1;
  const int c = lane & 15, s = lane >> 4;
  // GROUPED: the number of row tiles is known on the device alone; x holds whole tiles
  const int tiles_m = GROUPED ? __builtin_amdgcn_readfirstlane(*a.n_row_tiles) : a.tiles_m;
  const int M = GROUPED ? tiles_m * BM : a.M, N = a.N, K = a.K, I = N / 2;
  const int per_split = tiles_m * a.tiles_n;
  const int total = per_split * (MODE == 3 ? a.k_splits : 1);
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const int run = total >> 3, rest = total & 7;
  const int run_begin = xcd * run + min(xcd, rest), run_end = run_begin + run + (xcd < rest ? 1 : 0);
  // tile id -> (row tile, W tile): groups of W_GROUP_M row tiles, inside a group the row tiles
  // of one W tile next to each other
  auto tile_of = [&](int id, int* tm, int* tn) __attribute__((always_inline)) {
    if (MODE == 3) id %= per_split;  // the runs of K one after the other, each over all tiles
    const int per_group = W_GROUP_M * a.tiles_n;
    const int group = id / per_group, within = id - group * per_group;
    const int rows = min(W_GROUP_M, tiles_m - group * W_GROUP_M);
    *tn = within / rows;
    *tm = group * W_GROUP_M + (within - *tn * rows);
  };

  // Load i of a wave: MB blocks of x, every fourth, then the NB blocks of its half of W that hold the first or the last 8 rows
  // of the fragments. Lane: granule (lane & 7) of row lane / 8 of a block. The rows of a wave's loads lie fixed numbers of rows
  // apart, so few registers of addresses do (with 17 of them the widest tile's spilled, 5 us a tile).
  const int parity = wave & 1, half = wave >> 1, r = parity * 8 + (lane >> 3);
  const uint32_t granule_in = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
  const uint32_t x_at = (uint32_t)((int64_t)(half * 16 + r) * a.ldx * 2) + granule_in, x_step = (uint32_t)a.ldx * 64, w_row = (uint32_t)K * 2;
  constexpr int REGULAR = GATED ? NB & ~3 : NB & ~1;  // blocks whose rows wide_col deals alike; the others one more register
  auto w_first = [&](int ni) __attribute__((always_inline)) {
    const int col = half * (PER / 2) + wide_col<MODE, NB>(ni, r) - wide_col<MODE, NB>(ni, 0);
    return (uint32_t)((int64_t)(GATED && parity ? I + col : col) * K * 2) + granule_in;
  };
  const uint32_t w_at = w_first(0), w_at_rest = w_first(NB - 1);
  // stages of K before work item id's run
  auto stages_before = [&](int plane) __attribute__((always_inline)) { return MODE == 3 ? (int)((int64_t)(K / 64) * plane / a.k_splits) : 0; };
  int stages;  // of the work item that comes in
  __amdgpu_buffer_rsrc_t xr, wr;
  auto aim = [&](int id) __attribute__((always_inline)) {
    int tm, tn;
    tile_of(id, &tm, &tn);
    const int plane = MODE == 3 ? id / per_split : 0;
    const int64_t k0 = (int64_t)stages_before(plane) * 64;
    stages = MODE == 3 ? stages_before(plane + 1) - stages_before(plane) : K / 64;
    const int k_run = stages * 64;
    const int64_t x_row0 = (int64_t)tm * BM, w_row0 = (int64_t)tn * PER;
    // the descriptors begin at the run's first element of the tile's first row and end with the
    // run's last element of the matrix's last row: rows past the end read as zeros
    xr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.X + x_row0 * a.ldx + k0), 0,
                                           (int)(uint32_t)(((M - x_row0 - 1) * a.ldx + k_run) * 2), 0x00020000);
    const bf16_t* w_base = GROUPED ? a.W + (int64_t)__builtin_amdgcn_readfirstlane(a.tile_group[tm]) * a.w_group_stride : a.W;
    wr = __builtin_amdgcn_make_buffer_rsrc((void*)(w_base + w_row0 * K + k0), 0,
                                           (int)(uint32_t)(((N - w_row0 - 1) * (int64_t)K + k_run) * 2), 0x00020000);
  };
  auto fetch_as = [&](bool once, int stage, int slot, int i) __attribute__((always_inline)) {
    uint32_t apart = i < MB ? i * x_step : wide_col<MODE, NB>(i - MB, 0) * w_row;
    asm volatile("" : "+s"(apart));  // added here and now: the sums of all loads would take as many registers
    if (i < MB) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void_t*)(w_smem + slot + (i * 4 + wave) * W_BLOCK), 16, x_at + apart, stage * 128, 0, 0);
    } else {
      const int ni = i - MB;
      lds_void_t* to = (lds_void_t*)(w_smem + slot + (4 * MB + (half * NB + ni) * 2 + parity) * W_BLOCK);
      const uint32_t from = (ni < REGULAR ? w_at : w_at_rest) + apart;
      if (once) __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, to, 16, from, stage * 128, 0, 2);  // 2: nontemporal
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, to, 16, from, stage * 128, 0, 0);
    }
  };
  auto fetch_one = [&](int stage, int slot, int i) __attribute__((always_inline)) { fetch_as(false, stage, slot, i); };
  // (of fewer stages than slots the last comes in again: the number of loads in flight is what the waits count on)
  auto fetch_first_stages = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SLOTS; ++j)
#pragma unroll
      for (int i = 0; i < LOADS; ++i) fetch_one(min(j, stages - 1), j * STAGE, i);
  };

  constexpr int PRODUCTS = MB * NB, READS = MB + NB;
  f32x4_t acc[MB][NB];
  bf16x8_t xf[2][MB], wf[2][NB];
  auto x_set = [](int set, int mi) __attribute__((always_inline)) { return mi < MB / 2 ? 0 : set; };
  const unsigned char* x_base = w_smem + c * 128 + wm * MB * 2048;
  const unsigned char* w_base = w_smem + c * 128 + (2 * MB + wn * NB) * 2048;
  const int granule[2] = {((s) ^ ((c >> 1) & 7)) * 16, ((4 + s) ^ ((c >> 1) & 7)) * 16};
  // read i of a phase's fragments: W first, x in the order of its use
  auto read_one = [&](int slot, int half, int set, int i) __attribute__((always_inline)) {
    if (i < NB) wf[set][i] = *reinterpret_cast<const bf16x8_t*>(w_base + slot + granule[half] + i * 2048);
    else xf[x_set(set, i - NB)][i - NB] = *reinterpret_cast<const bf16x8_t*>(x_base + slot + granule[half] + (i - NB) * 2048);
  };
  // One phase: the products of register set ``set``, a tile's first ones if ``first``; with_read: the next phase's fragments, of half ``half`` of the stage
  // in ``read_slot``; loads from .. to of the wave's for stage ``stage`` into ``load_slot``.
  auto phase = [&](auto first_c, auto set_c, auto read_c, int read_slot, int half, auto from_c, auto to_c, int stage, int load_slot) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value, from = decltype(from_c)::value, count = decltype(to_c)::value - from;
    constexpr bool first = decltype(first_c)::value, with_read = decltype(read_c)::value;
#pragma unroll
    for (int g = 0; g < PRODUCTS; ++g) {
      const int mi = g / NB, ni = g % NB;
      if constexpr (PRODUCTS <= 64) {
        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][ni], xf[x_set(set, mi)][mi], first ? (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f} : acc[mi][ni], 0, 0, 0);
      } else {
        // More accumulators than there are accumulation registers: 62 live there and the others with the operands. Left to
        // itself the compiler keeps all in one kind and moves a hundred of them back and forth an iteration. It does not know
        // either that these are products, which may read what it has written two states before at the earliest; so their
        // first ones begin with a zero of their own, and nothing writes an accumulator but products. (tests/test_build.py looks
        // for operands written too late in the code as built.)
        if (first && g < 62) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&a"(acc[mi][ni]) : "v"(wf[set][ni]), "v"(xf[x_set(set, mi)][mi]));
        else if (first) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(acc[mi][ni]) : "v"(wf[set][ni]), "v"(xf[x_set(set, mi)][mi]));
        else if (g < 62) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[mi][ni]) : "v"(wf[set][ni]), "v"(xf[x_set(set, mi)][mi]));
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[mi][ni]) : "v"(wf[set][ni]), "v"(xf[x_set(set, mi)][mi]));
      }
      // reads and loads spread over the products (the texture path takes a load every 16 cycles; several in a row stall
      // the wave), the reads done a little before the end
      constexpr int SPAN = PRODUCTS - 3;
      const int r0 = min(g * READS / SPAN, READS), r1 = min((g + 1) * READS / SPAN, READS);
      const int l0 = (2 * g + 1) * count / (2 * PRODUCTS), l1 = (2 * g + 3) * count / (2 * PRODUCTS);
      if ((with_read && r0 < r1) || l0 < l1) {
        // the order of issue is the order written here: the scheduler may move nothing across
        __builtin_amdgcn_sched_barrier(0);
        if (with_read)
#pragma unroll
          for (int r = r0; r < r1; ++r) read_one(read_slot, half, set ^ 1, r);
#pragma unroll
        for (int l = l0; l < l1; ++l) fetch_one(stage, load_slot, from + l);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // what the compiler does not know of products that it has not written: their results need this long before a move of
    // accumulators (at the loop's ends) may read them
    if constexpr (PRODUCTS > 64) asm volatile("s_nop 15" ::: "memory");
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using Last = std::integral_constant<int, LOADS>;
  // two slots: all loads in the phase behind the barrier, else half of them in the next one
  using Split = std::integral_constant<int, SLOTS == 2 ? LOADS : (LOADS + 1) / 2>;
  using Yes = std::true_type;
  using No = std::false_type;
  auto next_slot = [](int slot) __attribute__((always_inline)) { return slot == (SLOTS - 1) * STAGE ? 0 : slot + STAGE; };

  int id = run_begin + local;
  if (id >= run_end) return;
  if constexpr (APART) {
    if (wave8 >= 4) {
      // Barrier n of the workgroup: stage n is in LDS, and the waves that multiply have read stage n - 1, whose slot
      // the next loads take. The stages of all its tiles are one row, so a tile's first come in while the last one's results go out.
      int ahead = 0, to = 0;
      // One or two row tiles, side by side on one XCD, read a matrix once: its lines need not stay in the caches, which are then x's and the
      // next kernels' (160 and 352 rows of 17920 x 1536 21.3 -> 20.4 us, 25.3 -> 24.6; with 7 row tiles 32 -> 39). From 32 MB on: smaller ones gain nothing and
      // partly wait longer (a step of 137 tokens of the 1.5B shape 2074 us with none so, 2082 with all, 2067 so; 100 tokens of the 7B shape 4611, 4400, 4283).
      const bool once = tiles_m <= 2 && (int64_t)N * K >= (1 << 24);
      for (; id < run_end; id += per_xcd) {
        aim(id);
        for (int t = 0; t < stages; ++t) {
          if (ahead == SLOTS - 1) {
            W_WAIT_LOADS((SLOTS - 2) * LOADS);
            W_BARRIER();
          } else {
            ++ahead;
          }
          if (once) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) fetch_as(true, t, to, i);
          } else {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) fetch_one(t, to, i);
          }
          to = next_slot(to);
        }
      }
      // the last ones, each as it comes in
      auto last = [&](auto behind_c) __attribute__((always_inline)) {
        constexpr int behind = decltype(behind_c)::value;
        if (behind < SLOTS - 1 && ahead > behind) {
          W_WAIT_LOADS((behind < SLOTS - 1 ? behind : 0) * LOADS);
          W_BARRIER();
        }
      };
      last(std::integral_constant<int, 4>{});
      last(std::integral_constant<int, 3>{});
      last(std::integral_constant<int, 2>{});
      last(std::integral_constant<int, 1>{});
      last(std::integral_constant<int, 0>{});
      return;
    }
  } else {
    aim(id);
    fetch_first_stages();
  }
  int slot = 0;
  for (bool first = true; id < run_end; id += per_xcd, first = false) {
    int tm, tn;
    tile_of(id, &tm, &tn);
    if constexpr (APART) {
      aim(id);  // (for its number of stages)
      W_BARRIER();
#pragma unroll
      for (int i = 0; i < READS; ++i) read_one(slot, 0, 0, i);
      phase(Yes{}, I0{}, Yes{}, slot, 1, I0{}, I0{}, 0, 0);
      for (int t = 1; t < stages; ++t) {
        W_WAIT_LDS();
        W_BARRIER();
        slot = next_slot(slot);
        phase(No{}, I1{}, Yes{}, slot, 0, I0{}, I0{}, 0, 0);
        phase(No{}, I0{}, Yes{}, slot, 1, I0{}, I0{}, 0, 0);
      }
      phase(No{}, I1{}, No{}, 0, 0, I0{}, I0{}, 0, 0);
      W_WAIT_LDS();
      slot = next_slot(slot);
    } else {
      // the first stage is in LDS (a tile's stores come after its successor's loads, and count as well)
      if (first) W_WAIT_LOADS((SLOTS - 1) * LOADS);
      else W_WAIT_LOADS(0);
      W_BARRIER();
#pragma unroll
      for (int i = 0; i < READS; ++i) read_one(0, 0, 0, i);
      slot = 0;
      int t = 0;
      phase(Yes{}, I0{}, Yes{}, slot, 1, I0{}, I0{}, 0, 0);
      // every wave has read stage t and its loads of stage t + 1 have landed
      W_WAIT_LOADS((SLOTS - 2) * LOADS);
      W_WAIT_LDS();
      W_BARRIER();
      for (; t + SLOTS < stages; ++t) {
        const int next = next_slot(slot);
        phase(No{}, I1{}, Yes{}, next, 0, I0{}, Split{}, t + SLOTS, slot);
        phase(No{}, I0{}, Yes{}, next, 1, Split{}, Last{}, t + SLOTS, slot);
        W_WAIT_LOADS((SLOTS - 2) * LOADS);
        W_WAIT_LDS();
        W_BARRIER();
        slot = next;
      }
      W_WAIT_LOADS(0);
      W_BARRIER();  // the last stages are in
      for (; t + 1 < stages; ++t) {
        const int next = next_slot(slot);
        phase(No{}, I1{}, Yes{}, next, 0, I0{}, I0{}, 0, 0);
        phase(No{}, I0{}, Yes{}, next, 1, I0{}, I0{}, 0, 0);
        slot = next;
      }
      phase(No{}, I1{}, No{}, 0, 0, I0{}, I0{}, 0, 0);
      W_WAIT_LDS();
      W_BARRIER();
      // every slot is free: the first stages of the next tile come in while this one's results go out
      if (id + per_xcd < run_end) {
        aim(id + per_xcd);
        fetch_first_stages();
      }
    }

    const int out_cols = GATED ? I : N;
    constexpr int ELEMENT = MODE == 3 ? 4 : 2;
    unsigned char* C = (unsigned char*)a.C + (MODE == 3 ? (int64_t)(id / per_split) * M * a.ldc * 4 : 0);
    const int64_t row0 = (int64_t)tm * BM + wm * (16 * MB);
    const int col0 = tn * PER + wn * (PER / 2);
    // Rows of 16-byte multiples: buffer stores, whose descriptor ends with the last row and drops what is told to lie beyond, so
    // nothing branches at a store. (With branches the last tile of a row, 32 of 96 columns, took the 1.5B shape's product of 512
    // rows from 36 to 43 us.)
    // ANY_ROWS: any other rows too, a value a store. (Two ends of a tile in one kernel keep so much alive that the widest tile's
    // registers spill, and what comes back from scratch waits for the next tile's first loads, 5 us a tile: that tile takes whole
    // rows only.)
    const bool whole = !ANY_ROWS || !(a.ldc & (16 / ELEMENT - 1)) && !((uintptr_t)a.C & 15) && !(out_cols & (16 / ELEMENT - 1)) && a.ldc < (1 << 20);
    const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(C + ((int64_t)tm * BM * a.ldc + tn * PER) * ELEMENT), 0,
        (int)(uint32_t)((min((int64_t)M - (int64_t)tm * BM - 1, (int64_t)BM) * a.ldc + min(PER, out_cols - tn * PER)) * ELEMENT), 0x00020000);
    const uint32_t c_row = (uint32_t)(((wm * 16 * MB + c) * a.ldc + wn * (PER / 2)) * ELEMENT), c_step = (uint32_t)(16 * a.ldc * ELEMENT);
    // count neighbouring columns from column n of the wave's part on, in row block mi
    auto store_whole = [&](int mi, uint32_t more, int n, const float* v, auto count_c) __attribute__((always_inline)) {
      constexpr int count = decltype(count_c)::value;
      const uint32_t to = col0 + n < out_cols ? c_row + mi * c_step + more + n * ELEMENT : 0x80000000u;
      if constexpr (MODE == 3) {
        const f32x4_t v4 = {v[0], v[1], v[2], v[3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v4), cr, to, 0, 0);
      } else if constexpr (count == 8) {
        const u32x4_t w4 = {w_pack_bf16(v[0], v[1]), w_pack_bf16(v[2], v[3]), w_pack_bf16(v[4], v[5]), w_pack_bf16(v[6], v[7])};
        __builtin_amdgcn_raw_buffer_store_b128(w4, cr, to, 0, 0);
      } else {
        const w_u32x2_t w2 = {w_pack_bf16(v[0], v[1]), w_pack_bf16(v[2], v[3])};
        __builtin_amdgcn_raw_buffer_store_b64(w2, cr, to, 0, 0);
      }
    };
    // the same for any tile: row m of C
    auto store = [&](int64_t m, bool live, int n, const float* v, auto count_c) __attribute__((always_inline)) {
      constexpr int count = decltype(count_c)::value;
      if (!live) return;
#pragma unroll
      for (int e = 0; e < count; ++e) {
        if (col0 + n + e >= out_cols) continue;
        if constexpr (MODE == 3) ((float*)C)[m * a.ldc + col0 + n + e] = v[e];
        else ((uint16_t*)C)[m * a.ldc + col0 + n + e] = (uint16_t)w_pack_bf16(v[e], 0.0f);
      }
    };
    using Four = std::integral_constant<int, 4>;
    using Eight = std::integral_constant<int, 8>;
    if constexpr (GATED) {
      auto all = [&](auto whole_c) __attribute__((always_inline)) {
        constexpr bool whole_tile = decltype(whole_c)::value;
        // gates of two accumulators and the ups to them, each in one lane
        auto gated = [&](const f32x4_t& p, const f32x4_t& q, float* v) __attribute__((always_inline)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const cw_u32x2_t gu = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[e]), __float_as_uint(q[e]), false, false);
            v[e] = w_gated<GATE>(__uint_as_float(gu[0]), __uint_as_float(gu[1]), a.act);
          }
        };
#pragma unroll
        for (int mi = 0; mi < MB; ++mi) {
          const int64_t m = row0 + mi * 16 + c;
#pragma unroll
          for (int q = 0; q + 3 < NB; q += 4) {
            float v[8];
            gated(acc[mi][q], acc[mi][q + 1], v);
            gated(acc[mi][q + 2], acc[mi][q + 3], v + 4);
            if (whole_tile) store_whole(mi, 0, q * 8 + s * 8, v, Eight{});
            else store(m, m < M, q * 8 + s * 8, v, Eight{});
          }
          if constexpr ((NB & 2) != 0) {
            float v[4];
            gated(acc[mi][NB & ~3], acc[mi][(NB & ~3) + 1], v);
            if (whole_tile) store_whole(mi, 0, (NB & ~3) * 8 + s * 4, v, Four{});
            else store(m, m < M, (NB & ~3) * 8 + s * 4, v, Four{});
          }
          if ((NB & 1) && !(mi & 1)) {
            // the last block alone: of this row block and of the next, if there is one
            const int other = mi + 1 < MB ? mi + 1 : mi;
            const int64_t m2 = m + (s >> 1) * 16;
            float v[4];
            gated(acc[mi][NB - 1], acc[other][NB - 1], v);
            if (whole_tile) {
              if (s < 2 || other != mi) store_whole(mi, (s >> 1) * c_step, (NB - 1) * 8 + (s & 1) * 4, v, Four{});
            } else {
              store(m2, m2 < M && (s < 2 || other != mi), (NB - 1) * 8 + (s & 1) * 4, v, Four{});
            }
          }
        }
      };
      if (whole) all(Yes{});
      else if constexpr (ANY_ROWS) all(No{});
    } else {
      auto all = [&](auto whole_c) __attribute__((always_inline)) {
        constexpr bool whole_tile = decltype(whole_c)::value;
#pragma unroll
        for (int mi = 0; mi < MB; ++mi) {
          int64_t m = row0 + mi * 16 + c;
          bool live = m < M;
          float row_factor = 1.0f;  // GROUPED: of the row that is being stored
          if (GROUPED && a.row_target != nullptr) {
            const int target = live ? a.row_target[m] : -1;
            live = target >= 0;
            row_factor = (live && a.row_factor != nullptr) ? a.row_factor[target] : 1.0f;
            m = live ? target : 0;
          }
          auto value = [&](int ni, float* v) __attribute__((always_inline)) {
            const int n0 = col0 + wide_col<MODE, NB>(ni, 4 * s);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v[e] = acc[mi][ni][e];
              if (MODE == 3) continue;
              if (a.bias != nullptr && n0 + e < N)
                v[e] += a.bias_f32 ? ((const float*)a.bias)[n0 + e] : __bfloat162float(((const bf16_t*)a.bias)[n0 + e]);
              if (GROUPED) v[e] *= row_factor;
              if (MODE == 5) {
                if (a.act > 0.0f) {
                  v[e] *= __builtin_amdgcn_rcpf(1.0f + __expf(-1.5957691216057308f * (v[e] + 0.044715f * v[e] * v[e] * v[e])));
                } else {
                  const float r = fmaxf(v[e], 0.0f);
                  v[e] = r * r;
                }
              }
            }
          };
          // GROUPED with targets: the rows lie apart
          auto put = [&](int n, const float* v, auto count_c) __attribute__((always_inline)) {
            if constexpr (GROUPED) {
              if (whole_tile) {
                if (live && col0 + n < out_cols) {
                  uint16_t* to = (uint16_t*)C + m * a.ldc + col0 + n;
                  if constexpr (decltype(count_c)::value == 8)
                    *reinterpret_cast<uint4*>(to) = make_uint4(w_pack_bf16(v[0], v[1]), w_pack_bf16(v[2], v[3]), w_pack_bf16(v[4], v[5]), w_pack_bf16(v[6], v[7]));
                  else
                    *reinterpret_cast<uint2*>(to) = make_uint2(w_pack_bf16(v[0], v[1]), w_pack_bf16(v[2], v[3]));
                }
              } else {
                store(m, live, n, v, count_c);
              }
            } else {
              if (whole_tile) store_whole(mi, 0, n, v, count_c);
              else store(m, live, n, v, count_c);
            }
          };
#pragma unroll
          for (int ni = 0; ni + 1 < NB; ni += 2) {
            float v[8];
            value(ni, v);
            value(ni + 1, v + 4);
            if constexpr (MODE == 3) {
              put(ni * 16 + s * 8, v, Four{});
              put(ni * 16 + s * 8 + 4, v + 4, Four{});
            } else {
              put(ni * 16 + s * 8, v, Eight{});
            }
          }
          if constexpr ((NB & 1) != 0) {
            float v[4];
            value(NB - 1, v);
            put((NB - 1) * 16 + s * 4, v, Four{});
          }
        }
      };
      if (whole) all(Yes{});
      else if constexpr (ANY_ROWS) all(No{});
    }
  }
}

static int w_tiles(int mode, int M, int N) {
  const int out_cols = mode == 2 ? N / 2 : N;
  const int per_tile = mode == 2 ? W_BN / 2 : W_BN;
  return ((M + W_BM - 1) / W_BM) * ((out_cols + per_tile - 1) / per_tile);
}

// Does the wide-tile kernel take this product? Returns its number of tiles of 256 x 192, or 0.
CW_EXPORT int cw_gemm_bf16_wide_tiles(int mode, int M, int N, int K, int64_t ldx) {
  if (M <= 0 || N <= 0 || (mode != 0 && mode != 2 && mode != 5) || (mode == 2 && (N & 1))) return 0;
  if ((K & 63) || K < 256 || (ldx & 7) || ldx < K) return 0;
  if ((int64_t)N * K * 2 >= (1ll << 32) || (int64_t)M * ldx * 2 >= (1ll << 32)) return 0;
  return w_tiles(mode, M, N);
}

// 1 if the wide-tile kernel sums this product in ``k_splits`` runs of K (cw_gemm_bf16_wide_partial).
CW_EXPORT int cw_gemm_bf16_wide_partial_ok(int M, int N, int K, int64_t ldx, int k_splits) {
  if (k_splits < 2 || k_splits > 16 || K % (64 * k_splits) || K / k_splits < 256) return 0;
  return cw_gemm_bf16_wide_tiles(0, M, N, K, ldx) > 0 ? 1 : 0;
}

// ``row_tiles``: GROUPED: how many there are at most
template <int MODE, int MB, int NB, int SLOTS, bool ANY_ROWS = true, bool GROUPED = false, int GATE = W_GATE_SILU>
static int w_launch(WideArgs a, int row_tiles, int workgroups, hipStream_t stream) {
  constexpr int SMEM = SLOTS * 4 * (MB + NB) * W_BLOCK;
  constexpr bool gated = MODE == 2;
  const int out_cols = gated ? a.N / 2 : a.N, per_tile = gated ? 16 * NB : 32 * NB;
  a.tiles_n = (out_cols + per_tile - 1) / per_tile;
  a.tiles_m = GROUPED ? 0 : (a.M + 32 * MB - 1) / (32 * MB);  // GROUPED: read on the device
  const int64_t total = (int64_t)(GROUPED ? row_tiles : a.tiles_m) * a.tiles_n * (MODE == 3 ? a.k_splits : 1);
  if (total > 0x3fffffff) return CW_ERR_SIZE;
  // a multiple of 8 workgroups, so that every XCD gets the same number of them
  int grid = total < workgroups ? (int)total : workgroups;
  grid = (grid + 7) & ~7;
  auto launch = [&](auto apart_c) -> int {
    constexpr bool APART = decltype(apart_c)::value;
    const auto kernel = gemm_wide_bf16_kernel<MODE, MB, NB, SLOTS, ANY_ROWS, GROUPED, GATE, APART>;
    static std::atomic<bool> allowed{false};
    const int status = cw_allow_lds(allowed, (const void*)kernel, SMEM);
    if (status != CW_OK) return status;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(APART ? 512 : 256), SMEM, stream, a);
    return cw_launch_status();
  };
  constexpr bool APART = w_loads_apart(MB, NB);
  // Of planes of more than four row tiles, which ask L2 for more than it gives in any case, only K whole or in two runs. Steps, us, loads by all waves / by waves
  // of their own: two planes, 2048 tokens of the 1.5B shape 6950 / 6917 and 6902 / 6874 (two cards), behind 4000 8754 / 8732, 2000 beside 15 requests
  // 7164 / 7140, of the 0.5B shape 3330 / 3313, 3318 / 3304, one or two, of the 7B shape 25339 / 25119, 25436 / 25211, 800 tokens 12229 / 11997; three
  // planes, 1000 tokens of the 1.5B shape behind 7000 5885 / 5975, 5800 / 5885, 5614 / 5593 (three cards; the product alone 32.3 / 31.0), behind none 4129 /
  // 4157; four, 700 and 800 tokens 3537 / 3530, 4373 / 4348.
  if constexpr (MODE == 3 && APART)
    if (a.tiles_m > 4 && a.k_splits > 2) return launch(std::false_type{});
  return launch(std::integral_constant<bool, APART>{});
}

// What a tile costs: ``fixed`` us of a work item and stage[q - 1] us a stage of 64 elements of K while q workgroups share a
// compute unit (the smallest tiles; the others have one to themselves). Fits over timings with operands from memory, 72 to
// 2048 rows of 26 shapes of the 0.5B to 14B models' layers and others (N 512 to 37888, K 512 to 18944); the fixed cost of 64 x 128
// after another 22000, 65 to 2048 rows of 38 shapes. Over those a tile's time (and a launch's beside) is off by 7.5 % in the mean;
// a tile that the rule names takes 1 to 1.6 % more than the fastest, the library among them, 24 % at worst (272 rows of 6144 x 1536 with
// a gate 18.4 by 160 x 96, 14.9 by 128 x 128; 704 rows of 1024 x 4096 and a norm 20.9, 17.9 by 96 x 96). A stage of the large tiles goes with BM + BN, 2.3 ns a row: its
// loads; 256 x 192 and 256 x 288 have two stages of them in LDS and wait longer, and gain by their few rounds.
// (Timed before tiles up to 192 x 160 had waves of their own for their loads, which took 5 % off them. Of 42 products of 100 to 2048 rows timed by
// every tile since, the rule's is the fastest for 38, and 1.6, 1.6, 4 and 9 % behind for four.)
struct TileRate {
  int bm, bn, modes, per_unit;  // modes: a bit each of 0, 2 and 3 (1, 2, 4); 8: rows of any length
  float fixed, stage[3];
};
static const TileRate TILE_RATES[] = {
    {64, 64, 15, 3, -1.63f, {0.342f, 0.556f, 0.809f}}, {64, 128, 12, 2, -0.9f, {0.475f, 0.835f}}, {96, 96, 5, 1, 0.12f, {0.399f}},
    {128, 96, 1, 1, 0.29f, {0.451f}},                  {128, 128, 12, 1, 0.34f, {0.592f}},        {160, 96, 2, 1, 0.53f, {0.507f}},
    {160, 128, 7, 1, 0.79f, {0.594f}},                 {160, 160, 2, 1, 1.39f, {0.686f}},         {192, 160, 7, 1, 1.48f, {0.782f}},
    {192, 192, 6, 1, 2.42f, {0.870f}},                 {256, 128, 4, 1, 1.62f, {0.803f}},         {256, 160, 1, 1, 3.59f, {0.898f}},
    {256, 192, 11, 1, 1.37f, {1.295f}},                {256, 288, 2, 1, 2.63f, {1.704f}},
};

// Time of a product's work items in microseconds, without what every launch costs: whole rounds over the compute units, the
// last one a little shorter for what it leaves idle, and the planes' way to memory and back.
static float tile_time(const TileRate& t, int mode, int M, int N, int K, int planes, int cus) {
  const int cols = mode == 2 ? N / 2 : N, per_tile = mode == 2 ? t.bn / 2 : t.bn;
  const int64_t items = (int64_t)((M + t.bm - 1) / t.bm) * ((cols + per_tile - 1) / per_tile) * planes;
  const int64_t rounds = items / ((int64_t)cus * t.per_unit), rest = items - rounds * cus * t.per_unit;
  const float stages = (float)((K / 64 + planes - 1) / planes);
  float time = (float)rounds * (t.fixed + stages * t.stage[t.per_unit - 1]);
  if (rest > 0) {
    const int share = (int)((rest + cus - 1) / cus);
    time += (t.fixed + stages * t.stage[share - 1]) * (0.79f + 0.21f * ((float)rest / (float)cus - (float)(share - 1)));
  }
  return time + (mode == 3 ? 1.8e-6f * (float)planes * (float)M * (float)N : 0.0f);
}

// The tile and the number of runs of K that take the least time; ``wide_only``: of the wide-tile kernel's. A long K of many rows is
// summed whole by tiles of 192 x 160 and more only: smaller ones have all units ask L2 for more than the 12 TB/s that it gives
// them, which a tile's cost does not know (7B shape's down product and norm, us: 1280 rows 199 by 160 x 128, 173 by 192 x 160 in three runs;
// 2048 rows 236 by 192 x 160, 251 in two runs).
static int tile_choice(int mode, int M, int N, int K, int most_planes, bool wide_only, bool whole, int cus) {
  int best = 0;
  float least = 0.0f;
  for (const TileRate& t : TILE_RATES) {
    if (!(t.modes & (mode == 0 ? 1 : mode == 2 ? 2 : 4)) || (wide_only && t.bm == 64) || !(whole || (t.modes & 8))) continue;
    for (int planes = 1; planes <= most_planes && (planes == 1 || K / planes >= 256); ++planes) {
      if (mode == 3 && planes == 1 && M > 640 && N >= 512 && K >= 3 * N && t.bm + t.bn < 352) continue;
      const float time = tile_time(t, mode, M, N, K, planes, cus);
      if (best == 0 || time < least) {
        least = time;
        best = t.bm | t.bn << 10 | planes << 20;
      }
    }
  }
  return best;
}

// The product by the tile of bm x bn (128 x 128 and 256 x 192 for rows of any length, the others for whole ones: 16-byte
// multiples), if there is such a tile for the mode. (No rule names 128 x 128 for mode 0; whoever asks for it by its size gets it.)
static int w_by_tile(int mode, int bm, int bn, bool whole, const WideArgs& a, int workgroups, hipStream_t stream) {
  const int gate = mode == 2 ? w_gate(a.act) : W_GATE_SILU;
#define CW_WIDE_GATE(MODE_, MB_, NB_, SLOTS_, ANY_, GATE_)                                                 \
  if (mode == MODE_ && gate == GATE_ && bm == 32 * MB_ && bn == 32 * NB_ && (whole || ANY_))               \
  return w_launch<MODE_, MB_, NB_, SLOTS_, ANY_, false, GATE_>(a, 0, workgroups, stream)
#define CW_WIDE(MODE_, MB_, NB_, SLOTS_, ANY_) CW_WIDE_GATE(MODE_, MB_, NB_, SLOTS_, ANY_, W_GATE_SILU)
#define CW_WIDE_GATED(MB_, NB_, SLOTS_, ANY_)               \
  CW_WIDE(2, MB_, NB_, SLOTS_, ANY_);                       \
  CW_WIDE_GATE(2, MB_, NB_, SLOTS_, ANY_, W_GATE_CLIPPED);  \
  CW_WIDE_GATE(2, MB_, NB_, SLOTS_, ANY_, W_GATE_RELU);     \
  CW_WIDE_GATE(2, MB_, NB_, SLOTS_, ANY_, W_GATE_GELU)
  CW_WIDE(0, 3, 3, 6, false);
  CW_WIDE(0, 4, 3, 5, false);
  CW_WIDE(0, 4, 4, 5, true);
  CW_WIDE(0, 5, 4, 4, false);
  CW_WIDE(0, 6, 5, 3, false);
  CW_WIDE(0, 8, 5, 3, false);
  CW_WIDE(0, 8, 6, 2, true);
  CW_WIDE_GATED(4, 4, 5, true);
  CW_WIDE_GATED(5, 3, 5, false);
  CW_WIDE_GATED(5, 4, 4, false);
  CW_WIDE_GATED(5, 5, 4, false);
  CW_WIDE_GATED(6, 5, 3, false);
  CW_WIDE_GATED(6, 6, 3, false);
  CW_WIDE_GATED(8, 6, 2, true);
  CW_WIDE_GATED(8, 9, 2, false);
  CW_WIDE(3, 3, 3, 6, false);
  CW_WIDE(3, 4, 4, 5, true);
  CW_WIDE(3, 5, 4, 4, false);
  CW_WIDE(3, 6, 5, 3, false);
  CW_WIDE(3, 6, 6, 3, false);
  CW_WIDE(3, 8, 4, 3, false);
  CW_WIDE(3, 8, 6, 2, true);
#undef CW_WIDE_GATED
#undef CW_WIDE
#undef CW_WIDE_GATE
  return CW_ERR_ARG;
}

// Rows of C that the tiles without ANY_ROWS take.
static bool w_whole(int mode, const void* C, int64_t ldc, int out_cols) {
  const int granule = mode == 3 ? 4 : 8;
  return !(ldc & (granule - 1)) && !(out_cols & (granule - 1)) && !((uintptr_t)C & 15) && ldc < (1 << 20);
}

// The same product as cw_gemm_bf16_tiled through the wide-tile kernel, for the shapes that
// cw_gemm_bf16_wide_tiles takes. ``workgroups``: how many to launch at most, the number of compute
// units of the GPU (one workgroup fills a unit).
CW_EXPORT int cw_gemm_bf16_wide(int mode, const void* X, int64_t ldx, const void* W, const void* bias, int bias_f32,
                                void* C, int64_t ldc, int M, int N, int K, float act, int workgroups, hipStream_t stream) {
  if (M < 0 || N <= 0 || K <= 0 || (mode != 0 && mode != 2 && mode != 5) || workgroups < 8 || !(act >= 0.0f || mode == 2)) return CW_ERR_ARG;
  if (((uintptr_t)X & 15) || ((uintptr_t)W & 15) || ((uintptr_t)C & 7)) return CW_ERR_ARG;
  if (mode == 2 && ((N & 1) || bias != nullptr)) return CW_ERR_ARG;
  if (ldc < (mode == 2 ? N / 2 : N)) return CW_ERR_ARG;
  if (M == 0) return CW_OK;
  if (cw_gemm_bf16_wide_tiles(mode, M, N, K, ldx) == 0) return CW_ERR_SIZE;
  WideArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, bias, bias_f32, C, ldc, M, N, K, 0, 0, 1};
  a.act = act;
  if (mode == 5) return w_launch<5, 8, 6, 2>(a, 0, workgroups, stream);
  const bool whole = w_whole(mode, C, ldc, mode == 2 ? N / 2 : N);
  const int tile = tile_choice(mode, M, N, K, 1, true, whole, workgroups);
  return w_by_tile(mode, tile & 1023, tile >> 10 & 1023, whole, a, workgroups, stream);
}

// parts[z] = x[:, run z of K] W[:, run z of K]^T for z < k_splits: float32 planes [k_splits, M, N]
// (rows ldc floats apart) whose sum, taken in the order of z, is the product. For the shapes that
// cw_gemm_bf16_wide_partial_ok takes.
CW_EXPORT int cw_gemm_bf16_wide_partial(const void* X, int64_t ldx, const void* W, float* parts, int64_t ldc, int M,
                                        int N, int K, int k_splits, int workgroups, hipStream_t stream) {
  if (M < 0 || N <= 0 || K <= 0 || workgroups < 8 || !parts || ldc < N) return CW_ERR_ARG;
  if (((uintptr_t)X & 15) || ((uintptr_t)W & 15) || ((uintptr_t)parts & 15)) return CW_ERR_ARG;
  if (M == 0) return CW_OK;
  if (!cw_gemm_bf16_wide_partial_ok(M, N, K, ldx, k_splits)) return CW_ERR_SIZE;
  WideArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, nullptr, 0, parts, ldc, M, N, K, 0, 0, k_splits};
  return w_launch<3, 8, 6, 2>(a, 0, workgroups, stream);
}

// Products of row tiles with matrices of their own through the wide-tile kernel: x holds
// ``*n_row_tiles`` (at most ``max_row_tiles``, a number on the device) tiles of 256 rows, and tile t
// multiplies matrix ``tile_group[t]`` of the stack W [groups, N, K] (``w_group_stride`` elements
// apart). mode 0: C[row_target[m]] = x[m] W_g^T (times row_factor[row_target[m]] when given; rows
// whose target is negative are not stored; row_target nullptr: C[m]). mode 2: W_g = [gate; up],
// C[m, i] = silu(gate_i . x_m) * (up_i . x_m). The grid depends on max_row_tiles alone, so a
// captured launch replays with other numbers of tiles. K a multiple of 64, at least 256.
CW_EXPORT int cw_gemm_bf16_wide_grouped(int mode, const void* X, int64_t ldx, const void* W, int64_t w_group_stride,
                                        void* C, int64_t ldc, int N, int K, const int* tile_group, const int* n_row_tiles,
                                        int max_row_tiles, const int* row_target, const float* row_factor, float act, int workgroups,
                                        hipStream_t stream) {
  if (!(act >= 0.0f) || N <= 0 || K <= 0 || (mode != 0 && mode != 2) || workgroups < 8 || max_row_tiles < 0) return CW_ERR_ARG;
  if (!X || !W || !C || !tile_group || !n_row_tiles || (row_factor && !row_target)) return CW_ERR_ARG;
  if (((uintptr_t)X & 15) || ((uintptr_t)W & 15) || ((uintptr_t)C & 7) || (w_group_stride & 7)) return CW_ERR_ARG;
  if (mode == 2 && (N & 1)) return CW_ERR_ARG;
  if (ldc < (mode == 2 ? N / 2 : N) || w_group_stride < (int64_t)N * K) return CW_ERR_ARG;
  if (max_row_tiles == 0) return CW_OK;
  if (cw_gemm_bf16_wide_tiles(mode, max_row_tiles * W_BM, N, K, ldx) == 0) return CW_ERR_SIZE;
  WideArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, nullptr, 0, C, ldc, 0, N, K, 0, 0, 1,
             tile_group, n_row_tiles, row_target, row_factor, w_group_stride, act};
  if (mode == 0) return w_launch<0, 8, 6, 2, true, true>(a, max_row_tiles, workgroups, stream);
  return act == 0.0f ? w_launch<2, 8, 6, 2, true, true>(a, max_row_tiles, workgroups, stream)
                     : w_launch<2, 8, 6, 2, true, true, W_GATE_CLIPPED>(a, max_row_tiles, workgroups, stream);
}

// rows of a tile of cw_gemm_bf16_wide_grouped
CW_EXPORT int cw_gemm_bf16_wide_rows(void) { return W_BM; }

// ------------------------------------------------------------------------------------------------
// Tiles for the steps between (65 to some 1000 rows): the wide tiles leave most compute units without one there,
// and so do the library's (a step of 256 rows of the 1.5B shape: 48 tiles for its down product, on 256 units).
//
// A workgroup of 4 waves owns BM rows of x by BN rows of W (64 or 128 each), a wave a quarter of it. K goes in stages
// of 64 elements straight into LDS, as blocks of 8 rows x 128 bytes (a load instruction each: whole lines, which come
// in a fifth to a third faster than the half lines of stages of 32) through a ring of three. The eight granules of a
// row change places by (row >> 1) & 7, so that the 16 lanes that read one granule of 16 rows touch every bank once.
// Workgroups are dealt to the 8 XCDs in turn; an XCD takes a run of neighbouring tiles, the row tiles of one W tile next
// to each other, so that W comes from memory once, into one L2.
// A product whose tiles leave compute units idle is cut over K (MODE 3): run z of every tile is a work item of its own
// and writes plane z of the partial sums, which the next norm kernel adds in their order.
// Bound by the loads into LDS, about 50 GB/s into each compute unit (deeper rings do not help): a tile's time goes
// with (BM + BN) K, which is what cw_gemm_bf16_mid_choice weighs.
// Measured on an MI355X with the norm behind it, library -> here (us): down product of the 0.5B shape 14.5 -> 11.7 for 144
// rows, 25.0 -> 18.0 for 640; of the 1.5B shape 28.1 -> 20.5 for 144, 35.8 -> 23.3 for 256, 44.0 -> 34.7 for 640; of the 7B
// shape 165 -> 52 for 144. Gate/up product and gate of the 0.5B shape 16.5 -> 10.9 for 144 rows; of the 1.5B shape
// 29.4 -> 26.3 for 144, and from 200 rows on the library's larger tiles, which read less, win.
#define MID_SLOTS 3
#define MID_MAX_PLANES 12

template <int MODE, int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_mid_bf16_kernel(WideArgs a) {
  extern __shared__ __align__(1024) unsigned char w_smem[];
  constexpr int XB = BM / 8, WB = BN / 8, LOADS = (XB + WB) / 4, STAGE = (XB + WB) * W_BLOCK;
  constexpr int TM = BM / 32, TN = BN / 32;  // 16 x 16 tiles of a wave
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int c = lane & 15, s = lane >> 4;
  const int M = a.M, N = a.N, K = a.K, I = N / 2;
  const int run = gridDim.x >> 3, rest = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int tile = xcd * run + min(xcd, rest) + (blockIdx.x >> 3);
  const int tm = tile % a.tiles_m, tn = tile / a.tiles_m % a.tiles_n, plane = tile / (a.tiles_m * a.tiles_n);
  constexpr bool PAIRS = MODE == 2 || MODE == 6;  // two rows of W a column
  const int m0 = tm * BM, w0 = tn * (PAIRS ? BN / 2 : BN);
  const int stages = K / 64;
  const int first = MODE == 3 ? (int)((int64_t)stages * plane / a.k_splits) : 0;
  const int last = (MODE == 3 ? (int)((int64_t)stages * (plane + 1) / a.k_splits) : stages) - 1;

  __amdgpu_buffer_rsrc_t xr, wr;
  xr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.X + (int64_t)m0 * a.ldx), 0,
                                         (int)(uint32_t)(((int64_t)(M - m0 - 1) * a.ldx + K) * 2), 0x00020000);
  const int w_from = MODE == 6 ? 0 : w0;
  wr = __builtin_amdgcn_make_buffer_rsrc((void*)(a.W + (int64_t)w_from * K), 0,
                                         (int)(uint32_t)((int64_t)(N - w_from) * K * 2), 0x00020000);
  // load i of a wave: block wave * LOADS + i of a stage, the x blocks first. (Of a size that hangs on no template
  // parameter, so that the host pass takes the loads below.)
  uint32_t at[8];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int block = wave * LOADS + i;
    int64_t from;
    if (block < XB) {
      from = (int64_t)(block * 8 + (lane >> 3)) * a.ldx;
    } else {
      const int rb = (block - XB) * 8 + (lane >> 3);
      if (PAIRS) {  // a wave's rows are gate rows followed by the up rows with the same indices (MODE 6: first and second halves)
        const int q = rb % (BN / 2), i2 = rb / (BN / 2) * (BN / 4) + q % (BN / 4);
        if (MODE == 6) from = min(pair_row(w0 + i2, a.hd) + (q < BN / 4 ? 0 : a.hd / 2), (int64_t)N) * K;
        else
        from = (int64_t)(q < BN / 4 ? i2 : I + i2) * K;
      } else {
        from = (int64_t)rb * K;
      }
    }
    at[i] = (uint32_t)((from + ((lane & 7) ^ ((block * 4 + (lane >> 4)) & 7)) * 8) * 2);
  }
  auto fetch = [&](int stage, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int block = wave * LOADS + i;
      unsigned char* to = w_smem + (slot * STAGE + block * W_BLOCK);
      if (block < XB) __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void_t*)to, 16, at[i], stage * 128, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void_t*)to, 16, at[i], stage * 128, 0, 0);
    }
  };
  f32x4_t acc[TM][TN];
#pragma unroll
  for (int mi = 0; mi < TM; ++mi)
#pragma unroll
    for (int ni = 0; ni < TN; ++ni) acc[mi][ni] = (f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
  // MODE 6: what the rotation and the stores need, asked for ahead of the tiles (asked for at the end, its trips to memory are 2 us)
  constexpr int PAIR_BLOCKS = MODE == 6 ? TN / 2 : 1;
  float4 cosines[TM][PAIR_BLOCKS], sines[TM][PAIR_BLOCKS];
  float bias_first[PAIR_BLOCKS][4], bias_second[PAIR_BLOCKS][4];
  int slot_of[TM];
  if constexpr (MODE == 6) {
#pragma unroll
    for (int ni = 0; ni < PAIR_BLOCKS; ++ni) {
      const int pair = min(w0 + wn * (BN / 4) + ni * 16, I - 16), head = pair / (a.hd / 2), d = pair - head * (a.hd / 2) + 4 * s;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t at_first = (int64_t)head * a.hd + d + e, at_second = at_first + a.hd / 2;
        bias_first[ni][e] = a.bias == nullptr ? 0.0f : a.bias_f32 ? ((const float*)a.bias)[at_first] : __bfloat162float(((const bf16_t*)a.bias)[at_first]);
        bias_second[ni][e] = a.bias == nullptr ? 0.0f : a.bias_f32 ? ((const float*)a.bias)[at_second] : __bfloat162float(((const bf16_t*)a.bias)[at_second]);
      }
#pragma unroll
      for (int mi = 0; mi < TM; ++mi) {
        const int64_t m = min(m0 + (wm * TM + mi) * 16 + c, M - 1);
        if (ni == 0) slot_of[mi] = a.slots[m];
        cosines[mi][ni] = make_float4(1.0f, 1.0f, 1.0f, 1.0f), sines[mi][ni] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (head < a.nh + a.nkv) {
          cosines[mi][ni] = *reinterpret_cast<const float4*>(a.angles + m * a.hd + d);
          sines[mi][ni] = *reinterpret_cast<const float4*>(a.angles + m * a.hd + a.hd / 2 + d);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MID_SLOTS - 1; ++i) fetch(min(first + i, last), i);
  int slot = 0;
  for (int t = first; t <= last; ++t) {
    // this wave's loads of the stage are in; behind the barrier every wave's are, and every wave has read the stage
    // before it, whose slot the next loads take (past the last stage it is asked for again, and nobody reads it:
    // the number of loads in flight stays what the wait counts on)
    W_WAIT_LOADS((MID_SLOTS - 2) * LOADS);
    W_BARRIER();
    fetch(min(t + MID_SLOTS - 1, last), (slot + MID_SLOTS - 1) % MID_SLOTS);
    const unsigned char* base = w_smem + slot * STAGE + c * 128;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int g = ((kk * 4 + s) ^ ((c >> 1) & 7)) * 16;
      bf16x8_t xf[TM], wf[TN];
#pragma unroll
      for (int ni = 0; ni < TN; ++ni) wf[ni] = *reinterpret_cast<const bf16x8_t*>(base + (XB * 1024 + (wn * TN + ni) * 2048) + g);
#pragma unroll
      for (int mi = 0; mi < TM; ++mi) xf[mi] = *reinterpret_cast<const bf16x8_t*>(base + (wm * TM + mi) * 2048 + g);
#pragma unroll
      for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int ni = 0; ni < TN; ++ni) acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ni], xf[mi], acc[mi][ni], 0, 0, 0);
    }
    slot = (slot + 1) % MID_SLOTS;
  }
  W_WAIT_LOADS(0);  // no load may reach LDS after the workgroup has gone

  // lane (c, s) holds columns 4 s .. 4 s + 3 of W block ni for row c of x block mi
  const int out_cols = PAIRS ? I : N;
#pragma unroll
  for (int mi = 0; mi < TM; ++mi) {
    const int m = m0 + (wm * TM + mi) * 16 + c;
    if (m >= M) continue;
    if constexpr (MODE == 6) {
#pragma unroll
      for (int ni = 0; ni < TN / 2; ++ni) {
        const int pair = w0 + wn * (BN / 4) + ni * 16, head = pair / (a.hd / 2), d = pair - head * (a.hd / 2) + 4 * s;  // 16 pairs of one head
        bf16_t* to = pair < I ? pair_target(a, m, head, slot_of[mi]) : nullptr;
        if (to == nullptr) continue;
        const f32x4_t first4 = acc[mi][ni], second4 = acc[mi][ni + TN / 2];
        const float co[4] = {cosines[mi][ni].x, cosines[mi][ni].y, cosines[mi][ni].z, cosines[mi][ni].w};
        const float si[4] = {sines[mi][ni].x, sines[mi][ni].y, sines[mi][ni].z, sines[mi][ni].w};
        float x[4], y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float f = first4[e] + bias_first[ni][e], g = second4[e] + bias_second[ni][e];
          const bool rotated = head < a.nh + a.nkv;   // (values pass as they are, infinities among them)
          x[e] = rotated ? f * co[e] - g * si[e] : f;
          y[e] = rotated ? g * co[e] + f * si[e] : g;
        }
        *reinterpret_cast<uint2*>(to + d) = make_uint2(w_pack_bf16(x[0], x[1]), w_pack_bf16(x[2], x[3]));
        *reinterpret_cast<uint2*>(to + a.hd / 2 + d) = make_uint2(w_pack_bf16(y[0], y[1]), w_pack_bf16(y[2], y[3]));
      }
      continue;
    }
#pragma unroll
    for (int ni = 0; ni < (MODE == 2 ? TN / 2 : TN); ++ni) {
      const int n = w0 + (MODE == 2 ? wn * (BN / 4) : wn * (BN / 2)) + ni * 16 + 4 * s;
      if (n >= out_cols) continue;
      f32x4_t v = acc[mi][ni];
      if (MODE == 3) {
        float* dst = (float*)a.C + ((int64_t)plane * M + m) * a.ldc + n;
        if (n + 4 <= N && !(a.ldc & 3)) {
          *reinterpret_cast<f32x4_t*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) dst[e] = v[e];
        }
        continue;
      }
      if (MODE == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = cw_gated(v[e], acc[mi][ni + (MODE == 2 ? TN / 2 : 0)][e], a.act);
      } else if (a.bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) v[e] += a.bias_f32 ? ((const float*)a.bias)[n + e] : __bfloat162float(((const bf16_t*)a.bias)[n + e]);
      }
      bf16_t* dst = (bf16_t*)a.C + (int64_t)m * a.ldc + n;
      const uint32_t lo = w_pack_bf16(v[0], v[1]), hi = w_pack_bf16(v[2], v[3]);
      if (n + 4 <= out_cols && !(a.ldc & 3)) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
      } else {
        const uint32_t w2[2] = {lo, hi};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < out_cols) ((uint16_t*)dst)[e] = (uint16_t)(w2[e >> 1] >> ((e & 1) * 16));
      }
    }
  }
}

template <int MODE, int BM, int BN>
static int mid_launch(WideArgs a, hipStream_t stream) {
  constexpr int SMEM = MID_SLOTS * (BM + BN) / 8 * W_BLOCK;
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_mid_bf16_kernel<MODE, BM, BN>, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM) != hipSuccess)
      return CW_ERR_LAUNCH;
    raised = true;
  }
  const int out_cols = MODE == 2 || MODE == 6 ? a.N / 2 : a.N;
  const int per_tile = MODE == 2 || MODE == 6 ? BN / 2 : BN;
  a.tiles_n = (out_cols + per_tile - 1) / per_tile;
  a.tiles_m = (a.M + BM - 1) / BM;
  const int64_t total = (int64_t)a.tiles_m * a.tiles_n * (MODE == 3 ? a.k_splits : 1);
  if (total > 0x7fffffff) return CW_ERR_SIZE;
  hipLaunchKernelGGL((gemm_mid_bf16_kernel<MODE, BM, BN>), dim3((unsigned)total), dim3(256), SMEM, stream, a);
  return cw_launch_status();
}

// y = x W^T through the tiles between. mode 0: bfloat16 [M, N], + bias [N] when given; 2: W = [gate; up], the gated
// product bfloat16 [M, N / 2] (``act`` as elsewhere); 3: float32 planes [k_splits, M, N] of partial sums over runs of K.
// bm, bn: 64 x 64, 64 x 128, 128 x 64, or a tile of the wide-tile kernel's (w_by_tile). K a multiple of 64 (of at least 64 elements a run), both matrices below 4 GiB.
CW_EXPORT int cw_gemm_bf16_mid(int mode, const void* X, int64_t ldx, const void* W, const void* bias, int bias_f32, void* C,
                               int64_t ldc, int M, int N, int K, float act, int k_splits, int bm, int bn, int workgroups, hipStream_t stream) {
  if (M < 0 || workgroups < 8 || N <= 0 || K <= 0 || (mode != 0 && mode != 2 && mode != 3) || !(act >= 0.0f || mode == 2)) return CW_ERR_ARG;
  if (((uintptr_t)X & 15) || ((uintptr_t)W & 15) || ((uintptr_t)C & (mode == 3 ? 15 : 7)) || !C) return CW_ERR_ARG;
  if ((mode == 2 && (N & 1)) || (mode != 0 && bias != nullptr)) return CW_ERR_ARG;
  if ((K & 63) || (ldx & 7) || ldx < K || ldc < (mode == 2 ? N / 2 : N)) return CW_ERR_ARG;
  if (mode == 3 ? (k_splits < 1 || k_splits > MID_MAX_PLANES || K / 64 < k_splits) : k_splits != 1) return CW_ERR_ARG;
  if ((int64_t)N * K * 2 >= (1ll << 32) || ((int64_t)M * ldx + 128 * ldx) * 2 >= (1ll << 32)) return CW_ERR_SIZE;
  if (M == 0) return CW_OK;
  WideArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, bias, bias_f32, C, ldc, M, N, K, 0, 0, k_splits};
  a.act = act;
#define CW_MID(BM_, BN_)                                                                                                        \
  if (bm == BM_ && bn == BN_)                                                                                                   \
    return mode == 0 ? mid_launch<0, BM_, BN_>(a, stream) : mode == 2 ? mid_launch<2, BM_, BN_>(a, stream) : mid_launch<3, BM_, BN_>(a, stream)
  CW_MID(64, 64);
  CW_MID(64, 128);
  CW_MID(128, 64);
#undef CW_MID
  return w_by_tile(mode, bm, bn, w_whole(mode, C, ldc, mode == 2 ? N / 2 : N), a, workgroups, stream);
}

// Which of this file's kernels a product of many rows should run on: 0 the library's, else bm | bn << 10 |
// planes << 20 (cw_gemm_bf16_mid; mode as there), by the table of tiles above. For results in rows of 16-byte multiples; for
// others, of which nothing is named here, cw_gemm_bf16_mid_choice is there.
// Where the lines lie, measured with operands from memory, 72 to 2048 rows (us, library -> here):
//  * mode 3 (a sum that the next norm adds up; times with that norm): K of two and a half times N and more, everywhere (1.5B
//    shape's down product, 72 rows 25.3 -> 15.3, 336 rows 40.3 -> 23.6, 1000 rows 55.8 -> 41.7, 2048 rows 83.3 -> 68.0; 7B
//    shape, 512 rows 204 -> 78, 2048 rows 385 -> 265) until M N is 8 M (14B shape, 1500 rows 223 -> 201, 2048 rows 267 -> 304),
//    2.1 M for outputs of more than 5120 columns (72B shape, 256 rows 293 -> 177, 640 rows 302 -> 370). A squarer matrix
//    while M N is below 1.2 M, 1.03 M for more than 1536 columns (2048 x 2048, 500 rows 17.5 -> 16.9, 522 rows 18.8 ->
//    20.2), and N at most 5120: beyond, mode 0 and a norm of its bfloat16 result are faster (1536 x 1536, 1000 rows 17.7,
//    11.2 and 4.6).
//  * mode 2: every shape measured up to the 7B one (72 rows of the 0.5B shape 15.1 -> 10.5, of the 1.5B shape 28.5 -> 20.1, of
//    the 7B shape 74.6 -> 53.0; 640 rows 27.1 -> 16.3, 51.0 -> 44.0, 194 -> 177). The 14B shape's 141 M elements: 128 rows 72 ->
//    66, 256 rows 100 -> 105, 384 rows 116 -> 125. A K of more than 1024 and half of N is a narrow output's (896 x 4864, 165 rows
//    15.0 -> 20.6).
//  * mode 0: a long K is summed faster by the library in parts (512 x 2048, 160 rows 8.4 -> 9.9), so K up to 512, up to 896
//    for 896 columns and more (q/k/v of the 0.5B shape 7.9 -> 6.1 for 160 rows, 11.0 -> 9.4 for 2048; 512 columns 5.3 -> 6.1); up to 1536
//    for 1536 columns and more from 0.5 M outputs on (q/k/v of the 1.5B shape, 160 rows 8.1 -> 8.4, 336 rows 9.4 -> 8.7, 2048 rows 18.3
//    -> 17.8; its output product, 2048 rows 17.4 -> 14.3; 4640 columns, 100 rows 11.6 -> 11.7, 128 rows 16.8 -> 12.0, 2048 rows 38.5 -> 31.6); up to
//    4096 for 2048 columns and more from 1.6 M on (4608 x 3584, 512 rows 34.4 -> 27.7, 1000 rows 47.0 -> 37.4; 3584 x 3584, 384 rows 23.1 -> 27.9),
//    with a K of more than 2048 up to 9.5 M (6144 x 3072, 1500 rows 59.3 -> 49.6, 1600 rows 53.1 -> 70.3, 2048 rows 62.8 -> 65.6; 5120 x 2048, 2048 rows 42.2 -> 36.9).
//    Beyond 8192 columns, and for the few outputs of 320 rows and more with a K of 1536 that are no 0.5 M, the 64 x 64 tiles by
//    their own lines (whole_sums_in_small_tiles): 8704 x 512, 72 rows 8.0 -> 5.9, 400 rows 12.4 -> 10.9; 16384 x 512, 160 rows 12.5 -> 10.8;
//    9728 x 896, 72 rows 11.9 -> 9.8, 160 rows 13.1 -> 11.1; 1536 x 1536, 325 rows 8.9 -> 8.3. From 512 tiles on with a K of more than
//    512 they lose as often as they win (9728 x 896, 256 rows 15.5 -> 16.3, 12288 x 896, 160 rows 13.3 -> 15.4; 9728 x 640, 256 rows
//    15.0 -> 13.3, 320 rows 14.3 -> 13.1); which, the number of tiles does not tell.
static int whole_sums_in_small_tiles(int M, int N, int K);
CW_EXPORT int cw_gemm_bf16_wide_choice(int mode, int M, int N, int K, int64_t ldx, int cus) {
  if (M <= 64 || M > 2048 || N <= 0 || K < 256 || (K & 63) || (ldx & 7) || ldx < K || cus < 8) return 0;
  if ((int64_t)N * K * 2 >= (1ll << 32) || ((int64_t)M * ldx + 128 * ldx) * 2 >= (1ll << 32)) return 0;
  if (N & (mode == 2 ? 15 : mode == 3 ? 3 : 7)) return 0;
  const int64_t elements = (int64_t)N * K, outputs = (int64_t)M * N;
  if (mode == 0) {
    const bool here = K <= 512 ? N >= 32 : K <= 896 ? N >= 896 : K <= 1536 ? N >= 1536 && outputs >= 500000 : K <= 4096 && N >= 2048 && outputs >= 1600000 && (K <= 2048 || outputs <= 9500000);
    if (!here || N > 8192) return whole_sums_in_small_tiles(M, N, K);
  } else if (mode == 2) {
    if ((N & 1) || (N < 2 * K && K > 1024) || elements > 136000000) return 0;
  } else if (mode == 3) {
    const int64_t most = 2 * (int64_t)K >= 5 * (int64_t)N ? (N <= 5120 ? 8000000 : 2100000) : N <= 1536 ? 1200000 : N <= 5120 ? 1030000 : 0;
    if (outputs > most) return 0;
  } else {
    return 0;
  }
  return tile_choice(mode, M, N, K, mode == 3 ? MID_MAX_PLANES : 1, false, true, cus);
}

// Time of a product's work items in microseconds as the choice below weighs them, without what every launch costs:
// rounds over the compute units, a stage of 64 elements of K taking what its loads take, and the planes' way to
// memory and back. The constants are fits (64 x 64 and 64 x 128 tiles share a compute unit with others, which covers
// for a part of their last round): over 72 to 1024 rows of eight shapes what they name takes 1.0 % more than the fastest
// tiles and counts do (2.9 % with 0.62 and 1.04 us a stage of the two largest: 700 rows of the 3B shape's down product
// went to 64 x 128 tiles, 67.7 us, where 128 x 128 ones take 59.7).
static float mid_time(int M, int N, int K, int bm, int bn, int planes, int cus) {
  const float stage = bm + bn == 128 ? 0.27f : bm + bn == 192 ? 0.38f : bm == 128 ? 0.55f : 0.9f;
  const int64_t items = (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * planes;
  const int64_t rounds = (items + cus - 1) / cus;
  const float share = rounds > 1 && bm + bn < 256 ? 0.95f : 1.0f;
  const int stages = (K / 64 + planes - 1) / planes;
  return share * (float)(rounds * stages) * stage + (planes > 1 ? 2.2e-6f * (float)planes * (float)M * (float)N : 0.0f);
}

// Which tiles a product of many rows should run on whose rows of results are no multiples of 16 bytes: 0 the library's, else
// bm | bn << 10 | planes << 20 (cw_gemm_bf16_mid). mode as there.
// Where the lines lie, measured with operands from memory, 72 to 2048 rows, for the layers of the 0.5B to 72B shapes
// and for outputs of 16 to 4096 columns with K of 256 to 16384 (us, library -> here):
//  * mode 3 (a sum that the next norm adds up): K of three times N and more. The library's product of that kind leaves
//    units idle (32B shape's down product, 256 rows 275 -> 116, 1536 rows 565 -> 384) until M N is large: 8 M (2048 rows
//    of the 32B shape 484 -> 513), 2.1 M for outputs of more than 5120 columns (72B shape, 256 rows 293 -> 177, 640 rows
//    302 -> 370). Beyond 1024 rows and columns on the wide tiles only (3B shape's down product, 1434 rows 98 -> 115 on
//    the small ones), which have to fill their rounds (7B shape, 1600 rows in 2.08 rounds 241 -> 273, 2048 in 2.4 386 ->
//    292; 3B shape, 1356 rows in 0.52 90 -> 103, 1600 in 0.6 112 -> 100); beyond 640 rows not as whole sums of K (2048 x
//    6144, 1000 rows 49.4 -> 54.5; as 2 planes on 128 x 128 tiles 43.6). A squarer matrix
//    while M N is below 1.2 M, 1.03 M for more than 1536 columns (2048 x 2048, 500 rows 17.5 -> 16.9, 522 rows 18.8 ->
//    20.2), and N at most 5120: beyond, the planes cost more than the library's idle units.
//  * mode 2: M N K up to 4.5e9 (72 rows of the 1.5B shape: 28.0 -> 22.9 us, 208 rows 32.2 -> 31.8), and up to 640 rows for
//    a matrix of at most 9 M elements; a K of more than 1024 and half of N is a narrow output's (896 x 4864, 165 rows
//    15.0 -> 20.6).
//  * mode 0 (whole sums of K on 64 x 64 tiles, 0.21 us a stage): a long K is summed faster by the library in parts (64 x
//    4096, 144 rows 11.6 -> 16.8), so K up to 512, up to 896 for 1024 columns and more (q/k/v of the 0.5B shape 8.0 ->
//    6.4 for 144 rows; 512 columns 5.3 -> 6.1), while a compute unit has three tiles or so (4096 x 896, 400 rows 10.6 ->
//    8.4, 700 rows 11.3 -> 12.1); and K up to 1536 for 1536 columns and more, 320 to 1024 rows (q/k/v of the 1.5B shape
//    14.0 -> 12.7 for 1000, 8.6 -> 8.8 for 144).
static int whole_sums_in_small_tiles(int M, int N, int K) {
  const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
  const bool short_k = M <= 1536 && N >= 32 && (K <= 512 || (K <= 896 && N >= 1024)) && tiles <= 1000 && tiles * K <= 600000;
  const bool qkv = K > 896 && K <= 1536 && N >= 1536 && (int64_t)N * K <= 4 << 20 && M >= 320 && M <= 1024;
  return short_k || qkv ? 64 | 64 << 10 | 1 << 20 : 0;
}

CW_EXPORT int cw_gemm_bf16_mid_choice(int mode, int M, int N, int K, int64_t ldx, int cus) {
  if (M <= 64 || M > 2048 || N <= 0 || K < 256 || (K & 63) || (ldx & 7) || ldx < K || cus < 8) return 0;
  if ((int64_t)N * K * 2 >= (1ll << 32) || ((int64_t)M * ldx + 128 * ldx) * 2 >= (1ll << 32)) return 0;
  const int64_t elements = (int64_t)N * K, outputs = (int64_t)M * N;
  if (mode == 0) return whole_sums_in_small_tiles(M, N, K);
  if (mode == 2) {
    if ((N & 1) || (N < 2 * K && K > 1024) || !((int64_t)M * elements <= 4500000000ll || (elements <= 9 << 20 && M <= 640))) return 0;
  } else if (mode == 3) {
    const int64_t most = K >= 3 * N ? (N <= 5120 ? 8000000 : 2100000) : N <= 1536 ? 1200000 : N <= 5120 ? 1030000 : 0;
    if (outputs > most) return 0;
  } else {
    return 0;
  }
  int best = 0;
  float least = 0.0f;
  for (int bm = 64; bm <= 128; bm += 64)
    for (int bn = 64; bn <= 128; bn += 64)
      for (int planes = 1; planes <= (mode == 3 ? MID_MAX_PLANES : 1) && K / planes >= 256; ++planes) {
        const float t = mid_time(M, N, K, bm, bn, planes, cus);
        if (best == 0 || t < least) {
          least = t;
          best = bm | bn << 10 | planes << 20;
        }
      }
  if (mode == 3 && M >= 512)
    for (int planes = 2; planes <= 8; ++planes)
      if (cw_gemm_bf16_wide_partial_ok(M, N, K, ldx, planes) && mid_time(M, N, K, W_BM, W_BN, planes, cus) < least) {
        least = mid_time(M, N, K, W_BM, W_BN, planes, cus);
        best = W_BM | W_BN << 10 | planes << 20;
      }
  if (mode == 3) {
    const int planes = best >> 20;
    if (planes == 1 && M > 640 && N >= 512 && K >= 3 * N) return 0;
    if ((best & 1023) != W_BM) return M > 1024 && N >= 1024 ? 0 : best;
    const int64_t items = (int64_t)((M + W_BM - 1) / W_BM) * ((N + W_BN - 1) / W_BN) * planes;
    if ((float)items < (items > cus ? 0.72f : M > 1024 ? 0.55f : 0.0f) * (float)(cus * ((items + cus - 1) / cus))) return 0;
  }
  return best;
}

// Does the product of the queries, keys and values of M tokens run with bias, rotation and cache write inside (cw_gemm_bf16_pairs)?
// In 64 x 64 tiles, where they are the ones for the product or nearly so: up to 576 of them and K of 2048. Where the lines lie (us, in a
// graph, operands from memory, the fastest product and the rotation kernel behind it -> here): 0.5B shape, 160 rows 9.5 -> 7.8, 1000 rows
// 12.1 -> 10.1, 2048 rows (576 tiles) 15.4 -> 14.5; 1.5B shape, 72 rows 10.9 -> 9.8, 336 rows 12.5 -> 10.4, 1000 rows (512) 16.2 -> 14.8, 1500
// rows (768) 21.4 -> 21.7; 3B shape (K 2048), 72 rows 12.4 -> 13.2, 160 rows 14.5 -> 12.5, 768 rows (480) 19.3 -> 17.9, 1000 rows (640)
// 21.4 -> 23.1; 7B shape (K 3584), 336 rows 29.7 -> 32.3. In tiles of 128 x 128 the rotation's end costs more than its kernel.
CW_EXPORT int cw_gemm_bf16_pairs_ok(int M, int N, int K, int64_t ldx, int hd) {
  if (M <= 64 || N <= 0 || K < 256 || (K & 63) || (ldx & 7) || ldx < K) return 0;
  if ((hd & 31) || hd < 32 || hd > 256 || N % hd || K > 2048 || (K > 1536 && M < 128)) return 0;
  return (int64_t)((M + 63) / 64) * ((N + 63) / 64) <= 576 ? 1 : 0;
}

// Rows of x W^T (+ bias) as heads of hd elements, nh of queries, then nkv of keys and nkv of values, queries and keys rotated by
// ``angles`` [M, 2, hd / 2] (cw_rope_angles): queries to Q [M, nh hd], keys and values to rows ``slots`` of the caches (negative
// or beyond cache_rows: nowhere). Heads of a multiple of 32 elements up to 256.
CW_EXPORT int cw_gemm_bf16_pairs(const void* X, int64_t ldx, const void* W, const void* bias, int bias_f32, const float* angles, const int* slots,
                                 void* Q, void* k_cache, void* v_cache, int64_t cache_rows, int M, int K, int nh, int nkv, int hd, hipStream_t stream) {
  if (M < 0 || K <= 0 || nh <= 0 || nkv <= 0 || hd <= 0 || cache_rows < 0) return CW_ERR_ARG;
  if (!X || !W || !angles || !slots || !Q || !k_cache || !v_cache) return CW_ERR_ARG;
  if (((uintptr_t)X & 15) || ((uintptr_t)W & 15) || ((uintptr_t)Q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15) || ((uintptr_t)angles & 15))
    return CW_ERR_ARG;
  const int64_t n = ((int64_t)nh + 2 * (int64_t)nkv) * hd;
  if (n > 0x7fffffff || (hd & 31) || hd > 256 || (K & 63) || (ldx & 7) || ldx < K) return CW_ERR_ARG;
  const int N = (int)n;
  if ((int64_t)N * K * 2 >= (1ll << 32) || ((int64_t)M * ldx + 256 * ldx) * 2 >= (1ll << 32)) return CW_ERR_SIZE;
  if (M == 0) return CW_OK;
  WideArgs a{(const bf16_t*)X, ldx, (const bf16_t*)W, bias, bias_f32, Q, (int64_t)nh * hd, M, N, K, 0, 0, 1};
  a.angles = angles;
  a.slots = slots;
  a.k_cache = (bf16_t*)k_cache;
  a.v_cache = (bf16_t*)v_cache;
  a.cache_rows = cache_rows;
  a.nh = nh;
  a.nkv = nkv;
  a.hd = hd;
  return mid_launch<6, 64, 64>(a, stream);
}
