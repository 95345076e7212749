// A linear recurrence with a matrix state per head and a decay per key channel, for gfx950:
//   S_t = diag(a_t) S_(t-1) + k_t v_t^T,   o_t = S_t^T (q_scale * q_t),   S in float32 [dim, vdim],
// with the decay made inside from a low-rank projection: a_t = sigmoid(z_t)^(1/tau),
// z_t = A2 u_t + b (u_t the token's ``rank`` inputs). o_t is optionally RMS-normed over vdim
// with a weight shared by the heads and multiplied by silu(g_t).
//
// Variants (LinRecForm), for a recurrence of another family:
//   decay_kind 1:  a_t = exp(-exp(z_t)) with z_t = A2 u_t + b;  2: the same with z_t = A2 tanh(u_t) + b.
//   bonus [heads, dim]:  the output reads the state BEFORE the token joins it, and the token itself
//                  through the bonus:  o_t = (S_(t-1) + diag(bonus) k_t v_t^T)^T q_t,  then
//                  S_t = diag(a_t) S_(t-1) + k_t v_t^T.
//   norm_w_stride: vdim when every head has norm weights of its own ([heads, vdim]), else 0.
//   u, u_stride:   the decay input as rows of a tensor of its own (else columns of proj).
// q, k, v and the gate may also lie in planes one behind the other, [4][T, heads * dim]: then
// stride is the plane's row and an offset a multiple of the plane's size.
//
// A workgroup owns one (request, head): the state lives in registers for the whole portion (a
// thread holds a run of rows of one column), tokens are walked in order, sixteen at a time: their
// q, k, v and decays are staged in LDS, the walk itself has no barrier, the outputs' partial sums
// over the row runs are added, normed and gated once per sixteen tokens. Decays, their logarithms,
// the state and the norm are float32 whatever the activation type T is.
#include "recurrence.h"

template <typename T, int RPT>
__global__ __launch_bounds__(256) void linear_recurrence_kernel(LinRecParams p, LinRecForm f) {
  extern __shared__ __align__(16) float smem[];
  const int D = p.dim, V = p.vdim, Hn = p.heads;
  const int r = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int row0 = p.cu_q[r], q_len = p.cu_q[r + 1] - row0;
  const int slot = p.state_slots[r];
  if (q_len <= 0 || slot < 0 || slot >= p.n_slots) return;
  const int DS = min(256 / V, D);            // row runs: threads that share a column
  const int v = tid % V, s = tid / V;
  const bool active = s < DS;
  const int d0 = s * RPT;                    // this thread's rows d0 .. d0 + RPT - 1 (those below D)

  float* qs = smem;                 // [TC][D]
  float* ks = qs + LR_TC * D;       // [TC][D]
  float* as = ks + LR_TC * D;       // [TC][D] decays
  float* vs = as + LR_TC * D;       // [TC][V]
  float* part = vs + LR_TC * V;     // [TC][DS][V]

  float S[RPT];
  float* st = p.state + (int64_t)slot * f.state_stride + ((int64_t)h * D) * V;
  float bonus[RPT];
#pragma unroll
  for (int rr = 0; rr < RPT; ++rr) {
    S[rr] = (active && d0 + rr < D) ? st[(int64_t)(d0 + rr) * V + v] : 0.0f;
    bonus[rr] = (f.bonus && active && d0 + rr < D) ? f.bonus[h * D + d0 + rr] : 0.0f;
  }

  const T* proj = (const T*)p.proj;
  const T* a2 = (const T*)p.a2;
  T* out = (T*)p.out;
  for (int t0 = 0; t0 < q_len; t0 += LR_TC) {
    const int nt = min(LR_TC, q_len - t0);
    __syncthreads();
    for (int idx = tid; idx < nt * D; idx += 256) {
      const int t = idx / D, d = idx - t * D;
      const T* row = proj + (int64_t)(row0 + t0 + t) * p.stride;
      qs[idx] = cw_to_float(row[p.q_off + h * D + d]) * p.q_scale;
      ks[idx] = cw_to_float(row[p.k_off + h * D + d]);
      float z = p.a2b ? p.a2b[h * D + d] : 0.0f;
      const T* w = a2 + (int64_t)(h * D + d) * p.rank;
      const T* u = f.u ? (const T*)f.u + (int64_t)(row0 + t0 + t) * f.u_stride : row + p.u_off;
      if (f.decay_kind == 2) {
        for (int c = 0; c < p.rank; ++c) z += cw_to_float(w[c]) * tanhf(cw_to_float(u[c]));
      } else {
        for (int c = 0; c < p.rank; ++c) z += cw_to_float(w[c]) * cw_to_float(u[c]);
      }
      as[idx] = lr_decay(z, f.decay_kind, p.inv_tau);
    }
    for (int idx = tid; idx < nt * V; idx += 256) {
      const int t = idx / V, c = idx - t * V;
      vs[idx] = cw_to_float(proj[(int64_t)(row0 + t0 + t) * p.stride + p.v_off + h * V + c]);
    }
    __syncthreads();
    if (active) {
      for (int t = 0; t < nt; ++t) {
        const float vv = vs[t * V + v];
        float po = 0.0f;
#pragma unroll
        for (int rr = 0; rr < RPT; ++rr) {
          const int d = d0 + rr;
          if (d < D) {
            const float kv = ks[t * D + d] * vv;
            if (f.bonus) po += qs[t * D + d] * (S[rr] + bonus[rr] * kv);
            S[rr] = as[t * D + d] * S[rr] + kv;
            if (!f.bonus) po += qs[t * D + d] * S[rr];
          }
        }
        part[(t * DS + s) * V + v] = po;
      }
    }
    __syncthreads();
    // a wave per token: sum the partial outputs, norm over vdim, gate, store
    const int wave = tid >> 6, lane = tid & 63;
    for (int t = wave; t < nt; t += 4) {
      float o[4];  // vdim <= 256
      float ss = 0.0f;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = lane + u * 64;
        float sum = 0.0f;
        if (c < V)
          for (int q = 0; q < DS; ++q) sum += part[(t * DS + q) * V + c];
        o[u] = sum;
        ss += sum * sum;
      }
      float inv = 1.0f;
      if (p.norm_w) inv = 1.0f / sqrtf(cw_wave_sum(ss) / (float)V + p.eps);
      const int64_t trow = row0 + t0 + t;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = lane + u * 64;
        if (c < V) {
          float val = o[u] * inv;
          if (p.norm_w) val *= p.norm_w[h * f.norm_w_stride + c];
          if (p.g_off >= 0) {
            const float g = cw_to_float(proj[trow * p.stride + p.g_off + h * V + c]);
            val *= g / (1.0f + expf(-g));
          }
          out[trow * (int64_t)(Hn * V) + h * V + c] = cw_from_float<T>(val);
        }
      }
    }
  }
  if (active) {
#pragma unroll
    for (int rr = 0; rr < RPT; ++rr)
      if (d0 + rr < D) st[(int64_t)(d0 + rr) * V + v] = S[rr];
  }
}

template <typename T, int RPT>
__global__ __launch_bounds__(256) void linear_recurrence_quads_kernel(LinRecParams p, LinRecForm f, bool rank_quads) {
  recurrence_quads<T, RPT>(p, f, rank_quads, blockIdx.x, blockIdx.y);
}

// vdim up to 256; dim up to 128 rows a thread: dim <= 128 * min(256 / vdim, dim).
CW_EXPORT int cw_linear_recurrence_supported(int dim, int vdim) {
  if (dim <= 0 || vdim <= 0 || vdim > 256) return 0;
  const int ds = 256 / vdim < dim ? 256 / vdim : dim;
  return (dim + ds - 1) / ds <= 128 ? 1 : 0;
}

// Checks the arguments and fills ``l``; l.rows is 0 where four columns a thread do not serve the sizes.
static int recurrence_launch(RecurrenceLaunch& l, int dtype, const void* proj, int64_t stride, int q_off, int k_off, int v_off, int g_off,
                             int u_off, const void* a2, const float* a2b, const float* norm_w, float* state, int n_slots,
                             const int* state_slots, const int* cu_q, void* out, int n_requests, int heads, int dim, int vdim, int rank,
                             float q_scale, float inv_tau, float eps, int decay_kind, const float* bonus, int norm_w_stride, const void* u,
                             int64_t u_stride, int64_t state_stride) {
  if (n_requests < 0 || !proj || !a2 || !state || !state_slots || !cu_q || !out) return CW_ERR_ARG;
  if (heads <= 0 || rank <= 0 || n_slots <= 0 || q_off < 0 || k_off < 0 || v_off < 0 || u_off < 0 || stride <= 0) return CW_ERR_ARG;
  if (q_off % stride + heads * dim > stride || k_off % stride + heads * dim > stride || v_off % stride + heads * vdim > stride ||
      (!u && u_off + rank > stride) || (g_off >= 0 && g_off % stride + heads * vdim > stride))
    return CW_ERR_ARG;
  if (decay_kind < 0 || decay_kind > 2 || (norm_w_stride != 0 && norm_w_stride != vdim) || (u && u_stride < rank) ||
      state_stride < (int64_t)heads * dim * vdim || state_stride > 0x7fffffff)
    return CW_ERR_ARG;
  if (!cw_linear_recurrence_supported(dim, vdim)) return CW_ERR_SIZE;
  l = RecurrenceLaunch{};
  l.f = {decay_kind, bonus, norm_w_stride, u, u_stride, (int)state_stride};
  LinRecParams& p = l.p;
  p.proj = proj; p.stride = stride; p.q_off = q_off; p.k_off = k_off; p.v_off = v_off; p.g_off = g_off; p.u_off = u_off;
  p.a2 = a2; p.a2b = a2b; p.norm_w = norm_w; p.state = state; p.state_slots = state_slots; p.cu_q = cu_q; p.out = out;
  p.heads = heads; p.dim = dim; p.vdim = vdim; p.rank = rank; p.n_slots = n_slots;
  p.q_scale = q_scale; p.inv_tau = inv_tau; p.eps = eps;
  l.dtype = dtype;
  l.requests = n_requests;
  // four columns a thread, where a wave's lanes divide evenly among them and the rows fit the registers
  const int vq = vdim / 4;
  if (vdim % 4 == 0 && (vq & (vq - 1)) == 0 && vq <= 64 && !((uintptr_t)state & 15) && state_stride % 4 == 0) {
    const int runs = 256 / vq < dim ? 256 / vq : dim;
    int rows = 1;
    while (rows * runs < dim) rows *= 2;
    const int ds = (dim + rows - 1) / rows < 256 / vq ? (dim + rows - 1) / rows : 256 / vq;
    l.rank_quads = rank % 16 == 0 && !((uintptr_t)a2 & 15) && !((uintptr_t)proj & 15) && !((uintptr_t)u & 15) &&
                   (u ? u_stride % 4 == 0 : stride % 4 == 0 && u_off % 4 == 0);
    l.lds = (int64_t)LR_TC * (3 * ds * rows + vdim + 4 * vdim) * sizeof(float);
    l.rows = rows;
  }
  return CW_OK;
}

CW_EXPORT int cw_linear_recurrence_prepared_bytes() { return sizeof(RecurrenceLaunch); }

// The launch of cw_linear_recurrence as ``prepared`` (cw_linear_recurrence_prepared_bytes()), for a kernel that runs it beside other
// work (cw_sink_decode_beside); CW_ERR_SIZE where there is none for these sizes: bfloat16, four columns and four or eight rows a thread.
CW_EXPORT int cw_linear_recurrence_prepare(int dtype, const void* proj, int64_t stride, int q_off, int k_off, int v_off, int g_off,
                                           int u_off, const void* a2, const float* a2b, const float* norm_w, float* state,
                                           int n_slots, const int* state_slots, const int* cu_q, void* out, int n_requests,
                                           int heads, int dim, int vdim, int rank, float q_scale, float inv_tau, float eps,
                                           int decay_kind, const float* bonus, int norm_w_stride, const void* u, int64_t u_stride,
                                           int64_t state_stride, void* prepared) {
  if (!prepared) return CW_ERR_ARG;
  RecurrenceLaunch l;
  const int rc = recurrence_launch(l, dtype, proj, stride, q_off, k_off, v_off, g_off, u_off, a2, a2b, norm_w, state, n_slots, state_slots,
                                   cu_q, out, n_requests, heads, dim, vdim, rank, q_scale, inv_tau, eps, decay_kind, bonus,
                                   norm_w_stride, u, u_stride, state_stride);
  if (rc != CW_OK) return rc;
  if (dtype != CW_BF16 || (l.rows != 4 && l.rows != 8)) return CW_ERR_SIZE;
  *(RecurrenceLaunch*)prepared = l;
  return CW_OK;
}

CW_EXPORT int cw_linear_recurrence(int dtype, const void* proj, int64_t stride, int q_off, int k_off, int v_off, int g_off,
                                   int u_off, const void* a2, const float* a2b, const float* norm_w, float* state,
                                   int n_slots, const int* state_slots, const int* cu_q, void* out, int n_requests,
                                   int heads, int dim, int vdim, int rank, float q_scale, float inv_tau, float eps,
                                   int decay_kind, const float* bonus, int norm_w_stride, const void* u, int64_t u_stride,
                                   int64_t state_stride, hipStream_t stream) {
  RecurrenceLaunch l;
  const int rc = recurrence_launch(l, dtype, proj, stride, q_off, k_off, v_off, g_off, u_off, a2, a2b, norm_w, state, n_slots, state_slots,
                                   cu_q, out, n_requests, heads, dim, vdim, rank, q_scale, inv_tau, eps, decay_kind, bonus,
                                   norm_w_stride, u, u_stride, state_stride);
  if (rc != CW_OK) return rc;
  if (n_requests == 0) return CW_OK;
  if (heads > 65535) return CW_ERR_SIZE;
  const LinRecParams& p = l.p;
  const LinRecForm& form = l.f;
  const int ds = 256 / vdim < dim ? 256 / vdim : dim;
  const int rpt = (dim + ds - 1) / ds;
  const size_t smem = ((size_t)LR_TC * (3 * dim + vdim) + (size_t)LR_TC * ds * vdim) * sizeof(float);
  dim3 grid(n_requests, heads), block(256);
  if (l.rows) {
    const int rows = l.rows;
    const size_t lds = (size_t)l.lds;
    const bool rank_quads = l.rank_quads != 0;
#define CW_QUADS(T_, RPT_)                                                                                          \
  do {                                                                                                              \
    if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)linear_recurrence_quads_kernel<T_, RPT_>,               \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) \
      return CW_ERR_LAUNCH;                                                                                         \
    hipLaunchKernelGGL((linear_recurrence_quads_kernel<T_, RPT_>), grid, block, lds, stream, p, form, rank_quads);  \
    return cw_launch_status();                                                                                      \
  } while (0)
#define CW_QUADS_BY_ROWS(T_)             \
  do {                                   \
    if (rows == 1) CW_QUADS(T_, 1);      \
    if (rows == 2) CW_QUADS(T_, 2);      \
    if (rows == 4) CW_QUADS(T_, 4);      \
    if (rows == 8) CW_QUADS(T_, 8);      \
    if (rows == 16) CW_QUADS(T_, 16);    \
    if (rows == 32) CW_QUADS(T_, 32);    \
  } while (0)
    if (dtype == CW_F32) CW_QUADS_BY_ROWS(float);
    if (dtype == CW_BF16) CW_QUADS_BY_ROWS(bf16_t);
#undef CW_QUADS_BY_ROWS
#undef CW_QUADS
  }
#define CW_LAUNCH(T_, RPT_)                                                                                        \
  do {                                                                                                             \
    if (smem > 48 * 1024 && hipFuncSetAttribute((const void*)linear_recurrence_kernel<T_, RPT_>,                   \
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) \
      return CW_ERR_LAUNCH;                                                                                        \
    hipLaunchKernelGGL((linear_recurrence_kernel<T_, RPT_>), grid, block, smem, stream, p, form);                        \
  } while (0)
#define CW_BY_ROWS(T_)                         \
  do {                                         \
    if (rpt <= 2) CW_LAUNCH(T_, 2);            \
    else if (rpt <= 4) CW_LAUNCH(T_, 4);       \
    else if (rpt <= 8) CW_LAUNCH(T_, 8);       \
    else if (rpt <= 16) CW_LAUNCH(T_, 16);     \
    else if (rpt <= 32) CW_LAUNCH(T_, 32);     \
    else if (rpt <= 64) CW_LAUNCH(T_, 64);     \
    else CW_LAUNCH(T_, 128);                   \
  } while (0)
  if (dtype == CW_F32) CW_BY_ROWS(float);
  else if (dtype == CW_BF16) CW_BY_ROWS(bf16_t);
  else return CW_ERR_DTYPE;
#undef CW_BY_ROWS
#undef CW_LAUNCH
  return cw_launch_status();
}

// ======================================================================================
// The same recurrence for long portions, cut into segments of tokens that run side by side. (Sizes that the matrix
// cores take run on the kernels behind these.)
//
//   prepare:   per token and key channel the decay a (float32, through log-sigmoid), the scaled
//              query and the key as float32 rows [T, heads * dim]: the walks below read them
//              with addresses that do not depend on the lane, so they arrive in scalar registers.
//   segments:  every (segment, head) walks its tokens from a zero state: what the segment adds to
//              the state (float32 [dim, vdim]) and the product of its decays per channel.
//   carry:     per request and head, segment after segment: start(s + 1) = decay(s) * start(s) +
//              added(s), from the request's state slot; the last one is the slot's new state.
//   outputs:   every (segment, head) walks its tokens again from its start state: o_t = S_t^T q_t.
//   finish:    RMS norm over vdim, weight, silu(gate), cast: one wave per (token, head).
//
// In the walks a thread owns one column of the state with all its rows in registers (dim <= 128),
// a wave 64 columns; nothing is exchanged between threads. The sums are the same as in the
// token-by-token kernel but for the place of the parentheses: S_t = A S_start + (local sum).
// ======================================================================================
#define LRS_MAX_DIM 128

struct SegParams {
  const void* proj;
  int64_t stride;
  int q_off, k_off, v_off, g_off, u_off;
  const void* a2;
  const float* a2b;
  const float* norm_w;
  float* state;
  const int* state_slots;
  const int* cu_q;
  const int* seg_items;   // [n_segments, 4]: request, first token of the segment (in the portion), tokens, index of the segment in its request
  const int* req_first;   // [R + 1]: first segment of each request in seg_items
  float* dec;             // [T, heads * dim] decays
  float* qf;              // [T, heads * dim] (the walks only, as kf and raw)
  float* kf;              // [T, heads * dim]
  float* added;           // [n_segments, heads, dim, vdim]
  float* seg_decay;       // [n_segments, heads, dim]
  float* raw;             // [T, heads * vdim] outputs before norm and gate
  void* out;
  int heads, dim, vdim, rank, n_slots, n_tokens;
  float q_scale, inv_tau, eps;
  int seg_tokens;         // the most tokens a segment has
  LinRecForm form;
};

template <typename T> struct LrVec;
template <> struct LrVec<float> {
  static constexpr int N = 4;
  __device__ static void load(const float* p, float* o) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
  }
};
template <> struct LrVec<bf16_t> {
  static constexpr int N = 8;
  __device__ static void load(const bf16_t* p, float* o) {
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) { o[2 * i] = __uint_as_float(w[i] << 16); o[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u); }
  }
};

template <typename T>
__global__ __launch_bounds__(256) void lrs_prepare_kernel(SegParams p) {
  const int HD = p.heads * p.dim;
  const int64_t n = (int64_t)p.n_tokens * HD;
  const T* proj = (const T*)p.proj;
  const T* a2 = (const T*)p.a2;
  constexpr int N = LrVec<T>::N;
  const bool vec = p.rank % N == 0 && !((uintptr_t)a2 & 15) &&
                   (p.form.u ? p.form.u_stride % N == 0 && !((uintptr_t)p.form.u & 15)
                             : p.u_off % N == 0 && p.stride % N == 0 && !((uintptr_t)proj & 15));
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < n; idx += (int64_t)gridDim.x * 256) {
    const int64_t t = idx / HD;
    const int c = (int)(idx - t * HD);
    const T* row = proj + t * p.stride;
    float z = p.a2b ? p.a2b[c] : 0.0f;
    const T* w = a2 + (int64_t)c * p.rank;
    const T* u = p.form.u ? (const T*)p.form.u + t * p.form.u_stride : row + p.u_off;
    if (p.form.decay_kind == 2) {
      for (int e = 0; e < p.rank; ++e) z += cw_to_float(w[e]) * tanhf(cw_to_float(u[e]));
    } else if (vec) {  // 16 bytes of the decay matrix's row and of the token's decay input at a time
      for (int e = 0; e < p.rank; e += N) {
        float wv[N], uv[N];
        LrVec<T>::load(w + e, wv);
        LrVec<T>::load(u + e, uv);
#pragma unroll
        for (int i = 0; i < N; ++i) z += wv[i] * uv[i];
      }
    } else {
      for (int e = 0; e < p.rank; ++e) z += cw_to_float(w[e]) * cw_to_float(u[e]);
    }
    p.dec[idx] = lr_decay(z, p.form.decay_kind, p.inv_tau);
    p.qf[idx] = cw_to_float(row[p.q_off + c]) * p.q_scale;
    p.kf[idx] = cw_to_float(row[p.k_off + c]);
  }
}

// MODE 0: from zero, leaves ``added`` and ``seg_decay``; MODE 1: from the start state in ``added``
// (the carry kernel has turned it into that), writes the raw outputs.
template <typename T, int DIM, int MODE>
__global__ __launch_bounds__(256) void lrs_walk_kernel(SegParams p) {
  extern __shared__ __align__(16) float tile[];  // the segment's decays, keys and queries: [3][tokens][D]
  const int seg = blockIdx.x, h = blockIdx.y;
  const int v = blockIdx.z * blockDim.x + threadIdx.x;
  const int r = p.seg_items[4 * seg], tok0 = p.seg_items[4 * seg + 1], ntok = p.seg_items[4 * seg + 2];
  const int q_len = p.cu_q[r + 1] - p.cu_q[r];
  const int slot = p.state_slots[r];
  if (tok0 >= q_len || slot < 0 || slot >= p.n_slots) return;
  const int nt = min(ntok, q_len - tok0);
  const int64_t row0 = p.cu_q[r] + tok0;
  const int D = p.dim, V = p.vdim, HD = p.heads * p.dim;
  const bool live = v < V;
  const int vc = live ? v : V - 1;
  float S[DIM];
  float* mine = p.added + (((int64_t)seg * p.heads + h) * D) * V;
  if (MODE == 1) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) S[d] = d < D ? mine[(int64_t)d * V + vc] : 0.0f;
  } else {
#pragma unroll
    for (int d = 0; d < DIM; ++d) S[d] = 0.0f;
  }
  float A[MODE == 0 ? DIM : 1];
  if (MODE == 0) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) A[d] = 1.0f;
  }
  const T* proj = (const T*)p.proj;
  // the waves of the workgroup (each 64 columns of the same head's state) share the segment's
  // decays, keys and queries through LDS: fetched once, in whole rows, then read by every lane at
  // the same address (a broadcast) while the tokens are walked
  float* As = tile;
  float* Kt = As + p.seg_tokens * D;
  float* Qt = Kt + p.seg_tokens * D;
  for (int i = threadIdx.x; i < nt * D; i += blockDim.x) {
    const int t = i / D, d = i - t * D;
    const int64_t at = (row0 + t) * HD + h * D + d;
    As[i] = p.dec[at];
    Kt[i] = p.kf[at];
    if (MODE == 1) Qt[i] = p.qf[at];
  }
  __syncthreads();
  // with a bonus the token's own share of its output is one number a token whatever the state's
  // column, (sum over d of q_d bonus_d k_d) v: lane t of every wave sums token t's, once a segment,
  // and hands it to the others when the token's turn comes (a segment has at most 64 tokens)
  float own = 0.0f;
  if (MODE == 1 && p.form.bonus) {
    const int lane = threadIdx.x & 63;
    if (lane < nt) {
      const float* bn = p.form.bonus + h * D;
      for (int i = 0; i < D; ++i) {
        const int d = (i + lane) % D;   // every lane a bank of its own
        own += Qt[lane * D + d] * bn[d] * Kt[lane * D + d];
      }
    }
  }
  const bool reads_before = MODE == 1 && p.form.bonus != nullptr;   // the output reads the state before the token joins it
  for (int t = 0; t < nt; ++t) {
    const int64_t row = row0 + t;
    const float* a = As + t * D;
    const float* k = Kt + t * D;
    const float* q = Qt + t * D;
    const float vv = cw_to_float(proj[row * p.stride + p.v_off + h * V + vc]);
    float o0 = 0.0f, o1 = 0.0f, o2 = 0.0f, o3 = 0.0f;
    if (reads_before) {
      o0 = __shfl(own, t, 64) * vv;
#pragma unroll
      for (int d = 0; d < DIM; d += 4) {
        if (d < D) {
          o0 += q[d] * S[d];
          o1 += q[d + 1] * S[d + 1];
          o2 += q[d + 2] * S[d + 2];
          o3 += q[d + 3] * S[d + 3];
          S[d] = a[d] * S[d] + k[d] * vv;
          S[d + 1] = a[d + 1] * S[d + 1] + k[d + 1] * vv;
          S[d + 2] = a[d + 2] * S[d + 2] + k[d + 2] * vv;
          S[d + 3] = a[d + 3] * S[d + 3] + k[d + 3] * vv;
        }
      }
    } else {
#pragma unroll
      for (int d = 0; d < DIM; d += 4) {
        if (d < D) {  // D is a multiple of 4 here (the host sees to it)
          S[d] = a[d] * S[d] + k[d] * vv;
          S[d + 1] = a[d + 1] * S[d + 1] + k[d + 1] * vv;
          S[d + 2] = a[d + 2] * S[d + 2] + k[d + 2] * vv;
          S[d + 3] = a[d + 3] * S[d + 3] + k[d + 3] * vv;
          if (MODE == 1) {
            o0 += q[d] * S[d];
            o1 += q[d + 1] * S[d + 1];
            o2 += q[d + 2] * S[d + 2];
            o3 += q[d + 3] * S[d + 3];
          } else if (threadIdx.x == 0 && blockIdx.z == 0) {
            A[d] *= a[d]; A[d + 1] *= a[d + 1]; A[d + 2] *= a[d + 2]; A[d + 3] *= a[d + 3];
          }
        }
      }
    }
    if (MODE == 1 && live) p.raw[row * (int64_t)(p.heads * V) + h * V + v] = (o0 + o1) + (o2 + o3);
  }
  if (MODE == 0) {
    if (live) {
#pragma unroll
      for (int d = 0; d < DIM; ++d)
        if (d < D) mine[(int64_t)d * V + v] = S[d];
    }
    if (threadIdx.x == 0 && blockIdx.z == 0) {
      float* sd = p.seg_decay + ((int64_t)seg * p.heads + h) * D;
#pragma unroll
      for (int d = 0; d < DIM; ++d)
        if (d < D) sd[d] = A[d];
    }
  }
}

// per (request, head, 256 state elements): walk the request's segments in order. Bound by the trips to memory of a
// chain that needs them not: eight segments' values are asked for together (64 segments of 12 heads of 64 x 128, one
// after another: 26.2 us, so 17.4).
__global__ __launch_bounds__(256) void lrs_carry_kernel(SegParams p) {
  const int r = blockIdx.x, h = blockIdx.y;
  const int64_t e = (int64_t)blockIdx.z * 256 + threadIdx.x;  // element d * V + v
  const int D = p.dim, V = p.vdim;
  const int slot = p.state_slots[r];
  const int q_len = p.cu_q[r + 1] - p.cu_q[r];
  if (e >= (int64_t)D * V || slot < 0 || slot >= p.n_slots || q_len <= 0) return;
  const int d = (int)(e / V);
  float* st = p.state + (int64_t)slot * p.form.state_stride + ((int64_t)h * D) * V + e;
  float S = *st;
  const int last = p.req_first[r + 1];
  for (int seg0 = p.req_first[r]; seg0 < last; seg0 += 8) {
    float add[8], decay[8];
    int begin[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t at = (int64_t)min(seg0 + u, last - 1) * p.heads + h;
      begin[u] = p.seg_items[4 * min(seg0 + u, last - 1) + 1];
      add[u] = p.added[at * D * V + e];
      decay[u] = p.seg_decay[at * D + d];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      // segments past the request's tokens (a batch of fixed shape) come after all others
      if (seg0 + u >= last || begin[u] >= q_len) break;
      p.added[((int64_t)(seg0 + u) * p.heads + h) * D * V + e] = S;  // the segment's start state, for the second walk
      S = decay[u] * S + add[u];
    }
  }
  *st = S;
}

template <typename T>
__global__ __launch_bounds__(256) void lrs_finish_kernel(SegParams p) {
  const int V = p.vdim, Hn = p.heads;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + wave;  // (token, head)
  if (item >= (int64_t)p.n_tokens * Hn) return;
  const int64_t t = item / Hn;
  const int h = (int)(item - t * Hn);
  const float* o = p.raw + t * (int64_t)(Hn * V) + h * V;
  float ss = 0.0f;
  for (int c = lane; c < V; c += 64) ss += o[c] * o[c];
  float inv = 1.0f;
  if (p.norm_w) inv = 1.0f / sqrtf(cw_wave_sum(ss) / (float)V + p.eps);
  const T* proj = (const T*)p.proj;
  T* out = (T*)p.out;
  for (int c = lane; c < V; c += 64) {
    float val = o[c] * inv;
    if (p.norm_w) val *= p.norm_w[h * p.form.norm_w_stride + c];
    if (p.g_off >= 0) {
      const float g = cw_to_float(proj[t * p.stride + p.g_off + h * V + c]);
      val *= g / (1.0f + expf(-g));
    }
    out[t * (int64_t)(Hn * V) + h * V + c] = cw_from_float<T>(val);
  }
}

// ======================================================================================
// The same on the matrix cores, for segments of up to 32 tokens, dim 16, 32, 64 or 128 and vdim a multiple of
// 16 up to 256, all in float32 (v_mfma_f32_16x16x4_f32). Within a chunk of 16 tokens
//   o_t = (q_t * A_t)^T S + sum over j <= t of P[t][j] v_j,   S' = diag(A_16) S + sum over j of (k_j * Z_j) v_j^T
// with A_t the product of the chunk's decays up to t, Z_j that of those behind j and P[t][j] = sum over d of
// q_t[d] k_j[d] (the product of the decays behind j up to t)[d]. Every factor is a product of decays, each at most 1,
// as in the walk: nothing is divided, so a decay that vanishes makes zeros and no infinity.
//
//   added:    (segment, head): decays (kept for ``outputs``), keys times the decays behind them, added = K'^T V.
//   carry:    as above.
//   outputs:  (segment, head): P on the vector unit, one thread a key and a run of channels, walking the chunk's
//             tokens; the products; norm over vdim, gate and cast.
// The walk takes 192 vector instructions and 48 reads of LDS a token, channel and column of 64; what bounds these
// two kernels is a chain of trips to memory and LDS a workgroup, with three workgroups a compute unit beside each other.
// Measured on an MI355X, 2048 tokens, 12 heads of 64 x 128, rank 32, bfloat16: prepare 21, walks 64 + 72, finish 14 and carry
// 17 us before, added 21, outputs 32 and carry 17 now; one call 188 -> 69 us, of 100 tokens (14 heads of 64 x 64) 133 -> 27.
// A wave owns 16 * VT columns; lane (c, s) = (l % 16, l / 16) holds, of a tile of the state, channels 4 s .. 4 s + 3 of
// column c, which is also what a product that contracts over channels wants of it.
typedef __attribute__((ext_vector_type(4))) float lrs_f32x4_t;
#define LRS_MFMA_SEG 32
#define LRS_MAX_STAGED 128  // ranks whose decay inputs the first kernel brings to LDS

// sum over the 16 lanes of a row of the wave; every lane gets it
__device__ __forceinline__ float lrs_row_sum(float v) {
#define LRS_ROR(n) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + (n), 0xf, 0xf, true))
  LRS_ROR(8);
  LRS_ROR(4);
  LRS_ROR(2);
  LRS_ROR(1);
#undef LRS_ROR
  return v;
}

// Elements of the wave's columns as a product's operand or result: token 16 b + 4 s + j, column col0 + 16 vt + c, of the
// head's columns from ``off`` on; zeros past the segment's tokens and past vdim (read from a place inside, so that no load
// hangs on a condition: one trip to memory for all of them).
template <typename T, int VT>
__device__ __forceinline__ void lrs_load_columns(const SegParams& p, int off, int64_t row0, int nt, int h, int col0, int c, int s,
                                                 float (&vf)[2][4][VT]) {
  const T* v = (const T*)p.proj + off + h * p.vdim + c;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const int t = 16 * b + 4 * s + j, col = col0 + 16 * vt;
        vf[b][j][vt] = cw_to_float(v[(row0 + min(t, nt - 1)) * p.stride + (col < p.vdim ? col : 0)]);
        vf[b][j][vt] = t < nt && col < p.vdim ? vf[b][j][vt] : 0.0f;
      }
}

template <typename T, int D, int VT>
__global__ __launch_bounds__(256) void lrs_added_kernel(SegParams p) {
  constexpr int LD = D + 4, G = 256 / D, TPG = LRS_MFMA_SEG / G;  // a thread makes TPG tokens' decays of one channel
  __shared__ __align__(16) float keys[LRS_MFMA_SEG * LD];
  __shared__ float total[G * D];
  const int seg = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, s = lane >> 4;
  const int r = p.seg_items[4 * seg], tok0 = p.seg_items[4 * seg + 1], ntok = p.seg_items[4 * seg + 2];
  const int begin = p.cu_q[r], q_len = p.cu_q[r + 1] - begin;
  const int slot = p.state_slots[r];
  if (tok0 >= q_len || slot < 0 || slot >= p.n_slots) return;
  const int nt = min(ntok, q_len - tok0);
  const int64_t row0 = begin + tok0;
  const int col0 = wave * 16 * VT;
  float vf[2][4][VT];
  lrs_load_columns<T, VT>(p, p.v_off, row0, nt, h, col0, c, s, vf);

  const int d = tid % D, g = tid / D, t0 = g * TPG, channel = h * D + d;
  const T* proj = (const T*)p.proj;
  const T* w = (const T*)p.a2 + (int64_t)channel * p.rank;
  constexpr int N = LrVec<T>::N;
  const bool vec = p.form.decay_kind != 2 && p.rank % N == 0 && p.rank <= LRS_MAX_STAGED && !((uintptr_t)p.a2 & 15) &&
                   (p.form.u ? p.form.u_stride % N == 0 && !((uintptr_t)p.form.u & 15)
                             : p.u_off % N == 0 && p.stride % N == 0 && !((uintptr_t)proj & 15));
  const T* u = p.form.u ? (const T*)p.form.u : proj + p.u_off;
  const int64_t u_stride = p.form.u ? p.form.u_stride : p.stride;
  float z[TPG], k[TPG];
  const float bias = p.a2b ? p.a2b[channel] : 0.0f;
#pragma unroll
  for (int i = 0; i < TPG; ++i) {
    z[i] = bias;
    k[i] = cw_to_float(proj[(row0 + min(t0 + i, nt - 1)) * p.stride + p.k_off + channel]);
  }
  if (vec) {  // 16 bytes of the channel's row and of each token's decay input at a time
    // (the tokens' inputs through LDS, as they are: every wave wants all of them)
    extern __shared__ __align__(16) unsigned char staged[];
    T* us = (T*)staged;
    const int pieces = p.rank / N;
    float wv[N];
    LrVec<T>::load(w, wv);
    for (int i = tid; i < LRS_MFMA_SEG * pieces; i += 256)
      reinterpret_cast<uint4*>(us)[i] = *reinterpret_cast<const uint4*>(u + (row0 + min(i / pieces, nt - 1)) * u_stride + i % pieces * N);
    __syncthreads();
    for (int e = 0; e < p.rank; e += N) {
      float next[N];
      LrVec<T>::load(w + min(e + N, p.rank - N), next);
#pragma unroll
      for (int i = 0; i < TPG; ++i) {
        float uv[N];
        LrVec<T>::load(us + (t0 + i) * p.rank + e, uv);
#pragma unroll
        for (int n = 0; n < N; ++n) z[i] += wv[n] * uv[n];
      }
#pragma unroll
      for (int n = 0; n < N; ++n) wv[n] = next[n];
    }
  } else {
    for (int e = 0; e < p.rank; ++e) {
      const float we = cw_to_float(w[e]);
#pragma unroll
      for (int i = 0; i < TPG; ++i) {
        const float ue = cw_to_float(u[(row0 + min(t0 + i, nt - 1)) * u_stride + e]);
        z[i] += we * (p.form.decay_kind == 2 ? tanhf(ue) : ue);
      }
    }
  }
  float run = 1.0f;  // the decays behind token i, of this thread's tokens
#pragma unroll
  for (int i = TPG - 1; i >= 0; --i) {
    const float a = lr_decay(z[i], p.form.decay_kind, p.inv_tau);
    k[i] = t0 + i < nt ? k[i] * run : 0.0f;
    if (t0 + i < nt) p.dec[(row0 + t0 + i) * (int64_t)(p.heads * D) + channel] = a;
    run *= t0 + i < nt ? a : 1.0f;
  }
  total[tid] = run;
  __syncthreads();
  float behind = 1.0f;
  for (int i = g + 1; i < G; ++i) behind *= total[i * D + d];
#pragma unroll
  for (int i = 0; i < TPG; ++i) keys[(t0 + i) * LD + d] = k[i] * behind;
  if (g == 0) p.seg_decay[((int64_t)seg * p.heads + h) * D + d] = run * behind;
  __syncthreads();
  float* mine = p.added + (((int64_t)seg * p.heads + h) * D) * p.vdim + col0 + c;
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) {
    lrs_f32x4_t acc[VT];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) acc[vt] = (lrs_f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = keys[(16 * b + 4 * s + j) * LD + 16 * dt + c];
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) acc[vt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vf[b][j][vt], acc[vt], 0, 0, 0);
      }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
      if (col0 + 16 * vt < p.vdim)
#pragma unroll
        for (int i = 0; i < 4; ++i) mine[(int64_t)(16 * dt + 4 * s + i) * p.vdim + 16 * vt] = acc[vt][i];
  }
}

template <typename T, int D, int VT>
__global__ __launch_bounds__(256, D * VT <= 128 ? 3 : 1) void lrs_outputs_kernel(SegParams p) {
  constexpr int LD = D + 4, DT = D / 16, PER = D / 16;  // PER: channels of a thread while P is made
  constexpr int UNITS = (4 * D + 255) / 256;            // runs of 8 tokens of a channel that a thread scales
  __shared__ __align__(16) float As[LRS_MFMA_SEG * LD], Qs[LRS_MFMA_SEG * LD], Ks[LRS_MFMA_SEG * LD];
  __shared__ __align__(16) float Ps[2 * 16 * 20], chunk_decay[2 * D];
  __shared__ float squares[4 * LRS_MFMA_SEG];
  const int seg = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, s = lane >> 4;
  const int r = p.seg_items[4 * seg], tok0 = p.seg_items[4 * seg + 1], ntok = p.seg_items[4 * seg + 2];
  const int begin = p.cu_q[r], q_len = p.cu_q[r + 1] - begin;
  const int slot = p.state_slots[r];
  if (tok0 >= q_len || slot < 0 || slot >= p.n_slots) return;
  const int nt = min(ntok, q_len - tok0);
  const int64_t row0 = begin + tok0;
  const int V = p.vdim, col0 = wave * 16 * VT;
  const bool before = p.form.bonus != nullptr;  // the output reads the state before the token joins it
  const T* proj = (const T*)p.proj;

  // decays, queries and keys of the segment; past its tokens decays of 1 and zeros
  constexpr int PIECES = LRS_MFMA_SEG * D / 256;
  {
    float a[PIECES], q[PIECES], k[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int idx = tid + 256 * i, t = idx / D, d = idx - t * D;
      const bool ok = t < nt;
      const int64_t row = row0 + (ok ? t : 0);
      const int channel = h * D + d;
      a[i] = p.dec[row * (int64_t)(p.heads * D) + channel];
      q[i] = cw_to_float(proj[row * p.stride + p.q_off + channel]);
      k[i] = cw_to_float(proj[row * p.stride + p.k_off + channel]);
      a[i] = ok ? a[i] : 1.0f;
      q[i] = ok ? q[i] * p.q_scale : 0.0f;
      k[i] = ok ? k[i] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int idx = tid + 256 * i, at = idx / D * LD + idx % D;
      As[at] = a[i];
      Qs[at] = q[i];
      Ks[at] = k[i];
    }
  }
  // what the products and the end need is asked for meanwhile
  float vf[2][4][VT];
  lrs_load_columns<T, VT>(p, p.v_off, row0, nt, h, col0, c, s, vf);
  lrs_f32x4_t S[DT][VT];
  const float* start = p.added + (((int64_t)seg * p.heads + h) * D) * V + col0 + c;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool live = col0 + 16 * vt < V;
        const float v = start[(int64_t)(16 * dt + 4 * s + i) * V + (live ? 16 * vt : -col0)];
        S[dt][vt][i] = live ? v : 0.0f;
      }
  float gate[2][4][VT], nw[VT];
  if (p.g_off >= 0) lrs_load_columns<T, VT>(p, p.g_off, row0, nt, h, col0, c, s, gate);
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) nw[vt] = p.norm_w && col0 + 16 * vt < V ? p.norm_w[h * p.form.norm_w_stride + col0 + 16 * vt + c] : 1.0f;
  __syncthreads();

  {  // P: thread = (key j of the chunk, run of PER channels), the 16 runs in neighbouring lanes
    const int j = tid >> 4, run = tid & 15;
    float bonus[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) bonus[e] = before ? p.form.bonus[h * D + run * PER + e] : 1.0f;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (16 * b >= nt) break;
      float w[PER], mine = 0.0f;
#pragma unroll
      for (int e = 0; e < PER; ++e) w[e] = Ks[(16 * b + j) * LD + run * PER + e];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const float* a = As + (16 * b + t) * LD + run * PER;
        const float* q = Qs + (16 * b + t) * LD + run * PER;
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < PER; ++e) {
          const float decayed = t > j ? w[e] * a[e] : w[e];
          sum += q[e] * (before ? (t == j ? bonus[e] * w[e] : w[e]) : decayed);
          w[e] = decayed;
        }
        sum = lrs_row_sum(sum);
        mine = t == run ? sum : mine;
      }
      Ps[(16 * b + run) * 20 + j] = run >= j ? mine : 0.0f;  // (a later key has no part in it, whatever it holds)
    }
  }
  // queries times the decays up to them, keys times those behind them, chunk by chunk
  float qn[UNITS][8], kn[UNITS][8], all[UNITS];
#pragma unroll
  for (int n = 0; n < UNITS; ++n) {
    const int unit = tid + 256 * n;
    const int d = unit % D, half = unit / D & 1, b = unit / (2 * D);
    if (b > 1) break;
    float other = 1.0f, a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a[i] = As[(16 * b + 8 * half + i) * LD + d];
      other *= As[(16 * b + 8 * (1 - half) + i) * LD + d];
    }
    float up = half ? other : 1.0f, down = half ? 1.0f : other;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float with = up * a[i];
      qn[n][i] = Qs[(16 * b + 8 * half + i) * LD + d] * (before ? up : with);
      up = with;
    }
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      kn[n][i] = Ks[(16 * b + 8 * half + i) * LD + d] * down;
      down *= a[i];
    }
    all[n] = down;
  }
  __syncthreads();
#pragma unroll
  for (int n = 0; n < UNITS; ++n) {
    const int unit = tid + 256 * n;
    const int d = unit % D, half = unit / D & 1, b = unit / (2 * D);
    if (b > 1) break;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      Qs[(16 * b + 8 * half + i) * LD + d] = qn[n][i];
      Ks[(16 * b + 8 * half + i) * LD + d] = kn[n][i];
    }
    if (!half) chunk_decay[b * D + d] = all[n];
  }
  __syncthreads();

  lrs_f32x4_t o[2][VT];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) o[b][vt] = (lrs_f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
    if (16 * b >= nt) continue;
    // Sums of every second or fourth tile of channels, and of the chunk's own keys, added at the end: one chain of additions
    // for all of them rounds further. Four tiles of columns a wave have registers for one sum beside the total, which
    // takes two tiles of channels at a time (none where three workgroups share a compute unit).
    constexpr bool TURNS = VT > 2;
    constexpr int SIDE = TURNS ? (D >= 64 ? 1 : 0) : D == 128 ? 4 : 2;
    lrs_f32x4_t apart[SIDE > 0 ? SIDE : 1][VT];
    auto sum_of = [&](int k, int vt) __attribute__((always_inline)) -> lrs_f32x4_t& { return k ? apart[k - 1][vt] : o[b][vt]; };
#pragma unroll
    for (int k = 0; k < SIDE; ++k)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) apart[k][vt] = (lrs_f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const lrs_f32x4_t q = *reinterpret_cast<const lrs_f32x4_t*>(Qs + (16 * b + c) * LD + 16 * dt + 4 * s);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          lrs_f32x4_t& to = sum_of(TURNS ? SIDE : dt % SIDE, vt);
          to = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i], S[dt][vt][i], to, 0, 0, 0);
        }
      if (TURNS && SIDE && dt & 1)
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          o[b][vt] += apart[0][vt];
          apart[0][vt] = (lrs_f32x4_t){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    bool finite = true;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) finite = finite && fabsf(vf[b][j][vt]) < INFINITY;
    if (__builtin_amdgcn_ballot_w64(!finite) == 0) {
      const lrs_f32x4_t w = *reinterpret_cast<const lrs_f32x4_t*>(Ps + (16 * b + c) * 20 + 4 * s);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) sum_of(SIDE, vt) = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], vf[b][j][vt], sum_of(SIDE, vt), 0, 0, 0);
    } else {  // an infinite value must not meet the zeros of the tokens before it
#pragma unroll
      for (int j = 0; j < 16; ++j)
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          const float v = __shfl(vf[b][j % 4][vt], (j / 4) * 16 + c, 64);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (4 * s + i >= j) sum_of(SIDE, vt)[i] = fmaf(Ps[(16 * b + 4 * s + i) * 20 + j], v, sum_of(SIDE, vt)[i]);
        }
    }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      if constexpr (SIDE == 4) {
        o[b][vt] += apart[0][vt];
        apart[0][vt] = apart[1][vt] + apart[2][vt];
      }
      if (!TURNS) o[b][vt] += apart[0][vt];
      if (SIDE) o[b][vt] += apart[SIDE - 1][vt];
    }
    if (b == 0 && nt > 16) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const lrs_f32x4_t a = *reinterpret_cast<const lrs_f32x4_t*>(chunk_decay + 16 * dt + 4 * s);
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) S[dt][vt] *= a;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float k = Ks[(4 * s + j) * LD + 16 * dt + c];
#pragma unroll
          for (int vt = 0; vt < VT; ++vt) S[dt][vt] = __builtin_amdgcn_mfma_f32_16x16x4f32(k, vf[0][j][vt], S[dt][vt], 0, 0, 0);
        }
      }
    }
  }

  if (p.norm_w) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float ss = 0.0f;
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) ss += o[b][vt][i] * o[b][vt][i];
        ss = lrs_row_sum(ss);
        if (c == 0) squares[wave * LRS_MFMA_SEG + 16 * b + 4 * s + i] = ss;
      }
    __syncthreads();
  }
  T* out = (T*)p.out;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * b + 4 * s + i;
      if (t >= nt) continue;
      float inv = 1.0f;
      if (p.norm_w) {
        const float* sq = squares + t;
        inv = 1.0f / sqrtf(((sq[0] + sq[LRS_MFMA_SEG]) + (sq[2 * LRS_MFMA_SEG] + sq[3 * LRS_MFMA_SEG])) / (float)V + p.eps);
      }
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const int col = col0 + 16 * vt + c;
        if (col0 + 16 * vt >= V) continue;
        float val = o[b][vt][i] * inv * nw[vt];
        if (p.g_off >= 0) val *= gate[b][i][vt] / (1.0f + expf(-gate[b][i][vt]));
        out[(row0 + t) * (int64_t)(p.heads * V) + h * V + col] = cw_from_float<T>(val);
      }
    }
}

template <typename T, int D>
static void lrs_launch_mfma(const SegParams& p, int n_segments, dim3 carry_grid, hipStream_t stream) {
  const dim3 grid(n_segments, p.heads), block(256);
  const size_t staged = p.rank <= LRS_MAX_STAGED ? (size_t)LRS_MFMA_SEG * p.rank * sizeof(T) : 0;
#define LRS_VT(VT_)                                                                                  \
  do {                                                                                               \
    hipLaunchKernelGGL((lrs_added_kernel<T, D, VT_>), grid, block, staged, stream, p);                  \
    hipLaunchKernelGGL(lrs_carry_kernel, carry_grid, block, 0, stream, p);                           \
    hipLaunchKernelGGL((lrs_outputs_kernel<T, D, VT_>), grid, block, 0, stream, p);                  \
  } while (0)
  if (p.vdim <= 64) LRS_VT(1);
  else if (p.vdim <= 128) LRS_VT(2);
  else LRS_VT(4);
#undef LRS_VT
}

// dim a multiple of 4 up to 128
CW_EXPORT int cw_linear_recurrence_segments_supported(int dim, int vdim) {
  return dim > 0 && dim <= LRS_MAX_DIM && dim % 4 == 0 && vdim > 0 ? 1 : 0;
}

// Do the matrix cores take segments of up to seg_tokens tokens of these sizes whole?
static bool lrs_takes_mfma(int seg_tokens, int dim, int vdim) {
  return seg_tokens <= LRS_MFMA_SEG && (dim == 16 || dim == 32 || dim == 64 || dim == 128) && vdim % 16 == 0 && vdim <= 256;
}

// floats of workspace: dec [T, heads * dim], added [segments, heads, dim, vdim] and seg_decay [segments, heads, dim], and for
// the walks qf, kf [T, heads * dim] each and raw [T, heads * vdim]
CW_EXPORT int64_t cw_linear_recurrence_segments_workspace_floats(int n_tokens, int n_segments, int heads, int dim, int vdim, int seg_tokens) {
  const int64_t both = (int64_t)n_tokens * heads * dim + (int64_t)n_segments * heads * dim * (vdim + 1);
  return lrs_takes_mfma(seg_tokens, dim, vdim) ? both : both + (int64_t)n_tokens * heads * (2 * dim + vdim);
}

CW_EXPORT int cw_linear_recurrence_segments(int dtype, const void* proj, int64_t stride, int q_off, int k_off, int v_off,
                                            int g_off, int u_off, const void* a2, const float* a2b, const float* norm_w,
                                            float* state, int n_slots, const int* state_slots, const int* cu_q,
                                            const int* seg_items, int n_segments, int seg_tokens, const int* req_first, float* workspace,
                                            void* out, int n_requests, int n_tokens, int heads, int dim, int vdim, int rank,
                                            float q_scale, float inv_tau, float eps, int decay_kind, const float* bonus,
                                            int norm_w_stride, const void* u, int64_t u_stride, int64_t state_stride,
                                            hipStream_t stream) {
  if (n_requests < 0 || n_tokens < 0 || n_segments < 0 || !proj || !a2 || !state || !state_slots || !cu_q || !seg_items ||
      !req_first || !workspace || !out)
    return CW_ERR_ARG;
  if (heads <= 0 || rank <= 0 || n_slots <= 0 || q_off < 0 || k_off < 0 || v_off < 0 || u_off < 0 || stride <= 0) return CW_ERR_ARG;
  if (q_off % stride + heads * dim > stride || k_off % stride + heads * dim > stride || v_off % stride + heads * vdim > stride ||
      (!u && u_off + rank > stride) || (g_off >= 0 && g_off % stride + heads * vdim > stride))
    return CW_ERR_ARG;
  if (decay_kind < 0 || decay_kind > 2 || (norm_w_stride != 0 && norm_w_stride != vdim) || (u && u_stride < rank) ||
      state_stride < (int64_t)heads * dim * vdim || state_stride > 0x7fffffff)
    return CW_ERR_ARG;
  if (!cw_linear_recurrence_segments_supported(dim, vdim)) return CW_ERR_SIZE;
  if (heads > 65535 || (vdim + 63) / 64 > 65535) return CW_ERR_SIZE;
  if (seg_tokens < 1 || (int64_t)3 * seg_tokens * dim * 4 > 48 * 1024 || (bonus && seg_tokens > 64)) return CW_ERR_SIZE;
  if (n_requests == 0 || n_tokens == 0 || n_segments == 0) return CW_OK;
  SegParams p;
  p.proj = proj; p.stride = stride; p.q_off = q_off; p.k_off = k_off; p.v_off = v_off; p.g_off = g_off; p.u_off = u_off;
  p.a2 = a2; p.a2b = a2b; p.norm_w = norm_w; p.state = state; p.state_slots = state_slots; p.cu_q = cu_q;
  p.seg_items = seg_items; p.req_first = req_first; p.out = out;
  p.heads = heads; p.dim = dim; p.vdim = vdim; p.rank = rank; p.n_slots = n_slots; p.n_tokens = n_tokens;
  p.q_scale = q_scale; p.inv_tau = inv_tau; p.eps = eps;
  p.form = LinRecForm{decay_kind, bonus, norm_w_stride, u, u_stride, (int)state_stride};
  const int64_t THD = (int64_t)n_tokens * heads * dim;
  const bool mfma = lrs_takes_mfma(seg_tokens, dim, vdim);
  p.dec = workspace; p.added = p.dec + THD;
  p.seg_decay = p.added + (int64_t)n_segments * heads * dim * vdim;
  p.qf = mfma ? nullptr : p.seg_decay + (int64_t)n_segments * heads * dim;
  p.kf = mfma ? nullptr : p.qf + THD;
  p.raw = mfma ? nullptr : p.kf + THD;
  int64_t pb = (THD + 255) / 256;
  if (pb > 65536) pb = 65536;
  p.seg_tokens = seg_tokens;
  const int walk_threads = vdim >= 256 ? 256 : 64 * ((vdim + 63) / 64);   // up to four waves share a segment's rows
  const dim3 walk_grid(n_segments, heads, (vdim + walk_threads - 1) / walk_threads);
  const size_t walk_lds = (size_t)3 * seg_tokens * dim * sizeof(float);
  const dim3 carry_grid(n_requests, heads, (unsigned)(((int64_t)dim * vdim + 255) / 256));
  const unsigned finish_blocks = (unsigned)(((int64_t)n_tokens * heads + 3) / 4);
  if (mfma) {
#define CW_MFMA(T_)                                                                       \
  do {                                                                                    \
    if (dim == 16) lrs_launch_mfma<T_, 16>(p, n_segments, carry_grid, stream);            \
    else if (dim == 32) lrs_launch_mfma<T_, 32>(p, n_segments, carry_grid, stream);       \
    else if (dim == 64) lrs_launch_mfma<T_, 64>(p, n_segments, carry_grid, stream);       \
    else lrs_launch_mfma<T_, 128>(p, n_segments, carry_grid, stream);                     \
  } while (0)
    if (dtype == CW_F32) CW_MFMA(float);
    else if (dtype == CW_BF16) CW_MFMA(bf16_t);
    else return CW_ERR_DTYPE;
#undef CW_MFMA
    return cw_launch_status();
  }
#define CW_WALK(T_, DIM_)                                                                          \
  do {                                                                                             \
    hipLaunchKernelGGL((lrs_walk_kernel<T_, DIM_, 0>), walk_grid, dim3(walk_threads), walk_lds, stream, p); \
    hipLaunchKernelGGL(lrs_carry_kernel, carry_grid, dim3(256), 0, stream, p);                     \
    hipLaunchKernelGGL((lrs_walk_kernel<T_, DIM_, 1>), walk_grid, dim3(walk_threads), walk_lds, stream, p); \
  } while (0)
#define CW_ALL(T_)                                                                                 \
  do {                                                                                             \
    hipLaunchKernelGGL((lrs_prepare_kernel<T_>), dim3((unsigned)pb), dim3(256), 0, stream, p);     \
    if (dim <= 16) CW_WALK(T_, 16);                                                                \
    else if (dim <= 32) CW_WALK(T_, 32);                                                           \
    else if (dim <= 64) CW_WALK(T_, 64);                                                           \
    else CW_WALK(T_, 128);                                                                         \
    hipLaunchKernelGGL((lrs_finish_kernel<T_>), dim3(finish_blocks), dim3(256), 0, stream, p);     \
  } while (0)
  if (dtype == CW_F32) CW_ALL(float);
  else if (dtype == CW_BF16) CW_ALL(bf16_t);
  else return CW_ERR_DTYPE;
#undef CW_ALL
#undef CW_WALK
  return cw_launch_status();
}
