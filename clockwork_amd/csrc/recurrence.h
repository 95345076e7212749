// The recurrence of linear_recurrence.hip for a workgroup of 256 threads that takes four columns a thread: for the kernel there and
// for those that run it beside other work.
#pragma once
#include "common.h"

#define LR_TC 16  // tokens staged at a time

struct LinRecForm {
  int decay_kind;        // 0: sigmoid(z)^(1/tau); 1: exp(-exp(z)); 2: exp(-exp(z)) with tanh on the decay input
  const float* bonus;    // [heads, dim] or null
  int norm_w_stride;     // 0 or vdim
  const void* u;         // decay input rows, or null: columns u_off .. of proj
  int64_t u_stride;
  int state_stride;      // floats between two slots' states (>= heads * dim * vdim)
};

__device__ __forceinline__ float lr_decay(float z, int kind, float inv_tau) {
  if (kind >= 1) return expf(-expf(z));
  // log(sigmoid(z)) without cancellation, then the 1/tau-th power
  const float ls = fminf(z, 0.0f) - log1pf(expf(-fabsf(z)));
  return expf(ls * inv_tau);
}

struct LinRecParams {
  const void* proj;   // [T, stride]: a token's q (heads * dim at q_off), k (k_off), v (heads * vdim at v_off),
  int64_t stride;     //   gate (heads * vdim at g_off, or g_off < 0) and decay input u (rank at u_off)
  int q_off, k_off, v_off, g_off, u_off;
  const void* a2;     // [heads * dim, rank], type T
  const float* a2b;   // [heads * dim] or null
  const float* norm_w;  // [vdim] or null: no norm
  float* state;       // [slots, heads, dim, vdim]
  const int* state_slots;  // [R]
  const int* cu_q;    // [R + 1]
  void* out;          // [T, heads * vdim]
  int heads, dim, vdim, rank, n_slots;
  float q_scale, inv_tau, eps;
};

// For vdim = 4 * a power of two, request r and head h, 256 threads: a thread holds RPT rows of four neighbouring columns, which it reads in
// pieces of 16 bytes, and takes a quarter of the values from LDS that a thread of one column takes. Four lanes share a
// channel's decay. A step of single tokens is bound by its trips to memory, one after another (slot, state and
// operands, decay, output): the state, the first values, gates and norm weights are asked for before anything waits.
// 8 requests, 12 heads of 64 x 128, rank 32: 18.1 us with a column a thread, 8.2 so.
template <typename T, int RPT>
__device__ __forceinline__ void recurrence_quads(const LinRecParams& p, const LinRecForm& f, bool rank_quads, int r, int h) {
  extern __shared__ __align__(16) float smem[];
  const int D = p.dim, V = p.vdim, Hn = p.heads, VQ = V / 4;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int row0 = p.cu_q[r], q_len = p.cu_q[r + 1] - row0;
  const int slot = p.state_slots[r];
  if (q_len <= 0 || slot < 0 || slot >= p.n_slots) return;
  const int DS = min(256 / VQ, (D + RPT - 1) / RPT), DP = DS * RPT;  // row runs; rows with those that pad the last run
  const int c4 = (tid & (VQ - 1)) * 4, s = tid / VQ, d0 = s * RPT;
  const bool active = s < DS;

  float* qs = smem;                 // [TC][DP]
  float* ks = qs + LR_TC * DP;      // [TC][DP]
  float* as = ks + LR_TC * DP;      // [TC][DP] decays
  float* vs = as + LR_TC * DP;      // [TC][V]
  float* part = vs + LR_TC * V;     // [TC][4 waves][V]

  float S[RPT][4];
  float* st = p.state + (int64_t)slot * f.state_stride + ((int64_t)h * D) * V + c4;
#pragma unroll
  for (int rr = 0; rr < RPT; ++rr) {
    if (active && d0 + rr < D) CwVec<float, 4>::load(st + (int64_t)(d0 + rr) * V, S[rr]);
    else S[rr][0] = S[rr][1] = S[rr][2] = S[rr][3] = 0.0f;
  }
  const T* proj = (const T*)p.proj;
  const T* a2 = (const T*)p.a2;
  T* out = (T*)p.out;
  // the rows past dim: nothing ever joins them
  for (int idx = tid; idx < LR_TC * (DP - D); idx += 256) {
    const int at = idx / (DP - D) * DP + D + idx % (DP - D);
    qs[at] = ks[at] = as[at] = 0.0f;
  }
  for (int t0 = 0; t0 < q_len; t0 += LR_TC) {
    const int nt = min(LR_TC, q_len - t0);
    const T* rows = proj + (int64_t)(row0 + t0) * p.stride;
    // a wave's first token's gate and norm weight, and a thread's first value
    float gate[4], nw[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = lane + u * 64;
      gate[u] = p.g_off >= 0 && wave < nt && c < V ? cw_to_float(rows[(int64_t)wave * p.stride + p.g_off + h * V + c]) : 0.0f;
      nw[u] = p.norm_w && c < V ? p.norm_w[h * f.norm_w_stride + c] : 1.0f;
    }
    const float v_first = tid < nt * V ? cw_to_float(rows[(int64_t)(tid / V) * p.stride + p.v_off + h * V + tid % V]) : 0.0f;
    if (t0) __syncthreads();
    for (int idx = tid; idx < nt * D * 4; idx += 256) {
      const int piece = idx & 3, t = (idx >> 2) / D, d = (idx >> 2) - t * D;
      const T* row = rows + (int64_t)t * p.stride;
      const float qk = cw_to_float(row[(piece == 1 ? p.k_off : p.q_off) + h * D + d]);
      const float z0 = p.a2b ? p.a2b[h * D + d] : 0.0f;
      const T* w = a2 + (int64_t)(h * D + d) * p.rank;
      const T* u = f.u ? (const T*)f.u + (int64_t)(row0 + t0 + t) * f.u_stride : row + p.u_off;
      float z = 0.0f;
      if (rank_quads) {
        for (int c = piece * 4; c < p.rank; c += 16) {
          float we[4], ue[4];
          CwVec<T, 4>::load(w + c, we);
          CwVec<T, 4>::load(u + c, ue);
#pragma unroll
          for (int e = 0; e < 4; ++e) z += we[e] * (f.decay_kind == 2 ? tanhf(ue[e]) : ue[e]);
        }
      } else {
        for (int c = piece; c < p.rank; c += 4) {
          const float ue = cw_to_float(u[c]);
          z += cw_to_float(w[c]) * (f.decay_kind == 2 ? tanhf(ue) : ue);
        }
      }
      z += __shfl_xor(z, 1, 64);
      z += __shfl_xor(z, 2, 64);
      if (piece == 0) {
        qs[t * DP + d] = qk * p.q_scale;
        as[t * DP + d] = lr_decay(z0 + z, f.decay_kind, p.inv_tau);
      } else if (piece == 1) {
        ks[t * DP + d] = qk;
      }
    }
    if (tid < nt * V) vs[tid] = v_first;
    for (int idx = tid + 256; idx < nt * V; idx += 256) {
      const int t = idx / V, c = idx - t * V;
      vs[idx] = cw_to_float(rows[(int64_t)t * p.stride + p.v_off + h * V + c]);
    }
    cw_lds_barrier();
    for (int t = 0; t < nt; ++t) {
      float po[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (active) {
        float vv[4];
        CwVec<float, 4>::load(vs + t * V + c4, vv);
#pragma unroll
        for (int rr = 0; rr < RPT; ++rr) {
          const float k = ks[t * DP + d0 + rr], a = as[t * DP + d0 + rr], q = qs[t * DP + d0 + rr];
          const float bonus = f.bonus && d0 + rr < D ? f.bonus[h * D + d0 + rr] : 0.0f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // (nothing for a row past dim, also where the value is infinite)
            const float kv = d0 + rr < D ? k * vv[e] : 0.0f;
            if (f.bonus) po[e] += q * (S[rr][e] + bonus * kv);
            S[rr][e] = a * S[rr][e] + kv;
            if (!f.bonus) po[e] += q * S[rr][e];
          }
        }
      }
      for (int off = VQ; off < 64; off <<= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) po[e] += __shfl_xor(po[e], off, 64);
      if (lane < VQ) CwVec<float, 4>::store(part + (t * 4 + wave) * V + c4, po);
    }
    cw_lds_barrier();
    // a wave per token: sum the partial outputs, norm over vdim, gate, store
    for (int t = wave; t < nt; t += 4) {
      float o[4], ss = 0.0f;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = lane + u * 64;
        const float* po = part + t * 4 * V + c;
        o[u] = c < V ? (po[0] + po[V]) + (po[2 * V] + po[3 * V]) : 0.0f;
        ss += o[u] * o[u];
      }
      const float inv = p.norm_w ? 1.0f / sqrtf(cw_wave_sum(ss) / (float)V + p.eps) : 1.0f;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = lane + u * 64;
        if (c < V) {
          float val = o[u] * inv * nw[u];
          if (p.g_off >= 0) {
            const float g = t == wave ? gate[u] : cw_to_float(rows[(int64_t)t * p.stride + p.g_off + h * V + c]);
            val *= g / (1.0f + expf(-g));
          }
          out[(int64_t)(row0 + t0 + t) * (int64_t)(Hn * V) + h * V + c] = cw_from_float<T>(val);
        }
      }
    }
  }
  if (active) {
#pragma unroll
    for (int rr = 0; rr < RPT; ++rr)
      if (d0 + rr < D) CwVec<float, 4>::store(st + (int64_t)(d0 + rr) * V, S[rr]);
  }
}

// A launch of the recurrence as cw_linear_recurrence_prepare leaves it for a kernel that runs it beside other work: a workgroup of
// 256 threads and ``lds`` bytes a (request, head).
struct RecurrenceLaunch {
  LinRecParams p;
  LinRecForm f;
  int64_t lds;
  int dtype, requests, rows, rank_quads;
};
