// One decode step of the recurrences with a matrix state per head, as a part of a launch: the launches of recurrent_step.hip, and attn_paged.hip's
// where a layer has both.
#pragma once

#include "common.h"
#include "typed.h"
#include "sigmoid_power.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

constexpr int kStepDim = 128;      // most key channels and values of a head
constexpr int kStepThreads = 512;
constexpr int kStepRows = 8;       // rows of S per thread
constexpr int kStepWaves = kStepThreads / 64;

// the channel's row of a second-stage matrix times the projected row's low-rank values: four neighbouring threads share it, `part` of four
template <typename A>
__device__ __forceinline__ float step_up(const A* w, const A* low, int rank, int rank_stride, int part) {
  float sum = 0.f;
#pragma unroll 2
  for (int c = part * 8; c < rank_stride; c += 32) {
    float wv[8], lv[8];
    Vec8<A>::load(w + c, wv);
    Vec8<A>::load(low + c, lv);
#pragma unroll
    for (int u = 0; u < 8; ++u) sum = fmaf(wv[u], c + u < rank ? lv[u] : 0.f, sum);
  }
  sum += __shfl_xor(sum, 1, kWave);
  return sum + __shfl_xor(sum, 2, kWave);
}

// a workgroup of kStepThreads: head h of entry e
template <typename A, typename Q, int KIND>
__device__ __forceinline__ void recurrent_step_block(const pegainfer_recurrent_step_desc& p, int h, int e) {
  constexpr bool kDelta = KIND != PEGAINFER_STEP_GATED, kChannel = KIND != PEGAINFER_STEP_DELTA;
  __shared__ float s_q[kStepDim], s_k[kStepDim], s_a[kStepDim], s_gate[kStepDim], s_ss[4], s_one[2], s_norm[2];
  __shared__ __attribute__((aligned(16))) float s_sk[kDelta ? kStepWaves : 1][kStepDim], s_sq[kStepWaves][kStepDim];
  __shared__ float s_kq[kStepWaves];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int H = p.heads, dim = p.dim, vdim = p.vdim, g0 = h / (H / p.kv_heads);
  const Q* x = static_cast<const Q*>(p.qkv) + (int64_t)e * p.qkv_stride;
  const A* pr = static_cast<const A*>(p.proj) + (int64_t)e * p.proj_stride;
  float* S_g = p.state + (int64_t)p.entry_slot[e] * p.slot_stride + (int64_t)h * dim * vdim;
  const int col = (tid & 31) * 4, r0 = tid >> 5;
  const bool live = col < vdim;
  float S[kStepRows][4], v[4] = {};
#pragma unroll
  for (int j = 0; j < kStepRows; ++j) {
    const int d = r0 + 16 * j;
    if (live && d < dim) ld4(S_g + (int64_t)d * vdim + col, S[j]);
    else {
#pragma unroll
      for (int u = 0; u < 4; ++u) S[j][u] = 0.f;
    }
  }
  if (live) ld4(x + p.v_off + (int64_t)h * vdim + col, v);
  // ---- the row: q and k, decays, the output's gate
  if (tid < 2 * kStepDim) {
    const int d = tid & (kStepDim - 1);
    const bool is_k = tid >= kStepDim;
    const float t = d < dim ? ld(x + (is_k ? p.k_off : p.q_off) + (int64_t)g0 * dim + d) : 0.f;
    (is_k ? s_k : s_q)[d] = t;
    if constexpr (kDelta) {
      const float ss = wave_sum(t * t);
      if (lane == 0) s_ss[wave] = ss;
    }
  }
  const int ch = tid >> 2, part = tid & 3;
  if constexpr (kChannel) {
    const int d = min(ch, dim - 1);
    const float z = p.w_up ? step_up(static_cast<const A*>(p.w_up) + ((int64_t)h * dim + d) * p.rank_stride, pr + p.low_off, p.rank, p.rank_stride, part)
                           : p.z[(int64_t)e * p.z_stride + (int64_t)h * dim + d];
    if (part == 0 && ch < dim) {
      const A* bias = static_cast<const A*>(p.z_bias);
      const float zb = z + (bias ? ld(bias + (int64_t)h * dim + d) : 0.f);
      if constexpr (kDelta) s_a[d] = expf(-expf(ld(static_cast<const A*>(p.A_log) + h)) * softplus_f(zb));
      else s_a[d] = sigmoid_power(zb, 1.0f / p.tau);
    }
  }
  {
    const int c = min(ch, vdim - 1);
    const float z = p.w_gate ? step_up(static_cast<const A*>(p.w_gate) + ((int64_t)h * vdim + c) * p.gate_rank_stride, pr + p.gate_low_off, p.gate_rank,
                                       p.gate_rank_stride, part)
                             : ld(static_cast<const A*>(p.gate) + (int64_t)e * p.gate_stride + (int64_t)h * vdim + c);
    if (part == 0 && ch < vdim) {
      A t;
      st(&t, z);                 // (a second stage's result is a stored value)
      const float zs = ld(&t);
      s_gate[c] = p.gate_kind == 0 ? silu_f(zs) : sigmoid_f(zs);
    }
  }
  if constexpr (kDelta) {
    if (tid == kStepThreads - 1) {
      s_one[0] = sigmoid_f(ld(pr + p.b_off + h));
      if constexpr (!kChannel)
        s_one[1] = expf(-expf(ld(static_cast<const A*>(p.A_log) + h)) * softplus_f(ld(pr + p.a_off + h) + ld(static_cast<const A*>(p.z_bias) + h)));
    }
  }
  const float wn = tid < vdim ? ld(static_cast<const A*>(p.norm_w) + tid) : 0.f;
  __syncthreads();
  // ---- the state
  float sk[4] = {}, sq[4] = {}, kq = 0.f, u[4];
  float sc_k = 1.f, sc_q = p.q_scale, beta = 0.f;
  if constexpr (kDelta) {
    sc_q = 1.0f / (sqrtf((float)dim) * sqrtf(s_ss[0] + s_ss[1] + 1e-6f));
    sc_k = 1.0f / sqrtf(s_ss[2] + s_ss[3] + 1e-6f);
    beta = s_one[0];
  }
#pragma unroll
  for (int j = 0; j < kStepRows; ++j) {
    const int d = r0 + 16 * j;
    if (d >= dim) continue;
    const float a = kChannel ? s_a[d] : s_one[1], kk = s_k[d] * sc_k, qq = s_q[d] * sc_q;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (kDelta) {
        S[j][c] *= a;
        sk[c] = fmaf(S[j][c], kk, sk[c]);
      } else {
        S[j][c] = fmaf(v[c], kk, a * S[j][c]);
      }
      sq[c] = fmaf(S[j][c], qq, sq[c]);
    }
    kq = fmaf(kk, qq, kq);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    sq[c] += __shfl_xor(sq[c], 32, kWave);
    if constexpr (kDelta) sk[c] += __shfl_xor(sk[c], 32, kWave);
  }
  if (lane < 32) {
    *reinterpret_cast<f32x4*>(&s_sq[wave][col]) = f32x4{sq[0], sq[1], sq[2], sq[3]};
    if constexpr (kDelta) *reinterpret_cast<f32x4*>(&s_sk[wave][col]) = f32x4{sk[0], sk[1], sk[2], sk[3]};
  }
  if constexpr (kDelta) {
    kq += __shfl_xor(kq, 32, kWave);
    if (lane == 0) s_kq[wave] = kq;
  }
  __syncthreads();
  if constexpr (kDelta) {
    float t[4] = {};
#pragma unroll
    for (int w = 0; w < kStepWaves; ++w) {
      const f32x4 part4 = *reinterpret_cast<const f32x4*>(&s_sk[w][col]);
#pragma unroll
      for (int c = 0; c < 4; ++c) t[c] += part4[c];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) u[c] = beta * (v[c] - t[c]);
  }
#pragma unroll
  for (int j = 0; j < kStepRows; ++j) {
    const int d = r0 + 16 * j;
    if (!live || d >= dim) continue;
    if constexpr (kDelta) {
      const float kk = s_k[d] * sc_k;
#pragma unroll
      for (int c = 0; c < 4; ++c) S[j][c] = fmaf(kk, u[c], S[j][c]);
    }
    st4(S_g + (int64_t)d * vdim + col, S[j]);
  }
  // ---- the read-out, a thread per value, normed over the head and gated
  float y = 0.f;
  if (tid < vdim) {
#pragma unroll
    for (int w = 0; w < kStepWaves; ++w) y += s_sq[w][tid];
    if constexpr (kDelta) {
      float t = 0.f, dot = 0.f;
#pragma unroll
      for (int w = 0; w < kStepWaves; ++w) {
        t += s_sk[w][tid];
        dot += s_kq[w];
      }
      y = fmaf(dot, beta * (ld(x + p.v_off + (int64_t)h * vdim + tid) - t), y);
    }
  }
  if (wave < 2) {
    const float ss = wave_sum(y * y);
    if (lane == 0) s_norm[wave] = ss;
  }
  __syncthreads();
  if (tid >= vdim) return;
  const float inv = 1.0f / sqrtf((s_norm[0] + s_norm[1]) / (float)vdim + p.eps);
  st(static_cast<A*>(p.out) + (int64_t)e * p.out_stride + (int64_t)h * vdim + tid, y * inv * wn * s_gate[tid] * p.factor);
}

// which steps these blocks take
inline bool recurrent_step_up_ok(const void* w, int32_t rank, int32_t rank_stride, const void* proj, int64_t proj_stride, int64_t low_off) {
  return w && rank > 0 && rank <= rank_stride && rank_stride % 8 == 0 && proj_stride % 8 == 0 && low_off % 8 == 0 && low_off + rank_stride <= proj_stride &&
         host_aligned16(w) && host_aligned16(proj);
}
inline bool recurrent_step_ok(const pegainfer_recurrent_step_desc* q) {
  if (!q || q->kind < 0 || q->kind > PEGAINFER_STEP_DELTA_CHANNEL) return false;
  const bool channel = q->kind != PEGAINFER_STEP_DELTA, delta = q->kind != PEGAINFER_STEP_GATED;
  return q->heads > 0 && q->kv_heads > 0 && q->heads % q->kv_heads == 0 && q->dim > 0 && q->dim <= kStepDim && q->vdim > 0 && q->vdim <= kStepDim &&
         q->vdim % 4 == 0 && q->n_entries >= 0 && q->n_entries <= 65535 && q->qkv && q->state && q->entry_slot && q->norm_w && q->out &&
         (q->gate || q->w_gate) && (delta || q->tau > 0.f) && (!channel || q->z || q->w_up) && (!delta || (q->A_log && q->proj && q->z_bias)) &&
         ((!q->w_up && !q->w_gate) || q->proj) &&
         (!channel || !q->w_up || recurrent_step_up_ok(q->w_up, q->rank, q->rank_stride, q->proj, q->proj_stride, q->low_off)) &&
         (!q->w_gate || recurrent_step_up_ok(q->w_gate, q->gate_rank, q->gate_rank_stride, q->proj, q->proj_stride, q->gate_low_off)) &&
         host_aligned16(q->qkv) && host_aligned16(q->state) && q->slot_stride % 4 == 0 && q->qkv_stride % 4 == 0 && q->v_off % 4 == 0;
}

}  // namespace pk
