// Recurrent matrix memories over ragged batches, fp32 state and fp32 arithmetic throughout.
//
// Both recurrences share one shape.  A workgroup of four waves owns 16 value columns of one (entry, head); a column's state
// S[:, col] is spread over the sixteen lanes of a DPP row (lane = 16 * column + r holds the NS consecutive rows
// d = r * NS + i), so a token costs each lane dim / 16 multiply-adds per product and a four-step DPP sum inside the row:
// the recurrence is a chain of dependent steps, so the work of one step is spread as wide as the wave allows and many small
// workgroups fill the chip.  The state stays in registers from the entry's first row to its last and touches HBM once on
// either side.  The tokens' keys, queries, values and gate values are staged 16 tokens at a time through LDS: the next round's
// global loads are issued before the current round is consumed and land in LDS after it.  Everything that does not depend on
// the state is computed before or beside the chain, once per token: unit vectors and gates of the delta rule by a prep
// launch over all rows, the matrix memory's running maximum by one lane per round and its three exponentials by sixteen.
// A round's sixteen outputs of a column leave in one store per lane.
//   delta_rule_kernel      S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q      (long entries with one decay per head: delta_chunk.hip)
//   matrix_memory_kernel   m' = max(f + m, i);  S <- e^(f + m - m') S + e^(i - m') k v^T;  n likewise;  o = S^T q / (max(|n.q|, e^-m') + 1e-6)
// A row's result depends only on the rows before it in its own request: the token order is fixed, and cutting a prompt into
// steps only moves where the state passes through HBM (exactly, it is fp32 either way).  The matrix memory (below) and the delta rule with one
// decay per head (delta_chunk.hip) also have a form in chunks for long portions; a portion's own length says which it takes, and that moves
// results by rounding only.
#include <algorithm>

#include "common.h"
#include "typed.h"
#include "delta_scan.h"
#include "head_rms_core.h"
#include "qk_prep_core.h"
#include "recurrent_core.h"
#include "scalar_chunks.h"
#include "sigmoid_power.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

__device__ __forceinline__ float logsigmoid_f(float x) { return fminf(x, 0.0f) - log1pf(expf(-fabsf(x))); }

template <typename A>
__global__ __launch_bounds__(256) void delta_prep_kernel(float* __restrict__ qkv, int64_t qkv_stride, const A* __restrict__ proj,
                                                         int64_t proj_stride, int64_t b_off, int64_t a_off,
                                                         const A* __restrict__ A_log, const A* __restrict__ dt_bias,
                                                         float* __restrict__ gates, int H, int G, int dim) {
  delta_prep_row<A>(blockIdx.x, blockIdx.y, gridDim.y, qkv, qkv_stride, proj, proj_stride, b_off, a_off, A_log, dt_bias, gates, H, G, dim);
}

// What delta_prep_row does for a decay per (head, key channel): gates[row] = [g: heads * dim | beta: heads], the decay inputs come as an fp32
// matrix `a` ([rows][heads * dim] at stride a_stride: the output of a low-rank projection pair), dt_bias has heads * dim values.
template <typename A>
__global__ __launch_bounds__(256) void delta_prep_channel_kernel(float* __restrict__ qkv, int64_t qkv_stride,
                                                                 const A* __restrict__ proj, int64_t proj_stride, int64_t b_off,
                                                                 const float* __restrict__ a, int64_t a_stride,
                                                                 const A* __restrict__ A_log, const A* __restrict__ dt_bias,
                                                                 float* __restrict__ gates, int H, int G, int dim) {
  const int row = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float* qk = qkv + (int64_t)row * qkv_stride;
  const float qs = 1.0f / sqrtf((float)dim);
  for (int hh = blockIdx.y * 4 + wave; hh < 2 * G; hh += 4 * gridDim.y) {
    float* x = qk + (int64_t)hh * dim;
    float ss = 0.f;
    for (int d = lane; d < dim; d += 64) ss = fmaf(x[d], x[d], ss);
    const float sc = (hh < G ? qs : 1.0f) / sqrtf(wave_sum(ss) + 1e-6f);
    for (int d = lane; d < dim; d += 64) x[d] *= sc;
  }
  const A* pr = proj + (int64_t)row * proj_stride;
  float* gr = gates + (int64_t)row * ((int64_t)H * dim + H);
  for (int i = blockIdx.y * 256 + threadIdx.x; i < H * dim; i += 256 * gridDim.y)
    gr[i] = expf(-expf(ld(A_log + i / dim)) * softplus_f(a[(int64_t)row * a_stride + i] + ld(dt_bias + i)));
  for (int h = blockIdx.y * 256 + threadIdx.x; h < H; h += 256 * gridDim.y) gr[(int64_t)H * dim + h] = sigmoid_f(ld(pr + b_off + h));
}

template <int NS, bool CH>
__global__ __launch_bounds__(256) void delta_rule_kernel(const float* __restrict__ qkv, int64_t qkv_stride,
                                                         const float* __restrict__ gates, float* __restrict__ state,
                                                         int64_t slot_stride, float* __restrict__ o, int H, int G, int dim,
                                                         int vdim, const int32_t* __restrict__ entry_row0,
                                                         const int32_t* __restrict__ entry_slot) {
  delta_rule_block<NS, CH>(blockIdx.x, blockIdx.y, blockIdx.z, qkv, qkv_stride, gates, state, slot_stride, o, H, G, dim, vdim, entry_row0, entry_slot);
}

// a token's log input and forget gate
template <typename A>
struct MemoryGates {
  const A* proj; int64_t proj_stride, i_off, f_off;
  float ib, fb, cap;
  int h;
  __device__ __forceinline__ float in(int64_t row) const { return cap * tanhf((ld(proj + row * proj_stride + i_off + h) + ib) / cap); }
  __device__ __forceinline__ float forget(int64_t row) const { return logsigmoid_f(cap * tanhf((ld(proj + row * proj_stride + f_off + h) + fb) / cap)); }
};

// A round's tc tokens, their gates in s_i / s_f: the running maxima s_m[1 ..] from s_m[0], then every token's factors (rows past tc leave S and
// n as they are).  Ends behind a barrier; s_m[0] is the round's last maximum.
__device__ __forceinline__ void memory_round(int tid, int tc, const float* s_i, const float* s_f, float* s_m, float* s_a, float* s_b, float* s_em) {
  if (tid == 0) {                 // the running maximum is a chain of one add and one max per token: one lane walks it
    float mm = s_m[0];
    for (int tt = 0; tt < tc; ++tt) {
      mm = fmaxf(s_f[tt] + mm, s_i[tt]);
      s_m[tt + 1] = mm;
    }
  }
  __syncthreads();
  if (tid < kRecTokens) {         // ... and the exponentials it feeds are computed side by side
    const bool live = tid < tc;   // rows past the entry's end: a = 1, b = 0 - a step that leaves S and n as they are
    const float mp = live ? s_m[tid] : 0.f, mn = live ? s_m[tid + 1] : 0.f;
    s_a[tid] = live ? expf(s_f[tid] + mp - mn) : 1.f;
    s_b[tid] = live ? expf(s_i[tid] - mn) : 0.f;
    s_em[tid] = live ? expf(-mn) : 1.f;
  }
  __syncthreads();
  if (tid == 0) s_m[0] = s_m[tc];
}

// n and the running maximum of an (entry, head) are read by every workgroup of the scan below that owns columns of it, so none of these may
// write them: where there are several, this launch behind the scan moves both on, by the same steps (a thread per value of n).
template <typename A>
__global__ __launch_bounds__(256) void memory_carry_kernel(const A* __restrict__ proj, int64_t proj_stride, int64_t k_off, int64_t i_off,
                                                           int64_t f_off, const A* __restrict__ i_bias, const A* __restrict__ f_bias, float cap,
                                                           float* __restrict__ state, int64_t slot_stride, int H, int dim, int vdim,
                                                           const int32_t* __restrict__ entry_row0, const int32_t* __restrict__ entry_slot,
                                                           int scan_max) {
  __shared__ float s_i[kRecTokens], s_f[kRecTokens], s_m[kRecTokens + 1], s_a[kRecTokens], s_b[kRecTokens], s_em[kRecTokens];
  const int e = blockIdx.y, h = blockIdx.x, tid = threadIdx.x;
  const int row0 = entry_row0[e], len = entry_row0[e + 1] - row0;
  if (scan_max > 0 && len > scan_max) return;      // the chunk form has this entry
  float* base = state + (int64_t)entry_slot[e] * slot_stride + (int64_t)H * dim * vdim;
  float *n_g = base + (int64_t)h * dim, *m_g = base + (int64_t)H * dim + h;
  const MemoryGates<A> gate{proj, proj_stride, i_off, f_off, ld(i_bias + h), ld(f_bias + h), cap, h};
  const int d = min(tid, dim - 1);
  float n = n_g[d];
  if (tid == 0) s_m[0] = *m_g;
  for (int t0 = 0; t0 < len; t0 += kRecTokens) {
    const int tc = min(kRecTokens, len - t0);
    float kk[kRecTokens];
#pragma unroll
    for (int t = 0; t < kRecTokens; ++t) kk[t] = ld(proj + (int64_t)(row0 + t0 + min(t, tc - 1)) * proj_stride + k_off + (int64_t)h * dim + d);
    __syncthreads();
    if (tid < tc) {
      s_i[tid] = gate.in(row0 + t0 + tid);
      s_f[tid] = gate.forget(row0 + t0 + tid);
    }
    __syncthreads();
    memory_round(tid, tc, s_i, s_f, s_m, s_a, s_b, s_em);
#pragma unroll
    for (int t = 0; t < kRecTokens; ++t)
      if (t < tc) n = fmaf(s_b[t], kk[t], s_a[t] * n);
  }
  __syncthreads();
  if (tid < dim) n_g[tid] = n;
  if (tid == 0) *m_g = s_m[0];
}

// of 256 threads: columns bx of nbx runs of sixteen, head h, entry e
template <int NS, typename A>
__device__ __forceinline__ void matrix_memory_block(int bx, int nbx, int h, int e, const A* __restrict__ proj, int64_t proj_stride, int64_t q_off,
                                                            int64_t k_off, int64_t v_off, int64_t i_off, int64_t f_off,
                                                            const A* __restrict__ i_bias, const A* __restrict__ f_bias,
                                                            float cap, float* __restrict__ state, int64_t slot_stride,
                                                            float* __restrict__ o, int H, int dim, int vdim,
                                                            const int32_t* __restrict__ entry_row0,
                                                            const int32_t* __restrict__ entry_slot, int scan_max) {
  constexpr int DP = kRecSlices * NS;
  __shared__ __attribute__((aligned(16))) float s_k[kRecTokens][DP], s_q[kRecTokens][DP];
  __shared__ float s_v[kRecTokens][kRecCols], s_i[kRecTokens], s_f[kRecTokens], s_m[kRecTokens + 1], s_a[kRecTokens],
      s_b[kRecTokens], s_em[kRecTokens];
  const int col0 = bx * kRecCols;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, cl = wave * 4 + (lane >> 4);
  const int col = col0 + cl;
  const int row0 = entry_row0[e], len = entry_row0[e + 1] - row0;
  if (scan_max > 0 && len > scan_max) return;      // the chunk form has this entry
  float* base = state + (int64_t)entry_slot[e] * slot_stride;
  float* S_g = base + (int64_t)h * dim * vdim;
  float* n_g = base + (int64_t)H * dim * vdim + (int64_t)h * dim;
  float* m_g = base + (int64_t)H * dim * vdim + (int64_t)H * dim + h;
  float S[NS], n[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int d = r * NS + i;
    S[i] = d < dim && col < vdim ? S_g[(int64_t)d * vdim + col] : 0.f;
    n[i] = d < dim ? n_g[d] : 0.f;
  }
  if (tid == 0) s_m[0] = *m_g;     // s_m[0] = the maximum before the round, s_m[t + 1] = after its token t
  const MemoryGates<A> gate{proj, proj_stride, i_off, f_off, ld(i_bias + h), ld(f_bias + h), cap, h};
  const float qs = 1.0f / sqrtf((float)dim);
  RoundFetch<NS> nxt;
  auto fetch = [&](int t0) {
    const A* base = proj + (int64_t)(row0 + t0) * proj_stride;
    nxt.issue(min(kRecTokens, len - t0), tid, dim,
              [=](int tt, int d) { return ld(base + (int64_t)tt * proj_stride + q_off + (int64_t)h * dim + d) * qs; },
              [=](int tt, int d) { return ld(base + (int64_t)tt * proj_stride + k_off + (int64_t)h * dim + d); },
              [=](int tt, int c) { return col0 + c < vdim ? ld(base + (int64_t)tt * proj_stride + v_off + (int64_t)h * vdim + col0 + c) : 0.f; });
  };
  fetch(0);
  for (int t0 = 0; t0 < len; t0 += kRecTokens) {
    const int tc = min(kRecTokens, len - t0);
    __syncthreads();
    nxt.land(tid, s_q, s_k, s_v);
    if (tid < tc) {
      s_i[tid] = gate.in(row0 + t0 + tid);
      s_f[tid] = gate.forget(row0 + t0 + tid);
    }
    __syncthreads();
    if (t0 + kRecTokens < len) fetch(t0 + kRecTokens);
    memory_round(tid, tc, s_i, s_f, s_m, s_a, s_b, s_em);
    float okeep = 0.f;
    // no token waits for the sums of the one before it here (only S and n carry over): four tokens per trip, their sums and
    // quotients in flight together
    for (int t4 = 0; t4 < tc; t4 += 4) {
#pragma unroll
     for (int uu = 0; uu < 4; ++uu) {
      const int tt = t4 + uu;
      const float a = s_a[tt], b = s_b[tt];
      const float bv = b * s_v[tt][cl];
      float num0 = 0.f, num1 = 0.f, nq0 = 0.f, nq1 = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const float kk = s_k[tt][r * NS + i], qq = s_q[tt][r * NS + i];
        S[i] = fmaf(bv, kk, a * S[i]);
        n[i] = fmaf(b, kk, a * n[i]);
        if (i & 1) { num1 = fmaf(S[i], qq, num1); nq1 = fmaf(n[i], qq, nq1); }
        else { num0 = fmaf(S[i], qq, num0); nq0 = fmaf(n[i], qq, nq0); }
      }
      const float num = row16_sum(num0 + num1), nq = row16_sum(nq0 + nq1);
      const float den = fmaxf(fabsf(nq), s_em[tt]) + 1e-6f;
      okeep = tt == r ? num / den : okeep;
     }
    }
    if (r < tc && col < vdim) o[(int64_t)(row0 + t0 + r) * ((int64_t)H * vdim) + (int64_t)h * vdim + col] = okeep;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int d = r * NS + i;
    if (d < dim && col < vdim) S_g[(int64_t)d * vdim + col] = S[i];
    if (nbx == 1 && tid < kRecSlices && d < dim) n_g[d] = n[i];
  }
  if (nbx == 1 && tid == 0) *m_g = s_m[0];   // (several workgroups read both: memory_carry_kernel writes them afterwards)
}
template <int NS, typename A>
__global__ __launch_bounds__(256) void matrix_memory_kernel(const A* __restrict__ proj, int64_t proj_stride, int64_t q_off,
                                                            int64_t k_off, int64_t v_off, int64_t i_off, int64_t f_off,
                                                            const A* __restrict__ i_bias, const A* __restrict__ f_bias,
                                                            float cap, float* __restrict__ state, int64_t slot_stride,
                                                            float* __restrict__ o, int H, int dim, int vdim,
                                                            const int32_t* __restrict__ entry_row0,
                                                            const int32_t* __restrict__ entry_slot, int scan_max) {
  matrix_memory_block<NS, A>(blockIdx.x, gridDim.x, blockIdx.y, blockIdx.z, proj, proj_stride, q_off, k_off, v_off, i_off, f_off, i_bias, f_bias, cap, state,
                             slot_stride, o, H, dim, vdim, entry_row0, entry_slot, scan_max);
}

// Decoding, a layer with an attention beside the memory: the scan and the preparation of the attention's rows, which write nothing that the other
// reads, in one grid (the scan's workgroups first), and behind the attention one launch for all that is left: the memory's n and maximum, the
// norm and gate of its read-out, the factor on the attention's rows.  One row, 16 heads over 4 of 256 beside 8 heads of 128 x 256:
// 5.1 + 8.6 and 4.8 + 4.8 + 3.9 us in launches of their own, 9.4 and 4.5 here.
template <int NS>
__global__ __launch_bounds__(256) void memory_beside_kernel(pegainfer_gated_matrix_memory_desc m, int nbx, int n_scan, pegainfer_qk_prep_desc p, PrepForm pf,
                                                            int per_row) {
  extern __shared__ float sm[];
  const int b = blockIdx.x;
  if (b < n_scan) {
    matrix_memory_block<NS, uint16_t>(b % nbx, nbx, b / nbx % m.heads, b / (nbx * m.heads), static_cast<const uint16_t*>(m.proj), m.proj_stride, m.q_off,
                                      m.k_off, m.v_off, m.i_off, m.f_off, static_cast<const uint16_t*>(m.i_bias),
                                      static_cast<const uint16_t*>(m.f_bias), m.cap, m.state, m.slot_stride, m.o, m.heads, m.dim, m.vdim, m.entry_row0,
                                      m.entry_slot, 0);
    return;
  }
  qk_prep_block<uint16_t, uint16_t, 2>(sm, (b - n_scan) / per_row, (b - n_scan) % per_row, per_row, p, pf);
}

// grid (heads + workgroups for the rows to scale, entries).  A head's workgroup: the first wave norms, the others move n on.
template <typename A, int V>
__global__ __launch_bounds__(256) void memory_finish_kernel(pegainfer_gated_matrix_memory_desc m, pegainfer_memory_finish_desc f) {
  const int e = blockIdx.y, h = blockIdx.x, tid = threadIdx.x, row = m.entry_row0[e];
  if (h >= m.heads) {
    const A* in = static_cast<const A*>(f.rows) + (int64_t)row * f.rows_stride;
    A* out = static_cast<A*>(f.scaled) + (int64_t)row * f.scaled_stride;
    for (int i = (h - m.heads) * 256 + tid; i < f.scale_cols; i += (gridDim.x - m.heads) * 256) st(out + i, ld(in + i) * f.scale);
    return;
  }
  if (tid < kWave) {
    head_rms_gate_wave<A, V>(row, h, m.o, static_cast<const A*>(f.norm_w), 1, static_cast<const A*>(f.gate), f.gate_stride, f.gate_kind, f.factor, f.eps,
                             static_cast<A*>(f.out), f.out_stride, m.heads, m.vdim, 0);
    return;
  }
  if (m.vdim <= kRecCols) return;                  // one workgroup per head has scanned: it has moved them on itself
  const A* proj = static_cast<const A*>(m.proj);
  float* base = m.state + (int64_t)m.entry_slot[e] * m.slot_stride + (int64_t)m.heads * m.dim * m.vdim;
  float *n_g = base + (int64_t)h * m.dim, *m_g = base + (int64_t)m.heads * m.dim + h;
  const MemoryGates<A> gate{proj, m.proj_stride, m.i_off, m.f_off, ld(static_cast<const A*>(m.i_bias) + h), ld(static_cast<const A*>(m.f_bias) + h), m.cap, h};
  const float gi = gate.in(row), gf = gate.forget(row), mp = *m_g, mn = fmaxf(gf + mp, gi), a = expf(gf + mp - mn), b = expf(gi - mn);
  for (int d = tid - kWave; d < m.dim; d += 256 - kWave)
    n_g[d] = fmaf(b, ld(proj + (int64_t)row * m.proj_stride + m.k_off + (int64_t)h * m.dim + d), a * n_g[d]);
  __syncthreads();                                 // the three waves that are left have read the maximum
  if (tid == kWave) *m_g = mn;
}

// ---- the matrix memory over long portions (scalar_chunks.h): with the running maxima known, the decays exp(f + m - m') and the factors
// exp(i - m') are numbers per head and token like any others.  1024 tokens, 8 heads of 128 x 256: the scan 468 us, gates 23, sums 14, walk 12 and
// outputs 39 us here; 4096 tokens 1851 and 311 us.
template <typename A>
struct MemIn {
  const A* proj; int64_t proj_stride, q_off, k_off, v_off;
  const float* gates;            // [chunk][head][decays | factors | floors of the norm][64]
  int H, dim, vdim;
  typedef A Row;
  static constexpr bool kNorm = true;
  __device__ __forceinline__ const A* rows() const { return proj; }
  __device__ __forceinline__ int64_t row_stride() const { return proj_stride; }
  __device__ __forceinline__ int64_t q_at(int h) const { return q_off + (int64_t)h * dim; }
  __device__ __forceinline__ int64_t k_at(int h) const { return k_off + (int64_t)h * dim; }
  __device__ __forceinline__ int64_t v_at(int h) const { return v_off + (int64_t)h * vdim; }
  __device__ __forceinline__ float q_factor() const { return 1.0f / sqrtf((float)dim); }
  __device__ __forceinline__ const float* gate(int c, int h, int k) const { return gates + (((int64_t)c * H + h) * 3 + k) * kDecayChunk; }
  __device__ __forceinline__ void steps(int c, int h, int, int, int lane, float* b, float* a) const {
    *a = gate(c, h, 0)[lane];
    *b = gate(c, h, 1)[lane];
  }
  __device__ __forceinline__ float floor_of(int c, int h, int i) const { return gate(c, h, 2)[i]; }
  __device__ __forceinline__ float skip(int) const { return 0.f; }
};

// One wave per (long entry, head) walks the entry's chunks: the running maximum m' = max(f + m, i) composes (a token maps m to
// max(F + m, M), two of them to F2 + F1 and max(F2 + M1, M2)), so 64 tokens take six steps; the next chunk's gate inputs are on their way.
template <typename A>
__global__ __launch_bounds__(64) void memory_gates_kernel(const A* __restrict__ proj, int64_t proj_stride, int64_t i_off, int64_t f_off,
                                                          const A* __restrict__ i_bias, const A* __restrict__ f_bias, float cap,
                                                          float* __restrict__ state, int64_t slot_stride, float* __restrict__ gates, int H, int dim,
                                                          int vdim, const int32_t* __restrict__ chunk_row0, const int32_t* __restrict__ chunk_rows,
                                                          const int32_t* __restrict__ long_chunk0, const int32_t* __restrict__ long_slot) {
  const int e = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  float* m_g = state + (int64_t)long_slot[e] * slot_stride + (int64_t)H * dim * (vdim + 1) + h;
  const float ib = ld(i_bias + h), fb = ld(f_bias + h);
  const int c_end = long_chunk0[e + 1];
  float m = *m_g, zi = 0.f, zf = 0.f;
  int n = 0;
  auto fetch = [&](int c) {
    n = chunk_rows[c];
    const A* pr = proj + (int64_t)(chunk_row0[c] + min(lane, n - 1)) * proj_stride;
    zi = ld(pr + i_off + h);
    zf = ld(pr + f_off + h);
  };
  int c = long_chunk0[e];
  if (c < c_end) fetch(c);
  for (; c < c_end; ++c) {
    const bool live = lane < n;
    const int last = n - 1;
    const float i = live ? cap * tanhf((zi + ib) / cap) : -INFINITY, f = live ? logsigmoid_f(cap * tanhf((zf + fb) / cap)) : 0.f;
    if (c + 1 < c_end) fetch(c + 1);
    float F = f, M = i;
#pragma unroll
    for (int x = 1; x < 64; x <<= 1) {
      const float Fo = __shfl_up(F, x, kWave), Mo = __shfl_up(M, x, kWave);
      if (lane >= x) { M = fmaxf(F + Mo, M); F += Fo; }
    }
    const float mn = fmaxf(F + m, M);
    float mp = __shfl_up(mn, 1, kWave);
    if (lane == 0) mp = m;
    float* g = gates + ((int64_t)c * H + h) * 3 * kDecayChunk + lane;
    g[0] = live ? expf(f + mp - mn) : 1.f;
    g[kDecayChunk] = live ? expf(i - mn) : 0.f;
    g[2 * kDecayChunk] = live ? expf(-mn) : 1.f;
    m = __shfl(mn, last, kWave);
  }
  if (lane == 0) *m_g = m;
}

}  // namespace pk

extern "C" {
using namespace pk;

#define PK_BAD ((pegainfer_status_t)hipErrorInvalidValue)

// workgroups per row of the launches before the recurrence
static int prep_parts(int rows, int heads) { return rows >= 256 ? 1 : std::max(1, std::min(ceil_div(heads, 4), 1024 / rows)); }

pegainfer_status_t pegainfer_delta_rule(float* qkv, int64_t qkv_stride, const void* proj, int64_t proj_stride, int64_t b_off,
                                        int64_t a_off, const void* A_log, const void* dt_bias, float* gates, float* state,
                                        int64_t slot_stride, float* o, int32_t heads, int32_t kv_heads, int32_t dim,
                                        int32_t vdim, int32_t n_rows, const int32_t* entry_row0, const int32_t* entry_slot,
                                        int32_t n_entries, int32_t dtype, pegainfer_stream_t stream) {
  if (n_entries <= 0 || n_rows <= 0) return 0;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > 256 || vdim <= 0 || heads > 65535 || n_entries > 65535)
    return PK_BAD;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        delta_prep_kernel<A><<<dim3(n_rows, prep_parts(n_rows, 2 * kv_heads)), 256, 0, as_stream(stream)>>>(qkv, qkv_stride, static_cast<const A*>(proj), proj_stride, b_off,
                                                                    a_off, static_cast<const A*>(A_log),
                                                                    static_cast<const A*>(dt_bias), gates, heads, kv_heads, dim);
      }))
    return PK_BAD;
  const dim3 grid(ceil_div(vdim, kRecCols), heads, n_entries);
  if (!by_slices(dim, [&](auto ns) {
        delta_rule_kernel<decltype(ns)::value, false><<<grid, 256, 0, as_stream(stream)>>>(qkv, qkv_stride, gates, state, slot_stride, o,
                                                                                    heads, kv_heads, dim, vdim, entry_row0,
                                                                                    entry_slot);
      }))
    return PK_BAD;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_delta_rule_channel(float* qkv, int64_t qkv_stride, const void* proj, int64_t proj_stride,
                                                int64_t b_off, const float* a, int64_t a_stride, const void* A_log,
                                                const void* dt_bias, float* gates, float* state, int64_t slot_stride, float* o,
                                                int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, int32_t n_rows,
                                                const int32_t* entry_row0, const int32_t* entry_slot, int32_t n_entries,
                                                int32_t dtype, pegainfer_stream_t stream) {
  if (n_entries <= 0 || n_rows <= 0) return 0;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > 256 || vdim <= 0 || heads > 65535 || n_entries > 65535)
    return PK_BAD;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        delta_prep_channel_kernel<A><<<dim3(n_rows, prep_parts(n_rows, 2 * kv_heads)), 256, 0, as_stream(stream)>>>(qkv, qkv_stride, static_cast<const A*>(proj), proj_stride,
                                                                            b_off, a, a_stride, static_cast<const A*>(A_log),
                                                                            static_cast<const A*>(dt_bias), gates, heads, kv_heads, dim);
      }))
    return PK_BAD;
  const dim3 grid(ceil_div(vdim, kRecCols), heads, n_entries);
  if (!by_slices(dim, [&](auto ns) {
        delta_rule_kernel<decltype(ns)::value, true><<<grid, 256, 0, as_stream(stream)>>>(qkv, qkv_stride, gates, state, slot_stride, o,
                                                                                          heads, kv_heads, dim, vdim, entry_row0,
                                                                                          entry_slot);
      }))
    return PK_BAD;
  return (pegainfer_status_t)hipGetLastError();
}

int64_t pegainfer_gated_matrix_memory_workspace(int32_t n_chunks, int32_t heads, int32_t dim, int32_t vdim) {
  return scalar_chunk_floats(n_chunks, heads, dim, vdim, true) + (int64_t)n_chunks * heads * 3 * kDecayChunk;
}

pegainfer_status_t pegainfer_gated_matrix_memory_form(const pegainfer_gated_matrix_memory_desc* q, pegainfer_stream_t stream) {
  if (!q) return PK_BAD;
  if (q->n_entries <= 0) return 0;
  const int H = q->heads, dim = q->dim, vdim = q->vdim;
  if (H <= 0 || dim <= 0 || dim > 256 || vdim <= 0 || H > 65535 || q->n_entries > 65535 || !(q->cap > 0.f)) return PK_BAD;
  const bool chunks = q->n_chunks > 0 && q->n_long > 0;
  if (chunks && (!q->workspace || !q->chunk_row0 || !q->chunk_rows || !q->long_chunk0 || !q->long_slot || q->scan_max <= 0)) return PK_BAD;
  hipStream_t st = as_stream(stream);
  bool ok = true;
  const bool known = by_dtype(q->dtype, [&](auto* t) {
    using A = std::remove_pointer_t<decltype(t)>;
    const A *proj = static_cast<const A*>(q->proj), *i_bias = static_cast<const A*>(q->i_bias), *f_bias = static_cast<const A*>(q->f_bias);
    if (q->n_entries > (chunks ? q->n_long : 0))
      ok = by_slices(dim, [&](auto ns) {
        matrix_memory_kernel<decltype(ns)::value, A><<<dim3(ceil_div(vdim, kRecCols), H, q->n_entries), 256, 0, st>>>(
            proj, q->proj_stride, q->q_off, q->k_off, q->v_off, q->i_off, q->f_off, i_bias, f_bias, q->cap, q->state, q->slot_stride, q->o, H, dim,
            vdim, q->entry_row0, q->entry_slot, chunks ? q->scan_max : 0);
      });
    if (ok && vdim > kRecCols && q->n_entries > (chunks ? q->n_long : 0))
      memory_carry_kernel<A><<<dim3(H, q->n_entries), 256, 0, st>>>(proj, q->proj_stride, q->k_off, q->i_off, q->f_off, i_bias, f_bias, q->cap,
                                                                    q->state, q->slot_stride, H, dim, vdim, q->entry_row0, q->entry_slot,
                                                                    chunks ? q->scan_max : 0);
    if (!ok || !chunks) return;
    float* gates = q->workspace + scalar_chunk_floats(q->n_chunks, H, dim, vdim, true);
    memory_gates_kernel<A><<<dim3(q->n_long, H), 64, 0, st>>>(proj, q->proj_stride, q->i_off, q->f_off, i_bias, f_bias, q->cap, q->state,
                                                              q->slot_stride, gates, H, dim, vdim, q->chunk_row0, q->chunk_rows, q->long_chunk0,
                                                              q->long_slot);
    const MemIn<A> in{proj, q->proj_stride, q->q_off, q->k_off, q->v_off, gates, H, dim, vdim};
    scalar_chunk_launch(in, q->workspace, q->state, q->slot_stride, q->o, q->chunk_row0, q->chunk_rows, q->n_chunks, q->long_chunk0, q->long_slot,
                        q->n_long, st);
  });
  return known && ok ? (pegainfer_status_t)hipGetLastError() : PK_BAD;
}

int32_t pegainfer_gated_matrix_memory_beside_ok(const pegainfer_gated_matrix_memory_desc* q, const pegainfer_qk_prep_desc* p) {
  return q && p && q->n_entries > 0 && q->n_entries <= 65535 && q->heads > 0 && q->dim > 0 && q->dim <= 256 && q->vdim > 0 && q->vdim <= 512 && q->cap > 0.f &&
         q->n_long == 0 && q->dtype == kDtBf16 && p->dtype == kDtBf16 && p->proj_dtype == kDtBf16 && p->n_rows > 0 && qk_prep_ok(p) && qk_prep_pairs(p) &&
         (int64_t)ceil_div(q->vdim, kRecCols) * q->heads * q->n_entries < (1 << 22);
}

pegainfer_status_t pegainfer_gated_matrix_memory_beside(const pegainfer_gated_matrix_memory_desc* q, const pegainfer_qk_prep_desc* p,
                                                        pegainfer_stream_t stream) {
  if (!pegainfer_gated_matrix_memory_beside_ok(q, p)) return PK_BAD;
  const int nbx = ceil_div(q->vdim, kRecCols), n_scan = nbx * q->heads * q->n_entries, per_row = qk_prep_per_row(*p);
  by_slices(q->dim, [&](auto ns) {
    memory_beside_kernel<decltype(ns)::value><<<n_scan + p->n_rows * per_row, 256, qk_prep_lds(*p), as_stream(stream)>>>(*q, nbx, n_scan, *p, qk_prep_form(*p),
                                                                                                                        per_row);
  });
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_gated_matrix_memory_finish(const pegainfer_gated_matrix_memory_desc* q, const pegainfer_memory_finish_desc* f,
                                                        pegainfer_stream_t stream) {
  if (!q || !f || q->n_entries <= 0 || q->n_entries > 65535 || q->heads <= 0 || q->dim <= 0 || q->vdim <= 0 || q->vdim > 512 || !f->norm_w || !f->gate || !f->out ||
      (f->rows && !f->scaled))
    return PK_BAD;
  const int scale = f->rows && f->scale_cols > 0 ? std::min(64, ceil_div(f->scale_cols, 256)) : 0;
  if (!by_dtype(q->dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        auto go = [&](auto kern) { kern<<<dim3(q->heads + scale, q->n_entries), 256, 0, as_stream(stream)>>>(*q, *f); };
        const int v = head_rms_values(q->o, f->norm_w, f->gate, f->gate_stride, f->out, f->out_stride, q->vdim);
        if (v == 4) go(memory_finish_kernel<A, 4>);
        else if (v == 2) go(memory_finish_kernel<A, 2>);
        else go(memory_finish_kernel<A, 1>);
      }))
    return PK_BAD;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_gated_matrix_memory(const void* proj, int64_t proj_stride, int64_t q_off, int64_t k_off,
                                                 int64_t v_off, int64_t i_off, int64_t f_off, const void* i_bias,
                                                 const void* f_bias, float cap, float* state, int64_t slot_stride, float* o,
                                                 int32_t heads, int32_t dim, int32_t vdim, const int32_t* entry_row0,
                                                 const int32_t* entry_slot, int32_t n_entries, int32_t dtype,
                                                 pegainfer_stream_t stream) {
  pegainfer_gated_matrix_memory_desc q{};
  q.proj = proj; q.proj_stride = proj_stride; q.q_off = q_off; q.k_off = k_off; q.v_off = v_off; q.i_off = i_off; q.f_off = f_off;
  q.i_bias = i_bias; q.f_bias = f_bias; q.cap = cap; q.state = state; q.slot_stride = slot_stride; q.o = o;
  q.heads = heads; q.dim = dim; q.vdim = vdim; q.entry_row0 = entry_row0; q.entry_slot = entry_slot; q.n_entries = n_entries; q.dtype = dtype;
  return pegainfer_gated_matrix_memory_form(&q, stream);
}

}  // extern "C"
