// The gated delta rule token by token, as a part of a launch: recurrent.hip's own, and delta_chunk.hip's for the short entries of a step that also has
// long ones.
#pragma once

#include "common.h"
#include "typed.h"
#include "recurrent_core.h"
#include "sigmoid_power.h"

namespace pk {

// the entry that holds a row: the last one that begins at or before it
__device__ __forceinline__ int entry_of_row(const int32_t* __restrict__ entry_row0, int n_entries, int row) {
  int lo = 0, hi = n_entries - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (entry_row0[mid] <= row) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Per row, before the recurrence: q and k heads made unit vectors in place (x / sqrt(sum(x^2) + 1e-6), q also * dim^-1/2),
// gates[row] = [g: heads | beta: heads].  A wave per head; a row's heads and gates are dealt over gridDim.y workgroups (few rows: as many
// as its heads fill - one workgroup took 10.0 us for a row of 32 heads of 128, eight take 4.2 us; from 256 rows on one).
// of 256 threads: workgroup y of ny of a row
template <typename A>
__device__ __forceinline__ void delta_prep_row(int row, int y, int ny, float* __restrict__ qkv, int64_t qkv_stride, const A* __restrict__ proj,
                                               int64_t proj_stride, int64_t b_off, int64_t a_off, const A* __restrict__ A_log,
                                               const A* __restrict__ dt_bias, float* __restrict__ gates, int H, int G, int dim) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float* qk = qkv + (int64_t)row * qkv_stride;
  const float qs = 1.0f / sqrtf((float)dim);
  for (int hh = y * 4 + wave; hh < 2 * G; hh += 4 * ny) {
    float* x = qk + (int64_t)hh * dim;
    float ss = 0.f;
    for (int d = lane; d < dim; d += 64) ss = fmaf(x[d], x[d], ss);
    const float sc = (hh < G ? qs : 1.0f) / sqrtf(wave_sum(ss) + 1e-6f);
    for (int d = lane; d < dim; d += 64) x[d] *= sc;
  }
  const A* pr = proj + (int64_t)row * proj_stride;
  for (int h = y * 256 + threadIdx.x; h < H; h += 256 * ny) {
    gates[(int64_t)row * 2 * H + h] = expf(-expf(ld(A_log + h)) * softplus_f(ld(pr + a_off + h) + ld(dt_bias + h)));
    gates[(int64_t)row * 2 * H + H + h] = sigmoid_f(ld(pr + b_off + h));
  }
}

// CH: the decay is one number per (head, key channel) - it scales the ROWS of S - and the gates row is laid out as
// delta_prep_channel_kernel leaves it; otherwise one number per head ([g: heads | beta: heads]).
// A chain of dependent steps with one wave per SIMD: whatever a step waits for beside its own arithmetic is lost time, so a round's gates
// come with its q | k | v (asked for when the round began, they held the chain up for a trip to memory), four values per load
// where the layout allows it, and a token's values leave LDS while the token before it is worked on.  Lane r's NS values lie in groups of
// four 64 floats apart, so that the lanes of a row read neighbouring 16 bytes.  1024 tokens of 32 heads of 128 x 128: 202 -> 180 us,
// 8 portions of 700 tokens at most with channel decays 169 -> 145 us.
// of 256 threads: columns bx of runs of sixteen, head h, entry e
template <int NS, bool CH>
__device__ __forceinline__ void delta_rule_block(int bx, int h, int e, const float* __restrict__ qkv, int64_t qkv_stride,
                                                 const float* __restrict__ gates, float* __restrict__ state, int64_t slot_stride,
                                                 float* __restrict__ o, int H, int G, int dim, int vdim, const int32_t* __restrict__ entry_row0,
                                                 const int32_t* __restrict__ entry_slot) {
  constexpr int DP = kRecSlices * NS;
  constexpr int V = NS >= 4 ? 4 : 1, NV = NS / V;      // values per load, loads of a thread
  __shared__ __attribute__((aligned(16))) float s_k[kRecTokens][DP], s_q[kRecTokens][DP];
  __shared__ __attribute__((aligned(16))) float s_gb[kRecTokens][2];
  __shared__ float s_v[kRecTokens][kRecCols];
  __shared__ __attribute__((aligned(16))) float s_gc[CH ? kRecTokens : 1][CH ? DP : 1];
  const int64_t gs = CH ? (int64_t)H * dim + H : (int64_t)2 * H;   // floats of one gates row
  const int col0 = bx * kRecCols;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, cl = wave * 4 + (lane >> 4);
  const int col = col0 + cl;
  const int g0 = h / (H / G);
  const int row0 = entry_row0[e], len = entry_row0[e + 1] - row0;
  float* S_g = state + (int64_t)entry_slot[e] * slot_stride + (int64_t)h * dim * vdim;
  float S[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int d = r * NS + i;
    S[i] = d < dim && col < vdim ? S_g[(int64_t)d * vdim + col] : 0.f;
  }
  const bool vec = V == 4 && (dim & 3) == 0 && (qkv_stride & 3) == 0 && aligned16(qkv);
  const bool vec_g = V == 4 && (dim & 3) == 0 && (gs & 3) == 0 && aligned16(gates);
  // thread t serves token t / 16 of a round: values V (t % 16 + 16 j) + 0 .. V of its query, key and decays, column t % 16 of its value
  const int ft = tid >> 4, part = tid & 15;
  struct Round { float q[NS], k[NS], gc[CH ? NS : 1], v, g, b; } nxt;
  auto fetch = [&](int t0) {           // rows past the entry's end and values past dim: some that are there, dropped by land()
    const int64_t row = row0 + min(t0 + ft, len - 1);
    auto take = [&](const float* p, bool wide, float (&x)[NS]) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int d = V * (part + 16 * j);
        if (V == 4 && wide) {
          ld4(p + (d < dim ? d : 0), &x[V * j]);
        } else {
#pragma unroll
          for (int u = 0; u < V; ++u) x[V * j + u] = p[d + u < dim ? d + u : 0];
        }
      }
    };
    const float* base = qkv + row * qkv_stride;
    take(base + (int64_t)g0 * dim, vec, nxt.q);
    take(base + (int64_t)(G + g0) * dim, vec, nxt.k);
    nxt.v = base[(int64_t)2 * G * dim + (int64_t)h * vdim + min(col0 + part, vdim - 1)];
    if constexpr (CH) take(gates + row * gs + (int64_t)h * dim, vec_g, nxt.gc);
    const float* gr = gates + (int64_t)(row0 + min(t0 + part, len - 1)) * gs + h;    // token t % 16 here: the first 16 threads keep it
    nxt.g = CH ? 1.f : gr[0];
    nxt.b = gr[CH ? (int64_t)H * dim : H];
  };
  // where value d of a row lies: lane d / NS holds it, as number d % NS
  auto place = [](int d) { return NS > 4 ? (d % NS / 4) * 64 + d / NS * 4 + d % 4 : d; };
  auto land = [&](int tc) {
    const bool live = ft < tc;
    auto put = [&](const float (&x)[NS], float* dst, float none) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int d = V * (part + 16 * j);
        if constexpr (V == 4) {
          f32x4 t;
#pragma unroll
          for (int u = 0; u < 4; ++u) t[u] = live && d + u < dim ? x[4 * j + u] : none;
          *reinterpret_cast<f32x4*>(dst + place(d)) = t;
        } else {
          dst[d] = live && d < dim ? x[j] : none;
        }
      }
    };
    put(nxt.q, s_q[ft], 0.f);
    put(nxt.k, s_k[ft], 0.f);
    if constexpr (CH) put(nxt.gc, s_gc[ft], 1.f);
    s_v[ft][part] = live && col0 + part < vdim ? nxt.v : 0.f;
    if (tid < kRecTokens) {   // rows past the entry's end: g = 1, beta = 0, zero key - a step that leaves S as it is
      s_gb[tid][0] = tid < tc ? nxt.g : 1.f;
      s_gb[tid][1] = tid < tc ? nxt.b : 0.f;
    }
  };
  struct Token { float k[NS], q[NS], gc[CH ? NS : 1], v, g, b; };
  auto read = [&](int tt, Token& x) {
    auto row = [&](const float* src, float (&y)[NS]) {
      if constexpr (V == 4) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          const f32x4 t = *reinterpret_cast<const f32x4*>(src + j * 64 + r * 4);
#pragma unroll
          for (int u = 0; u < 4; ++u) y[4 * j + u] = t[u];
        }
      } else {
#pragma unroll
        for (int i = 0; i < NS; ++i) y[i] = src[r * NS + i];
      }
    };
    row(s_k[tt], x.k);
    if constexpr (CH) row(s_gc[tt], x.gc);
    x.v = s_v[tt][cl];
    x.g = s_gb[tt][0];
    x.b = s_gb[tt][1];
    row(s_q[tt], x.q);
    asm volatile("" ::: "memory");     // asked for here, not where it is used
  };
  if (len > 0) fetch(0);
#pragma unroll
  for (int i = 0; i < NS; ++i) asm volatile("" : "+v"(S[i]));   // the state is waited for here: its wait must not land in the loop
  for (int t0 = 0; t0 < len; t0 += kRecTokens) {
    const int tc = min(kRecTokens, len - t0);
    __syncthreads();
    land(tc);
    __syncthreads();
    if (t0 + kRecTokens < len) fetch(t0 + kRecTokens);
    float okeep = 0.f;
    auto step = [&](int tt, const Token& x) {
      float a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        if constexpr (CH) S[i] *= x.gc[i]; else S[i] *= x.g;
        if (i & 1) a1 = fmaf(S[i], x.k[i], a1); else a0 = fmaf(S[i], x.k[i], a0);
      }
      const float u = x.b * (x.v - row16_sum(a0 + a1));
      float o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        S[i] = fmaf(x.k[i], u, S[i]);
        if (i & 1) o1 = fmaf(S[i], x.q[i], o1); else o0 = fmaf(S[i], x.q[i], o0);
      }
      const float oa = row16_sum(o0 + o1);
      okeep = tt == r ? oa : okeep;      // lane r of the column keeps token r of the round
    };
    // two tokens per trip: a token's first product starts while the read-out of the one before it is still being summed
    Token x, y;
    read(0, x);
    for (int t2 = 0; t2 < tc; t2 += 2) {
      read(t2 + 1, y);
      step(t2, x);
      read((t2 + 2) & (kRecTokens - 1), x);
      step(t2 + 1, y);
    }
    if (r < tc && col < vdim) o[(int64_t)(row0 + t0 + r) * ((int64_t)H * vdim) + (int64_t)h * vdim + col] = okeep;
  }
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int d = r * NS + i;
    if (d < dim && col < vdim) S_g[(int64_t)d * vdim + col] = S[i];
  }
}

}  // namespace pk
