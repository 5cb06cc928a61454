// The norm and gate of one head's read-out by one wave, as a part of a launch: seq_blocks.hip's own, and recurrent.hip's behind a step's scan.
#pragma once

#include "common.h"
#include "typed.h"

namespace pk {

// One wave per (row, head), vdim <= 512; a lane's values, gates and weights are all requested before the first is used, V at a time.  Bound by
// memory with many heads, by the launch with few: 8192 x 4 heads of 128 16.5 -> 12.6 us, one row of four groups of 512 9.7 -> 4.6 us (read
// value by value and a second time for the output before).
template <typename A, int V>
__device__ __forceinline__ void head_rms_gate_wave(int row, int h, const float* __restrict__ o, const A* __restrict__ w, int w_per_head,
                                                            const A* __restrict__ gate, int64_t gate_stride, int gate_kind,
                                                            float factor, float eps, A* __restrict__ out, int64_t out_stride,
                                                            int heads, int vdim, int gate_first) {
  constexpr int K = 8 / V;
  const int lane = threadIdx.x & 63;
  const float* p = o + ((int64_t)row * heads + h) * vdim;
  const A* gr = gate + (int64_t)row * gate_stride + (int64_t)h * vdim;
  const A* wr = w + (w_per_head ? (int64_t)h * vdim : 0);
  A* dst = out + (int64_t)row * out_stride + (int64_t)h * vdim;
  auto load = [&](const auto* q, float* t) {
    if constexpr (V == 4) ld4(q, t); else if constexpr (V == 2) ld2(q, t); else t[0] = ld(q);
  };
  float v[K][V], z[K][V], wv[K][V];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = (lane + 64 * k) * V;
    if (i < vdim) { load(p + i, v[k]); load(gr + i, z[k]); load(wr + i, wv[k]); }
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k)
    if ((lane + 64 * k) * V < vdim)
#pragma unroll
      for (int u = 0; u < V; ++u) {
        z[k][u] = gate_kind == 0 ? silu_f(z[k][u]) : sigmoid_f(z[k][u]);
        if (gate_first) v[k][u] *= z[k][u];   // gate_first: the gated values are what is normed
        ss = fmaf(v[k][u], v[k][u], ss);
      }
  ss = wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)vdim + eps);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = (lane + 64 * k) * V;
    if (i >= vdim) continue;
    float r[V];
    // (each order keeps its own sequence of roundings: norm, weight, gate, factor - or gate, norm, weight, factor)
#pragma unroll
    for (int u = 0; u < V; ++u) r[u] = gate_first ? v[k][u] * inv * wv[k][u] * factor : v[k][u] * inv * wv[k][u] * z[k][u] * factor;
    if constexpr (V == 4) st4(dst + i, r); else if constexpr (V == 2) st2(dst + i, r); else st(dst + i, r[0]);
  }
}

// as many values per access as rows, strides and pointers allow, without leaving lanes of a narrow head idle
inline int head_rms_values(const void* o, const void* w, const void* gate, int64_t gate_stride, const void* out, int64_t out_stride, int vdim) {
  const bool aligned = gate_stride % 4 == 0 && out_stride % 4 == 0 && host_aligned16(o) && host_aligned16(w) && host_aligned16(gate) && host_aligned16(out);
  return !aligned || vdim % 4 ? 1 : vdim > 128 ? 4 : vdim > 64 ? 2 : 1;
}

}  // namespace pk
