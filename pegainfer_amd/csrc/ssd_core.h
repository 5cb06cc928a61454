// The state-space scan of one run of columns, as a part of a launch: ssd.hip's own, and attn_paged.hip's where a layer has both halves.
#pragma once

#include "common.h"
#include "typed.h"
#include "recurrent_core.h"

namespace pk {

__device__ __forceinline__ float ssd_step(float raw, float bias) {   // softplus
  const float x = raw + bias;
  return x > 20.0f ? x : log1pf(expf(x));
}

// of 256 threads: columns bx of runs of sixteen, head h, entry e
template <int NS, typename A>
__device__ __forceinline__ void ssd_scan_block(int bx, int h, int e, const float* __restrict__ xbc, int64_t xbc_stride, const A* __restrict__ proj,
                                                       int64_t proj_stride, int64_t dt_off, const A* __restrict__ A_log,
                                                       const A* __restrict__ dt_bias, const A* __restrict__ Dskip,
                                                       float* __restrict__ state, int64_t slot_stride, float* __restrict__ o, int H,
                                                       int G, int dim, int vdim, const int32_t* __restrict__ entry_row0,
                                                       const int32_t* __restrict__ entry_slot, int scan_max) {
  constexpr int DP = kRecSlices * NS;
  __shared__ __attribute__((aligned(16))) float s_k[kRecTokens][DP], s_q[kRecTokens][DP];
  __shared__ float s_v[kRecTokens][kRecCols], s_a[kRecTokens], s_b[kRecTokens];
  const int col0 = bx * kRecCols;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, cl = wave * 4 + (lane >> 4);
  const int col = col0 + cl;
  const int g0 = h / (H / G);
  const int row0 = entry_row0[e], len = entry_row0[e + 1] - row0;
  if (scan_max > 0 && len > scan_max) return;      // the chunk form has this entry
  float* S_g = state + (int64_t)entry_slot[e] * slot_stride + (int64_t)h * dim * vdim;
  float S[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int d = r * NS + i;
    S[i] = d < dim && col < vdim ? S_g[(int64_t)d * vdim + col] : 0.f;
  }
  const float rate = -expf(ld(A_log + h)), dtb = ld(dt_bias + h), skip = ld(Dskip + h);
  const int64_t b_at = (int64_t)H * vdim + (int64_t)g0 * dim, c_at = (int64_t)H * vdim + (int64_t)(G + g0) * dim;
  RoundFetch<NS> nxt;
  auto fetch = [&](int t0) {
    const float* base = xbc + (int64_t)(row0 + t0) * xbc_stride;
    nxt.issue(min(kRecTokens, len - t0), tid, dim,
              [=](int tt, int d) { return base[(int64_t)tt * xbc_stride + c_at + d]; },
              [=](int tt, int d) { return base[(int64_t)tt * xbc_stride + b_at + d]; },
              [=](int tt, int c) { return col0 + c < vdim ? base[(int64_t)tt * xbc_stride + (int64_t)h * vdim + col0 + c] : 0.f; });
  };
  fetch(0);
  for (int t0 = 0; t0 < len; t0 += kRecTokens) {
    const int tc = min(kRecTokens, len - t0);
    __syncthreads();
    nxt.land(tid, s_q, s_k, s_v);
    if (tid < kRecTokens) {   // rows past the entry's end: a = 1, b = 0 - a step that leaves S as it is
      const bool live = tid < tc;
      const float dt = live ? ssd_step(ld(proj + (int64_t)(row0 + t0 + tid) * proj_stride + dt_off + h), dtb) : 0.f;
      s_a[tid] = live ? expf(rate * dt) : 1.f;
      s_b[tid] = dt;
    }
    __syncthreads();
    if (t0 + kRecTokens < len) fetch(t0 + kRecTokens);
    float okeep = 0.f;
    for (int t8 = 0; t8 < tc; t8 += 8) {       // (eight per trip measured 7 % faster than four: 182 against 196 us at 1024 tokens)
#pragma unroll
     for (int uu = 0; uu < 8; ++uu) {
      const int tt = t8 + uu;
      const float a = s_a[tt], xv = s_v[tt][cl];
      const float bv = s_b[tt] * xv;
      float y0 = 0.f, y1 = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const float kk = s_k[tt][r * NS + i], qq = s_q[tt][r * NS + i];
        S[i] = fmaf(bv, kk, a * S[i]);
        if (i & 1) y1 = fmaf(S[i], qq, y1); else y0 = fmaf(S[i], qq, y0);
      }
      const float y = fmaf(skip, xv, row16_sum(y0 + y1));
      okeep = tt == r ? y : okeep;
     }
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
