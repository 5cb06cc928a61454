// Selective state-space scan with one decay per head and token over ragged batches, fp32 state and fp32 arithmetic throughout:
//     a = exp(-exp(A_log) dt);  S <- a S + dt B x^T;  y = S^T C + D x          (dt = softplus(raw + bias))
// Two equivalent forms.  The scan is a serial chain of 0.18 us a token whatever the size; 1024 tokens of 32 heads of 128 states x 64 values
// take 180 us there and 65 us in chunks (sums 15, walk 10, outputs 37: the fp32 matrix-core products and the states' way through memory),
// 4096 tokens 703 and 208 us.
//   ssd_scan_kernel           token by token, the layout of recurrent.hip: decoding and short portions
//   ssd_chunk_sum_kernel      long portions, in chunks of <= 64 tokens that run side by side: U_c = sum_i w_i dt_i B_i x_i^T with w_i the
//                             product of the decays behind token i, and the product of all the chunk's decays
//   ssd_chunk_state_kernel    walks the chunks of an entry, S <- total_c S + U_c, and leaves the state BEFORE each in U_c's place
//   ssd_chunk_out_kernel      y_i = (a_1 .. a_i) S^T C_i + sum_{j <= i} (a_(j+1) .. a_i) dt_j (C_i . B_j) x_j + D x_i
// Decays enter the chunk form as products of the decays themselves, never as quotients or differences of logarithms: every factor is at
// most one, nothing cancels however fast a head forgets, and the roundings of a product are those of the scan's state.
// Products of the chunk form run on v_mfma_f32_16x16x4_f32 (chunk_core.h).  Its scores are computed transposed (keys as rows), which
// leaves lane l with the scores of query l % 16 against keys 4 (l / 16) + r: the A operand of the product with the values.
#include "common.h"
#include "typed.h"
#include "recurrent_core.h"
#include "chunk_core.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

__device__ __forceinline__ float ssd_step(float raw, float bias) {   // softplus
  const float x = raw + bias;
  return x > 20.0f ? x : log1pf(expf(x));
}

template <int NS, typename A>
__global__ __launch_bounds__(256) void ssd_scan_kernel(const float* __restrict__ xbc, int64_t xbc_stride, const A* __restrict__ proj,
                                                       int64_t proj_stride, int64_t dt_off, const A* __restrict__ A_log,
                                                       const A* __restrict__ dt_bias, const A* __restrict__ Dskip,
                                                       float* __restrict__ state, int64_t slot_stride, float* __restrict__ o, int H,
                                                       int G, int dim, int vdim, const int32_t* __restrict__ entry_row0,
                                                       const int32_t* __restrict__ entry_slot, int scan_max) {
  constexpr int DP = kRecSlices * NS;
  __shared__ __attribute__((aligned(16))) float s_k[kRecTokens][DP], s_q[kRecTokens][DP];
  __shared__ float s_v[kRecTokens][kRecCols], s_a[kRecTokens], s_b[kRecTokens];
  const int e = blockIdx.z, h = blockIdx.y, col0 = blockIdx.x * kRecCols;
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

template <typename A>
struct SsdIn {
  const float* xbc; int64_t xbc_stride;
  const A* proj; int64_t proj_stride, dt_off;
  const A *A_log, *dt_bias, *D;
  int H, G, dim, vdim;
  __device__ __forceinline__ int64_t b_at(int h) const { return (int64_t)H * vdim + (int64_t)(h / (H / G)) * dim; }
  __device__ __forceinline__ int64_t c_at(int h) const { return b_at(h) + (int64_t)G * dim; }
  // lane i of a wave: step size and decay of token i of a chunk (a step that changes nothing past the chunk's end)
  __device__ __forceinline__ void steps(int h, int row0, int n, int lane, float* dt, float* a) const {
    *dt = lane < n ? ssd_step(ld(proj + (int64_t)(row0 + lane) * proj_stride + dt_off + h), ld(dt_bias + h)) : 0.f;
    *a = lane < n ? expf(-expf(ld(A_log + h)) * *dt) : 1.f;
  }
};
constexpr int kSsdCols = 64;     // value columns of a workgroup of the chunk form
__host__ __device__ constexpr int ssd_cols(int vdim) { return (vdim + kSsdCols - 1) / kSsdCols * kSsdCols; }

// product of the lanes behind this one (exclusive), by doubling
__device__ __forceinline__ float product_behind(float a, int lane) {
#pragma unroll
  for (int x = 1; x < 64; x <<= 1) {
    const float o = __shfl_down(a, x, kWave);
    if (lane + x < 64) a *= o;
  }
  const float next = __shfl_down(a, 1, kWave);
  return lane < 63 ? next : 1.0f;
}

// One workgroup per (chunk, head, 64 value columns): a wave takes every fourth block of 16 state rows, all 64 columns.
template <typename A>
__global__ __launch_bounds__(256) void ssd_chunk_sum_kernel(SsdIn<A> in, float* __restrict__ ws, float* __restrict__ ws_total,
                                                            const int32_t* __restrict__ chunk_row0, const int32_t* __restrict__ chunk_rows) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ float s_w[kDecayChunk];
  const int c = blockIdx.x, h = blockIdx.y, col0 = blockIdx.z * kSsdCols, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l15 = lane & 15, lg = lane >> 4, row0 = chunk_row0[c], n = chunk_rows[c];
  const int dp = pad16(in.dim), vp = ssd_cols(in.vdim), sk = stride_rows4(in.dim), sv = stride_rows4(kSsdCols);
  float *s_k = sm, *s_v = sm + kDecayChunk * sk;
  if (wave == 0) {
    float dt, a;
    in.steps(h, row0, n, lane, &dt, &a);
    const float w = product_behind(a, lane);
    s_w[lane] = w * dt;
    if (lane == 0 && blockIdx.z == 0) ws_total[(int64_t)c * in.H + h] = w * a;
  }
  __syncthreads();
  auto same = [](float x) { return x; };
  stage_rows<4>(in.xbc, in.xbc_stride, in.b_at(h), row0, n, in.dim, dp, s_k, sk, s_w, tid, same);
  stage_rows<4>(in.xbc, in.xbc_stride, (int64_t)h * in.vdim + col0, row0, n, min(kSsdCols, in.vdim - col0), kSsdCols, s_v, sv, nullptr, tid, same);
  __syncthreads();
  float* U = ws + ((int64_t)c * in.H + h) * dp * vp + col0;
  const int steps = (n + 3) >> 2;
  for (int d0 = wave * 16; d0 < dp; d0 += 64) {
    f32x4 acc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float *ka = s_k + lg * sk + d0 + l15, *vb = s_v + lg * sv + l15;
#pragma unroll 4
    for (int i = 0; i < steps; ++i) {
      const float a = ka[4 * i * sk];
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, vb[4 * i * sv + 16 * b], acc[b], 0, 0, 0);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) U[(int64_t)(d0 + 4 * lg + r) * vp + 16 * b + l15] = acc[b][r];
  }
}

// One thread per element of the state: through the entry's chunks, the state before each left in U's place.
__global__ __launch_bounds__(256) void ssd_chunk_state_kernel(float* ws, const float* __restrict__ ws_total, float* __restrict__ state,
                                                              int64_t slot_stride, int H, int dim, int vdim,
                                                              const int32_t* __restrict__ long_chunk0, const int32_t* __restrict__ long_slot) {
  const int e = blockIdx.z, h = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
  if (i >= dim * vdim) return;
  const int dp = pad16(dim), vp = ssd_cols(vdim);
  float* sp = state + (int64_t)long_slot[e] * slot_stride + (int64_t)h * dim * vdim + i;
  const int64_t cs = (int64_t)H * dp * vp;
  float* u = ws + (int64_t)h * dp * vp + (int64_t)(i / vdim) * vp + i % vdim;
  const int c_end = long_chunk0[e + 1];
  float S = *sp;
  for (int c0 = long_chunk0[e]; c0 < c_end; c0 += 8) {      // eight chunks' loads in flight before the first store
    float t[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) t[k] = c0 + k < c_end ? u[(c0 + k) * cs] : 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (c0 + k < c_end) {
        u[(c0 + k) * cs] = S;
        S = fmaf(ws_total[(int64_t)(c0 + k) * H + h], S, t[k]);
      }
  }
  *sp = S;
}

// One workgroup per (chunk, head, 64 value columns), a wave per 16 queries.  Queries lie in registers (QB blocks of 16 state rows at most:
// lane (l15, lg) holds values 4 lg .. of each block, and the keys and the state before the chunk are read in the same numbering); keys
// and values in LDS.  A wave makes the decays between its own queries and all keys: lane j starts from the product of the decays between
// key j and the wave's first query and multiplies by one decay per query.
template <typename A, int QB>
__global__ __launch_bounds__(256) void ssd_chunk_out_kernel(SsdIn<A> in, const float* __restrict__ ws, float* __restrict__ o,
                                                            const int32_t* __restrict__ chunk_row0, const int32_t* __restrict__ chunk_rows) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  constexpr int sp = kDecayChunk + 4, sv = kSsdCols + 4;
  __shared__ __attribute__((aligned(16))) float s_p[kDecayChunk][sp];   // [query][key] decay between them, times the key's step size
  const int c = blockIdx.x, h = blockIdx.y, col0 = blockIdx.z * kSsdCols, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l15 = lane & 15, lg = lane >> 4, row0 = chunk_row0[c], n = chunk_rows[c], i0 = wave * 16;
  const int dim = in.dim, dp = pad16(dim), vp = ssd_cols(in.vdim), sk = stride_rows16(dim), vd = min(kSsdCols, in.vdim - col0);
  float *s_k = sm, *s_v = s_k + kDecayChunk * sk;
  f32x4 q[QB];
  {
    const float* src = in.xbc + (int64_t)(row0 + min(i0 + l15, n - 1)) * in.xbc_stride + in.c_at(h);
    const bool vec = aligned16(src) && (dim & 3) == 0;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      const int k = 16 * b + 4 * lg;
      if (vec) {
        q[b] = *reinterpret_cast<const f32x4*>(src + (k < dim ? k : 0));
        if (k >= dim) q[b] = f32x4{0.f, 0.f, 0.f, 0.f};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) q[b][e] = k + e < dim ? src[k + e] : 0.f;
      }
    }
  }
  auto same = [](float x) { return x; };
  stage_rows<4>(in.xbc, in.xbc_stride, in.b_at(h), row0, n, dim, dp, s_k, sk, nullptr, tid, same);
  stage_rows<4>(in.xbc, in.xbc_stride, (int64_t)h * in.vdim + col0, row0, n, vd, kSsdCols, s_v, sv, nullptr, tid, same);
  float before;                                      // product of the decays up to and with query i0 + l15
  {
    float dt, a;
    in.steps(h, row0, n, lane, &dt, &a);
    float f = a;
#pragma unroll
    for (int x = 1; x < 64; x <<= 1) {
      const float t = __shfl_up(f, x, kWave);
      if (lane >= x) f *= t;
    }
    before = __shfl(f, i0 + l15, kWave);
    float pr = product_behind(lane < i0 ? a : 1.0f, lane);     // keys before i0: the decays from there to the query before i0
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float ai = __shfl(a, i0 + k, kWave);
      pr = lane < i0 + k ? pr * ai : 1.0f;
      s_p[i0 + k][lane] = pr * dt;
    }
  }
  __syncthreads();
  if (i0 >= n) return;                               // no barrier follows
  f32x4 acc[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  {   // what the tokens before the chunk left; rows dim .. dp - 1 and columns past vdim of the state before a chunk are zeros
    const float* S = ws + ((int64_t)c * in.H + h) * dp * vp + col0 + (int64_t)(4 * lg) * vp + l15;
    float cur[4][4], nxt[4][4];
    auto fetch = [&](int k0, float (*t)[4]) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < 4; ++b) t[e][b] = S[(int64_t)(k0 + e) * vp + 16 * b];
    };
    fetch(0, cur);
#pragma unroll
    for (int kb = 0; kb < QB; ++kb) {
      if (16 * kb >= dp) break;
      fetch(min(16 * kb + 16, dp - 16), nxt);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = q[kb][e] * before;
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, cur[e][b], acc[b], 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < 4; ++b) cur[e][b] = nxt[e][b];
    }
  }
  for (int jb = 0; jb <= wave; ++jb) {               // the chunk's own tokens, 16 keys at a time
    f32x4 s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* kr = s_k + (jb * 16 + l15) * sk + 4 * lg;
#pragma unroll
    for (int kb = 0; kb < QB; ++kb) {
      if (16 * kb >= dp) break;
      const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + 16 * kb);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[e], q[kb][e], s[e], 0, 0, 0);
    }
    s[0] = (s[0] + s[1]) + (s[2] + s[3]);
    const f32x4 w = *reinterpret_cast<const f32x4*>(&s_p[i0 + l15][jb * 16 + 4 * lg]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = jb * 16 + 4 * lg + r;
      const float p = j <= i0 + l15 ? s[0][r] * w[r] : 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, s_v[j * sv + 16 * b + l15], acc[b], 0, 0, 0);
    }
  }
  const float skip = ld(in.D + h);
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int col = 16 * b + l15;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + 4 * lg + r;
      if (i < n && col < vd) o[(int64_t)(row0 + i) * ((int64_t)in.H * in.vdim) + (int64_t)h * in.vdim + col0 + col] = fmaf(skip, s_v[i * sv + col], acc[b][r]);
    }
  }
}

}  // namespace pk

extern "C" {
using namespace pk;

int64_t pegainfer_ssd_scan_workspace(int32_t n_chunks, int32_t heads, int32_t n_state, int32_t vdim) {
  return (int64_t)n_chunks * heads * ((int64_t)pad16(n_state) * ssd_cols(vdim) + 1);
}

pegainfer_status_t pegainfer_ssd_scan_form(const pegainfer_ssd_scan_desc* q, pegainfer_stream_t stream) {
  constexpr pegainfer_status_t bad = (pegainfer_status_t)hipErrorInvalidValue;
  if (!q) return bad;
  if (q->n_entries <= 0) return 0;
  const int H = q->heads, G = q->groups, dim = q->n_state, vdim = q->vdim;
  if (H <= 0 || G <= 0 || H % G || dim <= 0 || dim > 256 || vdim <= 0 || H > 65535 || q->n_entries > 65535) return bad;
  const bool chunks = q->n_chunks > 0 && q->n_long > 0;
  if (chunks && (!q->workspace || !q->chunk_row0 || !q->chunk_rows || !q->long_chunk0 || !q->long_slot || q->scan_max <= 0 || q->n_long > 65535))
    return bad;
  hipStream_t st = as_stream(stream);
  bool ok = true;
  const bool known = by_dtype(q->dtype, [&](auto* t) {
    using A = std::remove_pointer_t<decltype(t)>;
    const SsdIn<A> in{q->xbc, q->xbc_stride, static_cast<const A*>(q->proj), q->proj_stride, q->dt_off, static_cast<const A*>(q->A_log),
                      static_cast<const A*>(q->dt_bias), static_cast<const A*>(q->D), H, G, dim, vdim};
    if (q->n_entries > (chunks ? q->n_long : 0))
      ok = by_slices(dim, [&](auto ns) {
        ssd_scan_kernel<decltype(ns)::value, A><<<dim3(ceil_div(vdim, kRecCols), H, q->n_entries), 256, 0, st>>>(
            in.xbc, in.xbc_stride, in.proj, in.proj_stride, in.dt_off, in.A_log, in.dt_bias, in.D, q->state, q->slot_stride, q->o, H, G, dim, vdim,
            q->entry_row0, q->entry_slot, chunks ? q->scan_max : 0);
      });
    if (!ok || !chunks) return;
    float* totals = q->workspace + (int64_t)q->n_chunks * H * pad16(dim) * ssd_cols(vdim);
    const dim3 grid(q->n_chunks, H, ceil_div(vdim, kSsdCols));
    auto sums = &ssd_chunk_sum_kernel<A>;
    sums<<<grid, 256, with_lds(sums, (size_t)kDecayChunk * (stride_rows4(dim) + stride_rows4(kSsdCols)) * sizeof(float)), st>>>(
        in, q->workspace, totals, q->chunk_row0, q->chunk_rows);
    ssd_chunk_state_kernel<<<dim3(ceil_div((long)dim * vdim, 256), H, q->n_long), 256, 0, st>>>(
        q->workspace, totals, q->state, q->slot_stride, H, dim, vdim, q->long_chunk0, q->long_slot);
    auto out = [&](auto kern) {
      kern<<<grid, 256, with_lds(kern, (size_t)kDecayChunk * (stride_rows16(dim) + kSsdCols + 4) * sizeof(float)), st>>>(
          in, q->workspace, q->o, q->chunk_row0, q->chunk_rows);
    };
    if (dim <= 128) out(&ssd_chunk_out_kernel<A, 8>);
    else out(&ssd_chunk_out_kernel<A, 16>);
  });
  return known && ok ? (pegainfer_status_t)hipGetLastError() : bad;
}

pegainfer_status_t pegainfer_ssd_scan(const float* xbc, int64_t xbc_stride, const void* proj, int64_t proj_stride, int64_t dt_off,
                                      const void* A_log, const void* dt_bias, const void* D, float* state, int64_t slot_stride, float* o,
                                      int32_t heads, int32_t groups, int32_t n_state, int32_t vdim, const int32_t* entry_row0,
                                      const int32_t* entry_slot, int32_t n_entries, int32_t dtype, pegainfer_stream_t stream) {
  pegainfer_ssd_scan_desc q{};
  q.xbc = xbc; q.xbc_stride = xbc_stride; q.proj = proj; q.proj_stride = proj_stride; q.dt_off = dt_off;
  q.A_log = A_log; q.dt_bias = dt_bias; q.D = D; q.state = state; q.slot_stride = slot_stride; q.o = o;
  q.heads = heads; q.groups = groups; q.n_state = n_state; q.vdim = vdim;
  q.entry_row0 = entry_row0; q.entry_slot = entry_slot; q.n_entries = n_entries; q.dtype = dtype;
  return pegainfer_ssd_scan_form(&q, stream);
}

}  // extern "C"
