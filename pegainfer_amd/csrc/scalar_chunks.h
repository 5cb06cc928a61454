// The chunk form of linear recurrences with ONE decay per head and token (ssd.hip, recurrent.hip): S <- a S + b k v^T, read out by q, over
// long portions of ragged batches in chunks of <= 64 tokens that run side by side.
//   scalar_chunk_sum_kernel    U_c = sum_i w_i b_i k_i v_i^T with w_i the product of the decays behind token i, and the product of all
//                              the chunk's decays
//   scalar_chunk_state_kernel  walks the chunks of an entry that the run holds, S <- total_c S + U_c, and leaves the state BEFORE each in U_c's place
//   scalar_chunk_out_kernel    y_i = (a_1 .. a_i) S^T q_i + sum_{j <= i} (a_(j+1) .. a_i) b_j (q_i . k_j) v_j
// Decays enter as products of the decays themselves, never as quotients or differences of logarithms: every factor is at most one, nothing
// cancels however fast a head forgets, and the roundings of a product are those of a scan's state.
// Products run on v_mfma_f32_16x16x4_f32 (chunk_core.h).  Scores are computed transposed (keys as rows), which leaves lane l with the scores of
// query l % 16 against keys 4 (l / 16) + r: the A operand of the product with the values.  A later key's score is a zero there, so where a
// block of 16 tokens holds a value that is infinite or no number its own queries take the keys one by one (the product would bring it to the tokens
// before it): what is spoilt is what a token scan spoils.
// An In describes the recurrence: rows() / row_stride() of type Row with q_at, k_at, v_at of a head, q_factor; steps(chunk, head, row0, n, lane,
// &b, &a): lane i of a wave gets token i's factor and decay (0 and 1 past the chunk's end); H, dim, vdim; kNorm, floor_of, skip: see the outputs.
#pragma once

#include "common.h"
#include "typed.h"
#include "chunk_core.h"

namespace pk {

// [chunk][head][dim][columns] contributions, then states before the chunks; with a norm [chunk][head][dim] of the keys alone; totals
struct ScalarWs { float *state, *norm, *total; int first; };      // of the chunks from `first` on
constexpr int kScalarCols = 64;     // value columns of a workgroup
__host__ __device__ constexpr int scalar_cols(int vdim) { return (vdim + kScalarCols - 1) / kScalarCols * kScalarCols; }

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
template <typename In>
__global__ __launch_bounds__(256) void scalar_chunk_sum_kernel(In in, ScalarWs ws,
                                                            const int32_t* __restrict__ chunk_row0, const int32_t* __restrict__ chunk_rows) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ float s_w[kDecayChunk];
  const int slot = blockIdx.x, c = ws.first + slot, h = blockIdx.y, col0 = blockIdx.z * kScalarCols, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l15 = lane & 15, lg = lane >> 4, row0 = chunk_row0[c], n = chunk_rows[c];
  const int dp = pad16(in.dim), vp = scalar_cols(in.vdim), sk = stride_rows4(in.dim), sv = stride_rows4(kScalarCols);
  float *s_k = sm, *s_v = sm + kDecayChunk * sk;
  if (wave == 0) {
    float dt, a;
    in.steps(c, h, row0, n, lane, &dt, &a);
    const float w = product_behind(a, lane);
    s_w[lane] = w * dt;
    if (lane == 0 && blockIdx.z == 0) ws.total[(int64_t)slot * in.H + h] = w * a;
  }
  __syncthreads();
  auto same = [](float x) { return x; };
  stage_rows<4>(in.rows(), in.row_stride(), in.k_at(h), row0, n, in.dim, dp, s_k, sk, s_w, tid, same);
  stage_rows<4>(in.rows(), in.row_stride(), in.v_at(h) + col0, row0, n, min(kScalarCols, in.vdim - col0), kScalarCols, s_v, sv, nullptr, tid, same);
  __syncthreads();
  float* U = ws.state + ((int64_t)slot * in.H + h) * dp * vp + col0;
  if (In::kNorm && blockIdx.z == 0)                  // the keys alone: the state of a value that is one
    for (int d = tid; d < dp; d += 256) {
      float t = 0.f;
      for (int i = 0; i < n; ++i) t += s_k[i * sk + d];
      ws.norm[((int64_t)slot * in.H + h) * dp + d] = t;
    }
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
      for (int r = 0; r < 4; ++r) {
        const int d = d0 + 4 * lg + r;
        U[(int64_t)d * vp + 16 * b + l15] = d < in.dim ? acc[b][r] : 0.f;    // zeros of padding times an infinity would be no numbers
      }
  }
}

// One thread per element of the state: through the entry's chunks, the state before each left in U's place.
// NORM: dim more per head, the keys' own state behind the heads' matrices.
template <bool NORM>
__global__ __launch_bounds__(256) void scalar_chunk_state_kernel(ScalarWs ws, float* __restrict__ state, int64_t slot_stride, int H, int dim, int vdim,
                                                              const int32_t* __restrict__ long_chunk0, const int32_t* __restrict__ long_slot,
                                                              int n) {
  const int e = blockIdx.z, h = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
  const int j = i - dim * vdim;                            // >= 0: an element of the keys' state
  if (j >= (NORM ? dim : 0)) return;
  const int c_begin = max(long_chunk0[e] - ws.first, 0), c_end = min(long_chunk0[e + 1] - ws.first, n);     // places of the entry's chunks in this run
  if (c_begin >= c_end) return;
  const int dp = pad16(dim), vp = scalar_cols(vdim);
  float* sp = state + (int64_t)long_slot[e] * slot_stride + (j < 0 ? (int64_t)h * dim * vdim + i : (int64_t)H * dim * vdim + (int64_t)h * dim + j);
  const int64_t cs = (int64_t)H * dp * (j < 0 ? vp : 1);
  float* u = j < 0 ? ws.state + (int64_t)h * dp * vp + (int64_t)(i / vdim) * vp + i % vdim : ws.norm + (int64_t)h * dp + j;
  float S = *sp;
  for (int c0 = c_begin; c0 < c_end; c0 += 8) {      // eight chunks' loads in flight before the first store
    float t[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) t[k] = c0 + k < c_end ? u[(c0 + k) * cs] : 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (c0 + k < c_end) {
        u[(c0 + k) * cs] = S;
        S = fmaf(ws.total[(int64_t)(c0 + k) * H + h], S, t[k]);
      }
  }
  *sp = S;
}

// One workgroup per (chunk, head, 64 value columns), a wave per 16 queries.  Queries lie in registers (QB blocks of 16 state rows at most:
// lane (l15, lg) holds values 4 lg .. of each block, and the keys and the state before the chunk are read in the same numbering); keys
// and values in LDS.  A wave makes the decays between its own queries and all keys: lane j starts from the product of the decays between
// key j and the wave's first query and multiplies by one decay per query.
// In::kNorm: outputs divided by max(|n . q|, floor_of the token) + 1e-6, n = the keys' own state; its part inside the chunk is the sum of a
// query's scores, which the lanes of a query hold between them.
template <typename In, int QB>
__global__ __launch_bounds__(256) void scalar_chunk_out_kernel(In in, ScalarWs ws, float* __restrict__ o,
                                                            const int32_t* __restrict__ chunk_row0, const int32_t* __restrict__ chunk_rows) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  constexpr int sp = kDecayChunk + 4, sv = kScalarCols + 4;
  __shared__ __attribute__((aligned(16))) float s_p[kDecayChunk][sp];   // [query][key] decay between them, times the key's step size
  const int slot = blockIdx.x, c = ws.first + slot, h = blockIdx.y, col0 = blockIdx.z * kScalarCols, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l15 = lane & 15, lg = lane >> 4, row0 = chunk_row0[c], n = chunk_rows[c], i0 = wave * 16;
  const int dim = in.dim, dp = pad16(dim), vp = scalar_cols(in.vdim), sk = stride_rows16(dim), vd = min(kScalarCols, in.vdim - col0);
  float *s_k = sm, *s_v = s_k + kDecayChunk * sk;
  f32x4 q[QB];
  {
    const typename In::Row* src = in.rows() + (int64_t)(row0 + min(i0 + l15, n - 1)) * in.row_stride() + in.q_at(h);
    const bool vec = (reinterpret_cast<uintptr_t>(src) & (4 * sizeof(*src) - 1)) == 0 && (dim & 3) == 0;
    const float f = in.q_factor();
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      const int k = 16 * b + 4 * lg;
      if (vec) {
        float t[4];
        ld4(src + (k < dim ? k : 0), t);
        q[b] = f32x4{t[0], t[1], t[2], t[3]} * f;
        if (k >= dim) q[b] = f32x4{0.f, 0.f, 0.f, 0.f};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) q[b][e] = k + e < dim ? ld(src + k + e) * f : 0.f;
      }
    }
  }
  auto same = [](float x) { return x; };
  stage_rows<4>(in.rows(), in.row_stride(), in.k_at(h), row0, n, dim, dp, s_k, sk, nullptr, tid, same);
  stage_rows<4>(in.rows(), in.row_stride(), in.v_at(h) + col0, row0, n, vd, kScalarCols, s_v, sv, nullptr, tid, same);
  float before;                                      // product of the decays up to and with query i0 + l15
  {
    float dt, a;
    in.steps(c, h, row0, n, lane, &dt, &a);
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
    const float* S = ws.state + ((int64_t)slot * in.H + h) * dp * vp + col0 + (int64_t)(4 * lg) * vp + l15;
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
  float nq = 0.f;                                    // this lane's part of n . q
  if constexpr (In::kNorm) {
    const float* N = ws.norm + ((int64_t)slot * in.H + h) * dp + 4 * lg;
#pragma unroll
    for (int kb = 0; kb < QB; ++kb) {
      if (16 * kb >= dp) break;
      const f32x4 v = *reinterpret_cast<const f32x4*>(N + 16 * kb);
#pragma unroll
      for (int e = 0; e < 4; ++e) nq = fmaf(q[kb][e], v[e], nq);
    }
    nq *= before;
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
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = jb * 16 + 4 * lg + r <= i0 + l15 ? s[0][r] * w[r] : 0.f;
      if constexpr (In::kNorm) nq += p[r];
    }
    const float* vr = s_v + (jb * 16 + 4 * lg) * sv + l15;
    if (jb == wave) {
      bool spoilt = false;                           // a value that is infinite or no number: not for the queries before it
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int b = 0; b < 4; ++b) spoilt |= !(fabsf(vr[r * sv + 16 * b]) <= __FLT_MAX__);
      if (__any(spoilt)) {
        for (int k = 0; k < 16; ++k)                 // one key after the other, each query row of this lane on its own
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int src = (k >> 2) * 16 + 4 * lg + r;                     // the lane that holds p of query 4 lg + r and key k
            const float a = __shfl(p[0], src, kWave), c = __shfl(p[1], src, kWave), d = __shfl(p[2], src, kWave), e = __shfl(p[3], src, kWave);
            const float pk = (k & 2) ? ((k & 1) ? e : d) : ((k & 1) ? c : a);
            if (k <= 4 * lg + r) {
#pragma unroll
              for (int b = 0; b < 4; ++b) acc[b][r] = fmaf(pk, s_v[(jb * 16 + k) * sv + 16 * b + l15], acc[b][r]);
            }
          }
        continue;                                    // the last block of keys
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[r], vr[r * sv + 16 * b], acc[b], 0, 0, 0);
  }
  float den = 1.0f;                                  // of query i0 + l15
  if constexpr (In::kNorm) {
    nq += __shfl_xor(nq, 16, kWave);
    nq += __shfl_xor(nq, 32, kWave);
    den = fmaxf(fabsf(nq), in.floor_of(c, h, min(i0 + l15, n - 1))) + 1e-6f;
  }
  const float skip = In::kNorm ? 0.f : in.skip(h);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + 4 * lg + r;
    const float dr = In::kNorm ? __shfl(den, 4 * lg + r, kWave) : 1.0f;
    if (i >= n) continue;
    float* out = o + (int64_t)(row0 + i) * ((int64_t)in.H * in.vdim) + (int64_t)h * in.vdim + col0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int col = 16 * b + l15;
      if (col >= vd) continue;
      if constexpr (In::kNorm) out[col] = acc[b][r] / dr;
      else out[col] = fmaf(skip, s_v[i * sv + col], acc[b][r]);
    }
  }
}

// What the three launches of n_chunks chunks need, and they themselves.  A long step's chunks are walked in runs, one behind the other, whose
// states take 256 MB at most (or one chunk's): 256 chunks, 16 384 tokens, at 32 heads of 128 states x 64 values.
constexpr int64_t kScalarRunFloats = (int64_t)1 << 26;
inline int64_t scalar_chunk_each(int heads, int dim, int vdim, bool norm) {
  return (int64_t)heads * ((int64_t)pad16(dim) * (scalar_cols(vdim) + (norm ? 1 : 0)) + 1);
}
inline int scalar_chunk_run(int n_chunks, int heads, int dim, int vdim, bool norm) {
  const int64_t fit = kScalarRunFloats / scalar_chunk_each(heads, dim, vdim, norm);
  return (int)(fit >= n_chunks ? n_chunks : fit > 0 ? fit : 1);
}
inline int64_t scalar_chunk_floats(int n_chunks, int heads, int dim, int vdim, bool norm) {
  return n_chunks <= 0 ? 0 : scalar_chunk_run(n_chunks, heads, dim, vdim, norm) * scalar_chunk_each(heads, dim, vdim, norm);
}
template <typename In>
inline void scalar_chunk_launch(const In& in, float* workspace, float* state, int64_t slot_stride, float* o, const int32_t* chunk_row0,
                                const int32_t* chunk_rows, int n_chunks, const int32_t* long_chunk0, const int32_t* long_slot, int n_long,
                                hipStream_t st) {
  const int H = in.H, dim = in.dim, vdim = in.vdim, dp = pad16(dim), run = scalar_chunk_run(n_chunks, H, dim, vdim, In::kNorm);
  const int64_t slots = (int64_t)run * H;
  ScalarWs ws;
  ws.state = workspace;
  ws.norm = workspace + slots * dp * scalar_cols(vdim);
  ws.total = ws.norm + (In::kNorm ? slots * dp : 0);
  auto sums = &scalar_chunk_sum_kernel<In>;
  const size_t sum_lds = with_lds(sums, (size_t)kDecayChunk * (stride_rows4(dim) + stride_rows4(kScalarCols)) * sizeof(float));
  auto out = dim <= 128 ? &scalar_chunk_out_kernel<In, 8> : &scalar_chunk_out_kernel<In, 16>;
  const size_t out_lds = with_lds(out, (size_t)kDecayChunk * (stride_rows16(dim) + kScalarCols + 4) * sizeof(float));
  for (int c0 = 0; c0 < n_chunks; c0 += run) {
    const int n = n_chunks - c0 < run ? n_chunks - c0 : run;
    const dim3 grid(n, H, ceil_div(vdim, kScalarCols));
    ws.first = c0;
    sums<<<grid, 256, sum_lds, st>>>(in, ws, chunk_row0, chunk_rows);
    scalar_chunk_state_kernel<In::kNorm><<<dim3(ceil_div((long)dim * (vdim + (In::kNorm ? 1 : 0)), 256), H, n_long), 256, 0, st>>>(
        ws, state, slot_stride, H, dim, vdim, long_chunk0, long_slot, n);
    out<<<grid, 256, out_lds, st>>>(in, ws, o, chunk_row0, chunk_rows);
  }
}

}  // namespace pk
