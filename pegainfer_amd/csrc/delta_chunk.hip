// The gated delta rule of recurrent.hip (one decay per head) for prompts: 16 tokens at a time on fp32 matrix-core products.
//   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
// Token by token the recurrence is a chain of one state update per token, 374 cycles of it a token with one wave per SIMD (53 instructions of its
// own, waits for the rest).  Over a chunk the updates are known from the state S0 before it: with c_t = g_0 .. g_t and D[t][s] = g_{s+1} .. g_t
//   U = T' (V - diag(c) K S0),   T' = (I + L)^-1 diag(beta),   L[t][s] = beta_t D[t][s] k_t . k_s  (s < t)
//   O = diag(c) Q S0 + M U,      M[t][s] = D[t][s] q_t . k_s   (s <= t)
//   S = c_15 S0 + K^T diag(D[15][.]) U
// delta_chunk_prep_kernel brings q and k to unit length and makes T', M and the factors for every (chunk, head) side by side; delta_chunk_kernel walks the chunks of an (entry,
// head, 16 value columns), its four waves dim / 4 rows of S each.  All products are v_mfma_f32_16x16x4_f32 (plain fp32) and every decay is a product of
// gates at most 1, never a quotient, so strong decays only underflow as they do one by one.
// 1024 tokens of 32 heads of 128 x 128 over 16 key heads, prep and all: 187 us token by token, 88 here (traced 18 + 75); eight entries of 700 tokens, 8 heads
// over 4: 175 and 115.
// Against 64 bits the read-outs are off by 2.0e-7 with slow decays (2.3e-7 token by token), by 0.85 - 1.0e-7 with fast ones (1.1 - 1.2e-7): lengths and the
// products k . k, q . k are made in 64 bits and rounded once (in fp32 sums the fast ones were off by 1.2 - 1.4e-7).  fp32 logits of whole models are off by the
// same either way (0.9 - 1.8e-6).
// The triangular matrices hold zeros for later tokens, and a zero times what is infinite or no number is no number: such values are kept out of the
// products of the chunk they appear in and spoil its outputs from their own token on, column by column, as they do token by token.
#include <algorithm>

#include "common.h"
#include "typed.h"
#include "sigmoid_power.h"
#include "delta_scan.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kDc = 16;                        // tokens of a chunk
constexpr int kDcFloats = 2 * kDc * kDc + 2 * kDc + 32;  // of a (chunk, head): T', M, c, D[15][.], pad

// Chunks are numbered without a table: entry e's first is row0 / 16 + e (the next entry's first lies behind its last), so there are
// rows / 16 + entries numbers at most and some that stand for none.
__device__ __forceinline__ int delta_first_chunk(int row0, int e) { return row0 / kDc + e; }
// A long step's chunks are walked in runs, one behind the other, whose matrices take 256 MB at most (or one chunk's): 3640 chunks at 32 heads.
constexpr int64_t kDcRunFloats = (int64_t)1 << 26;
static int64_t delta_chunk_run(int64_t chunks, int heads) { return std::max<int64_t>(1, std::min(chunks, kDcRunFloats / ((int64_t)heads * kDcFloats))); }

// A wave per (chunk, key head): k . k and q . k of the chunk's tokens, then, sixteen lanes per value head, the triangular matrix and its inverse
// by forward substitution, a lane per column.
// MIXED: the entries of up to scan_max rows are prepared for the token-by-token form, by workgroups of their own behind the chunks'.
template <typename A, int NB, bool MIXED>
__global__ __launch_bounds__(256) void delta_chunk_prep_kernel(float* __restrict__ qkv, int64_t qkv_stride, const A* __restrict__ proj,
                                                               int64_t proj_stride, int64_t b_off, int64_t a_off, const A* __restrict__ A_log,
                                                               const A* __restrict__ dt_bias, float* __restrict__ ws, int H, int G,
                                                               const int32_t* __restrict__ entry_row0, int n_entries, int scan_max, int run0, int run, float* gates) {
  constexpr int DIM = 64 * NB;
  if (MIXED && (int)blockIdx.x >= run) {
    const int row = blockIdx.x - run, e = entry_of_row(entry_row0, n_entries, row);
    if (entry_row0[e + 1] - entry_row0[e] <= scan_max)
      delta_prep_row<A>(row, blockIdx.y, gridDim.y, qkv, qkv_stride, proj, proj_stride, b_off, a_off, A_log, dt_bias, gates, H, G, DIM);
    return;
  }
  __shared__ float s_kk[4][kDc][kDc + 1], s_qk[4][kDc][kDc + 1];
  __shared__ __attribute__((aligned(16))) float s_l[4][4][kDc][kDc + 4], s_gb[4][4][kDc][2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, t = lane & 15, j = lane >> 4;
  const int chunk = run0 + blockIdx.x, g = blockIdx.y * 4 + wave;
  int lo = 0, hi = n_entries - 1;              // the last entry whose first chunk is not behind this one
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (delta_first_chunk(entry_row0[mid], mid) <= chunk) lo = mid; else hi = mid - 1;
  }
  const int row0 = entry_row0[lo], len = entry_row0[lo + 1] - row0, at = (chunk - delta_first_chunk(row0, lo)) * kDc;
  if (at < 0 || at >= len || len <= scan_max || g >= G) return;   // (waves share nothing: there is no barrier below)
  const int tc = min(kDc, len - at);
  const int64_t row = row0 + at + min(t, tc - 1);
  const float live = t < tc ? 1.f : 0.f;
  // lane: token t, dims 16 b + 4 j .. + 3 - both operands of the products below
  f32x4 k[DIM / 16], q[DIM / 16];
  float *qp = qkv + row * qkv_stride + (int64_t)g * DIM + 4 * j, *kp = qp + (int64_t)G * DIM;
#pragma unroll
  for (int b = 0; b < DIM / 16; ++b) {
    k[b] = *reinterpret_cast<const f32x4*>(kp + 16 * b);
    q[b] = *reinterpret_cast<const f32x4*>(qp + 16 * b);
  }
  // Lengths and products in 64 bits, each rounded once: a read-out of strong decays is little more than q_t . k_t times its token's own update,
  // where token by token 128 roundings of S average out.
  double kss = 0, qss = 0;
#pragma unroll
  for (int b = 0; b < DIM / 16; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      k[b][r] = t < tc ? k[b][r] : 0.f;
      q[b][r] = t < tc ? q[b][r] : 0.f;
      kss = fma((double)k[b][r], (double)k[b][r], kss);
      qss = fma((double)q[b][r], (double)q[b][r], qss);
    }
  kss += __shfl_xor(kss, 16, kWave); kss += __shfl_xor(kss, 32, kWave);
  qss += __shfl_xor(qss, 16, kWave); qss += __shfl_xor(qss, 32, kWave);
  const float ik = (float)(1.0 / sqrt(kss + 1e-6)), iq = (float)(1.0 / sqrt((qss + 1e-6) * DIM));
  f64x4 kk[2] = {}, qk[2] = {};
#pragma unroll
  for (int b = 0; b < DIM / 16; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      k[b][r] *= ik;
      q[b][r] *= iq;
      const double kd = k[b][r], qd = q[b][r];
      kk[r & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(kd, kd, kk[r & 1], 0, 0, 0);
      qk[r & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(qd, kd, qk[r & 1], 0, 0, 0);
    }
  if (t < tc) {
#pragma unroll
    for (int b = 0; b < DIM / 16; ++b) {
      *reinterpret_cast<f32x4*>(kp + 16 * b) = k[b];
      *reinterpret_cast<f32x4*>(qp + 16 * b) = q[b];
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {                // lane: rows 4 r + j, column t (64-bit products leave them in that order)
    s_kk[wave][4 * r + j][t] = (float)(kk[0][r] + kk[1][r]);
    s_qk[wave][4 * r + j][t] = (float)(qk[0][r] + qk[1][r]);
  }
  const int per = H / G;
  for (int h0 = 0; h0 < per; h0 += 4) {
    const int h = g * per + min(h0 + j, per - 1);
    const bool own = h0 + j < per;
    const A* pr = proj + row * proj_stride;
    const float gt = live > 0.f ? expf(-expf(ld(A_log + h)) * softplus_f(ld(pr + a_off + h) + ld(dt_bias + h))) : 1.f;
    const float bt = live * sigmoid_f(ld(pr + b_off + h));
    s_gb[wave][j][t][0] = gt;
    s_gb[wave][j][t][1] = bt;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");          // a wave's own LDS writes, in its own order
    float* out = ws + ((int64_t)blockIdx.x * H + h) * kDcFloats;
    // lane: column t of head h; p = D[row][t]
    float p = 0.f;
#pragma unroll
    for (int i = 0; i < kDc; ++i) {
      const float gi = s_gb[wave][j][i][0], bi = s_gb[wave][j][i][1];
      p = i == t ? 1.f : p * gi;               // 0 above the diagonal
      s_l[wave][j][i][t] = i > t ? bi * p * s_kk[wave][i][t] : 0.f;
      if (own) out[kDc * kDc + i * kDc + t] = i >= t ? p * s_qk[wave][i][t] : 0.f;
      if (t == 0 && own) out[2 * kDc * kDc + i] = s_gb[wave][j][0][0] * p;     // c_i = g_0 D[i][0]
    }
    if (own) out[2 * kDc * kDc + kDc + t] = p;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    float T[kDc];
#pragma unroll
    for (int i = 0; i < kDc; ++i) {
      float sum[2] = {};
#pragma unroll
      for (int s4 = 0; s4 * 4 < i; ++s4) {
        const f32x4 l = *reinterpret_cast<const f32x4*>(&s_l[wave][j][i][4 * s4]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (4 * s4 + u < i) sum[u & 1] = fmaf(l[u], T[4 * s4 + u], sum[u & 1]);
      }
      T[i] = i == t ? 1.f : i > t ? -(sum[0] + sum[1]) : 0.f;
      if (own) out[i * kDc + t] = i >= t ? T[i] * bt : 0.f;      // (zeros also where bt is no number)
    }
  }
}

// Bound by its chain of products: 4 NB for K S0, as many for Q S0, 4 for U and 4 NB for S, 32 cycles each, and one exchange through LDS per chunk.
// S lies as the products leave it, which is also how they take it: accumulator r of block b is a wave's row NB (4 (lane / 16) + r) + b of S, so
// K and Q come as 16-byte loads in that order of k (and K's other operand, a lane per row, NB values at a time), and U's accumulators are
// the next product's operand in the same way.  Vector memory takes 16 cycles an instruction whatever it carries, so what all four waves need is
// fetched by a fifth, which also makes the outputs; nothing waits for those.  Operands are asked for two chunks ahead.
constexpr int kDcThreads = 320;
// MIXED: the workgroups of entries of up to scan_max rows go token by token, four of their five waves (a launch of its own would follow this one).
template <int NB, bool MIXED>
__global__ __launch_bounds__(kDcThreads) void delta_chunk_kernel(const float* qkv, int qkv_stride, const float* ws, float* __restrict__ state,
                                                                 int64_t slot_stride, float* __restrict__ o, int H, int G, int vdim,
                                                                 const int32_t* __restrict__ entry_row0, const int32_t* __restrict__ entry_slot, int scan_max, int run0, int run, const float* gates) {
  constexpr int DIM = 64 * NB;
  __shared__ f32x4 s_part[2][4][2][64];        // K S0 and Q S0 over a wave's rows of S
  __shared__ f32x4 s_common[2][4][64];         // by lane: values, T', c, D[15][.]
  __shared__ float s_end[2];
  const int e = blockIdx.z, h = blockIdx.y, col = blockIdx.x * 16 + (threadIdx.x & 15);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l15 = lane & 15, j = lane >> 4;
  int row0 = entry_row0[e], len = entry_row0[e + 1] - row0;
  if (len <= scan_max) {                       // (0: empty ones)
    if (MIXED && run0 == 0 && len > 0 && wave < 4) {
      constexpr int NS = NB == 1 ? 4 : NB == 2 ? 8 : 16;       // as by_slices does
      delta_rule_block<NS, false>(blockIdx.x, h, e, qkv, qkv_stride, gates, state, slot_stride, o, H, G, DIM, vdim, entry_row0, entry_slot);
    }
    return;
  }
  int place = delta_first_chunk(row0, e) - run0;               // of the entry's first chunk in this run
  {
    const int from = max(-place, 0), to = min((len + kDc - 1) / kDc, run - place);
    if (from >= to) return;
    row0 += from * kDc;
    len = min(len, to * kDc) - from * kDc;
    place += from;
  }
  const int n = (len + kDc - 1) / kDc, g0 = h / (H / G);
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };     // (not the loads of the chunks ahead)
  // rows past the entry's end: its last one, which T' leaves out
  auto row_at = [&](int c, int t) { return (int64_t)(row0 + min(c * kDc + t, len - 1)) * qkv_stride; };
  auto sum_of_waves = [&](int c, int which) {
    const auto& part = s_part[c & 1];
    return (part[0][which][lane] + part[1][which][lane]) + (part[2][which][lane] + part[3][which][lane]);
  };
  auto times = [&](const f32x4& a, const f32x4& b) {           // of a lower triangle and a chunk's rows
    f32x4 D = {};
#pragma unroll
    for (int s = 0; s < 4; ++s) D = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], D, 0, 0, 0);
    return D;
  };
  // The same for the outputs: what is not finite enters as zero, and the rows from the first such one of a column on are no numbers.  (For S the
  // plain product does: its column is no number anyway.)
  auto finite_times = [&](const f32x4& a, f32x4 b) {
    int first = kDc;
    const bool spoilt = __any(!(fabsf(b[0]) + fabsf(b[1]) + (fabsf(b[2]) + fabsf(b[3])) <= __FLT_MAX__));      // (or a sum past the largest number)
    if (spoilt) {
#pragma unroll
      for (int r = 3; r >= 0; --r)
        if (!(fabsf(b[r]) <= __FLT_MAX__)) { first = 4 * j + r; b[r] = 0.f; }
      first = min(first, __shfl_xor(first, 16, kWave));
      first = min(first, __shfl_xor(first, 32, kWave));
    }
    f32x4 D = times(a, b);
    if (spoilt) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * j + r >= first) D[r] = __builtin_nanf("");
    }
    return D;
  };
  // Chunk c's operands in x; those of c + 1 are on the way while it is worked on, those of c + 2 are asked for.  One loop with one way out: with
  // more, the compiler's waits at its head have to cover them all.  `whole`: all of the chunk's rows are there.
  auto walk = [&](auto& x, auto& y, auto& z, auto&& fetch, auto&& work) {
    fetch(x, 0);
    fetch(y, 1);
    int c = 0;
    for (; (c + 3) * kDc <= len; c += 3) {
      fetch(z, c + 2);
      work(x, c, std::true_type());
      fetch(x, c + 3);
      work(y, c + 1, std::true_type());
      fetch(y, c + 4);
      work(z, c + 2, std::true_type());
    }
    if (c + 2 < n) fetch(z, c + 2);
    if (c < n) work(x, c, std::false_type());
    if (c + 1 < n) work(y, c + 1, std::false_type());
    if (c + 2 < n) work(z, c + 2, std::false_type());
  };
  if (wave == 4) {
    const float *w0 = ws + ((int64_t)place * H + h) * kDcFloats, *v0 = qkv + (int64_t)2 * G * DIM + (int64_t)h * vdim + col;
    struct Chunk { f32x4 v, T, M, decay, left; float end; } x, y, z;
    auto fetch = [&](Chunk& x, int c) {
      // asked for here and in this order: the compiler would gather the loads of three chunks, whose waits are then one (the pointers are not
      // `__restrict__`, so that these hold)
      asm volatile("" ::: "memory");
      c = min(c, n - 1);
      const float *w = w0 + (int64_t)c * H * kDcFloats, *f = w + 2 * kDc * kDc;
#pragma unroll
      for (int s = 0; s < 4; ++s) x.v[s] = v0[row_at(c, 4 * j + s)];
      x.T = *reinterpret_cast<const f32x4*>(w + l15 * kDc + 4 * j);
      x.M = *reinterpret_cast<const f32x4*>(w + kDc * kDc + l15 * kDc + 4 * j);
      x.decay = *reinterpret_cast<const f32x4*>(f + 4 * j);
      x.left = *reinterpret_cast<const f32x4*>(f + kDc + 4 * j);
      x.end = f[kDc - 1];
      asm volatile("" ::: "memory");
    };
    auto work = [&](const Chunk& x, int c, auto whole) {
      auto& to = s_common[c & 1];
      to[0][lane] = x.v;
      to[1][lane] = x.T;
      to[2][lane] = x.decay;
      to[3][lane] = x.left;
      if (lane == 0) s_end[c & 1] = x.end;
      barrier();
      const f32x4 Q = sum_of_waves(c, 1);
      f32x4 O = finite_times(x.M, finite_times(x.T, x.v - x.decay * sum_of_waves(c, 0)));
#pragma unroll
      for (int r = 0; r < 4; ++r) O[r] = fmaf(x.decay[r], Q[r], O[r]);
      float* out = o + (int64_t)(row0 + c * kDc) * ((int64_t)H * vdim) + (int64_t)h * vdim + col;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (whole.value || c * kDc + 4 * j + r < len) out[(int64_t)(4 * j + r) * (H * vdim)] = O[r];
    };
    walk(x, y, z, fetch, work);
    return;
  }
  const int d0 = wave * 16 * NB;
  float* S_g = state + (int64_t)entry_slot[e] * slot_stride + (int64_t)h * DIM * vdim + col;
  f32x4 S[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[b][r] = S_g[(int64_t)(d0 + NB * (4 * j + r) + b) * vdim];
#pragma unroll
  for (int b = 0; b < NB; ++b) asm volatile("" : "+v"(S[b]));    // waited for here: the wait must not land in the loop
  const float *q0 = qkv + (int64_t)g0 * DIM + d0, *k0 = q0 + (int64_t)G * DIM;
  struct Chunk { float k[4 * NB], q[4 * NB], kt[4][NB]; } x, y, z;
  auto fetch = [&](Chunk& x, int c) {
    asm volatile("" ::: "memory");
    c = min(c, n - 1);
    const int64_t mine = row_at(c, l15) + 4 * NB * j;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      ld4(k0 + mine + 4 * b, &x.k[4 * b]);
      ld4(q0 + mine + 4 * b, &x.q[4 * b]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) __builtin_memcpy(x.kt[s], __builtin_assume_aligned(k0 + row_at(c, 4 * j + s) + NB * l15, NB % 4 == 0 ? 16 : NB % 2 == 0 ? 8 : 4), 4 * NB);
    asm volatile("" ::: "memory");
  };
  auto work = [&](const Chunk& x, int c, auto) {
    f32x4 P[4] = {}, Q[4] = {};
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        P[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[NB * r + b], S[b][r], P[r], 0, 0, 0);
        Q[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[NB * r + b], S[b][r], Q[r], 0, 0, 0);
      }
    s_part[c & 1][wave][0][lane] = (P[0] + P[1]) + (P[2] + P[3]);
    s_part[c & 1][wave][1][lane] = (Q[0] + Q[1]) + (Q[2] + Q[3]);
    barrier();
    const auto& from = s_common[c & 1];
    const f32x4 left = from[3][lane];
    const float end = s_end[c & 1];
    const f32x4 E = left * times(from[1][lane], from[0][lane] - from[2][lane] * sum_of_waves(c, 0));
    f32x4 X[NB] = {};                          // (a sum of its own, so that S is rounded once per chunk)
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int b = 0; b < NB; ++b) X[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[s][b], E[s], X[b], 0, 0, 0);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[b][r] = fmaf(end, S[b][r], X[b][r]);
  };
  walk(x, y, z, fetch, work);
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) S_g[(int64_t)(d0 + NB * (4 * j + r) + b) * vdim] = S[b][r];
}

template <typename F>
static bool by_rows_of_s(int dim, F&& fn) {
  if (dim == 64) fn(std::integral_constant<int, 1>());
  else if (dim == 128) fn(std::integral_constant<int, 2>());
  else if (dim == 192) fn(std::integral_constant<int, 3>());
  else if (dim == 256) fn(std::integral_constant<int, 4>());
  else return false;
  return true;
}

}  // namespace pk

extern "C" {
using namespace pk;

int64_t pegainfer_delta_rule_workspace(int32_t n_rows, int32_t n_entries, int32_t heads) {
  return n_rows <= 0 || n_entries <= 0 || heads <= 0 ? 0 : delta_chunk_run((int64_t)n_rows / kDc + n_entries, heads) * heads * kDcFloats;
}

int32_t pegainfer_delta_rule_chunked_ok(int32_t dim, int32_t vdim, const float* qkv, int64_t qkv_stride) {
  return (dim == 64 || dim == 128 || dim == 192 || dim == 256) && vdim > 0 && vdim % 16 == 0 && qkv_stride % 4 == 0 && qkv_stride <= INT32_MAX && host_aligned16(qkv);
}

pegainfer_status_t pegainfer_delta_rule_by_length(float* qkv, int64_t qkv_stride, const void* proj, int64_t proj_stride, int64_t b_off,
                                                  int64_t a_off, const void* A_log, const void* dt_bias, float* workspace, float* state,
                                                  int64_t slot_stride, float* o, int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim,
                                                  int32_t n_rows, const int32_t* entry_row0, const int32_t* entry_slot, int32_t n_entries,
                                                  int32_t scan_max, float* gates, int32_t dtype, pegainfer_stream_t stream) {
  constexpr pegainfer_status_t bad = (pegainfer_status_t)hipErrorInvalidValue;
  if (n_entries <= 0 || n_rows <= 0) return 0;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || heads > 65535 || (int64_t)heads * vdim > (1 << 24) || n_entries > 65535 || scan_max < 0 || (scan_max > 0 && !gates) || !workspace || !host_aligned16(workspace) ||
      !pegainfer_delta_rule_chunked_ok(dim, vdim, qkv, qkv_stride))
    return bad;
  hipStream_t st = as_stream(stream);
  const int chunks = n_rows / kDc + n_entries, run = (int)delta_chunk_run(chunks, heads);
  const bool known = by_dtype(dtype, [&](auto* ptr) {
    using A = std::remove_pointer_t<decltype(ptr)>;
    by_rows_of_s(dim, [&](auto nb) {
      constexpr int NB = decltype(nb)::value;
      auto go = [&](auto mixed) {
        constexpr bool MIXED = decltype(mixed)::value;
        for (int c = 0; c < chunks; c += run) {
          const int n = std::min(run, chunks - c), rows = MIXED && c == 0 ? n_rows : 0;
          delta_chunk_prep_kernel<A, NB, MIXED><<<dim3(n + rows, ceil_div(kv_heads, 4)), 256, 0, st>>>(
              qkv, qkv_stride, static_cast<const A*>(proj), proj_stride, b_off, a_off, static_cast<const A*>(A_log), static_cast<const A*>(dt_bias), workspace,
              heads, kv_heads, entry_row0, n_entries, scan_max, c, n, gates);
          delta_chunk_kernel<NB, MIXED><<<dim3(vdim / 16, heads, n_entries), kDcThreads, 0, st>>>(qkv, (int)qkv_stride, workspace, state, slot_stride, o, heads,
                                                                                                  kv_heads, vdim, entry_row0, entry_slot, scan_max, c, n, gates);
        }
      };
      if (scan_max > 0) go(std::true_type());
      else go(std::false_type());
    });
  });
  return known ? (pegainfer_status_t)hipGetLastError() : bad;
}

pegainfer_status_t pegainfer_delta_rule_chunked(float* qkv, int64_t qkv_stride, const void* proj, int64_t proj_stride, int64_t b_off,
                                                int64_t a_off, const void* A_log, const void* dt_bias, float* workspace, float* state,
                                                int64_t slot_stride, float* o, int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim,
                                                int32_t n_rows, const int32_t* entry_row0, const int32_t* entry_slot, int32_t n_entries,
                                                int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_delta_rule_by_length(qkv, qkv_stride, proj, proj_stride, b_off, a_off, A_log, dt_bias, workspace, state, slot_stride, o, heads, kv_heads,
                                        dim, vdim, n_rows, entry_row0, entry_slot, n_entries, 0, nullptr, dtype, stream);
}

}  // extern "C"
