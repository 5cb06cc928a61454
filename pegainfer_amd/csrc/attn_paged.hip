// Softmax attention over a paged key/value cache for any head sizes and grouped key/value heads, in a bf16 and an fp32
// storage instance; norms, angles, scores, softmax state and accumulators are fp32 in both.
//   qk_prep_paged_kernel       one or several workgroups per token row, a wave per head: optional bias, optional RMS norm over the head
//                              (plain weight), optional position-dependent query factor (query temperature), rotation
//                              of neighbouring pairs (2i, 2i + 1) of the first rot_dims values by position * inv_freq[i],
//                              queries to an fp32 buffer, keys and values into the cache entry of (request, position)
//   paged_attention_kernel     one workgroup per (row tile, key/value head): up to 16 (token, query head) rows that share the
//                              key/value head; key and value tiles of 64 positions are staged once in LDS (fp32) for all
//                              rows; a wave owns up to four rows and takes them through a tile together (a key or value
//                              read from LDS serves four products), a lane one key of the tile for the scores and value
//                              columns lane, lane + 64, ... for the output; running maximum / sum per row.  Options
//                              (AttnForm): keys restricted to the query's own run of `block` positions, a per-head sink
//                              logit in the denominator, two softmax maps over the same values combined as
//                              map 1 - lambda * map 2, an RMS norm of the head's output
//   paged_attention_mfma_kernel  the same tiles on the matrix cores, for a bf16 cache
//   paged_attention_rows_kernel  prompts over a bf16 cache: 32 or 64 rows per workgroup, the next tile's values on their way
// Keys are always visited in tiles of 64 from position 0, whatever the step's shape, so a row's arithmetic does not depend on
// how its prompt was cut or on what else runs in the step.
#include <algorithm>

#include "common.h"
#include "typed.h"
#include "qk_prep_core.h"
#include "head_rms_core.h"
#include "recurrent_step.h"
#include "ssd_core.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

template <typename A, typename I, int V>
__global__ __launch_bounds__(256) void qk_prep_paged_kernel(pegainfer_qk_prep_desc p, PrepForm pf) {
  extern __shared__ float sm[];
  qk_prep_block<A, I, V>(sm, blockIdx.x, blockIdx.y, gridDim.y, p, pf);
}

constexpr int kAttKeys = 64;    // keys per staged tile
constexpr int kAttRows = 16;    // (token, query head) rows per workgroup
constexpr int kAttRpw = 4;      // rows per wave

// What the general kernel can do beyond plain causal softmax attention; a zeroed struct is the plain form.
struct AttnForm {
  int block = 0;               // > 0: a key is visible only inside the query's own run of `block` positions (runs counted from
                               // position 0 of the sequence), and not after the query
  const void* sink = nullptr;  // [heads] logits (storage type) that join the softmax denominator, unscaled, without a value
  float lambda = 0.f;          // MAPS == 2: out = map 1 - lambda * map 2 (two softmax maps over the same values; a query /
                               // key head holds [map 1 : dim | map 2 : dim])
  int head_norm = 0;           // != 0: out / sqrt(mean(out^2) + norm_eps) over the head's vdim values, before `factor`
  float norm_eps = 0.f;
  float softcap = 0.f;         // > 0: score <- softcap * tanh(score / softcap), after the scale
  int window = 0;              // > 0: a key j is visible to position i only if i - j < window or j < keep_first (kept first
  int keep_first = 0;          // tokens stay visible at their true positions)
  const float* dist_bias = nullptr;   // fp32 [n_dist][heads], added to the (scaled, capped) score of query head h by distance:
  int n_dist = 0;                     // dist_bias[min(i - j, n_dist - 1)][h]
  const float* dist_slope = nullptr;  // fp32 [heads]: slope[h] * (i - j) is taken off the (scaled, capped) score
  const void* gate = nullptr;  // output gate logits (storage type), rows at gate_stride: the finished head is multiplied by
  int64_t gate_stride = 0;     // sigmoid(gate[row, h * vdim + c]) (gate_kind 1: one per value) or sigmoid(gate[row, h]) (2: one
  int gate_kind = 0;           // per head)
  int k_keep = 0;              // values of a key in the cache's key part; the key's values from there on are its value's (MAPS == 1, the
                               // whole key unless values are projected as keys and only a part of a key is rotated)
};

// first position of the run of keys that position `pos` sees (besides the kept first tokens)
__device__ __forceinline__ int attn_row_lo(const AttnForm& form, int pos) {
  int lo = form.block > 0 ? (pos / form.block) * form.block : 0;
  if (form.window > 0) lo = max(lo, pos - form.window + 1);
  return lo;
}
// a raw dot product turned into the score of (query position rpos, key position kp, query head qh)
// slope: the head's entry of form.dist_slope, read once per row by the caller
__device__ __forceinline__ float attn_score(const AttnForm& form, float dot, float scale, int rpos, int kp, int qh, int H, float slope) {
  float sc = dot * scale;
  if (form.softcap > 0.f) sc = form.softcap * tanhf(sc / form.softcap);
  if (form.dist_bias) sc += form.dist_bias[(int64_t)min(rpos - kp, form.n_dist - 1) * H + qh];
  if (form.dist_slope) sc = fmaf(-slope, (float)(rpos - kp), sc);
  return sc;
}

// cap * tanh(x / cap) of eight scores in fp32: an odd series where tanh is nearly its argument (next term below 3e-7 of it), beyond it
// 1 - 2 / (e^2u + 1), which runs into +-1 without an infinity in between.  Scores of a wave that all lie below 0.35 cap take the series alone.
__device__ __forceinline__ void soft_cap8(f32x4 (&x)[2], float cap, float inv_cap) {
  float u[8], small[8];
  bool near = true;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    u[i] = x[i >> 2][i & 3] * inv_cap;
    const float u2 = u[i] * u[i];
    near = near && u2 < 0.1225f;
    small[i] = u[i] * fmaf(u2, fmaf(u2, fmaf(u2, fmaf(u2, 0.021869489f, -0.053968254f), 0.13333333f), -0.33333333f), 1.0f);
  }
  if (!__all(near)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float big = fmaf(-2.0f, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(u[i] * 2.8853900818f) + 1.0f), 1.0f);
      if (!(u[i] * u[i] < 0.1225f)) small[i] = big;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i >> 2][i & 3] = cap * small[i];
}

// What a row's end reads beside its softmax states: the sink's logit and its gate, raw.  A kernel that waits for other loads first asks for
// these with them.
template <typename A>
struct AttnEnd {
  A sink, gate[4];
  __device__ __forceinline__ AttnEnd(const AttnForm& form, int row, int qh, int vdim, int lane) : sink(), gate() {
    if (form.sink) sink = static_cast<const A*>(form.sink)[qh];
    const A* g = static_cast<const A*>(form.gate) + (int64_t)row * form.gate_stride;
    if (form.gate_kind == 2) gate[0] = g[qh];
    if (form.gate_kind == 1) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (lane + 64 * c < vdim) gate[c] = g[(int64_t)qh * vdim + lane + 64 * c];
    }
  }
};
// A row's softmax states (one per map) turned into its output: the sink joins every denominator, the maps are combined, the
// head is normed, `factor` comes last.  The wave holds the row: lane l has columns l, l + 64, ...
template <typename A, int MAPS>
__device__ __forceinline__ void attn_finish_row(float* mrun, float* lrun, float (*acc)[4], const AttnForm& form, const AttnEnd<A>& end,
                                                int vdim, float factor, int lane, A* __restrict__ dst) {
  float res[4];
  if (form.sink) {   // rescale to the larger of the two maxima first
    const float sk = ld(&end.sink);
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
      const float mnew = fmaxf(mrun[m], sk);
      const float corr = mrun[m] == -INFINITY ? 0.f : expf(mrun[m] - mnew);
      lrun[m] = lrun[m] * corr + expf(sk - mnew);
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[m][c] *= corr;
    }
  }
  if constexpr (MAPS == 1) {
    const float invl = 1.0f / lrun[0];
#pragma unroll
    for (int c = 0; c < 4; ++c) res[c] = acc[0][c] * invl;
  } else {
    const float inv0 = 1.0f / lrun[0], inv1 = form.lambda / lrun[MAPS - 1];
#pragma unroll
    for (int c = 0; c < 4; ++c) res[c] = acc[0][c] * inv0 - acc[MAPS - 1][c] * inv1;
  }
  float post = factor;
  if (form.head_norm) {
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (lane + 64 * c < vdim) ss = fmaf(res[c], res[c], ss);
    post = factor / sqrtf(wave_sum(ss) / (float)vdim + form.norm_eps);
  }
  if (form.gate_kind == 2) post *= sigmoid_f(ld(&end.gate[0]));
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (lane + 64 * c < vdim) {
      float v = res[c] * post;
      if (form.gate_kind == 1) v *= sigmoid_f(ld(&end.gate[c]));
      st(dst + lane + 64 * c, v);
    }
}
// key tiles that the rows of a tile walk, counted from their first: a split past them has nothing to do and leaves nothing
__device__ __forceinline__ int attn_key_tiles(int kfirst, int kmax) { return (kmax - kfirst + kAttKeys - 1) / kAttKeys; }
__device__ __forceinline__ int attn_first_key(const AttnForm& form, int pos0) {
  return form.keep_first > 0 ? 0 : (attn_row_lo(form, pos0) / kAttKeys) * kAttKeys;
}

template <typename A, int MAPS>
__global__ __launch_bounds__(256) void paged_attention_kernel(
    const float* __restrict__ q, const A* __restrict__ cache, int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
    int page_size, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_entry,
    const int32_t* __restrict__ page_indptr, const int32_t* __restrict__ page_ids, int H, int G, int dim, int vdim, float scale,
    float factor, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok,
    const int32_t* __restrict__ tile_qh0, const int32_t* __restrict__ tile_nqh, A* __restrict__ out, int64_t out_stride,
    AttnForm form, int nsplit, float* __restrict__ part) {
  extern __shared__ float sm[];
  const int qd = MAPS * dim;                          // values of one query / key head (all maps)
  const int kd = qd + 1;                              // padded key row: a lane per key reads its row without bank conflicts
  float* s_k = sm;                                    // [64][qd + 1]
  float* s_v = s_k + kAttKeys * kd;                   // [64][vdim]
  float* s_q = s_v + kAttKeys * vdim;                 // [16][qd]
  float* s_p = s_q + kAttRows * qd;                   // [4 waves][MAPS][64 keys][4 rows of the wave]
  // 16-byte loads from the cache: every key / value row of the request starts at a multiple of eight values
  const int kw = form.k_keep;                         // values of a head in the cache's key part
  const bool tail = kw < qd;                          // the others are staged with the values
  const bool vec_k = (kw & 7) == 0 && (page_stride & 7) == 0 && (k_cache_off & 7) == 0 && aligned16(cache);
  const bool vec_v = (vdim & 7) == 0 && (kw & 7) == 0 && (page_stride & 7) == 0 && (v_cache_off & 7) == 0 && aligned16(cache);
  const int tile = blockIdx.x, g = blockIdx.y;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int row0 = tile_row0[tile], ntok = tile_ntok[tile], qh0 = tile_qh0[tile], nqh = tile_nqh[tile];
  const int nrows = ntok * nqh, per_group = H / G;
  const int e = row_entry[row0];
  const int32_t* pages = page_ids + page_indptr[e];
  const int kmax = positions[row0 + ntok - 1] + 1;    // keys 0 .. kmax - 1 are visible to the tile's last token
  // the first key any row of the tile sees, rounded down to the 64-key grid that starts at position 0
  const int lo0 = attn_row_lo(form, positions[row0]);   // rows of a tile are in position order: the lowest run start
  const int kfirst = attn_first_key(form, positions[row0]);
  if (nsplit > 1 && (int)blockIdx.z >= attn_key_tiles(kfirst, kmax)) return;
  for (int i = tid; i < nrows * qd; i += 256) {
    const int lr = i / qd, d = i % qd;
    const int tok = lr / nqh, qh = g * per_group + qh0 + lr % nqh;
    s_q[lr * qd + d] = q[((int64_t)(row0 + tok) * H + qh) * qd + d];
  }
  float mrun[kAttRpw][MAPS], lrun[kAttRpw][MAPS], acc[kAttRpw][MAPS][4];
  int rpos[kAttRpw], rlo[kAttRpw], rqh[kAttRpw];
  float rsl[kAttRpw];
#pragma unroll
  for (int i = 0; i < kAttRpw; ++i) {
    const int lr = wave + 4 * i;
    rpos[i] = lr < nrows ? positions[row0 + lr / nqh] : -1;
    rlo[i] = rpos[i] >= 0 ? attn_row_lo(form, rpos[i]) : 0;
    rqh[i] = g * per_group + qh0 + (lr < nrows ? lr % nqh : 0);
    rsl[i] = form.dist_slope ? form.dist_slope[rqh[i]] : 0.f;
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
      mrun[i][m] = -INFINITY;
      lrun[i][m] = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[i][m][c] = 0.f;
    }
  }
  // nsplit > 1: workgroup z of the tile takes key tiles z, z + nsplit, ... (the count of splits does not depend on the
  // context's length, so a recorded launch serves every later length) and leaves its softmax state to the merge kernel
  for (int k0 = kfirst + (int)blockIdx.z * kAttKeys; k0 < kmax; k0 += kAttKeys * nsplit) {
    const int nk = min(kAttKeys, kmax - k0);
    // a tile between the kept first tokens and the lowest run start is seen by no row (uniform over the workgroup)
    if (k0 >= form.keep_first && k0 + kAttKeys <= lo0) continue;
    __syncthreads();
    {   // staging: four threads per key; one page lookup per thread and tile, 16-byte loads where the layout allows
      const int j = tid >> 2, sub = tid & 3;
      if (j < nk) {
        const int p = k0 + j;
        const int64_t pg = (int64_t)pages[p / page_size] * page_stride;
        const A* kp = cache + pg + k_cache_off + ((int64_t)(p % page_size) * G + g) * kw;
        const A* vp = cache + pg + v_cache_off + ((int64_t)(p % page_size) * G + g) * vdim;
        float* dk = s_k + j * kd;
        float* dv = s_v + j * vdim;
        if (vec_k && vec_v) {
          // 128 values of the key and of the value requested before the first is stored (one chunk at a time: 19.4 -> 17.0 us for two decoded
          // fp32 tokens of 8 heads of 128, 77 -> 70 us for their prompts of 470)
          for (int d0 = sub * 8; d0 < max(kw, vdim); d0 += 128) {
            float tk[4][8], tv[4][8];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              if (d0 + 32 * c < kw) Vec8<A>::load(kp + d0 + 32 * c, tk[c]);
              if (d0 + 32 * c < vdim) Vec8<A>::load(vp + d0 + 32 * c, tv[c]);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const int d = d0 + 32 * c;
              if (d < kw) {
#pragma unroll
                for (int u = 0; u < 8; ++u) dk[d + u] = tk[c][u];
              }
              if (d < vdim) {
#pragma unroll
                for (int u = 0; u < 8; ++u) dv[d + u] = tv[c][u];
                if (tail && d >= kw) {
#pragma unroll
                  for (int u = 0; u < 8; ++u) dk[d + u] = tv[c][u];
                }
              }
            }
          }
        } else {
          // one side off: the other keeps its 16-byte loads (two fp32 prompts of 470, 8 heads, keys of 128 and values of 100: 127 us, 142 with
          // single values on both sides)
          if (vec_k) {
            for (int d = sub * 8; d < kw; d += 32) {
              float t[8];
              Vec8<A>::load(kp + d, t);
#pragma unroll
              for (int u = 0; u < 8; ++u) dk[d + u] = t[u];
            }
          } else {
            for (int d = sub; d < kw; d += 4) dk[d] = ld(kp + d);
          }
          if (vec_v) {
            for (int d = sub * 8; d < vdim; d += 32) {
              float t[8];
              Vec8<A>::load(vp + d, t);
#pragma unroll
              for (int u = 0; u < 8; ++u) {
                dv[d + u] = t[u];
                if (tail && d >= kw) dk[d + u] = t[u];
              }
            }
          } else {
            for (int d = sub; d < vdim; d += 4) {
              const float t = ld(vp + d);
              dv[d] = t;
              if (tail && d >= kw) dk[d] = t;
            }
          }
        }
      }
    }
    __syncthreads();
    // the wave's (up to) four rows go through the tile together: a key value read from LDS serves four products
    // (bound by the latency of its LDS reads: unrolled, so that several are on their way, two decoded fp32 tokens of 8 heads of 128 over five
    // tiles 18.0 -> 14.5 us, their prompts of 470 tokens 67 -> 53; the same sums in the same order)
    bool act[kAttRpw];
    int jlo = nk, jhi = 0;
    bool any = false;
#pragma unroll
    for (int i = 0; i < kAttRpw; ++i) {
      const int lr = wave + 4 * i;
      // a row whose position lies before the tile, or whose run of visible keys begins after it, is left as it is
      act[i] = lr < nrows && k0 <= rpos[i] && (k0 + nk > rlo[i] || k0 < form.keep_first);
      if (act[i]) {
        any = true;
        jlo = min(jlo, k0 < form.keep_first ? 0 : max(0, rlo[i] - k0));
        jhi = max(jhi, min(nk, rpos[i] - k0 + 1));
      }
    }
    if (!any) continue;       // uniform over the wave; the barriers are at the head of the loop, which every wave reaches
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
      float a[kAttRpw] = {0.f, 0.f, 0.f, 0.f};
      if (lane < nk) {
        const float* kr = s_k + lane * kd + m * dim;
        const float* qb = s_q + wave * qd + m * dim;        // row i of the wave: + 4 * i * qd
        if ((dim & 3) == 0) {
#pragma unroll 4
          for (int d = 0; d < dim; d += 4) {
            const float k0v = kr[d], k1v = kr[d + 1], k2v = kr[d + 2], k3v = kr[d + 3];
#pragma unroll
            for (int i = 0; i < kAttRpw; ++i) {
              const f32x4 qv = *reinterpret_cast<const f32x4*>(qb + 4 * i * qd + d);
              a[i] = fmaf(qv.x, k0v, a[i]);
              a[i] = fmaf(qv.y, k1v, a[i]);
              a[i] = fmaf(qv.z, k2v, a[i]);
              a[i] = fmaf(qv.w, k3v, a[i]);
            }
          }
        } else {
          for (int d = 0; d < dim; ++d) {
            const float kv = kr[d];
#pragma unroll
            for (int i = 0; i < kAttRpw; ++i) a[i] = fmaf(qb[4 * i * qd + d], kv, a[i]);
          }
        }
      }
      float* pw = s_p + (wave * MAPS + m) * (64 * kAttRpw);   // [key][row of the wave]
      float corr[kAttRpw];
#pragma unroll
      for (int i = 0; i < kAttRpw; ++i) {
        corr[i] = 1.0f;
        float pv = 0.f;
        if (act[i]) {
          const int kp_ = k0 + lane;
          const bool seen = lane < nk && kp_ <= rpos[i] && (kp_ >= rlo[i] || kp_ < form.keep_first);
          const float sc = seen ? attn_score(form, a[i], scale, rpos[i], kp_, rqh[i], H, rsl[i]) : -INFINITY;
          const float mnew = fmaxf(mrun[i][m], wave_max(sc));
          pv = sc == -INFINITY ? 0.f : expf(sc - mnew);
          corr[i] = mrun[i][m] == -INFINITY ? 0.f : expf(mrun[i][m] - mnew);
          lrun[i][m] = lrun[i][m] * corr[i] + wave_sum(pv);
          mrun[i][m] = mnew;
        }
        pw[lane * kAttRpw + i] = pv;
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int col = lane + 64 * c;
        if (col < vdim) {
          float o0 = act[0] ? acc[0][m][c] * corr[0] : acc[0][m][c], o1 = act[1] ? acc[1][m][c] * corr[1] : acc[1][m][c],
                o2 = act[2] ? acc[2][m][c] * corr[2] : acc[2][m][c], o3 = act[3] ? acc[3][m][c] * corr[3] : acc[3][m][c];
#pragma unroll 8
          for (int j = jlo; j < jhi; ++j) {    // weights outside a row's own range are exact zeros: they add nothing
            const f32x4 pj = *reinterpret_cast<const f32x4*>(pw + j * kAttRpw);
            const float v = s_v[j * vdim + col];
            o0 = fmaf(pj.x, v, o0);
            o1 = fmaf(pj.y, v, o1);
            o2 = fmaf(pj.z, v, o2);
            o3 = fmaf(pj.w, v, o3);
          }
          acc[0][m][c] = o0; acc[1][m][c] = o1; acc[2][m][c] = o2; acc[3][m][c] = o3;
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  if (nsplit > 1) {   // [tile][kv head][split][row][map][vdim values | maximum | sum]
    float* pb = part + (((int64_t)(tile * G + g) * nsplit + blockIdx.z) * kAttRows) * MAPS * (vdim + 2);
#pragma unroll
    for (int i = 0; i < kAttRpw; ++i) {
      const int lr = wave + 4 * i;
      if (lr >= nrows) continue;
#pragma unroll
      for (int m = 0; m < MAPS; ++m) {
        float* pr = pb + ((int64_t)lr * MAPS + m) * (vdim + 2);
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (lane + 64 * c < vdim) pr[lane + 64 * c] = acc[i][m][c];
        if (lane == 0) { pr[vdim] = mrun[i][m]; pr[vdim + 1] = lrun[i][m]; }
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < kAttRpw; ++i) {
    const int lr = wave + 4 * i;
    if (lr >= nrows) continue;
    const int tok = lr / nqh, qh = g * per_group + qh0 + lr % nqh;
    attn_finish_row<A, MAPS>(mrun[i], lrun[i], acc[i], form, AttnEnd<A>(form, row0 + tok, qh, vdim, lane), vdim, factor, lane,
                             out + (int64_t)(row0 + tok) * out_stride + (int64_t)qh * vdim);
  }
}

// The same attention on the matrix cores, for a bf16 cache (v_mfma_f32_16x16x16_bf16 for both products).  Same tiles: up to 16
// (token, query head) rows of one key/value head per workgroup, key tiles of 64 positions on the grid that starts at position 0.
// Each of the four waves owns 16 keys of a tile and is a softmax stream of its own over them (its own running maximum, sum and
// output block for all 16 rows), so a tile costs no exchange between waves; the four streams are folded once, after the last
// tile, through LDS.  A wave computes S^T = K Q^T: the result leaves lane l with the scores of row l % 16 against keys
// 4 (l / 16) .. + 3 - exactly the A operand (weights, rounded to bf16) the second product P V wants from it; its B operand comes
// from a transposed copy of the value tile in LDS.  Scores, maxima, sums and outputs are fp32; q and the weights are rounded to
// bf16 where they enter the matrix cores, and the row sum is taken over the rounded weights.  dim is padded to a multiple of
// 16 per map, vdim to NCB * 16 columns (zeros).
typedef short v4s_t __attribute__((ext_vector_type(4)));
constexpr int kMfVs = kAttKeys + 4;     // row stride of the transposed value tile (bf16 values; 8-byte aligned rows)

// a workgroup of 256 threads: key/value head g of a tile, split z of its keys
template <int MAPS, int NCB>
__device__ __forceinline__ void paged_attention_mfma_block(
    int tile, int g, int z0,
    const float* __restrict__ q, const uint16_t* __restrict__ cache, int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
    int page_size, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_entry,
    const int32_t* __restrict__ page_indptr, const int32_t* __restrict__ page_ids, int H, int G, int dim, int vdim, float scale,
    float factor, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok,
    const int32_t* __restrict__ tile_qh0, const int32_t* __restrict__ tile_nqh, uint16_t* __restrict__ out, int64_t out_stride,
    AttnForm form, int nsplit, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smraw[];
  constexpr int VP = NCB * 16;
  const int qd = MAPS * dim, dp = (dim + 15) & ~15, ks = MAPS * dp + 4;
  uint16_t* s_k = reinterpret_cast<uint16_t*>(smraw);        // [64][ks]
  uint16_t* s_q = s_k + kAttKeys * ks;                         // [16][ks]
  uint16_t* s_vt = s_q + kAttRows * ks;                        // [VP][kMfVs]: value column major
  float* f_buf = reinterpret_cast<float*>(smraw);              // after the last tile: [2][MAPS][16][VP] partial outputs,
  float* f_st = f_buf + 2 * MAPS * kAttRows * VP;              //   [4 waves][MAPS][16][2] maxima and sums, [MAPS][16][2] folded
  float* f_fin = f_st + 4 * MAPS * kAttRows * 2;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lrow = lane & 15, lgrp = lane >> 4;
  const int row0 = tile_row0[tile], ntok = tile_ntok[tile], qh0 = tile_qh0[tile], nqh = tile_nqh[tile];
  const int nrows = ntok * nqh, per_group = H / G;
  const int e = row_entry[row0];
  const int32_t* pages = page_ids + page_indptr[e];
  const int kmax = positions[row0 + ntok - 1] + 1;
  const int lo0 = attn_row_lo(form, positions[row0]);   // rows of a tile are in position order: the lowest run start
  const int kfirst = attn_first_key(form, positions[row0]);
  if (nsplit > 1 && z0 >= attn_key_tiles(kfirst, kmax)) return;
  const int kw = form.k_keep;                       // values of a head in the cache's key part
  const bool tail = kw < qd;                        // the others are staged with the values (one map then)
  const bool vec_k = (dim & 7) == 0 && (kw & 7) == 0 && (page_stride & 7) == 0 && (k_cache_off & 7) == 0 && aligned16(cache);
  const bool vec_v = (vdim & 7) == 0 && (kw & 7) == 0 && (page_stride & 7) == 0 && (v_cache_off & 7) == 0 && aligned16(cache);
  // four threads per key, each with every fourth 16-byte chunk; a tile is requested whole (not a chunk at a time, each waited for), the first
  // before anything else is done and the next before the products of the one in LDS
  const int j = tid >> 2, sub = tid & 3;
  constexpr int kVc = NCB / 2, kKc = 8;      // chunks of a thread: vdim <= 16 NCB, a key's maps hold 256 values at most
  u32x4 rk[kKc], rv[kVc];
  auto key_row = [&](int k0) { return cache + (int64_t)pages[(k0 + j) / page_size] * page_stride + k_cache_off + ((int64_t)((k0 + j) % page_size) * G + g) * kw; };
  auto value_row = [&](int k0) { return cache + (int64_t)pages[(k0 + j) / page_size] * page_stride + v_cache_off + ((int64_t)((k0 + j) % page_size) * G + g) * vdim; };
  auto request = [&](int k0) {
    if (!(vec_k && vec_v) || k0 + j >= kmax) return;
    const uint16_t *kp = key_row(k0), *vp = value_row(k0);
#pragma unroll
    for (int c = 0; c < kKc; ++c)
      if (sub * 8 + 32 * c < kw) rk[c] = *reinterpret_cast<const u32x4*>(kp + sub * 8 + 32 * c);
#pragma unroll
    for (int c = 0; c < kVc; ++c)
      if (sub * 8 + 32 * c < vdim) rv[c] = *reinterpret_cast<const u32x4*>(vp + sub * 8 + 32 * c);
  };
  // the next key tile of this split that a row of the tile sees (uniform over the workgroup)
  auto seen_from = [&](int k0) {
    while (k0 < kmax && k0 >= form.keep_first && k0 + kAttKeys <= lo0) k0 += kAttKeys * nsplit;
    return k0;
  };
  int k0 = seen_from(kfirst + z0 * kAttKeys);
  if (nsplit > 1 && k0 >= kmax) {                   // no row sees any of its tiles: the states say so, the values are not read
    if (tid < nrows * MAPS) {
      float* pr = part + ((((int64_t)(tile * G + g) * nsplit + z0) * kAttRows) * MAPS + tid) * (vdim + 2);
      pr[vdim] = -INFINITY;
      pr[vdim + 1] = 0.f;
    }
    return;
  }
  request(k0);
  const bool q4 = (dim & 3) == 0 && aligned16(q);
  auto q_row = [&](int lr) { return q + ((int64_t)(row0 + lr / nqh) * H + g * per_group + qh0 + lr % nqh) * qd; };
  float tq[4][4];                                    // a wave's rows (w, w + 4, ...): four values of each per lane (qd <= 256)
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (wave + 4 * i < nrows && q4 && lane * 4 < qd) ld4(q_row(wave + 4 * i) + lane * 4, tq[i]);
  // zeros everywhere first: padding columns, rows past the tile's, keys past the context's end must multiply as zeros
  {   // (the tiles' bytes are a multiple of 16: ks is a multiple of 4 values, the row counts of 16, VP * kMfVs of 8)
    u32x4* z = reinterpret_cast<u32x4*>(smraw);
    for (int i = tid; i < ((kAttKeys + kAttRows) * ks + VP * kMfVs) / 8; i += 256) z[i] = u32x4{0u, 0u, 0u, 0u};
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lr = wave + 4 * i, c = lane * 4;
    if (lr >= nrows) break;
    if (q4) {                                        // four values lie in one map, 8-byte aligned (dp and ks are multiples of 4)
      if (c < qd) st4(s_q + lr * ks + (MAPS > 1 && c >= dim ? dp + c - dim : c), tq[i]);
    } else {
      for (int d = lane; d < qd; d += 64) s_q[lr * ks + (MAPS > 1 && d >= dim ? dp + d - dim : d)] = f2bf(q_row(lr)[d]);
    }
  }
  const int rpos = lrow < nrows ? positions[row0 + lrow / nqh] : -1;      // this lane's row (as a column of S^T)
  const int rlo = rpos >= 0 ? attn_row_lo(form, rpos) : 0;
  const int lqh = g * per_group + qh0 + (lrow < nrows ? lrow % nqh : 0);
  const float lsl = form.dist_slope ? form.dist_slope[lqh] : 0.f;
  float mrun[MAPS], lrun[MAPS];
  f32x4 o[MAPS][NCB];
#pragma unroll
  for (int m = 0; m < MAPS; ++m) {
    mrun[m] = -INFINITY;
    lrun[m] = 0.f;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) o[m][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (; k0 < kmax;) {
    const int nk = min(kAttKeys, kmax - k0);
    __syncthreads();
    if (j < nk) {                                    // staging; the value tile is written transposed
      uint16_t* dk = s_k + j * ks;
      auto put_v = [&](int c, const u32x4& t) {
        const uint32_t w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          s_vt[(c + 2 * u) * kMfVs + j] = (uint16_t)(w[u] & 0xFFFFu);
          s_vt[(c + 2 * u + 1) * kMfVs + j] = (uint16_t)(w[u] >> 16);
        }
        if (tail && c >= kw) {
          *reinterpret_cast<u32x2*>(dk + c) = u32x2{t.x, t.y};
          *reinterpret_cast<u32x2*>(dk + c + 4) = u32x2{t.z, t.w};
        }
      };
      auto put_k = [&](int c, const u32x4& t) {
        uint16_t* dst = dk + (MAPS > 1 && c >= dim ? dp + c - dim : c);   // 8-byte aligned (ks * 2 is a multiple of 8 only)
        *reinterpret_cast<u32x2*>(dst) = u32x2{t.x, t.y};
        *reinterpret_cast<u32x2*>(dst + 4) = u32x2{t.z, t.w};
      };
      if (vec_k && vec_v) {
#pragma unroll
        for (int c = 0; c < kKc; ++c)
          if (sub * 8 + 32 * c < kw) put_k(sub * 8 + 32 * c, rk[c]);
#pragma unroll
        for (int c = 0; c < kVc; ++c)
          if (sub * 8 + 32 * c < vdim) put_v(sub * 8 + 32 * c, rv[c]);
      } else {                                       // one side or both off 16 bytes
        const uint16_t *kp = key_row(k0), *vp = value_row(k0);
        if (vec_k) {
          for (int c = sub * 8; c < kw; c += 32) put_k(c, *reinterpret_cast<const u32x4*>(kp + c));
        } else {
          for (int c = sub; c < kw; c += 4) dk[MAPS > 1 && c >= dim ? dp + c - dim : c] = kp[c];
        }
        if (vec_v) {
          for (int c = sub * 8; c < vdim; c += 32) put_v(c, *reinterpret_cast<const u32x4*>(vp + c));
        } else {
          for (int c = sub; c < vdim; c += 4) {
            const uint16_t t = vp[c];
            s_vt[c * kMfVs + j] = t;
            if (tail && c >= kw) dk[c] = t;
          }
        }
      }
    }
    __syncthreads();
    const int kt = k0, kb = wave * 16;              // this tile, and this wave's keys of it
    k0 = seen_from(k0 + kAttKeys * nsplit);
    request(k0);
    if (kt + kb >= kmax) continue;                  // uniform over the wave; barriers sit at the loop's head
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
      f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
      const uint16_t* ka = s_k + (kb + lrow) * ks + m * dp + 4 * lgrp;
      const uint16_t* qb = s_q + lrow * ks + m * dp + 4 * lgrp;
      for (int kk = 0; kk < dp; kk += 16)
        sc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*reinterpret_cast<const v4s_t*>(ka + kk), *reinterpret_cast<const v4s_t*>(qb + kk),
                                                       sc, 0, 0, 0);
      float sv[4] = {sc.x, sc.y, sc.z, sc.w};
      float tmax = -INFINITY;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kp_ = kt + kb + 4 * lgrp + r;
        sv[r] = (kp_ <= rpos && (kp_ >= rlo || kp_ < form.keep_first)) ? attn_score(form, sv[r], scale, rpos, kp_, lqh, H, lsl) : -INFINITY;
        tmax = fmaxf(tmax, sv[r]);
      }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, kWave));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, kWave));
      const float mnew = fmaxf(mrun[m], tmax);
      const float corr = mnew == -INFINITY ? 1.0f : (mrun[m] == -INFINITY ? 0.f : expf(mrun[m] - mnew));
      uint16_t pb[4];
      float psum = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pb[r] = f2bf(sv[r] == -INFINITY ? 0.f : expf(sv[r] - mnew));
        psum += bf2f(pb[r]);
      }
      psum += __shfl_xor(psum, 16, kWave);
      psum += __shfl_xor(psum, 32, kWave);
      lrun[m] = lrun[m] * corr + psum;
      mrun[m] = mnew;
      // the output block holds rows 4 (l / 16) + r: their factors sit in the lanes of those numbers
      float cr[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) cr[r] = __shfl(corr, 4 * lgrp + r, kWave);
      v4s_t pa;
      pa.x = (short)pb[0]; pa.y = (short)pb[1]; pa.z = (short)pb[2]; pa.w = (short)pb[3];
      const uint16_t* vb = s_vt + lrow * kMfVs + kb + 4 * lgrp;
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) {
        f32x4 t = o[m][cb];
        t.x *= cr[0]; t.y *= cr[1]; t.z *= cr[2]; t.w *= cr[3];
        o[m][cb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, *reinterpret_cast<const v4s_t*>(vb + cb * 16 * kMfVs), t, 0, 0, 0);
      }
    }
  }
  __syncthreads();                                  // the tiles' LDS is free: the four streams are folded through it
  if (lane < 16) {
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
      f_st[((wave * MAPS + m) * kAttRows + lane) * 2] = mrun[m];
      f_st[((wave * MAPS + m) * kAttRows + lane) * 2 + 1] = lrun[m];
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MAPS; ++m) {
    float mall = -INFINITY, lall = 0.f, mine = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) mall = fmaxf(mall, f_st[((w * MAPS + m) * kAttRows + lrow) * 2]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = f_st[((w * MAPS + m) * kAttRows + lrow) * 2];
      const float sw = mw == -INFINITY ? 0.f : expf(mw - mall);
      lall += f_st[((w * MAPS + m) * kAttRows + lrow) * 2 + 1] * sw;
      if (w == wave) mine = sw;
    }
    if (wave == 0 && lane < 16) {
      f_fin[(m * kAttRows + lane) * 2] = mall;
      f_fin[(m * kAttRows + lane) * 2 + 1] = lall;
    }
    float cr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) cr[r] = __shfl(mine, 4 * lgrp + r, kWave);
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) { o[m][cb].x *= cr[0]; o[m][cb].y *= cr[1]; o[m][cb].z *= cr[2]; o[m][cb].w *= cr[3]; }
  }
  // element (map m, row 4 (l / 16) + r, column 16 cb + l % 16) of a wave's block
  auto slot = [&](int b, int m, int cb, int r) { return f_buf + ((b * MAPS + m) * kAttRows + 4 * lgrp + r) * VP + cb * 16 + lrow; };
  auto put = [&](int b) {
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) { *slot(b, m, cb, 0) = o[m][cb].x; *slot(b, m, cb, 1) = o[m][cb].y; *slot(b, m, cb, 2) = o[m][cb].z; *slot(b, m, cb, 3) = o[m][cb].w; }
  };
  auto take = [&](int b) {
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) { o[m][cb].x += *slot(b, m, cb, 0); o[m][cb].y += *slot(b, m, cb, 1); o[m][cb].z += *slot(b, m, cb, 2); o[m][cb].w += *slot(b, m, cb, 3); }
  };
  if (wave >= 2) put(wave - 2);
  __syncthreads();
  if (wave < 2) take(wave);
  __syncthreads();
  if (wave == 1) put(0);
  __syncthreads();
  if (wave == 0) { take(0); put(0); }
  __syncthreads();
  // rows go back to the layout of the plain kernel: wave w finishes rows w, w + 4, ...; a lane holds columns l, l + 64, ...
  float* pbase = nsplit > 1 ? part + (((int64_t)(tile * G + g) * nsplit + z0) * kAttRows) * MAPS * (vdim + 2) : nullptr;
  for (int lr = wave; lr < nrows; lr += 4) {
    float fm[MAPS], fl[MAPS], acc[MAPS][4];
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
      fm[m] = f_fin[(m * kAttRows + lr) * 2];
      fl[m] = f_fin[(m * kAttRows + lr) * 2 + 1];
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[m][c] = lane + 64 * c < vdim ? f_buf[(m * kAttRows + lr) * VP + lane + 64 * c] : 0.f;
    }
    if (nsplit > 1) {
#pragma unroll
      for (int m = 0; m < MAPS; ++m) {
        float* pr = pbase + ((int64_t)lr * MAPS + m) * (vdim + 2);
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (lane + 64 * c < vdim) pr[lane + 64 * c] = acc[m][c];
        if (lane == 0) { pr[vdim] = fm[m]; pr[vdim + 1] = fl[m]; }
      }
      continue;
    }
    const int tok = lr / nqh, qh = g * per_group + qh0 + lr % nqh;
    attn_finish_row<uint16_t, MAPS>(fm, fl, acc, form, AttnEnd<uint16_t>(form, row0 + tok, qh, vdim, lane), vdim, factor, lane,
                                    out + (int64_t)(row0 + tok) * out_stride + (int64_t)qh * vdim);
  }
}
template <int MAPS, int NCB>
__global__ __launch_bounds__(256) void paged_attention_mfma_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ cache, int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
    int page_size, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_entry,
    const int32_t* __restrict__ page_indptr, const int32_t* __restrict__ page_ids, int H, int G, int dim, int vdim, float scale,
    float factor, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok,
    const int32_t* __restrict__ tile_qh0, const int32_t* __restrict__ tile_nqh, uint16_t* __restrict__ out, int64_t out_stride,
    AttnForm form, int nsplit, float* __restrict__ part) {
  paged_attention_mfma_block<MAPS, NCB>(blockIdx.x, blockIdx.y, blockIdx.z, q, cache, page_stride, k_cache_off, v_cache_off, page_size, positions,
                                        row_entry, page_indptr, page_ids, H, G, dim, vdim, scale, factor, tile_row0, tile_ntok, tile_qh0,
                                        tile_nqh, out, out_stride, form, nsplit, part);
}

// The same attention and, beside it, a decode step of a recurrence that reads and writes nothing of it: a layer with both halves has two
// launches that each leave most of the chip idle and wait on chains of their own.  One grid: the attention's workgroups first (theirs is the
// longer chain), then one per (head, entry) of the step.  A workgroup has the step's 512 threads; the upper half of an attention one ends at once
// (a barrier waits for the waves that are left).  Eight rows, 8 heads on each side: 10.1 and 8.2 us one after the other, and a step of a model with
// two such layers 268 us; 48 steps behind their prompts 14.45 -> 13.85 ms with the two in one launch.
template <int NCB>
__global__ __launch_bounds__(kStepThreads) void paged_attention_beside_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ cache, int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
    int page_size, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_entry,
    const int32_t* __restrict__ page_indptr, const int32_t* __restrict__ page_ids, int H, int G, int dim, int vdim, float scale,
    float factor, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok,
    const int32_t* __restrict__ tile_qh0, const int32_t* __restrict__ tile_nqh, uint16_t* __restrict__ out, int64_t out_stride,
    AttnForm form, int nsplit, float* __restrict__ part, int n_tiles, pegainfer_recurrent_step_desc step) {
  const int n_attention = n_tiles * G * nsplit, b = blockIdx.x;
  if (b >= n_attention) {
    recurrent_step_block<uint16_t, uint16_t, PEGAINFER_STEP_GATED>(step, (b - n_attention) % step.heads, (b - n_attention) / step.heads);
    return;
  }
  if (threadIdx.x >= 256) return;
  paged_attention_mfma_block<1, NCB>(b % n_tiles, b / n_tiles % G, b / (n_tiles * G), q, cache, page_stride, k_cache_off, v_cache_off, page_size,
                                     positions, row_entry, page_indptr, page_ids, H, G, dim, vdim, scale, factor, tile_row0, tile_ntok, tile_qh0,
                                     tile_nqh, out, out_stride, form, nsplit, part);
}

// bytes of LDS the matrix-core kernel needs: the tiles while the keys are walked, the fold buffers afterwards
static size_t mfma_attention_lds(int maps, int dim, int ncb) {
  const size_t ks = (size_t)maps * ((dim + 15) & ~15) + 4, vp = (size_t)ncb * 16;
  const size_t tiles = ((kAttKeys + kAttRows) * ks + vp * kMfVs) * sizeof(uint16_t);
  const size_t fold = (2 * maps * kAttRows * vp + 4 * maps * kAttRows * 2 + maps * kAttRows * 2) * sizeof(float);
  return std::max(tiles, fold);
}

// Prompts: the same attention with 16 RG rows per workgroup (32 or 64), for a bf16 cache, one map or two, sizes in multiples of 8.
// Two waves per 16 rows, each on 32 of a tile's 64 keys, two softmax streams per row folded once at the end.  Keys and values travel by
// LDS-DMA into a ring of S tiles, row-major, requested S - 1 tiles ahead (their page numbers one tile further, in scalar registers: a vector
// load beside the DMAs could only be waited for together with them): a tile costs one barrier and a counted wait, no LDS writes.  A row's 16-byte chunks are XORed with bits of its number (the DMA
// fetches the chunk that belongs in its place), so 16 rows of one column lie in 16 different bank groups.
// Products on v_mfma_f32_16x16x32_bf16: S^T = K Q^T leaves lane l with the scores of row l % 16, and O^T = V^T P^T takes them as they
// are - which of its 32 keys sits in which place of the product is free, so a lane's two runs of four keys are its eight places (the
// value fragments come from ds_read_b64_tr_b16 of the same row-major tile) - and leaves the outputs of row l % 16 in the same lane.  The
// running maximum follows only when a score passes it by more than 2^8: weights up to 256 keep their relative precision, and a tile
// without a jump needs no exchange between lanes; the row sums stay per lane until the end.
// Bound by each wave's chain through a tile (LDS reads, products, weights, products) at two waves per SIMD: 43 % of the waves' cycles are waits, a
// third of the LDS cycles repeat for bank conflicts.  1024 rows x 16 heads of 128: 28 us
// causal (153 TFLOP/s), 86 us behind 3072 cached tokens, 103 us with a cap - against 39, 131 and 160 us with both tiles
// passing through registers, values transposed on the way, scores shaped one by one and the maximum exchanged in every tile.
// Two maps (of P / 2 values each, a key's halves): a stream per map, every value fragment read once for both.  Eight prompts of 350 - 700 tokens, 8 heads of
// 2 x 64 over 128 values: 195 -> 58 us against tiles of 16 rows; the same prompts' block-masked layer of one map 65 -> 29 us.
template <int P, int RG>
struct RowsShape {
  static constexpr int N = RG * 128, CH = P / 8, S = P == 256 || RG == 2 ? 2 : 3;   // threads, chunks of a row, tiles in the ring
  static constexpr int kTile = kAttKeys * P * 2;                                  // bytes of a key (or value) tile
  static constexpr int kLoads = 2 * (kTile / 1024) / (2 * RG);                    // DMA instructions per wave and tile
};
template <int P, int RG, int MAPS>
__global__ __launch_bounds__(RG * 128) void paged_attention_rows_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ cache, int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
    int page_size, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_entry,
    const int32_t* __restrict__ page_indptr, const int32_t* __restrict__ page_ids, int H, int G, int dim, int vdim, float scale,
    float factor, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok,
    const int32_t* __restrict__ tile_qh0, const int32_t* __restrict__ tile_nqh, uint16_t* __restrict__ out, int64_t out_stride,
    AttnForm form) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smraw[];
  typedef RowsShape<P, RG> Sh;
  constexpr int N = Sh::N, NCB = P / 16, CH = Sh::CH, S = Sh::S;     // LDS: ring [S][keys | values][64][P]
  // Two maps: the maximum never lags.  A largest weight of exactly one is not rounded, and the difference of the maps (normed, often) shows it: 3 % nearer to
  // 64-bit results, as near as 16-row tiles within 2 % (which keep four streams a row, these two); 56 -> 58 us.
  constexpr float kLog2e = 1.44269504088896341f, kJump = MAPS == 2 ? 0.0f : 8.0f;
  const int tile = gridDim.x - 1 - blockIdx.x, g = blockIdx.y;        // the longest rows of keys first
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, lg = lane >> 4;
  const int rg = wave % RG, kh = wave / RG;
  const int row0 = tile_row0[tile], ntok = tile_ntok[tile], qh0 = tile_qh0[tile], nqh = tile_nqh[tile];
  const int nrows = ntok * nqh, per_group = H / G;
  const int32_t* pages = page_ids + page_indptr[row_entry[row0]];
  const int kmax = positions[row0 + ntok - 1] + 1;
  const int lo0 = attn_row_lo(form, positions[row0]);                 // rows of a tile are in position order: the lowest run start
  auto next_tile = [&](int k) {                                       // the next tile that any row sees
    k += kAttKeys;
    return k >= form.keep_first && k + kAttKeys <= lo0 ? (lo0 / kAttKeys) * kAttKeys : k;
  };
  const int kfirst = form.keep_first > 0 ? 0 : (lo0 / kAttKeys) * kAttKeys;
  const int kw = form.k_keep, qd = MAPS * dim;        // two maps: qd = P
  // this wave's rows
  const int lr = rg * 16 + l15;
  const bool mine = lr < nrows;
  const int rpos = mine ? positions[row0 + lr / nqh] : -1, rlo = mine ? attn_row_lo(form, rpos) : 0;
  const int rqh = g * per_group + qh0 + (mine ? lr % nqh : 0);
  const float rsl = form.dist_slope ? form.dist_slope[rqh] : 0.f;
  const float inv_cap = form.softcap > 0.f ? 1.0f / form.softcap : 0.f;
  // uniform: no key after `last` concerns the wave; keys of [all_lo, all_hi] are seen by all of its rows, without a look at each
  const int last = rg * 16 < nrows ? positions[row0 + min(rg * 16 + 15, nrows - 1) / nqh] : -1;
  const int first_lo = last >= 0 ? attn_row_lo(form, positions[row0 + rg * 16 / nqh]) : 0;      // the lowest key of any of its rows
  const int all_lo = last >= 0 ? attn_row_lo(form, last) : 0, all_hi = rg * 16 + 15 < nrows ? positions[row0 + rg * 16 / nqh] : -1;
  bf16x8_t qf[P / 32];
  {
    const float* qr = q + ((int64_t)(row0 + (mine ? lr / nqh : 0)) * H + rqh) * qd;
#pragma unroll
    for (int st = 0; st < P / 32; ++st) {
      const int c = st * 32 + lg * 8;
      float t[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (mine && c < qd) Vec8<float>::load(qr + c, t);
      qf[st] = __builtin_bit_cast(bf16x8_t, u32x4{pack_bf2(t[0], t[1]), pack_bf2(t[2], t[3]), pack_bf2(t[4], t[5]), pack_bf2(t[6], t[7])});
    }
  }
  if (qd < P || vdim < P) {       // chunks past a row's end are never fetched: they stay zero
    for (int i = tid; i < S * 2 * Sh::kTile / 16; i += N) reinterpret_cast<u32x4*>(smraw)[i] = u32x4{0u, 0u, 0u, 0u};
  }
  // swizzle of row j: CH 16 - its low four bits; CH 8 - two rows share 256 bytes, the three bits above the lowest
  auto swz = [](int j) { return CH == 8 ? (j >> 1) & 7 : j & 15; };
  // a wave's DMA instructions: kLoads / 2 of the key tile, as many of the value tile; lane l fills the 16 bytes l of a run of 64
  constexpr int kHalf = Sh::kLoads / 2;
  int src_j[kHalf], src_c[kHalf], off_k[kHalf], off_v[kHalf];
  // the rows of one instruction share a page and lie at the same place in it for every tile (pages of 16: always)
  const bool even = page_size % (64 / CH) == 0 && kAttKeys % page_size == 0;
#pragma unroll
  for (int i = 0; i < kHalf; ++i) {
    const int unit = (wave * kHalf + i) * 64 + lane;
    src_j[i] = unit / CH;
    src_c[i] = ((unit % CH) ^ swz(src_j[i])) * 8;
    const int slot = (src_j[i] % page_size) * G + g;
    off_k[i] = src_c[i] < kw ? slot * kw + src_c[i] : slot * vdim + src_c[i];
    off_v[i] = slot * vdim + src_c[i];
  }
  const uint16_t *kbase = cache + k_cache_off, *vbase = cache + v_cache_off;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  const uint32_t ring = (uint32_t)(uintptr_t)(lds_ptr_t)smraw;
  auto dma = [&](const uint16_t* src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :: "v"(src), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory", "m0");
  };
  // page numbers of a tile's instructions, uniform over the wave (even pages)
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  auto page_numbers = [&](int k0, int (&pn)[kHalf]) {
#pragma unroll
    for (int i = 0; i < kHalf; ++i) pn[i] = even ? pages[min(k0 + (wave_u * kHalf + i) * (64 / CH), kmax - 1) / page_size] : 0;
  };
  // kLoads instructions per wave, whatever the tile: keys past the end fetch the last key's row again
  auto fetch = [&](int i, int64_t page, int ok, int ov, int stage) {
    const int c = src_c[i];
    const uint32_t dst = ring + (uint32_t)(stage * 2 * Sh::kTile + (wave_u * kHalf + i) * 1024);
    if (c < qd) dma((c < kw ? kbase : vbase) + page + ok, dst);
    if (c < vdim) dma(vbase + page + ov, dst + Sh::kTile);
  };
  auto fetch_at = [&](int i, int p, int page, int stage) {     // the general form: a key's own page and place
    const int slot = (p % page_size) * G + g, c = src_c[i];
    fetch(i, (int64_t)page * page_stride, c < kw ? slot * kw + c : slot * vdim + c, slot * vdim + c, stage);
  };
  auto request = [&](int k0, const int (&pn)[kHalf], int stage) {
    if (even && k0 + kAttKeys <= kmax) {             // uniform; paths of their own: a vector load of page numbers would be waited for in both
#pragma unroll
      for (int i = 0; i < kHalf; ++i) fetch(i, (int64_t)pn[i] * page_stride, off_k[i], off_v[i], stage);
    } else if (even) {
#pragma unroll
      for (int i = 0; i < kHalf; ++i) fetch_at(i, min(k0 + src_j[i], kmax - 1), pn[i], stage);
    } else {
#pragma unroll
      for (int i = 0; i < kHalf; ++i) {
        const int p = min(k0 + src_j[i], kmax - 1);
        fetch_at(i, p, pages[p / page_size], stage);
      }
    }
  };
  float mrun[MAPS], lrun[MAPS];                       // log2 units; lrun: this lane's part of the row sum
  f32x4 o[MAPS][NCB];
#pragma unroll
  for (int m = 0; m < MAPS; ++m) {
    mrun[m] = -INFINITY;
    lrun[m] = 0.f;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) o[m][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int krow = 32 * kh + l15, vrow = 32 * kh + 4 * lg + (l15 >> 2);
  // byte addresses inside a tile: swz(row + 16) = swz(row) for both row widths, so the second half of the keys lies 16 rows on
  const uint32_t ka = (uint32_t)(krow * P * 2 + ((lg ^ swz(krow)) << 4));
  const uint32_t va = (uint32_t)(vrow * P * 2 + ((((l15 & 3) >> 1) ^ swz(vrow)) << 4) + (l15 & 1) * 8);
  // masked: some row of the wave does not see some of these keys.  Values of keys that none of them sees go in as zeros: an infinity or no number
  // times a weight of zero would reach rows that the form of 16-row tiles keeps it from.  Two bodies, chosen at the top: masking inside one
  // cost 13 % (the branch, or 32 instructions a tile, stands between the weights and the second products); 77 us behind 3072 tokens so, 79 unmasked.
  auto multiply_keys = [&](int kb, int stage, auto masked) {
    const unsigned char* kt = smraw + stage * 2 * Sh::kTile;
    f32x4 maps[MAPS][2] = {};
#pragma unroll
    for (int st = 0; st < P / 32; ++st)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        maps[st * 32 * MAPS / P][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4*>(kt + 16 * t * P * 2 + (ka ^ (uint32_t)(st << 6)))), qf[st], maps[st * 32 * MAPS / P][t], 0, 0, 0);
    // dot products -> scores times log2(e); each option in a pass of its own: one uniform branch per tile, its loads in flight together
    const int dist = rpos - kb - 4 * lg;             // of this lane's key (t, r): dist - 16 t - r
    const bool options = form.softcap > 0.f || form.dist_bias || form.dist_slope;
    const float f0 = options ? scale : scale * kLog2e;
    uint32_t see[4];
    bf16x8_t pf[MAPS];
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
      f32x4 (&sc)[2] = maps[m];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[t][r] *= f0;
      if (form.softcap > 0.f) soft_cap8(sc, form.softcap, inv_cap);
      if (form.dist_bias) {
        float bias[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) bias[t][r] = form.dist_bias[(int64_t)max(0, min(dist - 16 * t - r, form.n_dist - 1)) * H + rqh];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[t][r] += bias[t][r];
      }
      if (form.dist_slope) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[t][r] = fmaf(-rsl, (float)(dist - 16 * t - r), sc[t][r]);
      }
      if (options) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[t][r] *= kLog2e;
      }
      if constexpr (decltype(masked)::value) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int kp = kb + 16 * t + 4 * lg + r;
            if (!(kp <= rpos && (kp >= rlo || kp < form.keep_first))) sc[t][r] = -INFINITY;
          }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kp = kb + 16 * (i >> 1) + 4 * lg + 2 * (i & 1);
          auto seen = [&](int j) { return j <= last && (j >= first_lo || j < form.keep_first); };
          see[i] = (seen(kp) ? 0xFFFFu : 0u) | (seen(kp + 1) ? 0xFFFF0000u : 0u);
        }
      }
      float tmax = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])), fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
      if (__any(!(tmax <= mrun[m] + kJump))) {            // uniform; the first keys of a row always, a NaN too
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, kWave));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, kWave));
        const float mnew = fmaxf(mrun[m], tmax);
        const float corr = __builtin_amdgcn_exp2f(mrun[m] - (mnew == -INFINITY ? 0.f : mnew));   // a row that has met no key yet: 0, and nothing to scale
        lrun[m] *= corr;
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) { o[m][cb].x *= corr; o[m][cb].y *= corr; o[m][cb].z *= corr; o[m][cb].w *= corr; }
        mrun[m] = mnew;
      }
      const float mref = mrun[m] == -INFINITY ? 0.f : mrun[m];
      uint32_t pb[4];
      float psum = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          const uint32_t w = pack_bf2(__builtin_amdgcn_exp2f(sc[t][r] - mref), __builtin_amdgcn_exp2f(sc[t][r + 1] - mref));
          pb[2 * t + (r >> 1)] = w;
          psum += bf_lo(w) + bf_hi(w);                 // the sum of the weights as they are multiplied
        }
      lrun[m] += psum;
      pf[m] = __builtin_bit_cast(bf16x8_t, u32x4{pb[0], pb[1], pb[2], pb[3]});
    }
    typedef v4s_t __attribute__((address_space(3)))* lds_v4_t;
    const uint32_t vt = ring + (uint32_t)(stage * 2 * Sh::kTile + Sh::kTile);
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      const uint32_t at = vt + (va ^ (uint32_t)(cb << 5));
      u32x2 v0 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(uintptr_t)at));
      u32x2 v1 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(uintptr_t)(at + 16 * P * 2)));
      if constexpr (decltype(masked)::value) { v0.x &= see[0]; v0.y &= see[1]; v1.x &= see[2]; v1.y &= see[3]; }
#pragma unroll
      for (int m = 0; m < MAPS; ++m)
        o[m][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, u32x4{v0.x, v0.y, v1.x, v1.y}), pf[m], o[m][cb], 0, 0, 0);
    }
  };
  auto multiply = [&](int k0, int stage) {           // uniform over the wave
    const int kb = k0 + 32 * kh;
    if (kb > last || kb >= kmax) return;
    if (kb < all_lo || kb + 31 > all_hi) multiply_keys(kb, stage, std::true_type{});
    else multiply_keys(kb, stage, std::false_type{});
  };
  int k[S + 1];                                      // k[i]: the tile i ahead
  k[0] = kfirst;
#pragma unroll
  for (int i = 1; i <= S; ++i) k[i] = next_tile(k[i - 1]);
  int pn[kHalf];
  __syncthreads();                                   // the zeros are in LDS
#pragma unroll
  for (int i = 0; i < S - 1; ++i) {
    page_numbers(k[i], pn);
    request(k[i], pn, i);
  }
  page_numbers(k[S - 1], pn);
  int stage = 0;
  while (true) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * Sh::kLoads) : "memory");   // this wave's part of tile k[0] has landed
    __syncthreads();                                 // everybody's has; the stage of the tile before is free
    request(k[S - 1], pn, stage == 0 ? S - 1 : stage - 1);
    page_numbers(k[S], pn);
    multiply(k[0], stage);
    if (k[1] >= kmax) break;                         // uniform over the workgroup
#pragma unroll
    for (int i = 0; i < S; ++i) k[i] = k[i + 1];
    k[S] = next_tile(k[S]);
    stage = stage + 1 == S ? 0 : stage + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may land in the memory that is reused below
  __syncthreads();                                   // the tiles' LDS is free
  f32x4* f_o = reinterpret_cast<f32x4*>(smraw);      // [MAPS][RG][NCB][64]
  float* f_ml = reinterpret_cast<float*>(f_o + MAPS * RG * NCB * 64);        // [MAPS][RG][64][2]
#pragma unroll
  for (int m = 0; m < MAPS; ++m) {
    lrun[m] += __shfl_xor(lrun[m], 16, kWave);
    lrun[m] += __shfl_xor(lrun[m], 32, kWave);
    if (kh == 1) {
#pragma unroll
      for (int cb = 0; cb < NCB; ++cb) f_o[((m * RG + rg) * NCB + cb) * 64 + lane] = o[m][cb];
      f_ml[((m * RG + rg) * 64 + lane) * 2] = mrun[m];
      f_ml[((m * RG + rg) * 64 + lane) * 2 + 1] = lrun[m];
    }
  }
  __syncthreads();
  if (kh == 1 || rg * 16 >= nrows) return;
  float i0[MAPS], i1[MAPS];
#pragma unroll
  for (int m = 0; m < MAPS; ++m) {
    const float m1 = f_ml[((m * RG + rg) * 64 + lane) * 2], l1 = f_ml[((m * RG + rg) * 64 + lane) * 2 + 1];
    float mall = fmaxf(mrun[m], m1), sink = -INFINITY;
    if (form.sink && mine) {
      sink = bf2f(static_cast<const uint16_t*>(form.sink)[rqh]) * kLog2e;
      mall = fmaxf(mall, sink);
    }
    const float w0 = mrun[m] == -INFINITY ? 0.f : exp2f(mrun[m] - mall), w1 = m1 == -INFINITY ? 0.f : exp2f(m1 - mall);
    const float l = lrun[m] * w0 + l1 * w1 + (sink == -INFINITY ? 0.f : exp2f(sink - mall));
    i0[m] = w0 / l;
    i1[m] = w1 / l;
  }
  float ss = 0.f;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const f32x4 t = f_o[(rg * NCB + cb) * 64 + lane];
    f32x4 v = {};
    if constexpr (MAPS == 2) v = f_o[((RG + rg) * NCB + cb) * 64 + lane];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[0][cb][r] = o[0][cb][r] * i0[0] + t[r] * i1[0];
      if constexpr (MAPS == 2) o[0][cb][r] -= form.lambda * (o[1][cb][r] * i0[1] + v[r] * i1[1]);
      if (16 * cb + 4 * lg + r < vdim) ss = fmaf(o[0][cb][r], o[0][cb][r], ss);
    }
  }
  float post = factor;
  if (form.head_norm) {
    ss += __shfl_xor(ss, 16, kWave);
    ss += __shfl_xor(ss, 32, kWave);
    post = factor / sqrtf(ss / (float)vdim + form.norm_eps);
  }
  if (!mine) return;
  const int row = row0 + lr / nqh;
  const uint16_t* gate = static_cast<const uint16_t*>(form.gate) + (int64_t)row * form.gate_stride;
  if (form.gate_kind == 2) post *= sigmoid_f(bf2f(gate[rqh]));
  uint16_t* dst = out + (int64_t)row * out_stride + (int64_t)rqh * vdim;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
    const int c = 16 * cb + 4 * lg;
    if (c >= vdim) continue;                         // vdim is a multiple of 8
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v[r] = o[0][cb][r] * post;
      if (form.gate_kind == 1) v[r] *= sigmoid_f(bf2f(gate[(int64_t)rqh * vdim + c + r]));
    }
    st4(dst + c, v);
  }
}
template <int P, int RG, int MAPS>
static constexpr size_t rows_attention_lds() {
  typedef RowsShape<P, RG> Sh;
  return std::max((size_t)Sh::S * 2 * Sh::kTile, (size_t)MAPS * RG * 64 * (P + 8));
}

// The states that the live splits of a tile have left, brought to their common maximum and summed, then finished like an unsplit row.  A
// workgroup per row: wave w takes splits w, w + 4, ..., eight splits' values on their way with everything else that the row needs before
// anything is waited for; the waves' sums meet in LDS in wave order.  Launch- and latency-bound: against a
// wave per row, splits one batch of loads after another, 8 rows of 8 heads with two maps 8.3 -> 6.8 us; one row over 64 splits 5.6 (over 16 5.8).
// of 256 threads: row lr of key/value head g of a tile
template <typename A, int MAPS>
__device__ __forceinline__ void paged_attention_merge_block(
    int tile, int g, int lr,
    const float* __restrict__ part, int nsplit, int H, int G, int vdim, float factor, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok, const int32_t* __restrict__ tile_qh0,
    const int32_t* __restrict__ tile_nqh, A* __restrict__ out, int64_t out_stride, AttnForm form) {
  __shared__ float s_acc[3][MAPS][256];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row0 = tile_row0[tile], ntok = tile_ntok[tile], qh0 = tile_qh0[tile], nqh = tile_nqh[tile];
  if (lr >= ntok * nqh) return;
  const int row = row0 + lr / nqh, qh = g * (H / G) + qh0 + lr % nqh;
  const int live = min(nsplit, attn_key_tiles(attn_first_key(form, positions[row0]), positions[row0 + ntok - 1] + 1));
  const AttnEnd<A> end(form, row, qh, vdim, lane);
  const int64_t zs = (int64_t)kAttRows * MAPS * (vdim + 2);        // floats between two splits of a row
  float mrun[MAPS], lrun[MAPS], acc[MAPS][4];
#pragma unroll
  for (int m = 0; m < MAPS; ++m) {
    // lane z reads split z's maximum and sum (nsplit <= 64): every split's weight follows without a dependent load
    const float* pr = part + ((((int64_t)(tile * G + g) * nsplit) * kAttRows + lr) * MAPS + m) * (vdim + 2);
    const float mz = lane < live ? pr[lane * zs + vdim] : -INFINITY;
    const float lz = lane < live ? pr[lane * zs + vdim + 1] : 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[m][c] = 0.f;
    float wz = 0.f;
    for (int z0 = wave; z0 < live; z0 += 32) {
      float val[8][4];
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          val[u][c] = z0 + 4 * u < live && lane + 64 * c < vdim ? pr[(z0 + 4 * u) * zs + lane + 64 * c] : 0.f;
      if (z0 == wave) {
        mrun[m] = wave_max(mz);
        wz = mz == -INFINITY ? 0.f : expf(mz - mrun[m]);            // none: a split that met no visible key, its values are not written
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float w = __shfl(wz, min(z0 + 4 * u, 63), kWave), top = __shfl(mz, min(z0 + 4 * u, 63), kWave);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[m][c] = top == -INFINITY ? acc[m][c] : fmaf(val[u][c], w, acc[m][c]);
      }
    }
    if (wave == 0) lrun[m] = wave_sum(lz * wz);                     // wave 0 has a split: live >= 1
    else {
#pragma unroll
      for (int c = 0; c < 4; ++c) s_acc[wave - 1][m][lane + 64 * c] = acc[m][c];
    }
  }
  __syncthreads();
  if (wave) return;
#pragma unroll
  for (int m = 0; m < MAPS; ++m)
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[m][c] += s_acc[w][m][lane + 64 * c];
  attn_finish_row<A, MAPS>(mrun, lrun, acc, form, end, vdim, factor, lane, out + (int64_t)row * out_stride + (int64_t)qh * vdim);
}
template <typename A, int MAPS>
__global__ __launch_bounds__(256) void paged_attention_merge_kernel(
    const float* __restrict__ part, int nsplit, int H, int G, int vdim, float factor, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok, const int32_t* __restrict__ tile_qh0,
    const int32_t* __restrict__ tile_nqh, A* __restrict__ out, int64_t out_stride, AttnForm form) {
  paged_attention_merge_block<A, MAPS>(blockIdx.x, blockIdx.y, blockIdx.z, part, nsplit, H, G, vdim, factor, positions, tile_row0, tile_ntok, tile_qh0, tile_nqh, out, out_stride, form);
}

// Decoding, a layer with a state-space scan beside its attention: the scan's workgroups behind the attention's in one grid, and the norm and gate of its
// read-out behind the merge's.  One row, 16 heads over 4 of 128 beside 32 heads of 128 x 64: 9.0 + 6.6 and 5.6 + 3.7 us one after the other,
// 9.6 and 5.6 here.
template <int NCB, int NS>
__global__ __launch_bounds__(256) void paged_attention_scan_kernel(
    const float* __restrict__ q, const uint16_t* __restrict__ cache, int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
    int page_size, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_entry,
    const int32_t* __restrict__ page_indptr, const int32_t* __restrict__ page_ids, int H, int G, int dim, int vdim, float scale,
    float factor, const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok,
    const int32_t* __restrict__ tile_qh0, const int32_t* __restrict__ tile_nqh, uint16_t* __restrict__ out, int64_t out_stride,
    AttnForm form, int nsplit, float* __restrict__ part, int n_tiles, pegainfer_ssd_scan_desc d, int nbx) {
  const int n_attention = n_tiles * G * nsplit, b = blockIdx.x;
  if (b >= n_attention) {
    const int i = b - n_attention;
    ssd_scan_block<NS, uint16_t>(i % nbx, i / nbx % d.heads, i / (nbx * d.heads), d.xbc, d.xbc_stride, static_cast<const uint16_t*>(d.proj), d.proj_stride,
                                 d.dt_off, static_cast<const uint16_t*>(d.A_log), static_cast<const uint16_t*>(d.dt_bias),
                                 static_cast<const uint16_t*>(d.D), d.state, d.slot_stride, d.o, d.heads, d.groups, d.n_state, d.vdim, d.entry_row0,
                                 d.entry_slot, 0);
    return;
  }
  paged_attention_mfma_block<1, NCB>(b % n_tiles, b / n_tiles % G, b / (n_tiles * G), q, cache, page_stride, k_cache_off, v_cache_off, page_size, positions, row_entry, page_indptr, page_ids, H, G, dim, vdim, scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh, out, out_stride, form, nsplit, part);
}
template <int V>
__global__ __launch_bounds__(256) void paged_attention_merge_norm_kernel(
    const float* __restrict__ part, int nsplit, int H, int G, int vdim, float factor, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ tile_row0, const int32_t* __restrict__ tile_ntok, const int32_t* __restrict__ tile_qh0,
    const int32_t* __restrict__ tile_nqh, uint16_t* __restrict__ out, int64_t out_stride, AttnForm form, int n_tiles, pegainfer_scan_beside_desc d, const float* o_scan) {
  const int n_merge = n_tiles * G * kAttRows, b = blockIdx.x;
  if (b >= n_merge) {
    const int rh = (b - n_merge) * 4 + (threadIdx.x >> 6);
    if (rh < d.rows * d.heads)
      head_rms_gate_wave<uint16_t, V>(rh / d.heads, rh % d.heads, o_scan, static_cast<const uint16_t*>(d.norm_w), d.w_per_head,
                                      static_cast<const uint16_t*>(d.gate), d.gate_stride, d.gate_kind, d.factor, d.eps, static_cast<uint16_t*>(d.out),
                                      d.out_stride, d.heads, d.vdim, d.gate_first);
    return;
  }
  paged_attention_merge_block<uint16_t, 1>(b % n_tiles, b / n_tiles % G, b / (n_tiles * G), part, nsplit, H, G, vdim, factor, positions, tile_row0, tile_ntok, tile_qh0, tile_nqh, out, out_stride, form);
}

// out[row, :cols] = in[row, :cols] * factor, rows of either side at their own stride
template <typename A>
__global__ __launch_bounds__(256) void scale_rows_kernel(const A* __restrict__ in, int64_t in_stride, A* __restrict__ out,
                                                         int64_t out_stride, int cols, float factor) {
  const int row = blockIdx.x;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < cols; i += gridDim.y * 256)
    st(out + (int64_t)row * out_stride + i, ld(in + (int64_t)row * in_stride + i) * factor);
}

}  // namespace pk

extern "C" {
using namespace pk;

#define PK_BAD ((pegainfer_status_t)hipErrorInvalidValue)

pegainfer_status_t pegainfer_qk_prep_paged(const void* proj, int64_t proj_stride, int64_t q_off, int64_t k_off, int64_t v_off,
                                          int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, const void* q_norm,
                                          const void* k_norm, float eps, const void* q_bias, const void* k_bias,
                                          const void* v_bias, float qt_coef, int32_t qt_every, const float* inv_freq,
                                          int32_t rot_dims, const int32_t* positions, const int32_t* row_entry,
                                          const int32_t* page_indptr, const int32_t* page_ids, void* cache, int64_t page_stride,
                                          int64_t k_cache_off, int64_t v_cache_off, int32_t page_size, float* q_out,
                                          void* q_out_stored, int32_t n_rows, int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_qk_prep_paged_form(proj, dtype, proj_stride, q_off, k_off, v_off, heads, kv_heads, dim, vdim, q_norm, k_norm,
                                      PEGAINFER_QKNORM_HEAD_WEIGHT, eps, q_bias, k_bias, v_bias, qt_coef, qt_every, inv_freq, rot_dims,
                                      PEGAINFER_ROT_PAIRS, positions, row_entry, page_indptr, page_ids, cache, page_stride, k_cache_off,
                                      v_cache_off, page_size, q_out, q_out_stored, n_rows, dtype, stream);
}

pegainfer_status_t pegainfer_qk_prep_paged_form(const void* proj, int32_t proj_dtype, int64_t proj_stride, int64_t q_off,
                                               int64_t k_off, int64_t v_off, int32_t heads, int32_t kv_heads, int32_t dim,
                                               int32_t vdim, const void* q_norm, const void* k_norm, int32_t norm_kind, float eps,
                                               const void* q_bias, const void* k_bias, const void* v_bias, float qt_coef,
                                               int32_t qt_every, const float* inv_freq, int32_t rot_dims, int32_t rot_layout,
                                               const int32_t* positions, const int32_t* row_entry, const int32_t* page_indptr,
                                               const int32_t* page_ids, void* cache, int64_t page_stride, int64_t k_cache_off,
                                               int64_t v_cache_off, int32_t page_size, float* q_out, void* q_out_stored,
                                               int32_t n_rows, int32_t dtype, pegainfer_stream_t stream) {
  pegainfer_qk_prep_desc p{};
  p.proj = proj; p.proj_dtype = proj_dtype; p.proj_stride = proj_stride; p.q_off = q_off; p.k_off = k_off; p.v_off = v_off;
  p.heads = heads; p.kv_heads = kv_heads; p.dim = dim; p.vdim = vdim;
  p.q_norm = q_norm; p.k_norm = k_norm; p.norm_kind = norm_kind; p.eps = eps;
  p.q_bias = q_bias; p.k_bias = k_bias; p.v_bias = v_bias; p.qt_coef = qt_coef; p.qt_every = qt_every;
  p.inv_freq = inv_freq; p.rot_dims = rot_dims; p.rot_layout = rot_layout; p.rot_amp = 1.0f;
  p.positions = positions; p.row_entry = row_entry; p.page_indptr = page_indptr; p.page_ids = page_ids;
  p.cache = cache; p.page_stride = page_stride; p.k_cache_off = k_cache_off; p.v_cache_off = v_cache_off; p.page_size = page_size;
  p.q_out = q_out; p.q_out_stored = q_out_stored; p.n_rows = n_rows; p.dtype = dtype;
  return pegainfer_qk_prep(&p, stream);
}

pegainfer_status_t pegainfer_qk_prep(const pegainfer_qk_prep_desc* p, pegainfer_stream_t stream) {
  if (!p) return PK_BAD;
  if (p->n_rows <= 0) return 0;
  if (!qk_prep_ok(p)) return PK_BAD;
  const PrepForm pf = qk_prep_form(*p);
  const bool two = qk_prep_pairs(p);
  bool ok = true;
  const bool known = by_dtype(p->dtype, [&](auto* t) {
    using A = std::remove_pointer_t<decltype(t)>;
    ok = by_dtype(p->proj_dtype, [&](auto* ti) {
      using I = std::remove_pointer_t<decltype(ti)>;
      auto go = [&](auto kern) { kern<<<dim3(p->n_rows, qk_prep_per_row(*p)), 256, qk_prep_lds(*p), as_stream(stream)>>>(*p, pf); };
      two ? go(qk_prep_paged_kernel<A, I, 2>) : go(qk_prep_paged_kernel<A, I, 1>);
    });
  });
  return known && ok ? (pegainfer_status_t)hipGetLastError() : PK_BAD;
}

pegainfer_status_t pegainfer_qk_norm_rope_paged(const void* proj, int64_t proj_stride, int64_t q_off, int64_t k_off,
                                                int64_t v_off, int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim,
                                                const void* q_norm, const void* k_norm, float eps, const float* inv_freq,
                                                int32_t rot_dims, const int32_t* positions, const int32_t* row_entry,
                                                const int32_t* page_indptr, const int32_t* page_ids, void* cache,
                                                int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
                                                int32_t page_size, float* q_out, void* q_out_stored, int32_t n_rows,
                                                int32_t dtype, pegainfer_stream_t stream) {
  if (!q_norm || !k_norm) return PK_BAD;
  return pegainfer_qk_prep_paged(proj, proj_stride, q_off, k_off, v_off, heads, kv_heads, dim, vdim, q_norm, k_norm, eps, nullptr,
                                 nullptr, nullptr, 0.f, 0, inv_freq, rot_dims, positions, row_entry, page_indptr, page_ids, cache,
                                 page_stride, k_cache_off, v_cache_off, page_size, q_out, q_out_stored, n_rows, dtype, stream);
}

pegainfer_status_t pegainfer_paged_attention_ex(const float* q, const void* cache, int64_t page_stride, int64_t k_cache_off,
                                                int64_t v_cache_off, int32_t page_size, const int32_t* positions,
                                                const int32_t* row_entry, const int32_t* page_indptr, const int32_t* page_ids,
                                                int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, float scale,
                                                float factor, const int32_t* tile_row0, const int32_t* tile_ntok,
                                                const int32_t* tile_qh0, const int32_t* tile_nqh, int32_t n_tiles, void* out,
                                                int64_t out_stride, int32_t maps, float lambda, int32_t block, const void* sink,
                                                int32_t head_norm, float norm_eps, int32_t n_split, float* workspace,
                                                int32_t plain, int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_paged_attention_masked(q, cache, page_stride, k_cache_off, v_cache_off, page_size, positions, row_entry, page_indptr,
                                          page_ids, heads, kv_heads, dim, vdim, scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh,
                                          n_tiles, out, out_stride, maps, lambda, block, sink, head_norm, norm_eps, 0.f, 0, 0, nullptr, 0,
                                          nullptr, 0, 0, n_split, workspace, plain, dtype, stream);
}

pegainfer_status_t pegainfer_paged_attention_masked(const float* q, const void* cache, int64_t page_stride, int64_t k_cache_off,
                                                    int64_t v_cache_off, int32_t page_size, const int32_t* positions,
                                                    const int32_t* row_entry, const int32_t* page_indptr, const int32_t* page_ids,
                                                    int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, float scale,
                                                    float factor, const int32_t* tile_row0, const int32_t* tile_ntok,
                                                    const int32_t* tile_qh0, const int32_t* tile_nqh, int32_t n_tiles, void* out,
                                                    int64_t out_stride, int32_t maps, float lambda, int32_t block, const void* sink,
                                                    int32_t head_norm, float norm_eps, float softcap, int32_t window,
                                                    int32_t keep_first, const float* dist_bias, int32_t n_dist, const void* gate,
                                                    int64_t gate_stride, int32_t gate_kind, int32_t n_split, float* workspace,
                                                    int32_t plain, int32_t dtype, pegainfer_stream_t stream) {
  pegainfer_attn_options o{};
  o.maps = maps; o.lambda = lambda; o.block = block; o.sink = sink; o.head_norm = head_norm; o.norm_eps = norm_eps;
  o.softcap = softcap; o.window = window; o.keep_first = keep_first; o.dist_bias = dist_bias; o.n_dist = n_dist;
  o.gate = gate; o.gate_stride = gate_stride; o.gate_kind = gate_kind; o.n_split = n_split; o.workspace = workspace; o.plain = plain;
  return pegainfer_paged_attention_opt(q, cache, page_stride, k_cache_off, v_cache_off, page_size, positions, row_entry, page_indptr,
                                          page_ids, heads, kv_heads, dim, vdim, scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh,
                                          n_tiles, out, out_stride, &o, dtype, stream);
}

int32_t pegainfer_paged_attention_beside_ok(const pegainfer_attn_options* o, int32_t dtype) {
  const pegainfer_recurrent_step_desc* q = o ? o->beside : nullptr;
  return q && dtype == kDtBf16 && o->maps <= 1 && !o->plain && o->tile_rows <= kAttRows && q->kind == PEGAINFER_STEP_GATED && q->dtype == dtype &&
         recurrent_step_ok(q) && q->n_entries > 0;
}

int32_t pegainfer_paged_attention_scan_ok(const pegainfer_attn_options* o, int32_t dtype) {
  const pegainfer_scan_beside_desc* d = o ? o->scan_beside : nullptr;
  const pegainfer_ssd_scan_desc* q = d ? d->scan : nullptr;
  return q && dtype == kDtBf16 && o->maps <= 1 && !o->plain && o->tile_rows <= kAttRows && o->n_split > 1 && q->dtype == dtype && q->n_long == 0 && q->heads > 0 &&
         q->groups > 0 && q->heads % q->groups == 0 && q->n_state > 32 && q->n_state <= 128 && q->vdim > 0 && q->n_entries > 0 && q->n_entries <= 65535 &&
         (int64_t)ceil_div(q->vdim, kRecCols) * q->heads * q->n_entries < (1 << 22) && q->o && d->norm_w && d->gate && d->out && d->heads > 0 && d->vdim > 0 &&
         d->vdim <= 512 && d->rows > 0 && (int64_t)d->rows * d->heads < (1 << 24);
}

// the kernel for prompts with two maps: a map's share of a key is a whole number of its 32-wide products, known at compile time
static bool rows_two_maps_ok(int dim, int vdim) { return (dim == 32 && vdim <= 64) || (dim == 64 && vdim <= 128); }

static pegainfer_status_t paged_attention(const float* q, const void* cache, int64_t page_stride, int64_t k_cache_off,
                                         int64_t v_cache_off, int32_t page_size, const int32_t* positions,
                                         const int32_t* row_entry, const int32_t* page_indptr, const int32_t* page_ids,
                                         int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, float scale,
                                         float factor, const int32_t* tile_row0, const int32_t* tile_ntok,
                                         const int32_t* tile_qh0, const int32_t* tile_nqh, int32_t n_tiles, void* out,
                                         int64_t out_stride, const pegainfer_attn_options* opt, int32_t dtype,
                                         pegainfer_stream_t stream,
                                         bool two_wide) {
  if (n_tiles <= 0) return 0;
  if (!opt) return PK_BAD;
  const int32_t maps = opt->maps > 0 ? opt->maps : 1, block = opt->block, window = opt->window, keep_first = opt->keep_first,
                gate_kind = opt->gate_kind, plain = opt->plain;
  int32_t n_split = opt->n_split;
  float* workspace = opt->workspace;
  if (gate_kind < 0 || gate_kind > 2 || (gate_kind && !opt->gate)) return PK_BAD;
  if (window < 0 || keep_first < 0 || (keep_first > 0 && window <= 0) || opt->softcap < 0.f || (opt->dist_bias && opt->n_dist < 1)) return PK_BAD;
  if (opt->beside && !pegainfer_paged_attention_beside_ok(opt, dtype)) return PK_BAD;
  if (opt->scan_beside && (opt->beside || !pegainfer_paged_attention_scan_ok(opt, dtype))) return PK_BAD;
  if (n_split < 1) n_split = 1;
  if (n_split > 1 && (!workspace || n_split > 64)) return PK_BAD;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || (maps != 1 && maps != 2) || maps * dim > 256 || vdim <= 0 ||
      vdim > 256 || page_size <= 0 || kv_heads > 65535 || block < 0 || opt->shared_tail < 0 || opt->shared_tail > dim ||
      (opt->shared_tail > 0 && (maps != 1 || vdim != dim)))
    return PK_BAD;
  const int qd = maps * dim;
  const size_t smem = ((size_t)kAttKeys * (qd + 1) + (size_t)kAttKeys * vdim + (size_t)kAttRows * qd + 4 * maps * 64 * kAttRpw) * sizeof(float);
  const dim3 grid(n_tiles, kv_heads, n_split);
  AttnForm form;
  form.block = block;
  form.sink = opt->sink;
  form.lambda = opt->lambda;
  form.head_norm = opt->head_norm;
  form.norm_eps = opt->norm_eps;
  form.softcap = opt->softcap;
  form.window = window;
  form.keep_first = window > 0 ? keep_first : 0;
  form.dist_bias = opt->dist_bias;
  form.n_dist = opt->n_dist;
  form.dist_slope = opt->dist_slope;
  form.gate = opt->gate;
  form.gate_stride = opt->gate_stride;
  form.gate_kind = gate_kind;
  form.k_keep = qd - opt->shared_tail;
  bool ok = true;
  if (opt->tile_rows > kAttRows) {    // tables cut for the prompts' kernel
    if ((opt->tile_rows != 32 && opt->tile_rows != 64) || (maps != 1 && !(two_wide && rows_two_maps_ok(dim, vdim))) || n_split != 1 || plain || dtype != kDtBf16 || out_stride % 4 ||
        !host_aligned16(out) || !host_aligned16(q) || !host_aligned16(cache) || k_cache_off % 8 ||
        !pegainfer_paged_attention_rows_ok(qd, vdim, opt->shared_tail, page_stride, v_cache_off, page_size))
      return PK_BAD;
    auto launch = [&](auto kern, size_t lds, int rg) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
        ok = false;
        return;
      }
      kern<<<dim3(n_tiles, kv_heads), rg * 128, lds, as_stream(stream)>>>(
          q, static_cast<const uint16_t*>(cache), page_stride, k_cache_off, v_cache_off, page_size, positions, row_entry, page_indptr, page_ids,
          heads, kv_heads, dim, vdim, scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh, static_cast<uint16_t*>(out), out_stride, form);
    };
    auto by_size = [&](auto rg) {
      constexpr int RG = decltype(rg)::value;
      const int most = std::max(qd, vdim);
      if (maps == 2 && most <= 64) launch(paged_attention_rows_kernel<64, RG, 2>, rows_attention_lds<64, RG, 2>(), RG);
      else if (maps == 2) launch(paged_attention_rows_kernel<128, RG, 2>, rows_attention_lds<128, RG, 2>(), RG);
      else if (most <= 64) launch(paged_attention_rows_kernel<64, RG, 1>, rows_attention_lds<64, RG, 1>(), RG);
      else if (most <= 128) launch(paged_attention_rows_kernel<128, RG, 1>, rows_attention_lds<128, RG, 1>(), RG);
      else launch(paged_attention_rows_kernel<256, RG, 1>, rows_attention_lds<256, RG, 1>(), RG);
    };
    if (opt->tile_rows == 64) by_size(std::integral_constant<int, 4>());
    else by_size(std::integral_constant<int, 2>());
    return ok ? (pegainfer_status_t)hipGetLastError() : PK_BAD;
  }
  if (dtype == kDtBf16 && !plain) {   // bf16 cache: the matrix-core kernel; same tiles, same splits, same merge
    const int ncb = vdim <= 32 ? 2 : vdim <= 64 ? 4 : vdim <= 128 ? 8 : 16;
    const size_t lds = mfma_attention_lds(maps, dim, ncb);
    // own: what the kernel has besides, at most; 64 KB in all need no request
    auto launch_as = [&](auto kern, dim3 blocks, int threads, size_t own, auto... more) {
      if (lds + own > 64 * 1024 &&
          hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
        ok = false;
        return;
      }
      kern<<<blocks, threads, lds, as_stream(stream)>>>(q, static_cast<const uint16_t*>(cache), page_stride, k_cache_off, v_cache_off, page_size,
                                                        positions, row_entry, page_indptr, page_ids, heads, kv_heads, dim, vdim, scale, factor,
                                                        tile_row0, tile_ntok, tile_qh0, tile_nqh, static_cast<uint16_t*>(out), out_stride, form,
                                                        n_split, workspace, more...);
    };
    auto launch = [&](auto kern) { launch_as(kern, grid, 256, 16 * 1024); };
    if (const pegainfer_recurrent_step_desc* step = opt->beside) {
      const dim3 blocks((unsigned)((int64_t)n_tiles * kv_heads * n_split + (int64_t)step->heads * step->n_entries));
      auto both = [&](auto kern) { launch_as(kern, blocks, kStepThreads, 16 * 1024, (int)n_tiles, *step); };
      if (ncb == 2) both(paged_attention_beside_kernel<2>);
      else if (ncb == 4) both(paged_attention_beside_kernel<4>);
      else if (ncb == 8) both(paged_attention_beside_kernel<8>);
      else both(paged_attention_beside_kernel<16>);
    } else if (const pegainfer_scan_beside_desc* d = opt->scan_beside) {
      const pegainfer_ssd_scan_desc& scan = *d->scan;
      const int nbx = ceil_div(scan.vdim, kRecCols);
      const dim3 blocks((unsigned)((int64_t)n_tiles * kv_heads * n_split + (int64_t)nbx * scan.heads * scan.n_entries));
      auto both = [&](auto kern) { launch_as(kern, blocks, 256, 24 * 1024, (int)n_tiles, scan, nbx); };
      auto by_states = [&](auto cols) {
        constexpr int NCB = decltype(cols)::value;
        if (scan.n_state > 64) both(paged_attention_scan_kernel<NCB, 8>);
        else both(paged_attention_scan_kernel<NCB, 4>);
      };
      if (ncb == 2) by_states(std::integral_constant<int, 2>());
      else if (ncb == 4) by_states(std::integral_constant<int, 4>());
      else if (ncb == 8) by_states(std::integral_constant<int, 8>());
      else by_states(std::integral_constant<int, 16>());
      if (!ok) return PK_BAD;
      const unsigned merge = (unsigned)((int64_t)n_tiles * kv_heads * kAttRows + ceil_div((long)d->rows * d->heads, 4));
      auto finish = [&](auto kern) {
        kern<<<merge, 256, 0, as_stream(stream)>>>(workspace, n_split, heads, kv_heads, vdim, factor, positions, tile_row0, tile_ntok, tile_qh0, tile_nqh,
                                                   static_cast<uint16_t*>(out), out_stride, form, (int)n_tiles, *d, scan.o);
      };
      const int v = head_rms_values(scan.o, d->norm_w, d->gate, d->gate_stride, d->out, d->out_stride, d->vdim);
      if (v == 4) finish(paged_attention_merge_norm_kernel<4>);
      else if (v == 2) finish(paged_attention_merge_norm_kernel<2>);
      else finish(paged_attention_merge_norm_kernel<1>);
      return (pegainfer_status_t)hipGetLastError();
    } else {
    auto by_cols = [&](auto maps_c) {
      constexpr int M = decltype(maps_c)::value;
      if (ncb == 2) launch(paged_attention_mfma_kernel<M, 2>);
      else if (ncb == 4) launch(paged_attention_mfma_kernel<M, 4>);
      else if (ncb == 8) launch(paged_attention_mfma_kernel<M, 8>);
      else launch(paged_attention_mfma_kernel<M, 16>);
    };
    if (maps == 1) by_cols(std::integral_constant<int, 1>());
    else by_cols(std::integral_constant<int, 2>());
    }
    if (ok && n_split > 1) {
      if (maps == 1)
        paged_attention_merge_kernel<uint16_t, 1><<<dim3(n_tiles, kv_heads, kAttRows), 256, 0, as_stream(stream)>>>(
            workspace, n_split, heads, kv_heads, vdim, factor, positions, tile_row0, tile_ntok, tile_qh0, tile_nqh, static_cast<uint16_t*>(out), out_stride, form);
      else
        paged_attention_merge_kernel<uint16_t, 2><<<dim3(n_tiles, kv_heads, kAttRows), 256, 0, as_stream(stream)>>>(
            workspace, n_split, heads, kv_heads, vdim, factor, positions, tile_row0, tile_ntok, tile_qh0, tile_nqh, static_cast<uint16_t*>(out), out_stride, form);
    }
    return ok ? (pegainfer_status_t)hipGetLastError() : PK_BAD;
  }
  const bool known = by_dtype(dtype, [&](auto* t) {
    using A = std::remove_pointer_t<decltype(t)>;
    auto go = [&](auto kern) {
      if (smem > 48 * 1024 &&
          hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
        ok = false;
        return;
      }
      kern<<<grid, 256, smem, as_stream(stream)>>>(q, static_cast<const A*>(cache), page_stride, k_cache_off, v_cache_off,
                                                   page_size, positions, row_entry, page_indptr, page_ids, heads, kv_heads, dim,
                                                   vdim, scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh,
                                                   static_cast<A*>(out), out_stride, form, n_split, workspace);
    };
    auto merge = [&](auto kern) {
      kern<<<dim3(n_tiles, kv_heads, kAttRows), 256, 0, as_stream(stream)>>>(workspace, n_split, heads, kv_heads, vdim, factor, positions, tile_row0,
                                                                    tile_ntok, tile_qh0, tile_nqh, static_cast<A*>(out), out_stride, form);
    };
    if (maps == 1) {
      go(paged_attention_kernel<A, 1>);
      if (ok && n_split > 1) merge(paged_attention_merge_kernel<A, 1>);
    } else {
      go(paged_attention_kernel<A, 2>);
      if (ok && n_split > 1) merge(paged_attention_merge_kernel<A, 2>);
    }
  });
  return known && ok ? (pegainfer_status_t)hipGetLastError() : PK_BAD;
}

pegainfer_status_t pegainfer_paged_attention_opt(const float* q, const void* cache, int64_t page_stride, int64_t k_cache_off,
                                                 int64_t v_cache_off, int32_t page_size, const int32_t* positions,
                                                 const int32_t* row_entry, const int32_t* page_indptr, const int32_t* page_ids,
                                                 int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, float scale,
                                                 float factor, const int32_t* tile_row0, const int32_t* tile_ntok,
                                                 const int32_t* tile_qh0, const int32_t* tile_nqh, int32_t n_tiles, void* out,
                                                 int64_t out_stride, const pegainfer_attn_options* opt, int32_t dtype,
                                                 pegainfer_stream_t stream) {
  return paged_attention(q, cache, page_stride, k_cache_off, v_cache_off, page_size, positions, row_entry, page_indptr, page_ids, heads, kv_heads, dim, vdim,
                         scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh, n_tiles, out, out_stride, opt, dtype, stream, false);
}

pegainfer_status_t pegainfer_paged_attention_maps(const float* q, const void* cache, int64_t page_stride, int64_t k_cache_off,
                                                  int64_t v_cache_off, int32_t page_size, const int32_t* positions,
                                                  const int32_t* row_entry, const int32_t* page_indptr, const int32_t* page_ids,
                                                  int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, float scale,
                                                  float factor, const int32_t* tile_row0, const int32_t* tile_ntok,
                                                  const int32_t* tile_qh0, const int32_t* tile_nqh, int32_t n_tiles, void* out,
                                                  int64_t out_stride, const pegainfer_attn_options* opt, int32_t dtype,
                                                  pegainfer_stream_t stream) {
  return paged_attention(q, cache, page_stride, k_cache_off, v_cache_off, page_size, positions, row_entry, page_indptr, page_ids, heads, kv_heads, dim, vdim,
                         scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh, n_tiles, out, out_stride, opt, dtype, stream, true);
}

int32_t pegainfer_paged_attention_maps_rows_ok(int32_t maps, int32_t dim, int32_t vdim, int64_t page_stride, int64_t v_cache_off,
                                               int32_t page_size) {
  return (maps == 1 || (maps == 2 && rows_two_maps_ok(dim, vdim))) &&
         pegainfer_paged_attention_rows_ok(maps * dim, vdim, 0, page_stride, v_cache_off, page_size);
}

int32_t pegainfer_paged_attention_rows_ok(int32_t dim, int32_t vdim, int32_t shared_tail, int64_t page_stride, int64_t v_cache_off,
                                          int32_t page_size) {
  return dim > 0 && dim <= 256 && dim % 8 == 0 && vdim > 0 && vdim <= 256 && vdim % 8 == 0 && shared_tail % 8 == 0 && page_stride % 8 == 0 &&
         v_cache_off % 8 == 0 && page_size > 0;
}

int64_t pegainfer_paged_attention_workspace(int32_t n_tiles, int32_t kv_heads, int32_t vdim, int32_t maps, int32_t n_split) {
  return n_split > 1 ? (int64_t)n_tiles * kv_heads * n_split * kAttRows * maps * (vdim + 2) : 0;
}

pegainfer_status_t pegainfer_paged_attention(const float* q, const void* cache, int64_t page_stride, int64_t k_cache_off,
                                             int64_t v_cache_off, int32_t page_size, const int32_t* positions,
                                             const int32_t* row_entry, const int32_t* page_indptr, const int32_t* page_ids,
                                             int32_t heads, int32_t kv_heads, int32_t dim, int32_t vdim, float scale,
                                             float factor, const int32_t* tile_row0, const int32_t* tile_ntok,
                                             const int32_t* tile_qh0, const int32_t* tile_nqh, int32_t n_tiles, void* out,
                                             int64_t out_stride, int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_paged_attention_ex(q, cache, page_stride, k_cache_off, v_cache_off, page_size, positions, row_entry, page_indptr,
                                      page_ids, heads, kv_heads, dim, vdim, scale, factor, tile_row0, tile_ntok, tile_qh0, tile_nqh,
                                      n_tiles, out, out_stride, 1, 0.f, 0, nullptr, 0, 0.f, 1, nullptr, 1, dtype, stream);
}

pegainfer_status_t pegainfer_scale_rows(const void* in, int64_t in_stride, void* out, int64_t out_stride, int32_t cols,
                                        int32_t rows, float factor, int32_t dtype, pegainfer_stream_t stream) {
  if (rows <= 0 || cols <= 0) return 0;
  const dim3 grid(rows, std::min(8, ceil_div(cols, 256)));
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        scale_rows_kernel<A><<<grid, 256, 0, as_stream(stream)>>>(static_cast<const A*>(in), in_stride, static_cast<A*>(out),
                                                                  out_stride, cols, factor);
      }))
    return PK_BAD;
  return (pegainfer_status_t)hipGetLastError();
}

}  // extern "C"
