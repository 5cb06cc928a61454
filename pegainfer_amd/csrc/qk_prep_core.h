// The preparation of a token row's queries, keys and values, as a part of a launch: attn_paged.hip's own, and recurrent.hip's where a layer has both halves.
#pragma once

#include "common.h"
#include "typed.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

// how qk_prep_paged_kernel norms and rotates
struct PrepForm {
  int norm_kind = 0;    // 0: per head before the rotation, times a weight [dim] (when weights are given); 1: per head AFTER the
                        // rotation, no weight (unit root mean square); 2: over ALL heads of the projection at once before the
                        // rotation, times a weight [heads * dim] / [kv_heads * dim]
  int rot_halves = 0;   // 0: neighbours (2i, 2i + 1) are rotated together; 1: value i with value i + rot_dims / 2
  float rot_amp = 1.f;  // factor of every cosine and sine
  int k_keep = 0;       // leading values of a key that go to the key part of the cache (dim unless the rest is the value's)
};

// I: type of the projection rows read (the storage type, or float for rows that an fp32 stage such as a convolution left).  V: neighbouring
// values that a lane takes at once (2 where every offset, stride and pointer allows it).
// Bound by the launch with few rows and by memory with many; what kept it from either was one head's chain of loads after another (page
// number, angles, barrier, then the head's values, then its weights).  A wave's next head is on its way while the present one is worked on, the
// first one and the values before the angles: one row with a norm over all heads 9.3 -> 6.0 us, eight rows 5.1 -> 4.4 us,
// 1024 rows 22.6 -> 16.6 us (norms per head) and 18.3 -> 13.4 us (over all heads).
// of 256 threads: row, workgroup by of nby of the row; sm: (4 dim + rot_dims) floats of LDS
template <typename A, typename I, int V>
__device__ __forceinline__ void qk_prep_block(
    float* sm, int row, int by, int nby,
    const I* __restrict__ proj, int64_t proj_stride, int64_t q_off, int64_t k_off, int64_t v_off, int H, int G, int dim, int vdim,
    const A* __restrict__ q_norm, const A* __restrict__ k_norm, float eps, const float* __restrict__ inv_freq, int rot_dims,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ row_entry, const int32_t* __restrict__ page_indptr,
    const int32_t* __restrict__ page_ids, A* __restrict__ cache, int64_t page_stride, int64_t k_cache_off, int64_t v_cache_off,
    int page_size, float* __restrict__ q_out, A* __restrict__ q_out_stored, const A* __restrict__ q_bias,
    const A* __restrict__ k_bias, const A* __restrict__ v_bias, float qt_coef, int qt_every, PrepForm pf) {
  constexpr int C = 4 / V;        // dim <= 256: a lane's values i = V lane + u + 64 V c
  // sm: [4 waves][dim], then the row's cosines and sines [rot_dims / 2] each
  __shared__ float red[8];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  auto load = [&](const auto* p, float* t) {
    if constexpr (V == 2) ld2(p, t); else t[0] = ld(p);
  };
  auto store = [&](auto* p, const float* t) {
    if constexpr (V == 2) st2(p, t); else st(p, t[0]);
  };
  const I* pr = proj + (int64_t)row * proj_stride;
  float* buf = sm + wave * dim;
  struct Head { float x[C][V], b[C][V], w[C][V]; };
  auto fetch = [&](int hh, Head& n) {
    const bool is_q = hh < H;
    const int hd = is_q ? hh : hh - H;
    const I* src = pr + (is_q ? q_off : k_off) + (int64_t)hd * dim;
    const A* bs = is_q ? q_bias : k_bias;
    const A* nw = is_q ? q_norm : k_norm;
    if (pf.norm_kind == 2) nw += (int64_t)hd * dim;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = V * (lane + 64 * c);
      if (i >= dim) continue;
      load(src + i, n.x[c]);
      if (bs) load(bs + (int64_t)hd * dim + i, n.b[c]);
      if (nw && pf.norm_kind != 1) load(nw + i, n.w[c]);
    }
  };
  Head next;
  int hh = by * 4 + wave;   // the row's heads are dealt to the workgroups of its grid column, a wave per head
  if (hh < H + G) fetch(hh, next);
  const int pos = positions[row], e = row_entry[row];
  // the projected values: two groups of a thread are kept until the page is known
  constexpr int kValues = 2;
  float vals[kValues][V], vb[kValues][V];
  const int v_step = 256 * V * nby, v_first = (by * 256 + threadIdx.x) * V;
#pragma unroll
  for (int c = 0; c < kValues; ++c) {
    const int i = v_first + c * v_step;
    if (i >= G * vdim) continue;
    load(pr + v_off + i, vals[c]);
    if (v_bias) load(v_bias + i, vb[c]);
  }
  const int64_t page = page_ids[page_indptr[e] + pos / page_size];
  const int slot = pos % page_size;
  // query temperature: a factor on the whole query that grows with the logarithm of the position's block number
  const float qt = qt_every > 0 ? 1.0f + qt_coef * logf((float)((pos + 1) / qt_every) + 1.0f) : 1.0f;
  float inv_all_q = 1.f, inv_all_k = 1.f;
  if (pf.norm_kind == 2) {   // root mean squares over the whole q and the whole k projection
    auto squares = [&](const I* src, const A* bias, int n) {
      float ss = 0.f;
#pragma unroll 4
      for (int i = threadIdx.x * V; i < n; i += 256 * V) {
        float v[V], b[V];
        load(src + i, v);
        if (bias) load(bias + i, b);
#pragma unroll
        for (int u = 0; u < V; ++u) {
          const float t = v[u] + (bias ? b[u] : 0.f);
          ss = fmaf(t, t, ss);
        }
      }
      return wave_sum(ss);
    };
    const float sq = squares(pr + q_off, q_bias, H * dim), sk = squares(pr + k_off, k_bias, G * dim);
    if (lane == 0) { red[wave] = sq; red[4 + wave] = sk; }
  }
  const int half = rot_dims >> 1;
  float *s_cs = sm + 4 * dim, *s_sn = s_cs + half;   // every head turns by the same angles
  for (int f = threadIdx.x; f < half; f += 256) {
    const float ang = (float)pos * inv_freq[f];
    s_cs[f] = cosf(ang) * pf.rot_amp;
    s_sn[f] = sinf(ang) * pf.rot_amp;
  }
  __syncthreads();
  if (pf.norm_kind == 2) {
    inv_all_q = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)(H * dim) + eps);
    inv_all_k = 1.0f / sqrtf((red[4] + red[5] + red[6] + red[7]) / (float)(G * dim) + eps);
  }
  for (; hh < H + G; hh += 4 * nby) {
    const bool is_q = hh < H;
    const int hd = is_q ? hh : hh - H;
    const bool biased = is_q ? q_bias : k_bias;
    const Head cur = next;
    if (hh + 4 * nby < H + G) fetch(hh + 4 * nby, next);
    float x[C][V], ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int u = 0; u < V; ++u) {
        x[c][u] = V * (lane + 64 * c) < dim ? cur.x[c][u] + (biased ? cur.b[c][u] : 0.f) : 0.f;
        ss = fmaf(x[c][u], x[c][u], ss);
      }
    const bool weighted = pf.norm_kind == 2 || (pf.norm_kind == 0 && q_norm);
    const float inv = pf.norm_kind == 2 ? (is_q ? inv_all_q : inv_all_k) : weighted ? 1.0f / sqrtf(wave_sum(ss) / (float)dim + eps) : 1.0f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = V * (lane + 64 * c);
      if (i >= dim) continue;
#pragma unroll
      for (int u = 0; u < V; ++u) {
        if (weighted) x[c][u] = x[c][u] * inv * cur.w[c][u];
        if (is_q && qt_every > 0) x[c][u] *= qt;
        buf[i + u] = x[c][u];
      }
    }
    __builtin_amdgcn_wave_barrier();
    float ss2 = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const int i = V * (lane + 64 * c) + u;
        if (i < rot_dims) {          // rot_dims <= dim
          if (pf.rot_halves) {
            const int f = i < half ? i : i - half;
            const float cs = s_cs[f], sn = s_sn[f];
            x[c][u] = i < half ? x[c][u] * cs - buf[i + half] * sn : x[c][u] * cs + buf[i - half] * sn;
          } else {
            const float cs = s_cs[i >> 1], sn = s_sn[i >> 1];
            x[c][u] = (i & 1) ? x[c][u] * cs + buf[i - 1] * sn : x[c][u] * cs - buf[i + 1] * sn;
          }
        }
        ss2 = fmaf(x[c][u], x[c][u], ss2);
      }
    const float post = pf.norm_kind == 1 ? 1.0f / sqrtf(wave_sum(ss2) / (float)dim + eps) : 1.0f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = V * (lane + 64 * c);
      if (i >= dim) continue;
#pragma unroll
      for (int u = 0; u < V; ++u) x[c][u] *= post;
      if (is_q) {
        if (q_out_stored) store(q_out_stored + ((int64_t)row * H + hh) * dim + i, x[c]);
        else store(q_out + ((int64_t)row * H + hh) * dim + i, x[c]);
      } else if (i < pf.k_keep)
        store(cache + page * page_stride + k_cache_off + ((int64_t)slot * G + hd) * pf.k_keep + i, x[c]);
    }
    __builtin_amdgcn_wave_barrier();
  }
  A* dst = cache + page * page_stride + v_cache_off + (int64_t)slot * G * vdim;
#pragma unroll
  for (int c = 0; c < kValues; ++c) {
    const int i = v_first + c * v_step;
    if (i >= G * vdim) continue;
#pragma unroll
    for (int u = 0; u < V; ++u) vals[c][u] += v_bias ? vb[c][u] : 0.f;
    store(dst + i, vals[c]);
  }
  for (int i = v_first + kValues * v_step; i < G * vdim; i += v_step) {
    float v[V], b[V];
    load(pr + v_off + i, v);
    if (v_bias) load(v_bias + i, b);
#pragma unroll
    for (int u = 0; u < V; ++u) v[u] += v_bias ? b[u] : 0.f;
    store(dst + i, v);
  }
}

// workgroups of a row: with few rows (decoding) its heads spread over several, four heads each; many rows fill the chip alone (two or three
// workgroups for each of a thousand rows: 13.4 -> 16.1 us)
inline int qk_prep_per_row(const pegainfer_qk_prep_desc& p) { return p.n_rows >= 512 ? 1 : std::min(16, ceil_div(p.heads + p.kv_heads, 4)); }
inline size_t qk_prep_lds(const pegainfer_qk_prep_desc& p) { return ((size_t)4 * p.dim + p.rot_dims) * sizeof(float); }
inline PrepForm qk_prep_form(const pegainfer_qk_prep_desc& p) {
  PrepForm pf;
  pf.norm_kind = p.norm_kind;
  pf.rot_halves = p.rot_layout == PEGAINFER_ROT_HALVES;
  pf.rot_amp = p.rot_amp;
  pf.k_keep = p.dim - p.shared_tail;
  return pf;
}
inline bool qk_prep_ok(const pegainfer_qk_prep_desc* p) {
  return !(p->heads <= 0 || p->kv_heads <= 0 || p->dim <= 0 || p->dim > 256 || p->vdim <= 0 || p->rot_dims < 0 || p->rot_dims > p->dim ||
           (p->rot_dims & 1) || p->page_size <= 0 || (p->rot_dims > 0 && !p->inv_freq) || (!p->q_norm) != (!p->k_norm) || p->norm_kind < 0 ||
           p->norm_kind > 2 || (p->norm_kind == PEGAINFER_QKNORM_ALL_WEIGHT && !p->q_norm) ||
           (p->rot_layout != PEGAINFER_ROT_PAIRS && p->rot_layout != PEGAINFER_ROT_HALVES) || p->shared_tail < 0 || p->shared_tail > p->dim);
}
// two values per lane where rows, offsets and pointers allow it
inline bool qk_prep_pairs(const pegainfer_qk_prep_desc* p) {
  return !((p->dim | p->vdim | (p->dim - p->shared_tail) | p->proj_stride | p->q_off | p->k_off | p->v_off | p->page_stride | p->k_cache_off |
            p->v_cache_off) & 1) && host_aligned8(p->proj) && host_aligned8(p->q_norm) && host_aligned8(p->k_norm) &&
         host_aligned8(p->cache) && host_aligned8(p->q_out) && host_aligned8(p->q_out_stored) && host_aligned8(p->q_bias) &&
         host_aligned8(p->k_bias) && host_aligned8(p->v_bias);
}
// the block on a description's pointers
template <typename A, typename I, int V>
__device__ __forceinline__ void qk_prep_block(float* sm, int row, int by, int nby, const pegainfer_qk_prep_desc& p, const PrepForm& pf) {
  qk_prep_block<A, I, V>(sm, row, by, nby, static_cast<const I*>(p.proj), p.proj_stride, p.q_off, p.k_off, p.v_off, p.heads, p.kv_heads, p.dim, p.vdim,
                         static_cast<const A*>(p.q_norm), static_cast<const A*>(p.k_norm), p.eps, p.inv_freq, p.rot_dims, p.positions, p.row_entry,
                         p.page_indptr, p.page_ids, static_cast<A*>(p.cache), p.page_stride, p.k_cache_off, p.v_cache_off, p.page_size, p.q_out,
                         static_cast<A*>(p.q_out_stored), static_cast<const A*>(p.q_bias), static_cast<const A*>(p.k_bias),
                         static_cast<const A*>(p.v_bias), p.qt_coef, p.qt_every, pf);
}

}  // namespace pk
