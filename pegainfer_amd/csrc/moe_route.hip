// Routed feed-forward: the router and the bookkeeping around the expert GEMMs (which run on the grouped form of
// pegainfer_gemm_strided).
//   route_kernel    one workgroup per token row: fp32 router logits (a wave per expert, lanes over the width), sigmoid
//                   scores, the correction added for the CHOICE only, group scores = the two largest choices of a group,
//                   the best `keep` groups stay eligible, then the `top` largest eligible choices; weights = the plain
//                   sigmoid scores of the chosen experts.  Selection runs on one wave: a lane per group for the group
//                   scores and ranks, then a lane per expert that counts the choices ahead of its own (beyond 64 experts
//                   `top` wave-wide arg-max steps); ties go to the lower index.
//   sort_kernel     (row, choice) pairs bucketed by expert with LDS counters, an exclusive scan, and the table of <= 64-row
//                   tiles the grouped GEMM walks.  The order of pairs inside an expert comes from atomics; every pair owns
//                   its output row, so results do not depend on it.  Tiles hold <= 64 or <= 128 rows, as the GEMM form that walks them wants, or no
//                   more than a step of few rows has: an expert gets more pairs than that when a row without eligible experts fills its choices.
//   combine_kernel  out[row] = sum over the row's choices, in choice order, of weight * expert output (fp32 sum), plus a row
//                   every token gets (a shared expert), optionally times the sigmoid of a per-row gate logit.
// Options of the selection: a group's score = its two largest choices (default) or its largest; the chosen weights as they
// are (default) or divided by their sum, times a factor.  Expert numbers past the experts that have tensors are identity experts:
// they get no position in the sort, and the combine takes the feed-forward's input row for them.
//   route_plan_kernel  selection and sort in one launch for steps of up to 16 rows
#include <algorithm>

#include "route_core.h"

namespace pk {

// Few rows: sixteen waves of two experts each, four loads of the width ahead; many rows fill the chip with four waves of four experts.
// 4 rows of 2048, 32 experts: 20.0 us with four waves -> 9.8 us.  The order of a logit's sum is the lanes' alone.
template <typename A, int N, int EB>
__global__ __launch_bounds__(N) void route_kernel(const A* __restrict__ h, const A* __restrict__ wr,
                                                  const A* __restrict__ corr, int32_t* __restrict__ out_e,
                                                  float* __restrict__ out_w, int d, int E, int G, int keep, int top,
                                                  int score) {
  extern __shared__ float sm[];
  float* s = sm;            // [E] sigmoid scores
  float* ch = sm + E;       // [E] choice scores (eligible) or -inf
  float* gs = sm + 2 * E;   // [G] group scores
  const int row = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const A* x = h + (size_t)row * d;
  const bool vec = (d & 7) == 0 && aligned16(x) && aligned16(wr);
  // a wave takes EB experts at a time (independent weight streams in flight), waves interleaved over the groups of EB
  for (int e0 = wave * EB; e0 < E; e0 += N / 64 * EB) {
    float a[EB] = {};
    if (vec) {
#pragma unroll 4
      for (int i = lane * 8; i < d; i += 512) {
        float xv[8];
        Vec8<A>::load(x + i, xv);
#pragma unroll
        for (int q = 0; q < EB; ++q) {
          float wv[8];
          Vec8<A>::load(wr + (size_t)min(e0 + q, E - 1) * d + i, wv);
#pragma unroll
          for (int k = 0; k < 8; ++k) a[q] = fmaf(xv[k], wv[k], a[q]);
        }
      }
    } else {
      for (int i = lane; i < d; i += 64) {
        const float xv = ld(x + i);
#pragma unroll
        for (int q = 0; q < EB; ++q) a[q] = fmaf(xv, ld(wr + (size_t)min(e0 + q, E - 1) * d + i), a[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < EB; ++q) {
      const float z = wave_sum(a[q]);
      const int e = e0 + q;
      if (lane == 0 && e < E) {
        const float sc = score == PEGAINFER_SCORE_SOFTMAX ? z : sigmoid_f(z);   // softmax: the logit for now
        s[e] = sc;
        ch[e] = corr ? sc + ld(corr + e) : sc;
      }
    }
  }
  __syncthreads();
  if (wave != 0) return;
  route_select_wave(s, ch, gs, corr, out_e, out_w, row, lane, E, G, keep, top, score);
}

// The same selection from router logits that a GEMM has left in fp32 ([rows][E] at a stride), by one wave with LDS of its own.
struct RouteForm {
  int E, G, keep, top, score, group_kind, renorm;
  float factor;
  int64_t logits_stride;
};
template <typename A>
__device__ __forceinline__ void route_row_from_logits(const float* __restrict__ logits, const A* __restrict__ corr, int32_t* out_e,
                                                      float* out_w, const RouteForm& f, int row, int lane, float* s, int* pairs = nullptr) {
  float *ch = s + f.E, *gs = s + 2 * f.E;
  for (int e = lane; e < f.E; e += 64) {
    const float z = logits[(size_t)row * f.logits_stride + e];
    const float sc = f.score == PEGAINFER_SCORE_SOFTMAX ? z : sigmoid_f(z);
    s[e] = sc;
    ch[e] = corr ? sc + ld(corr + e) : sc;
  }
  __builtin_amdgcn_wave_barrier();
  route_select_wave(s, ch, gs, corr, out_e, out_w, row, lane, f.E, f.G, f.keep, f.top, f.score, f.group_kind, f.renorm, f.factor, pairs);
}
// a wave per row, four rows per workgroup
template <typename A>
__global__ __launch_bounds__(256) void route_from_logits_kernel(const float* __restrict__ logits, const A* __restrict__ corr,
                                                                int32_t* __restrict__ out_e, float* __restrict__ out_w, int rows,
                                                                RouteForm f) {
  extern __shared__ float sm[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + wave;
  if (row >= rows) return;
  route_row_from_logits(logits, corr, out_e, out_w, f, row, lane, sm + wave * (2 * f.E + f.G));
}

struct SortOut {
  int32_t *pos_pair, *pos_row, *tile_group, *tile_row0, *tile_rows, *n_tiles;
  int max_tiles, per_tile;
};
// Pairs whose expert number is E or more (identity experts) get no position.  One workgroup of N threads; cnt: [2 E] of LDS.
template <int N>
__device__ __forceinline__ void route_sort_block(const int32_t* expert, int n_pairs, int top, int E, const SortOut& o, int* cnt) {
  int* cur = cnt + E;            // [E] counts, then [E] cursors
  for (int e = threadIdx.x; e < E; e += N) cnt[e] = 0;
  __syncthreads();
  constexpr int kKeep = 4;       // a thread's first choices stay in registers between the two walks
  int mine[kKeep];
#pragma unroll
  for (int k = 0; k < kKeep; ++k) {
    const int p = threadIdx.x + N * k;
    mine[k] = p < n_pairs ? expert[p] : E;
  }
#pragma unroll
  for (int k = 0; k < kKeep; ++k)
    if (mine[k] < E) atomicAdd(&cnt[mine[k]], 1);
  for (int p = threadIdx.x + N * kKeep; p < n_pairs; p += N) {
    const int e = expert[p];
    if (e < E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < 64) {        // offsets and tiles by two scans over the experts, 64 at a time
    const int lane = threadIdx.x;
    int off = 0, nt = 0;         // before this run of 64
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane, c = e < E ? cnt[e] : 0, tiles = (c + o.per_tile - 1) / o.per_tile;
      int c_sum = c, t_sum = tiles;
#pragma unroll
      for (int x = 1; x < 64; x <<= 1) {
        const int a = __shfl_up(c_sum, x, kWave), b = __shfl_up(t_sum, x, kWave);
        if (lane >= x) { c_sum += a; t_sum += b; }
      }
      const int first = off + c_sum - c, tile0 = nt + t_sum - tiles;
      if (e < E) cur[e] = first;
      for (int k = 0; k < tiles && tile0 + k < o.max_tiles; ++k) {
        o.tile_group[tile0 + k] = e;
        o.tile_row0[tile0 + k] = first + k * o.per_tile;
        o.tile_rows[tile0 + k] = min(o.per_tile, c - k * o.per_tile);
      }
      off += __shfl(c_sum, 63, kWave);
      nt += __shfl(t_sum, 63, kWave);
    }
    if (lane == 0) *o.n_tiles = min(nt, o.max_tiles);
  }
  __syncthreads();
  auto place = [&](int p, int e) {
    if (e >= E) return;
    const int at = atomicAdd(&cur[e], 1);
    o.pos_pair[at] = p;
    o.pos_row[at] = p / top;
  };
#pragma unroll
  for (int k = 0; k < kKeep; ++k) place(threadIdx.x + N * k, mine[k]);
  for (int p = threadIdx.x + N * kKeep; p < n_pairs; p += N) place(p, expert[p]);
}
constexpr int kSortThreads = 1024;
__global__ __launch_bounds__(kSortThreads) void route_sort_kernel(const int32_t* __restrict__ expert, int n_pairs, int top, int E, SortOut o) {
  extern __shared__ int cnt[];
  route_sort_block<kSortThreads>(expert, n_pairs, top, E, o, cnt);
}
// Few rows (decoding): selection and sort in one launch of one workgroup, a wave per row; the choices pass to the sort through LDS.
// 8 rows, 16 experts and an identity one: 14.6 us (four waves in turn, choices and weights read back from memory, one thread laying out
// the tiles) -> 6.2 us; selection and sort in two launches 13.0 us.
template <typename A>
__global__ __launch_bounds__(kSortThreads) void route_plan_kernel(const float* __restrict__ logits, const A* __restrict__ corr, int32_t* out_e,
                                                                  float* out_w, int rows, RouteForm f, int sort_experts, SortOut o) {
  extern __shared__ float sm[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, per = 2 * f.E + f.G;
  int* pairs = reinterpret_cast<int*>(sm + rows * per);
  if (wave < rows) route_row_from_logits(logits, corr, out_e, out_w, f, wave, lane, sm + wave * per, pairs);
  __syncthreads();               // the selection's LDS is free
  route_sort_block<kSortThreads>(pairs, rows * f.top, f.top, sort_experts, o, reinterpret_cast<int*>(sm));
}
constexpr int kPlanRows = kSortThreads / 64;

// expert / same: pairs that chose an expert number of same_from or more take the row of `same` (the feed-forward's own input) instead
// of a y_pairs row
// V columns per thread; up to four pairs' values are on their way at once (fp32 pairs of 1024 rows of 2560, three experts: 23.2 -> 9.8 us,
// 3421 rows of 1024 22.4 -> 12.3 us against a column and a pair at a time; bound by the pairs' bytes)
template <typename A, int V>
__global__ __launch_bounds__(256) void route_combine_kernel(const float* __restrict__ y, const float* __restrict__ w,
                                                            const A* __restrict__ add, A* __restrict__ out, int d, int top,
                                                            const float* __restrict__ add_gate, int64_t add_gate_stride,
                                                            const int32_t* __restrict__ expert, int same_from,
                                                            const A* __restrict__ same, int64_t same_stride,
                                                            const float* __restrict__ add_pairs, int n_add) {
  const int row = blockIdx.x;
  const float gate = (add || n_add) && add_gate ? sigmoid_f(add_gate[(size_t)row * add_gate_stride]) : 1.0f;
  auto load = [&](const auto* p, float* t) {
    if constexpr (V == 4) ld4(p, t); else t[0] = ld(p);
  };
  for (int i = (blockIdx.y * 256 + threadIdx.x) * V; i < d; i += gridDim.y * 256 * V) {
    float a[V] = {};
    if (add) load(add + (size_t)row * d + i, a);
    for (int j = 0; j < n_add; ++j) {
      float t[V];
      load(add_pairs + ((size_t)j * gridDim.x + row) * d + i, t);
#pragma unroll
      for (int u = 0; u < V; ++u) a[u] += t[u];
    }
#pragma unroll
    for (int u = 0; u < V; ++u) a[u] *= gate;
    for (int c0 = 0; c0 < top; c0 += 4) {
      float v[4][V], wt[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int c = c0 + k;
        if (c >= top) continue;
        const bool own = same && expert[(size_t)row * top + c] >= same_from;      // uniform over the workgroup
        if (own) load(same + (size_t)row * same_stride + i, v[k]); else load(y + ((size_t)row * top + c) * d + i, v[k]);
        wt[k] = w[(size_t)row * top + c];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (c0 + k < top)
#pragma unroll
          for (int u = 0; u < V; ++u) a[u] = fmaf(wt[k], v[k][u], a[u]);
    }
    if constexpr (V == 4) st4(out + (size_t)row * d + i, a); else st(out + (size_t)row * d + i, a[0]);
  }
}

}  // namespace pk

extern "C" {
using namespace pk;

int32_t pegainfer_router_tail_ok(int32_t experts, int32_t has_gate, int32_t d, int32_t dtype) {
  return router_tail_pays(experts, has_gate, d, dtype);
}

// 64 or 128, or for few rows whatever no tile of the table may pass
static bool tile_rows_ok(int n) { return n == 64 || n == 128 || (n >= 1 && n <= 16); }

pegainfer_status_t pegainfer_route_topk(const void* h, const void* w_router, const void* correction, int32_t* out_expert,
                                        float* out_weight, int32_t d, int32_t experts, int32_t n_groups, int32_t keep_groups,
                                        int32_t top, int32_t rows, int32_t score_kind, int32_t dtype, pegainfer_stream_t stream) {
  if (rows <= 0) return 0;
  if (score_kind != PEGAINFER_SCORE_SIGMOID && score_kind != PEGAINFER_SCORE_SOFTMAX) return (pegainfer_status_t)hipErrorInvalidValue;
  if (n_groups < 1) n_groups = 1;
  if (experts <= 0 || experts % n_groups || top <= 0 || top > experts || keep_groups < 1 || keep_groups > n_groups ||
      (size_t)(2 * experts + n_groups) * 4 > 60000)
    return (pegainfer_status_t)hipErrorInvalidValue;
  const size_t smem = (size_t)(2 * experts + n_groups) * sizeof(float);
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        auto run = [&](auto kern, int threads) {
          kern<<<rows, threads, smem, as_stream(stream)>>>(static_cast<const A*>(h), static_cast<const A*>(w_router),
                                                           static_cast<const A*>(correction), out_expert, out_weight, d, experts, n_groups,
                                                           keep_groups, top, score_kind);
        };
        if (rows <= device_cus()) run(&route_kernel<A, 1024, 2>, 1024);
        else run(&route_kernel<A, 256, 4>, 256);
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_route_plan(const pegainfer_route_plan_desc* q, pegainfer_stream_t stream) {
  constexpr pegainfer_status_t bad = (pegainfer_status_t)hipErrorInvalidValue;
  if (!q) return bad;
  if (q->rows <= 0) return 0;
  const int E = q->experts, groups = std::max(1, q->n_groups), keep = q->n_groups < 1 ? 1 : q->keep_groups, top = q->top;
  if (!q->logits || !q->out_expert || !q->out_weight || E <= 0 || E % groups || top <= 0 || top > E || keep < 1 || keep > groups ||
      q->logits_stride < E || (size_t)(2 * E + groups) * 16 > 60000 ||
      (q->score_kind != PEGAINFER_SCORE_SIGMOID && q->score_kind != PEGAINFER_SCORE_SOFTMAX) ||
      (q->group_kind != PEGAINFER_GROUP_TOP2_SUM && q->group_kind != PEGAINFER_GROUP_MAX))
    return bad;
  const int64_t pairs = (int64_t)q->rows * top;
  const bool sorted = q->sort_experts > 0;
  if (sorted && (!tile_rows_ok(q->rows_per_tile) || q->sort_experts > 7000 || pairs > 0x7FFFFFFF || !q->pos_pair ||
                 !q->pos_row || !q->tile_group || !q->tile_row0 || !q->tile_rows || !q->n_tiles ||
                 q->max_tiles < std::min<int64_t>(pairs, (pairs + q->rows_per_tile - 1) / q->rows_per_tile + q->sort_experts)))
    return bad;
  const RouteForm f{E, groups, keep, top, q->score_kind, q->group_kind, q->renorm, q->factor, q->logits_stride};
  const SortOut o{q->pos_pair, q->pos_row, q->tile_group, q->tile_row0, q->tile_rows, q->n_tiles, q->max_tiles, q->rows_per_tile};
  const size_t smem = (size_t)4 * (2 * E + groups) * sizeof(float), sort_smem = (size_t)2 * std::max(0, q->sort_experts) * sizeof(int);
  if (!by_dtype(q->dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        const A* corr = static_cast<const A*>(q->correction);
        // the sort's tables take the selection's place in LDS, the choices lie behind both
        const size_t rows_smem = (size_t)q->rows * (2 * E + groups) * sizeof(float), plan_smem = rows_smem + (size_t)pairs * sizeof(int);
        if (sorted && q->rows <= kPlanRows && sort_smem <= rows_smem && plan_smem <= 60000) {
          route_plan_kernel<A><<<1, kSortThreads, plan_smem, as_stream(stream)>>>(q->logits, corr, q->out_expert, q->out_weight, q->rows, f,
                                                                                  q->sort_experts, o);
          return;
        }
        route_from_logits_kernel<A><<<ceil_div(q->rows, 4), 256, smem, as_stream(stream)>>>(q->logits, corr, q->out_expert, q->out_weight,
                                                                                            q->rows, f);
        if (sorted)
          route_sort_kernel<<<1, kSortThreads, sort_smem, as_stream(stream)>>>(q->out_expert, (int)pairs, top, q->sort_experts, o);
      }))
    return bad;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_route_from_logits_ex(const float* logits, int64_t logits_stride, const void* correction,
                                                  int32_t* out_expert, float* out_weight, int32_t experts, int32_t n_groups,
                                                  int32_t keep_groups, int32_t top, int32_t rows, int32_t score_kind,
                                                  int32_t group_kind, int32_t renorm, int32_t dtype, pegainfer_stream_t stream) {
  pegainfer_route_plan_desc q{};
  q.logits = logits; q.logits_stride = logits_stride; q.correction = correction; q.out_expert = out_expert; q.out_weight = out_weight;
  q.experts = experts; q.n_groups = n_groups; q.keep_groups = keep_groups; q.top = top; q.rows = rows; q.score_kind = score_kind;
  q.group_kind = group_kind; q.renorm = renorm; q.factor = 1.0f; q.dtype = dtype;
  return pegainfer_route_plan(&q, stream);
}

pegainfer_status_t pegainfer_route_from_logits(const float* logits, const void* correction, int32_t* out_expert, float* out_weight,
                                               int32_t experts, int32_t n_groups, int32_t keep_groups, int32_t top, int32_t rows,
                                               int32_t score_kind, int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_route_from_logits_ex(logits, experts, correction, out_expert, out_weight, experts, n_groups, keep_groups, top, rows,
                                        score_kind, PEGAINFER_GROUP_TOP2_SUM, 0, dtype, stream);
}

pegainfer_status_t pegainfer_route_sigmoid_grouped(const void* h, const void* w_router, const void* correction,
                                                   int32_t* out_expert, float* out_weight, int32_t d, int32_t experts,
                                                   int32_t n_groups, int32_t keep_groups, int32_t top, int32_t rows,
                                                   int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_route_topk(h, w_router, correction, out_expert, out_weight, d, experts, n_groups, keep_groups, top, rows,
                              PEGAINFER_SCORE_SIGMOID, dtype, stream);
}

pegainfer_status_t pegainfer_route_sort(const int32_t* expert, int32_t n_pairs, int32_t top, int32_t experts,
                                        int32_t* pos_pair, int32_t* pos_row, int32_t* tile_group, int32_t* tile_row0,
                                        int32_t* tile_rows, int32_t* n_tiles, int32_t max_tiles, int32_t rows_per_tile,
                                        pegainfer_stream_t stream) {
  if (n_pairs <= 0) return 0;
  if (!tile_rows_ok(rows_per_tile) || experts <= 0 || experts > 7000 ||
      max_tiles < (n_pairs + rows_per_tile - 1) / rows_per_tile + experts)
    return (pegainfer_status_t)hipErrorInvalidValue;
  const SortOut o{pos_pair, pos_row, tile_group, tile_row0, tile_rows, n_tiles, max_tiles, rows_per_tile};
  route_sort_kernel<<<1, kSortThreads, (size_t)2 * experts * sizeof(int), as_stream(stream)>>>(expert, n_pairs, top, experts, o);
  return (pegainfer_status_t)hipGetLastError();
}

static pegainfer_status_t combine_launch(const float* y_pairs, const float* weight, const int32_t* expert, int32_t same_from, const void* same,
                                         int64_t same_stride, const void* add, const float* add_pairs, int32_t n_add, const float* add_gate,
                                         int64_t add_gate_stride, void* out, int32_t d, int32_t top, int32_t rows, int32_t dtype,
                                         pegainfer_stream_t stream) {
  if (rows <= 0) return 0;
  if (same && !expert) return (pegainfer_status_t)hipErrorInvalidValue;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        auto go = [&](auto kern, int per_row) {
          kern<<<dim3(rows, per_row), 256, 0, as_stream(stream)>>>(y_pairs, weight, static_cast<const A*>(add), static_cast<A*>(out), d, top,
                                                                   add_gate, add_gate_stride, expert, same_from,
                                                                   static_cast<const A*>(same), same_stride, add_pairs, n_add);
        };
        // many rows: four columns per thread where rows and pointers allow it; few rows (decoding) are cut over as many threads as there
        // are columns
        const bool vec = d % 4 == 0 && (!same || same_stride % 4 == 0) && host_aligned16(y_pairs) && host_aligned16(add) &&
                         host_aligned16(same) && host_aligned16(add_pairs) && host_aligned16(out);
        if (vec && rows >= 256) go(route_combine_kernel<A, 4>, std::min(16, ceil_div(d, 1024)));
        else go(route_combine_kernel<A, 1>, rows >= 256 ? 1 : std::min(16, ceil_div(d, 256)));
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_route_combine_gated(const float* y_pairs, const float* weight, const void* add,
                                                 const float* add_gate, int64_t add_gate_stride, void* out, int32_t d,
                                                 int32_t top, int32_t rows, int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_route_combine_same(y_pairs, weight, nullptr, 0, nullptr, 0, add, add_gate, add_gate_stride, out, d, top, rows, dtype, stream);
}

pegainfer_status_t pegainfer_route_combine_same(const float* y_pairs, const float* weight, const int32_t* expert, int32_t same_from,
                                                const void* same, int64_t same_stride, const void* add, const float* add_gate,
                                                int64_t add_gate_stride, void* out, int32_t d, int32_t top, int32_t rows, int32_t dtype,
                                                pegainfer_stream_t stream) {
  return combine_launch(y_pairs, weight, expert, same_from, same, same_stride, add, nullptr, 0, add_gate, add_gate_stride, out, d, top, rows, dtype,
                        stream);
}

pegainfer_status_t pegainfer_route_combine_pairs(const float* y_pairs, const float* weight, const float* add_pairs, int32_t n_add,
                                                 const float* add_gate, int64_t add_gate_stride, void* out, int32_t d, int32_t top,
                                                 int32_t rows, int32_t dtype, pegainfer_stream_t stream) {
  if (n_add < 0 || (n_add > 0 && !add_pairs)) return (pegainfer_status_t)hipErrorInvalidValue;
  return combine_launch(y_pairs, weight, nullptr, 0, nullptr, 0, nullptr, add_pairs, n_add, add_gate, add_gate_stride, out, d, top, rows, dtype,
                        stream);
}
pegainfer_status_t pegainfer_route_combine_add(const float* y_pairs, const float* weight, const void* add, void* out, int32_t d,
                                               int32_t top, int32_t rows, int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_route_combine_gated(y_pairs, weight, add, nullptr, 0, out, d, top, rows, dtype, stream);
}

pegainfer_status_t pegainfer_route_combine(const float* y_pairs, const float* weight, void* out, int32_t d, int32_t top,
                                           int32_t rows, int32_t dtype, pegainfer_stream_t stream) {
  return pegainfer_route_combine_add(y_pairs, weight, nullptr, out, d, top, rows, dtype, stream);
}

}  // extern "C"
