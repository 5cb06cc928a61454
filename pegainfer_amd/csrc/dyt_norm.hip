// Dynamic-Tanh normalisation over an fp32 residual stream (beside the RMSNorm family of norm.hip):
//   dyt(x) = tanh(alpha * x) * w + b        - elementwise: no mean, no variance, no reduction, so no row-wide barrier.
// Three forms, all one pass over the row, fp32 arithmetic, storage type of the activations / weights a template parameter:
//   embed_f32          token rows of the embedding table widened into the fp32 stream
//   dyt_norm           out = dyt(x)
//   dyt_add_norm       x += dyt_post(y); out = dyt_next(x)   (post-norm + residual sum + the next sublayer's pre-norm:
//                      the sublayer boundary costs one launch and one read of y, one read-modify-write of x)
//   dyt_step           all of these around one row: the stream read in place, through a row index or as an embedding row; a stored output or the
//                      routed experts' weighted sum joins it; the next pre-norm
// Memory-bound: 4 B read + 2-4 B written per element.
#include "route_core.h"

namespace pk {

template <typename A>
__global__ __launch_bounds__(256) void embed_f32_kernel(const A* __restrict__ embed, const uint32_t* __restrict__ ids,
                                                        float* __restrict__ out, int width) {
  const A* src = embed + (size_t)ids[blockIdx.x] * width;
  float* dst = out + (size_t)blockIdx.x * width;
  for (int i = threadIdx.x; i < width; i += 256) dst[i] = ld(src + i);
}

// (beside the stream itself, both halves of the rows that a projection of [stream | embedding] reads: one launch for three)
template <typename A>
__global__ __launch_bounds__(256) void embed_f32_pair_kernel(const A* __restrict__ embed, const uint32_t* __restrict__ ids,
                                                             float* __restrict__ out, float* __restrict__ pair, int width) {
  const int i = blockIdx.y * 256 + threadIdx.x;
  if (i >= width) return;
  const float v = ld(embed + (size_t)ids[blockIdx.x] * width + i);
  if (out) out[(size_t)blockIdx.x * width + i] = v;
  pair[(size_t)blockIdx.x * 2 * width + i] = v;
  pair[(size_t)blockIdx.x * 2 * width + width + i] = v;
}

template <typename A>
__global__ __launch_bounds__(256) void dyt_norm_kernel(const float* __restrict__ x, const A* __restrict__ alpha,
                                                       const A* __restrict__ w, const A* __restrict__ b,
                                                       A* __restrict__ out, int d, long n) {
  const float a = ld(alpha);
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
    const int c = (int)(i % d);
    st(out + i, tanhf(a * x[i]) * ld(w + c) + ld(b + c));
  }
}

template <typename A, bool NEXT>
__global__ __launch_bounds__(256) void dyt_add_norm_kernel(float* __restrict__ x, const A* __restrict__ y,
                                                           const A* __restrict__ pa, const A* __restrict__ pw,
                                                           const A* __restrict__ pb, const A* __restrict__ na,
                                                           const A* __restrict__ nw, const A* __restrict__ nb,
                                                           A* __restrict__ out, int d, long n) {
  const float a = ld(pa);
  const float a2 = NEXT ? ld(na) : 0.f;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
    const int c = (int)(i % d);
    const float v = x[i] + (tanhf(a * ld(y + i)) * ld(pw + c) + ld(pb + c));
    x[i] = v;
    if (NEXT) st(out + i, tanhf(a2 * v) * ld(nw + c) + ld(nb + c));
  }
}

// Four neighbouring values per thread, a workgroup per row and 1024 of its channels.  Memory-bound with many rows: 2404 rows of 2048, output, sum and
// next norm 23.5 -> 17.7 us (one value per thread and a division per value before), with a routed sum of four 24.6 (30 + 25); launch-bound
// with few: 4 rows with the routed sum 4.6 us (4.6 + 4.5).
template <typename A>
struct DytStep {
  float* x; const A* embed; const uint32_t* ids; const int32_t* row_index;
  const A* y; const float *pairs, *weight; int top;
  const A *pa, *pw, *pb, *na, *nw, *nb;
  A* out;
  int d;
};
// T: the router of the feed-forward behind the row, which then lies in one workgroup
template <typename A, int N = 256, typename T = NoTail>
__global__ __launch_bounds__(N) void dyt_step_kernel(DytStep<A> p, RouterTail router) {
  __shared__ typename T::Shared sh;
  if (T::helps(router, p.d)) return;
  T tail;
  const int row = blockIdx.x, i = (blockIdx.y * N + threadIdx.x) * 4;
  const int64_t at = (int64_t)row * p.d + i;
  const bool on = i < p.d, joins = p.y || p.pairs;
  float v[4], pw[4], pb[4], nw[4], nb[4], y[4] = {0.f, 0.f, 0.f, 0.f};
  if (on) {
    if (p.embed) ld4(p.embed + (int64_t)p.ids[row] * p.d + i, v);
    else ld4(p.x + (p.row_index ? (int64_t)p.row_index[row] * p.d + i : at), v);
    if (joins) { ld4(p.pw + i, pw); ld4(p.pb + i, pb); }
    if (p.nw) { ld4(p.nw + i, nw); ld4(p.nb + i, nb); }
    if (p.y) ld4(p.y + at, y);
  }
  tail.request(router, p.d);
  if (on) {
    if (joins) {
      if (!p.y) {
#pragma unroll 4
        for (int c = 0; c < p.top; ++c) {
          const float w = p.weight[(int64_t)row * p.top + c];
          float t[4];
          ld4(p.pairs + ((int64_t)row * p.top + c) * p.d + i, t);
#pragma unroll
          for (int u = 0; u < 4; ++u) y[u] = fmaf(w, t[u], y[u]);
        }
        if constexpr (sizeof(A) == 2) {      // as a stored sum: a router behind it sees the same rows whichever launch made the sum
#pragma unroll
          for (int u = 0; u < 4; ++u) y[u] = bf16_round_f(y[u]);
        }
      }
      const float a = ld(p.pa);
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] += tanhf(a * y[u]) * pw[u] + pb[u];
    }
    if (!p.row_index && (joins || p.embed)) st4(p.x + at, v);
    if (p.nw) {
      const float a = ld(p.na);
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = tanhf(a * v[u]) * nw[u] + nb[u];
      st4(p.out + at, v);
      tail.put(sh, i, v);
    }
  }
  tail.finish(router, sh, p.d, row);
}

__global__ __launch_bounds__(256) void gather_rows_f32_kernel(const float* __restrict__ x, const int32_t* __restrict__ idx,
                                                              float* __restrict__ out, int d) {
  const float* src = x + (size_t)idx[blockIdx.x] * d;
  float* dst = out + (size_t)blockIdx.x * d;
  for (int i = threadIdx.x; i < d; i += 256) dst[i] = src[i];
}

// eight values per thread where the pointers allow it: 2404 rows of 8192 in place 20.1 -> 13.7 us
template <typename A, int V>
__global__ __launch_bounds__(256) void relu_sq_kernel(const A* x, A* out, long n) {
  for (long i = ((long)blockIdx.x * 256 + threadIdx.x) * V; i < n; i += (long)gridDim.x * 256 * V) {
    if (V == 8 && i + V <= n) {
      float v[8];
      Vec8<A>::load(x + i, v);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        v[u] = fmaxf(v[u], 0.f);
        v[u] *= v[u];
      }
      Vec8<A>::store(out + i, v);
      continue;
    }
    for (long k = i; k < std::min<long>(i + V, n); ++k) {
      const float v = fmaxf(ld(x + k), 0.f);
      st(out + k, v * v);
    }
  }
}

static inline int grid_for(long n) { return (int)std::min<long>((n + 255) / 256, 8192); }

}  // namespace pk

extern "C" {
using namespace pk;

pegainfer_status_t pegainfer_embed_f32(const void* embed, const uint32_t* token_ids, float* out, int32_t width,
                                       int32_t n_tokens, int32_t dtype, pegainfer_stream_t stream) {
  if (n_tokens <= 0) return 0;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        embed_f32_kernel<A><<<n_tokens, 256, 0, as_stream(stream)>>>(static_cast<const A*>(embed), token_ids, out, width);
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_embed_f32_pair(const void* embed, const uint32_t* token_ids, float* out, float* pair, int32_t width,
                                            int32_t n_tokens, int32_t dtype, pegainfer_stream_t stream) {
  if (n_tokens <= 0) return 0;
  if (width <= 0 || !pair || ceil_div(width, 256) > 65535) return (pegainfer_status_t)hipErrorInvalidValue;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        embed_f32_pair_kernel<A><<<dim3(n_tokens, ceil_div(width, 256)), 256, 0, as_stream(stream)>>>(static_cast<const A*>(embed), token_ids, out,
                                                                                                     pair, width);
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_dyt_norm(const float* x, const void* alpha, const void* w, const void* b, void* out,
                                      int32_t d, int32_t rows, int32_t dtype, pegainfer_stream_t stream) {
  const long n = (long)d * rows;
  if (n <= 0) return 0;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        dyt_norm_kernel<A><<<grid_for(n), 256, 0, as_stream(stream)>>>(x, static_cast<const A*>(alpha), static_cast<const A*>(w),
                                                                       static_cast<const A*>(b), static_cast<A*>(out), d, n);
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_dyt_add_norm(float* x, const void* y, const void* post_alpha, const void* post_w,
                                          const void* post_b, const void* next_alpha, const void* next_w,
                                          const void* next_b, void* out, int32_t d, int32_t rows, int32_t dtype,
                                          pegainfer_stream_t stream) {
  const long n = (long)d * rows;
  if (n <= 0) return 0;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        auto c = [](const void* p) { return static_cast<const A*>(p); };
        if (next_w)
          dyt_add_norm_kernel<A, true><<<grid_for(n), 256, 0, as_stream(stream)>>>(
              x, c(y), c(post_alpha), c(post_w), c(post_b), c(next_alpha), c(next_w), c(next_b), static_cast<A*>(out), d, n);
        else
          dyt_add_norm_kernel<A, false><<<grid_for(n), 256, 0, as_stream(stream)>>>(
              x, c(y), c(post_alpha), c(post_w), c(post_b), nullptr, nullptr, nullptr, nullptr, d, n);
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

static pegainfer_status_t dyt_step_launch(const pegainfer_dyt_step_desc* q, const pegainfer_router_tail_desc* router, pegainfer_stream_t stream) {
  constexpr pegainfer_status_t bad = (pegainfer_status_t)hipErrorInvalidValue;
  if (!q) return bad;
  if (q->rows <= 0) return 0;
  const bool joins = q->y || q->y_pairs;
  if (q->d <= 0 || q->d % 4 || (!q->x && !q->embed) || (q->embed && (!q->token_ids || q->row_index || !q->x)) || (q->row_index && joins) ||
      (q->y && q->y_pairs) || (q->y_pairs && (!q->weight || q->top <= 0)) || (joins && (!q->post_alpha || !q->post_w || !q->post_b)) ||
      (q->next_w && (!q->next_alpha || !q->next_b || !q->out)))
    return bad;
  const void* stored[] = {q->embed, q->y, q->post_w, q->post_b, q->next_w, q->next_b, q->out};
  for (const void* v : stored)
    if (reinterpret_cast<uintptr_t>(v) & (q->dtype == kDtF32 ? 15u : 7u)) return bad;
  if (!host_aligned16(q->x) || !host_aligned16(q->y_pairs)) return bad;
  RouterTail tail{};
  if (router && (!q->next_w || q->y_pairs || !router_tail(router, q->rows, q->d, q->dtype, &tail))) return bad;
  if (!by_dtype(q->dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        auto c = [](const void* p) { return static_cast<const A*>(p); };
        const DytStep<A> p{q->x, c(q->embed), q->token_ids, q->row_index, c(q->y), q->y_pairs, q->weight, q->top, c(q->post_alpha), c(q->post_w),
                           c(q->post_b), c(q->next_alpha), c(q->next_w), c(q->next_b), static_cast<A*>(q->out), q->d};
        if constexpr (sizeof(A) == 2) {
          if (router) {
            auto behind = [&](auto n) {
              constexpr int N = decltype(n)::value;
              const int blocks = tail_blocks(tail, q->d);
              if (tail.E + tail.extra <= 32) dyt_step_kernel<A, N, RouteTail<N, 2>><<<blocks, N, 0, as_stream(stream)>>>(p, tail);
              else dyt_step_kernel<A, N, RouteTail<N, 3>><<<blocks, N, 0, as_stream(stream)>>>(p, tail);
            };
            if (q->d <= 1024) behind(std::integral_constant<int, 256>());
            else if (q->d <= 2048) behind(std::integral_constant<int, 512>());
            else behind(std::integral_constant<int, 1024>());
            return;
          }
        }
        dyt_step_kernel<A><<<dim3(q->rows, ceil_div(q->d, 1024)), 256, 0, as_stream(stream)>>>(p, tail);
      }))
    return bad;
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_dyt_step(const pegainfer_dyt_step_desc* q, pegainfer_stream_t stream) { return dyt_step_launch(q, nullptr, stream); }
pegainfer_status_t pegainfer_dyt_step_routed(const pegainfer_dyt_step_desc* q, const pegainfer_router_tail_desc* router, pegainfer_stream_t stream) {
  return router ? dyt_step_launch(q, router, stream) : (pegainfer_status_t)hipErrorInvalidValue;
}

pegainfer_status_t pegainfer_gather_rows_f32(const float* x, const int32_t* rows_index, float* out, int32_t d,
                                             int32_t n_rows, pegainfer_stream_t stream) {
  if (n_rows <= 0) return 0;
  gather_rows_f32_kernel<<<n_rows, 256, 0, as_stream(stream)>>>(x, rows_index, out, d);
  return (pegainfer_status_t)hipGetLastError();
}

pegainfer_status_t pegainfer_relu_sq(const void* x, void* out, int64_t n, int32_t dtype, pegainfer_stream_t stream) {
  if (n <= 0) return 0;
  if (!by_dtype(dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        if (n >= 8 * 64 * 1024 && host_aligned16(x) && host_aligned16(out))   // (a wave for each SIMD)
          relu_sq_kernel<A, 8><<<grid_for((n + 7) / 8), 256, 0, as_stream(stream)>>>(static_cast<const A*>(x), static_cast<A*>(out), n);
        else
          relu_sq_kernel<A, 1><<<grid_for(n), 256, 0, as_stream(stream)>>>(static_cast<const A*>(x), static_cast<A*>(out), n);
      }))
    return (pegainfer_status_t)hipErrorInvalidValue;
  return (pegainfer_status_t)hipGetLastError();
}

}  // extern "C"
