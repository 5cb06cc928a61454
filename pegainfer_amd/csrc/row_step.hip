// Decode steps, in which every entry brings one row: what lies between two matrix products, a workgroup per row.
//   row_scalar_step_kernel  residual sum with a constant factor (+ bias, + extra rows, + one extra vector), RMS norm with one number as its gain,
//                           the input convolution of the sublayer that follows (four taps, tail moved on)
//   row_group_step_kernel   RMS norm in groups of a sublayer's output, residual sum, weighted sum over earlier streams, the same convolution
// The sublayer's output may be the weighted sum of routed experts, made on the way.  A step's first row comes from the embedding table itself (in a
// launch of its own: 3.7 us a step of 264), and the last is normed for the output table without a convolution.
// Bound by latency and launches: a thread holds four neighbouring channels (NV times), everything that the row needs - output, stream, earlier
// streams, weights, the convolution's tail - is requested before the first sum and stays in registers, so a row costs one memory latency, one or
// two block sums and one round of stores.  8 rows of 1024: routed sum, residual with norm and convolution took 4.2 + 4.4 + 4.5 us in three launches,
// here 5.2; without a routed sum 4.4 + 4.5, here 3.5.  One row of 2560 with earlier streams: 4.5 + 5.8 + 4.5, here 6.8; without a routed
// sum 4.6 + 4.5, here 4.8.
#include <algorithm>
#include <type_traits>

#include "route_core.h"

namespace pk {

constexpr int kStepTaps = 4;
constexpr int kStepGroups = 64;

template <typename A>
struct RowStep {
  const float* x_in; const int32_t* row_index; float* x_out;
  const A* embed; const uint32_t* ids;                       // in place of x_in: a row is its token's embedding row
  const A* y; const A* bias; float mult;
  const float *pairs, *weight; int top;                      // routed: in place of y
  const A* add; const float* add_pairs; int n_add; const float* add_gate; int64_t add_gate_stride;
  const float* add_rows; const A* add_vec;
  const A* gain; int groups; float eps; float* n_out; A* xb_out;
  const float* stack; int64_t stack_stride; const A* coef; int n_mix; float* mix_out;
  const A* conv_w; float* conv_state; int64_t slot_stride; const int32_t* slot; A* conv_out;
  int d, rows;
};

// a thread's chunks of four channels, the first at 4 tid, the next 4 N further
template <int N, int NV, typename F>
__device__ __forceinline__ void each_chunk(int d, F&& f) {
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int i = (threadIdx.x + N * k) * 4;
    if (i < d) f(k, i);
  }
}

// four taps on a row: the tail and the weights are asked for early, the sum runs oldest first
template <typename A, int N, int NV>
struct StepConv {
  float t[kStepTaps - 1][NV][4], w[NV][4 * kStepTaps];
  float* tail;
  __device__ __forceinline__ void request(const RowStep<A>& p, int row) {
    tail = p.conv_state + (int64_t)p.slot[row] * p.slot_stride;
    each_chunk<N, NV>(p.d, [&](int k, int i) {
#pragma unroll
      for (int j = 0; j < kStepTaps - 1; ++j) ld4(tail + (int64_t)j * p.d + i, t[j][k]);
#pragma unroll
      for (int q = 0; q < kStepTaps; ++q) ld4(p.conv_w + (int64_t)i * kStepTaps + 4 * q, w[k] + 4 * q);
    });
  }
  // seen(i, o): the four values of a chunk as they are left
  template <typename F>
  __device__ __forceinline__ void finish(const RowStep<A>& p, int row, const float (&cur)[NV][4], F&& seen) const {
    each_chunk<N, NV>(p.d, [&](int k, int i) {
      float o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < kStepTaps - 1; ++j) acc = fmaf(w[k][u * kStepTaps + j], t[j][k][u], acc);
        o[u] = fmaf(w[k][u * kStepTaps + kStepTaps - 1], cur[k][u], acc) + cur[k][u];
      }
#pragma unroll
      for (int j = 1; j < kStepTaps - 1; ++j) st4(tail + (int64_t)(j - 1) * p.d + i, t[j][k]);
      st4(tail + (int64_t)(kStepTaps - 2) * p.d + i, cur[k]);
      st4(p.conv_out + (int64_t)row * p.d + i, o);
      seen(i, o);
    });
  }
};

// the sublayer's output of a row: as stored (with its bias), or the routed experts' weighted sum in choice order
template <typename A, int N, int NV, bool ROUTED>
__device__ __forceinline__ void step_output(const RowStep<A>& p, int row, float (&y)[NV][4]) {
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) y[k][u] = 0.f;
  if constexpr (!ROUTED) {
    if (!p.y) return;
    each_chunk<N, NV>(p.d, [&](int k, int i) { ld4(p.y + (int64_t)row * p.d + i, y[k]); });
    if (p.bias)
      each_chunk<N, NV>(p.d, [&](int k, int i) {
        float b[4];
        ld4(p.bias + i, b);
#pragma unroll
        for (int u = 0; u < 4; ++u) y[k][u] += b[u];
      });
  } else {
    if (p.add) each_chunk<N, NV>(p.d, [&](int k, int i) { ld4(p.add + (int64_t)row * p.d + i, y[k]); });
#pragma unroll 2
    for (int j = 0; j < p.n_add; ++j)
      each_chunk<N, NV>(p.d, [&](int k, int i) {
        float v[4];
        ld4(p.add_pairs + ((int64_t)j * p.rows + row) * p.d + i, v);
#pragma unroll
        for (int u = 0; u < 4; ++u) y[k][u] += v[u];
      });
    const float g = (p.add || p.n_add) && p.add_gate ? sigmoid_f(p.add_gate[(int64_t)row * p.add_gate_stride]) : 1.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
      for (int u = 0; u < 4; ++u) y[k][u] *= g;
#pragma unroll 4
    for (int c = 0; c < p.top; ++c) {
      const int64_t at = (int64_t)row * p.top + c;
      const float w = p.weight[at];
      each_chunk<N, NV>(p.d, [&](int k, int i) {
        float v[4];
        ld4(p.pairs + at * p.d + i, v);
#pragma unroll
        for (int u = 0; u < 4; ++u) y[k][u] = fmaf(w, v[u], y[k][u]);
      });
    }
  }
}

template <typename A, int N, int NV, bool ROUTED, typename T = NoTail>
__global__ __launch_bounds__(N) void row_scalar_step_kernel(RowStep<A> p, RouterTail router) {
  __shared__ float red[N / 64];
  __shared__ typename T::Shared sh;
  if (T::helps(router, p.d)) return;
  T tail;
  const int row = blockIdx.x;
  const int64_t src = (int64_t)(p.row_index ? p.row_index[row] : row) * p.d, base = (int64_t)row * p.d;
  StepConv<A, N, NV> conv;
  float r[NV][4], y[NV][4];
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) r[k][u] = 0.f;
  if (ROUTED || p.x_in) {
    each_chunk<N, NV>(p.d, [&](int k, int i) { ld4(p.x_in + src + i, r[k]); });
  } else {
    const A* e = p.embed + (int64_t)p.ids[row] * p.d;
    each_chunk<N, NV>(p.d, [&](int k, int i) { ld4(e + i, r[k]); });
  }
  if (p.conv_w) conv.request(p, row);
  step_output<A, N, NV, ROUTED>(p, row, y);
  tail.request(router, p.d);
  float ss = 0.f;
  each_chunk<N, NV>(p.d, [&](int k, int i) {
    float a[4] = {}, v[4] = {};
    if (p.add_rows) ld4(p.add_rows + base + i, a);
    if (p.add_vec) ld4(p.add_vec + i, v);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      r[k][u] = fmaf(p.mult, y[k][u], r[k][u]);
      if (p.add_rows) r[k][u] += a[u];
      if (p.add_vec) r[k][u] += v[u];
      ss = fmaf(r[k][u], r[k][u], ss);
    }
    if (p.x_out) st4(p.x_out + base + i, r[k]);
  });
  if (!p.gain) return;                             // uniform over the grid
  const float sc = ld(p.gain) / sqrtf(block_sum<N / 64>(ss, red) / (float)p.d + p.eps);
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) r[k][u] *= sc;
  if (p.n_out) each_chunk<N, NV>(p.d, [&](int k, int i) { st4(p.n_out + base + i, r[k]); });
  if (p.conv_w) conv.finish(p, row, r, [&](int i, const float* o) { tail.put(sh, i, o); });
  tail.finish(router, sh, p.d, row);
}

template <typename A, int N, int NV, bool ROUTED, typename T = NoTail>
__global__ __launch_bounds__(N) void row_group_step_kernel(RowStep<A> p, RouterTail router) {
  __shared__ typename T::Shared sh;
  if (T::helps(router, p.d)) return;
  T tail;
  __shared__ float part[N * NV], inv[kStepGroups];
  const int row = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, gs = p.d / p.groups;
  const int64_t base = (int64_t)row * p.d;
  StepConv<A, N, NV> conv;
  float r[NV][4], y[NV][4], w[NV][4], m[NV][4];
#pragma unroll
  for (int k = 0; k < NV; ++k)
#pragma unroll
    for (int u = 0; u < 4; ++u) m[k][u] = 0.f;
  each_chunk<N, NV>(p.d, [&](int k, int i) {
    ld4(p.x_in + base + i, r[k]);
    ld4(p.gain + i, w[k]);
  });
  if (p.conv_w) conv.request(p, row);
  step_output<A, N, NV, ROUTED>(p, row, y);
  tail.request(router, p.d);
  each_chunk<N, NV>(p.d, [&](int k, int i) { part[i >> 2] = fmaf(y[k][0], y[k][0], fmaf(y[k][1], y[k][1], fmaf(y[k][2], y[k][2], y[k][3] * y[k][3]))); });
#pragma unroll 4
  for (int j = 0; j < p.n_mix - 1; ++j) {
    const float c = ld(p.coef + j);
    each_chunk<N, NV>(p.d, [&](int k, int i) {
      float v[4];
      ld4(p.stack + (int64_t)j * p.stack_stride + base + i, v);
#pragma unroll
      for (int u = 0; u < 4; ++u) m[k][u] = fmaf(c, v[u], m[k][u]);
    });
  }
  __syncthreads();
  for (int g = wave; g < p.groups; g += N / 64) {
    float ss = 0.f;
    for (int i = lane; i < gs / 4; i += 64) ss += part[g * (gs / 4) + i];
    ss = wave_sum(ss);
    if (lane == 0) inv[g] = 1.0f / sqrtf(ss / (float)gs + p.eps);
  }
  __syncthreads();
  const float own = p.n_mix > 0 ? ld(p.coef + p.n_mix - 1) : 0.f;
  each_chunk<N, NV>(p.d, [&](int k, int i) {
    const float sc = inv[i / gs];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      r[k][u] += y[k][u] * sc * w[k][u];
      m[k][u] = fmaf(own, r[k][u], m[k][u]);
    }
    if (p.x_out) st4(p.x_out + base + i, r[k]);
    if (p.xb_out) st4(p.xb_out + base + i, r[k]);
    tail.put(sh, i, r[k]);
    if (p.n_mix > 0 && p.mix_out) st4(p.mix_out + base + i, m[k]);
  });
  if (p.conv_w) conv.finish(p, row, m, [](int, const float*) {});
  tail.finish(router, sh, p.d, row);
}

}  // namespace pk

extern "C" {
using namespace pk;

int32_t pegainfer_row_step_ok(int32_t d, int32_t groups, int32_t taps, int64_t state_off, int64_t slot_stride) {
  return d > 0 && d % 4 == 0 && d <= 8192 && groups >= 0 && groups <= kStepGroups && (groups == 0 || (d % groups == 0 && d / groups % 4 == 0)) &&
         taps == kStepTaps && state_off % 4 == 0 && slot_stride % 4 == 0;
}

static pegainfer_status_t row_step_launch(const pegainfer_row_step_desc* q, const pegainfer_router_tail_desc* router, const void* embed, const uint32_t* ids,
                                          pegainfer_stream_t stream) {
  constexpr pegainfer_status_t bad = (pegainfer_status_t)hipErrorInvalidValue;
  if (!q) return bad;
  if (q->rows <= 0) return 0;
  const bool routed = q->y_pairs != nullptr, grouped = q->groups > 0;
  const void* vectors[] = {q->x_in, q->x_out, q->y, q->bias, q->y_pairs, q->add, q->add_pairs, q->add_rows, q->add_vec, q->n_out, q->xb_out, q->stack,
                           q->mix_out, q->conv_w, q->conv_state, q->conv_out, grouped ? q->gain : nullptr, embed};
  for (const void* v : vectors)
    if (reinterpret_cast<uintptr_t>(v) & (q->dtype == kDtF32 ? 15u : 7u)) return bad;       // fp32 rows: on 16 bytes, below
  const void* wide[] = {q->x_in, q->x_out, q->y_pairs, q->add_pairs, q->add_rows, q->n_out, q->stack, q->mix_out, q->conv_state};
  for (const void* v : wide)
    if (!host_aligned16(v)) return bad;
  if (!pegainfer_row_step_ok(q->d, q->groups, kStepTaps, 0, q->conv_w ? q->conv_slot_stride : 0) || (!q->x_in && !embed) || (routed && (!q->weight || q->top <= 0 || q->y)) ||
      q->n_add < 0 || (q->n_add > 0 && (!q->add_pairs || q->add || !routed)) || (q->add && !routed) ||
      (q->conv_w && (!q->conv_state || !q->conv_slot || !q->conv_out || !q->gain)) ||
      (grouped && (!q->gain || (!q->y && !routed) || q->n_mix < 0 || (q->n_mix > 0 && !q->coef) || (q->n_mix > 1 && !q->stack) ||
                   (q->conv_w && q->n_mix < 1) || q->stack_stride % 4)))
    return bad;
  // what the other form alone works on, and rows picked from a matrix that other workgroups write
  if (grouped ? q->row_index || q->add_rows || q->add_vec || q->n_out : q->stack || q->coef || q->mix_out || q->xb_out) return bad;
  if (q->bias && !q->y) return bad;
  if (embed && (!ids || q->x_in || q->row_index || routed || grouped || router)) return bad;
  if (q->row_index && q->x_out == q->x_in) return bad;
  RouterTail tail{};
  if (router && (routed || (grouped ? !q->xb_out : !q->conv_w) || !router_tail(router, q->rows, q->d, q->dtype, &tail))) return bad;
  if (!by_dtype(q->dtype, [&](auto* t) {
        using A = std::remove_pointer_t<decltype(t)>;
        auto a = [](const void* p) { return static_cast<const A*>(p); };
        const RowStep<A> p{q->x_in, q->row_index, q->x_out, a(embed), ids, a(q->y), a(q->bias), q->mult, q->y_pairs, q->weight, q->top, a(q->add), q->add_pairs, q->n_add,
                           q->add_gate, q->add_gate_stride, q->add_rows, a(q->add_vec), a(q->gain), q->groups, q->eps, q->n_out,
                           static_cast<A*>(q->xb_out), q->stack, q->stack_stride, a(q->coef), q->n_mix, q->mix_out, a(q->conv_w), q->conv_state,
                           q->conv_slot_stride, q->conv_slot, static_cast<A*>(q->conv_out), q->d, q->rows};
        auto shape = [&](auto n, auto nv) {
          constexpr int N = decltype(n)::value, NV = decltype(nv)::value;
          auto launch = [&](auto kern) { kern<<<router ? tail_blocks(tail, q->d) : q->rows, N, 0, as_stream(stream)>>>(p, tail); };
          if constexpr (sizeof(A) == 2 && NV == 1) {
            if (router) {
              auto behind = [&](auto* t) {
                using T = std::remove_pointer_t<decltype(t)>;
                grouped ? launch(row_group_step_kernel<A, N, NV, false, T>) : launch(row_scalar_step_kernel<A, N, NV, false, T>);
              };
              tail.E + tail.extra <= 32 ? behind(static_cast<RouteTail<N, 2>*>(nullptr)) : behind(static_cast<RouteTail<N, 3>*>(nullptr));
              return;
            }
          }
          if (grouped) routed ? launch(row_group_step_kernel<A, N, NV, true>) : launch(row_group_step_kernel<A, N, NV, false>);
          else routed ? launch(row_scalar_step_kernel<A, N, NV, true>) : launch(row_scalar_step_kernel<A, N, NV, false>);
        };
        typedef std::integral_constant<int, 1> One;
        if (q->d <= 1024) shape(std::integral_constant<int, 256>(), One());
        else if (q->d <= 2048) shape(std::integral_constant<int, 512>(), One());
        else if (q->d <= 4096) shape(std::integral_constant<int, 1024>(), One());
        else shape(std::integral_constant<int, 1024>(), std::integral_constant<int, 2>());
      }))
    return bad;
  return (pegainfer_status_t)hipGetLastError();
}
pegainfer_status_t pegainfer_row_step(const pegainfer_row_step_desc* q, pegainfer_stream_t stream) { return row_step_launch(q, nullptr, nullptr, nullptr, stream); }
pegainfer_status_t pegainfer_row_step_routed(const pegainfer_row_step_desc* q, const pegainfer_router_tail_desc* router, pegainfer_stream_t stream) {
  return router ? row_step_launch(q, router, nullptr, nullptr, stream) : (pegainfer_status_t)hipErrorInvalidValue;
}
pegainfer_status_t pegainfer_row_step_embed(const pegainfer_row_step_desc* q, const void* embed, const uint32_t* token_ids, pegainfer_stream_t stream) {
  return embed ? row_step_launch(q, nullptr, embed, token_ids, stream) : (pegainfer_status_t)hipErrorInvalidValue;
}

}  // extern "C"
