// Selective state-space scan with one decay per head and token over ragged batches, fp32 state and fp32 arithmetic throughout:
//     a = exp(-exp(A_log) dt);  S <- a S + dt B x^T;  y = S^T C + D x          (dt = softplus(raw + bias))
// Two equivalent forms.  The scan is a serial chain of 0.18 us a token whatever the size; 1024 tokens of 32 heads of 128 states x 64 values
// take 180 us there and 65 us in chunks (sums 15, walk 10, outputs 37: the fp32 matrix-core products and the states' way through memory),
// 4096 tokens 703 and 208 us.
//   ssd_scan_kernel           token by token, the layout of recurrent.hip: decoding and short portions
//   scalar_chunks.h           long portions, in chunks of <= 64 tokens that run side by side, with B as keys, C as queries, x as values
#include "common.h"
#include "typed.h"
#include "ssd_core.h"
#include "scalar_chunks.h"
#include "pegainfer_kernels_blocks.h"

namespace pk {

template <int NS, typename A>
__global__ __launch_bounds__(256) void ssd_scan_kernel(const float* __restrict__ xbc, int64_t xbc_stride, const A* __restrict__ proj,
                                                       int64_t proj_stride, int64_t dt_off, const A* __restrict__ A_log,
                                                       const A* __restrict__ dt_bias, const A* __restrict__ Dskip,
                                                       float* __restrict__ state, int64_t slot_stride, float* __restrict__ o, int H,
                                                       int G, int dim, int vdim, const int32_t* __restrict__ entry_row0,
                                                       const int32_t* __restrict__ entry_slot, int scan_max) {
  ssd_scan_block<NS, A>(blockIdx.x, blockIdx.y, blockIdx.z, xbc, xbc_stride, proj, proj_stride, dt_off, A_log, dt_bias, Dskip, state, slot_stride, o, H, G, dim, vdim, entry_row0, entry_slot, scan_max);
}

template <typename A>
struct SsdIn {
  const float* xbc; int64_t xbc_stride;
  const A* proj; int64_t proj_stride, dt_off;
  const A *A_log, *dt_bias, *D;
  int H, G, dim, vdim;
  typedef float Row;
  static constexpr bool kNorm = false;
  __device__ __forceinline__ const float* rows() const { return xbc; }
  __device__ __forceinline__ int64_t row_stride() const { return xbc_stride; }
  __device__ __forceinline__ float q_factor() const { return 1.0f; }
  __device__ __forceinline__ int64_t v_at(int h) const { return (int64_t)h * vdim; }
  __device__ __forceinline__ int64_t k_at(int h) const { return (int64_t)H * vdim + (int64_t)(h / (H / G)) * dim; }
  __device__ __forceinline__ int64_t q_at(int h) const { return k_at(h) + (int64_t)G * dim; }
  __device__ __forceinline__ void steps(int, int h, int row0, int n, int lane, float* dt, float* a) const {
    *dt = lane < n ? ssd_step(ld(proj + (int64_t)(row0 + lane) * proj_stride + dt_off + h), ld(dt_bias + h)) : 0.f;
    *a = lane < n ? expf(-expf(ld(A_log + h)) * *dt) : 1.f;
  }
  __device__ __forceinline__ float floor_of(int, int, int) const { return 0.f; }
  __device__ __forceinline__ float skip(int h) const { return ld(D + h); }
};
}  // namespace pk

extern "C" {
using namespace pk;

int64_t pegainfer_ssd_scan_workspace(int32_t n_chunks, int32_t heads, int32_t n_state, int32_t vdim) {
  return scalar_chunk_floats(n_chunks, heads, n_state, vdim, false);
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
    scalar_chunk_launch(in, q->workspace, q->state, q->slot_stride, q->o, q->chunk_row0, q->chunk_rows, q->n_chunks, q->long_chunk0, q->long_slot,
                        q->n_long, st);
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
