// One decode step of the recurrences with a matrix state per head (recurrent.hip's delta rules, gated_linear.hip), every entry one row: what
// prepares the row (unit vectors, decays, second stages of low-rank projections), the state's update, the read-out and its norm and gate in one
// launch.  A workgroup of eight waves owns a whole (entry, head), so that the norm over the head's values needs no second launch; a thread
// holds four neighbouring columns of every sixteenth row of S.  With no chain over tokens to follow, all of S and every input is requested
// before the first barrier.  The delta rules take S^T k and S^T q of the decayed state in one pass:  S'^T q = S^T q + (k . q) u.
// Bound by the launch and by S through one CU (128 x 128 values, 64 KB each way).  One row, 32 heads of 128 x 128: 4.6 + 5.7 + 4.2 us for
// preparation, scan and norm, 7.2 us here; eight rows of 8 heads with decays per channel and both second stages 5.4 + 5.2 + 4.4 + 10.0 + 4.2 and
// 9.9 us; eight rows of 8 heads of gated linear attention 11.3 + 4.5 and 8.2 us.
#include "recurrent_step.h"

namespace pk {

template <typename A, typename Q, int KIND>
__global__ __launch_bounds__(kStepThreads) void recurrent_step_kernel(pegainfer_recurrent_step_desc p) {
  recurrent_step_block<A, Q, KIND>(p, blockIdx.x, blockIdx.y);
}

}  // namespace pk

extern "C" {
using namespace pk;

int32_t pegainfer_recurrent_step_up_ok(const void* w, int32_t rank, int32_t rank_stride, const void* proj, int64_t proj_stride, int64_t low_off) {
  return recurrent_step_up_ok(w, rank, rank_stride, proj, proj_stride, low_off);
}

int32_t pegainfer_recurrent_step_ok(const pegainfer_recurrent_step_desc* q) { return recurrent_step_ok(q); }

pegainfer_status_t pegainfer_recurrent_step(const pegainfer_recurrent_step_desc* q, pegainfer_stream_t stream) {
  constexpr pegainfer_status_t bad = (pegainfer_status_t)hipErrorInvalidValue;
  if (!recurrent_step_ok(q)) return bad;
  if (q->n_entries == 0) return 0;
  hipStream_t st = as_stream(stream);
  const bool known = by_dtype(q->dtype, [&](auto* t) {
    using A = std::remove_pointer_t<decltype(t)>;
    auto go = [&](auto kern) { kern<<<dim3(q->heads, q->n_entries), kStepThreads, 0, st>>>(*q); };
    if (q->kind == PEGAINFER_STEP_GATED) go(recurrent_step_kernel<A, A, PEGAINFER_STEP_GATED>);
    else if (q->kind == PEGAINFER_STEP_DELTA) go(recurrent_step_kernel<A, float, PEGAINFER_STEP_DELTA>);
    else go(recurrent_step_kernel<A, float, PEGAINFER_STEP_DELTA_CHANNEL>);
  });
  return known ? (pegainfer_status_t)hipGetLastError() : bad;
}

}  // extern "C"
