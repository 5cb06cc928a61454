// The end of a capture: what was recorded becomes an executable graph.  The recording itself is let go of in every case, also where a launch of it was
// refused (recorded = false) or the capture failed.
#pragma once

#include <hip/hip_runtime.h>

namespace pst {

inline hipError_t end_capture(hipStream_t stream, bool recorded, hipGraphExec_t* exec) {
  hipGraph_t g = nullptr;
  *exec = nullptr;
  hipError_t e = hipStreamEndCapture(stream, &g);
  if (e == hipSuccess && recorded) e = hipGraphInstantiate(exec, g, nullptr, nullptr, 0);
  if (e != hipSuccess) *exec = nullptr;
  if (g) (void)hipGraphDestroy(g);
  return e;
}

}  // namespace pst
