// Device scratch that a step is faster with and can do without.
#pragma once

#include <cstddef>

namespace pq {

struct OptionalScratch {
  float* p = nullptr;
  size_t cap = 0;   // floats

  // Room for `need` floats; false: there is no memory for it, and the step goes the way that needs none.
  // alloc(bytes) -> pointer or nullptr, leaving no error behind; release(pointer) once nothing uses it any more.
  template <typename Alloc, typename Release>
  bool grow(size_t need, Alloc&& alloc, Release&& release) {
    if (need <= cap) return true;
    drop(release);
    p = static_cast<float*>(alloc(need * sizeof(float)));
    if (p) cap = need;
    return p != nullptr;
  }
  template <typename Release>
  void drop(Release&& release) {
    if (p) release(p);
    p = nullptr;
    cap = 0;
  }
};

}  // namespace pq
