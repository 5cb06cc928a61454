// What a step exchanges with the host: its packed metadata block on the way in, its greedy tokens on the way out.  Both sides of the block are
// kept here, the host's in pinned memory; tokens are stored to pinned memory by the kernel that finds them, so they are there when the step
// is waited for.  A captured step begins with a kernel that fetches the block from the host's side (its length lies before it): the copy
// commands around a replay, one each way, cost more than the fetch - 40 launches of 5 us with 4 KB in and 32 bytes out 252 -> 236 us.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "pegainfer_kernels_blocks.h"

namespace pst {

class StepIo {
 public:
  StepIo() = default;
  StepIo(const StepIo&) = delete;
  StepIo& operator=(const StepIo&) = delete;
  ~StepIo() { drop(); }     // after the stream that reads it has been waited for

  int32_t* host() const { return block_ + kHeader; }
  const int32_t* dev() const { return dev_; }
  int32_t* tokens() const { return tokens_; }
  size_t words() const { return words_; }
  // room for so many words; what was recorded over the old block is void.  Nothing may be in flight.
  hipError_t grow(size_t words) {
    size_t c = PEGAINFER_FETCH_WORDS;
    while (c < words) c *= 2;
    if (block_) (void)hipHostFree(block_);
    if (dev_) (void)hipFree(dev_);
    block_ = dev_ = nullptr;
    words_ = 0;
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&block_), (c + kHeader) * 4, hipHostMallocCoherent);
    if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&dev_), c * 4);
    if (e == hipSuccess) words_ = c;
    return e;
  }
  hipError_t grow_tokens(size_t n) {
    if (tokens_) (void)hipHostFree(tokens_);
    tokens_ = nullptr;
    return hipHostMalloc(reinterpret_cast<void**>(&tokens_), n * 4, hipHostMallocCoherent);
  }
  // the first `words` of the block are the step's: copied now, or fetched by a captured step's own first launch
  hipError_t send(size_t words, bool captured, hipStream_t stream) {
    block_[0] = (int32_t)words;
    return captured ? hipSuccess : hipMemcpyAsync(dev_, host(), words * 4, hipMemcpyHostToDevice, stream);
  }
  pegainfer_status_t fetch(pegainfer_stream_t stream) const { return pegainfer_fetch_words(dev_, host(), block_, stream); }
  void drop() {
    if (block_) (void)hipHostFree(block_);
    if (tokens_) (void)hipHostFree(tokens_);
    if (dev_) (void)hipFree(dev_);
    block_ = dev_ = tokens_ = nullptr;
    words_ = 0;
  }

 private:
  static constexpr size_t kHeader = 4;     // the length, and 16-byte alignment of what follows
  int32_t *block_ = nullptr, *dev_ = nullptr, *tokens_ = nullptr;
  size_t words_ = 0;
};

}  // namespace pst
