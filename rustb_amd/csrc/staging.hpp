// Pinned staging of a call's small transfers (staging.cpp).
#pragma once

#include "rtb_internal.hpp"

namespace rtb {

constexpr size_t kStagingBytes = size_t(2) << 20;

// One call's transfers on its stream.  Sources of h2d may be reused at once
// unless they exceed the buffer (then as hipMemcpyAsync of pageable memory);
// targets of d2h hold their values after finish(), which waits for the stream
// and empties the buffer.
class Staging {
 public:
  explicit Staging(hipStream_t st);
  ~Staging();
  Staging(const Staging&) = delete;
  Staging& operator=(const Staging&) = delete;
  int h2d(void* dst, const void* src, size_t bytes);
  int d2h(void* dst, const void* src, size_t bytes);
  int finish();

 private:
  struct Out {
    void* dst;
    const void* src;
    size_t bytes;
  };
  char* take(size_t bytes);
  hipStream_t st_ = nullptr;
  char* buf_ = nullptr;
  size_t off_ = 0;
  std::vector<Out> out_;
};

}  // namespace rtb
