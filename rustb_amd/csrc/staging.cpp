// Pinned staging of a call's small transfers.  A pageable copy goes through
// the runtime's own staging one at a time, each waiting for the stream (a
// call's k-points, tables, outputs and counters: 5 copies of 24 us each, of a
// 225 us call at one k-point).  A call leases one pinned buffer: uploads are
// copied into it and left to the stream, downloads land in it and are handed
// over together after the one synchronisation that ends the call or its chunk.
// Transfers that do not fit what is left of the buffer take the pageable path.
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "staging.hpp"

namespace rtb {

namespace {
std::mutex g_mu;
std::vector<void*> g_idle;  // at most one per concurrent call is ever made

void release_idle() {
  std::vector<void*> drop;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    drop.swap(g_idle);
  }
  for (void* p : drop) (void)hipHostFree(p);
}
const bool g_hook = (workspace_release_hook() = &release_idle, true);
}  // namespace

Staging::Staging(hipStream_t st) : st_(st) {
  (void)g_hook;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_idle.empty()) {
      buf_ = static_cast<char*>(g_idle.back());
      g_idle.pop_back();
      return;
    }
  }
  void* p = nullptr;
  if (hipHostMalloc(&p, kStagingBytes, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    return;  // no buffer: every transfer takes the pageable path
  }
  buf_ = static_cast<char*>(p);
}

Staging::~Staging() {
  if (!buf_) return;
  (void)hipStreamSynchronize(st_);  // an early return may leave copies in flight
  std::lock_guard<std::mutex> lock(g_mu);
  g_idle.push_back(buf_);
}

char* Staging::take(size_t bytes) {
  const size_t b = (bytes + 63) / 64 * 64;
  if (!buf_ || off_ + b > kStagingBytes) return nullptr;
  char* p = buf_ + off_;
  off_ += b;
  return p;
}

int Staging::h2d(void* dst, const void* src, size_t bytes) {
  char* p = take(bytes);
  if (p) std::memcpy(p, src, bytes);
  RTB_HIP(hipMemcpyAsync(dst, p ? p : src, bytes, hipMemcpyHostToDevice, st_));
  return RTB_OK;
}

int Staging::d2h(void* dst, const void* src, size_t bytes) {
  char* p = take(bytes);
  RTB_HIP(hipMemcpyAsync(p ? p : dst, src, bytes, hipMemcpyDeviceToHost, st_));
  if (p) out_.push_back({dst, p, bytes});
  return RTB_OK;
}

int Staging::finish() {
  RTB_HIP(hipStreamSynchronize(st_));
  for (const Out& o : out_) std::memcpy(o.dst, o.src, o.bytes);
  out_.clear();
  off_ = 0;
  return RTB_OK;
}

}  // namespace rtb
