// Parts of the one-launch scans: the decoupled look-back over a launch's chunks
// (Merrill and Garland, "Single-pass parallel prefix scan with decoupled
// look-back", 2016) and the pinned buffers that their totals go to the host
// through.
#pragma once

#include <mutex>

#include "sp_common.h"

namespace sp {

// Small pinned host buffers that kernels write their counts to, kept between
// calls (one per call in flight, whatever the thread or device): a copy of the
// counts from device memory costs a launch and ~4 us before the host goes on.
// At most kIdle of 256 bytes are kept; what more calls in flight needed is freed.
struct PinnedPool {
  static constexpr int kIdle = 64;
  std::mutex m;
  void* idle[kIdle];
  int n = 0;
};
inline PinnedPool& pinned_pool() {
  static PinnedPool* p = new PinnedPool;  // (outlives the threads that return buffers to it)
  return *p;
}
class PinnedCounts {
 public:
  static constexpr size_t kBytes = 256;
  int take() {
    {
      std::lock_guard<std::mutex> lock(pinned_pool().m);
      if (pinned_pool().n > 0) {
        p_ = pinned_pool().idle[--pinned_pool().n];
        return SP_OK;
      }
    }
    SP_HIP(hipHostMalloc(&p_, kBytes, hipHostMallocPortable | hipHostMallocMapped));
    return SP_OK;
  }
  ~PinnedCounts() {
    if (!p_) return;
    {
      std::lock_guard<std::mutex> lock(pinned_pool().m);
      if (pinned_pool().n < PinnedPool::kIdle) {
        pinned_pool().idle[pinned_pool().n++] = p_;
        return;
      }
    }
    (void)hipHostFree(p_);
  }
  uint64_t* data() const { return static_cast<uint64_t*>(p_); }

 private:
  void* p_ = nullptr;
};

// A chunk's state is one 64-bit word, status in the top two bits (0: nothing
// yet), so no fence orders it.  The chunk's first wave publishes its own sum
// first, then adds up the chunks before it, 64 at a time, until one knows its
// prefix.  Chunks are numbered by a counter as workgroups start, so every
// chunk waited for belongs to a running workgroup that publishes its sum
// before it waits itself.
constexpr uint64_t kScanSum = uint64_t(1) << 62, kScanPrefix = uint64_t(2) << 62;
__device__ __forceinline__ uint64_t scan_lookback(uint64_t* state, int64_t chunk, int lane) {
  uint64_t base = 0;
  for (int64_t top = chunk - 1; top >= 0; top -= 64) {
    const int64_t at = top - lane;
    uint64_t v = kScanPrefix;  // (before the first chunk: a prefix of none)
    for (;;) {
      if (at >= 0)
        v = __hip_atomic_load(&state[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (!__ballot((v >> 62) == 0)) break;
      __builtin_amdgcn_s_sleep(1);
    }
    const uint64_t known = __ballot((v >> 62) == 2);
    const int last = known ? __builtin_ctzll(known) : 63;
    uint64_t part = lane <= last ? v & (kScanSum - 1) : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
    base += part;
    if (known) break;
  }
  return base;
}

}  // namespace sp
