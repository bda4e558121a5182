// Ids handed over in pageable host memory (csrc/core/preprocess.cu:98-99 of the reference copies them with one
// cudaMemcpyAsync): the copy to the device, through a pinned staging buffer filled by several threads, with the
// transfers of the pieces that are ready issued behind them.  The runtime's own path for pageable memory stages with one
// thread; at 13.6 MB of ids per batch that copy is as long as the rest of the training step.
#pragma once
#include "common.h"

namespace hctr {

class HostStager {
 public:
  HostStager() = default;
  ~HostStager();
  HostStager(const HostStager &) = delete;
  HostStager &operator=(const HostStager &) = delete;

  // Enqueues on `s` the transfer of `bytes` bytes at pageable `src` to device memory `dst` and returns once `src` has
  // been read (the caller may reuse it).  The staging buffer is reused by the next call on this object, which first
  // waits for the transfers enqueued here.
  // narrow_ids: `src` holds 64-bit ids and `dst` receives bytes / 2 bytes of 32-bit ones, half the bytes on the bus;
  // an id that does not fit (a negative one too) arrives as 0xffffffff.  What is narrowed is looked at on the way:
  // largest() says afterwards how large an id arrived.
  void copy(void *dst, const void *src, size_t bytes, hipStream_t s, bool narrow_ids = false);

  // The same without the transfer, for kLendUpTo bytes at most: returns the staging buffer, filled, at the address a kernel
  // launched on `s` reads it through the bus.  The caller waits for that kernel before the next call on this object (preprocess
  // does: for the whole index of the batch before).
  // A training step whose ids arrive this way against one with the transfer (rows of 64 floats, MI355X): 53 k ids 73 us
  // instead of 110, 213 k 129 (168), 262 k -- the most that are lent -- 146 (184), all while preprocess still waited for the kernel
  // that reads the ids.  Since it returns when they are staged, two steps lent and transferred: 426 k ids 340 and 378 us, 852 k
  // 564 and 554, 1.7 M 1016 and 955, of 128 floats 1425 and 1335.  The line could be half a million ids.
  static constexpr size_t kLendUpTo = 2 << 20;
  const void *lend(const void *src, size_t bytes, hipStream_t s, bool narrow_ids);
  uint32_t largest() const { return largest_; } // of the ids the last call narrowed, as 32-bit ones

 private:
  uint32_t largest_ = 0;
  void reserve(size_t bytes, hipStream_t reader);
  unsigned char *pinned_ = nullptr;
  size_t cap_ = 0;
  hipEvent_t sent_ = nullptr; // behind the last transfer out of the staging buffer
};

// threads that fill staging buffers, the calling one included; HETUCTR_COPY_THREADS (1..64), default 8
int host_copy_threads();

} // namespace hctr
