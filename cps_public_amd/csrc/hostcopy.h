// Copies between pageable host vectors and the device.
#pragma once
#include <cstddef>

#include "cps_hip_internal.h"

namespace cpship {

// Staged copies for one owner.  A call takes a ring of pinned buffers from a
// pool that all owners share (allocating one takes about 10 ms) and puts it
// back when its transfers have ended; the pool keeps at most two idle rings
// (64 MiB) and frees them with the last owner.  Safe from several threads.
struct HostStager {
  static constexpr int WORKERS = 8, BUFS = 2;
  static constexpr size_t CHUNK = size_t(2) << 20;
  HostStager();
  HostStager(const HostStager&) = delete;
  HostStager& operator=(const HostStager&) = delete;
  ~HostStager();
  // Order as hipMemcpyAsync on st; `host` has been read when to_device
  // returns, and written when to_host returns (which waits for st).
  hipError_t to_device(void* dev, const void* host, size_t bytes, hipStream_t st);
  hipError_t to_host(void* host, const void* dev, size_t bytes, hipStream_t st);
};

}  // namespace cpship
