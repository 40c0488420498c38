// Copies between pageable host vectors and the device.
#pragma once
#include <cstddef>

#include "cps_hip_internal.h"

namespace cpship {

// Ring of pinned buffers that large copies are staged through, allocated at
// the first one and given back with its owner.  Not for concurrent use.
struct HostStager {
  static constexpr int WORKERS = 8, BUFS = 2;
  static constexpr size_t CHUNK = size_t(2) << 20;
  char* pinned = nullptr;   // WORKERS * BUFS chunks
  hipEvent_t done[WORKERS * BUFS] = {};
  HostStager() = default;
  HostStager(const HostStager&) = delete;
  HostStager& operator=(const HostStager&) = delete;
  ~HostStager();
  // Order as hipMemcpyAsync on st; `host` has been read when to_device
  // returns, and written when to_host returns (which waits for st).
  hipError_t to_device(void* dev, const void* host, size_t bytes, hipStream_t st);
  hipError_t to_host(void* host, const void* dev, size_t bytes, hipStream_t st);

 private:
  bool ready();
  hipError_t run(char* dev, char* host, size_t bytes, hipStream_t st, bool up);
};

}  // namespace cpship
