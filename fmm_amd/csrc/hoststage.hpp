// hoststage.hpp -- downloads into a caller's pageable memory through pinned staging.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

namespace fmmh {

struct HostCopy {
  void *dst;        // host
  const void *src;  // device
  size_t bytes;
};

// Keeps the pinned buffers alive while an operator that may use them lives; the last user to
// go gives them back.
class HostStageUser {
 public:
  HostStageUser();
  ~HostStageUser();
  HostStageUser(const HostStageUser &) = delete;
  HostStageUser &operator=(const HostStageUser &) = delete;

  // The copies in order on stream s of device `device`, complete on return.  Safe from
  // several threads: each call takes a buffer of its own.
  void download(int device, hipStream_t s, const std::vector<HostCopy> &copies);
};

}  // namespace fmmh
