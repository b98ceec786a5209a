// devbuf.hpp -- device buffers and row lists owned by the operators.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace fmmh {

void hip_check(hipError_t e, const char *what);

template <typename T>
struct DevBuf {
  T *ptr = nullptr;
  size_t count = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  DevBuf(DevBuf &&o) noexcept : ptr(o.ptr), count(o.count) {
    o.ptr = nullptr;
    o.count = 0;
  }
  DevBuf &operator=(DevBuf &&o) noexcept {
    if (this != &o) {
      release();
      ptr = o.ptr;
      count = o.count;
      o.ptr = nullptr;
      o.count = 0;
    }
    return *this;
  }
  ~DevBuf() { release(); }
  void release() {
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    count = 0;
  }
  void alloc(size_t n) {
    release();
    count = n;
    if (n) hip_check(hipMalloc(&ptr, n * sizeof(T)), "hipMalloc");
  }
  void upload(const std::vector<T> &v) {
    alloc(v.size());
    if (!v.empty()) hip_check(hipMemcpy(ptr, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice), "upload");
  }
  size_t bytes() const { return count * sizeof(T); }
};

// A row list for the leaf kernels: rows with an output (box or leaf) and CSR entries.
struct Rows {
  uint32_t rows = 0;
  DevBuf<uint32_t> row_id, row_cell, row_off, row_ent;
};

}  // namespace fmmh
