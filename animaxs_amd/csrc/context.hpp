// Execution context and device workspace (MetalContext + BufferPool analog,
// AnimaXS/Runtime/Metal/MetalContext.swift:14-104).
#pragma once

#include <vector>

#include "common.hpp"

struct anima_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
};

namespace anima {

// RAII guard making the context's device current for the duration of a call.
struct DeviceGuard {
  int prev = -1;
  explicit DeviceGuard(const anima_ctx* ctx) {
    ANIMA_HIP(hipGetDevice(&prev));
    if (prev != ctx->device) ANIMA_HIP(hipSetDevice(ctx->device));
  }
  ~DeviceGuard() {
    int cur = -1;
    if (hipGetDevice(&cur) == hipSuccess && cur != prev && prev >= 0) (void)hipSetDevice(prev);
  }
};

// A device scratch buffer that grows on demand and is freed on destruction
// (the reference's BufferPool grows and never frees, MetalContext.swift:86-104).
// Growing synchronises the stream first so in-flight kernels never see the old
// allocation freed under them; an allocation that a captured call was given stays until
// destruction, since the graph writes to it on every replay (each is more than 1/8 larger than
// the one before, so all of them together are less than ten times the last).
class Workspace {
 public:
  Workspace() = default;
  Workspace(const Workspace&) = delete;
  Workspace& operator=(const Workspace&) = delete;
  ~Workspace() { release(); }

  void* get(int64_t bytes, hipStream_t stream) {
    if (bytes > capacity_) grow(bytes, stream);
    if (!captured_) captured_ = capturing(stream);
    return ptr_;
  }
  // Whether get(bytes, stream) can serve: nothing can be allocated while the stream is captured.
  bool available(int64_t bytes, hipStream_t stream) const { return bytes <= capacity_ || !capturing(stream); }
  int64_t capacity() const { return capacity_ + retired_bytes_; }

 private:
  void grow(int64_t bytes, hipStream_t stream) {
    if (ptr_ && !captured_) {
      ANIMA_HIP(hipStreamSynchronize(stream));
      free_current();
    }
    retired_.reserve(retired_.size() + 1);
    int64_t cap = bytes + (bytes >> 3);
    cap = (cap + 4095) & ~int64_t(4095);
    void* p = nullptr;
    ANIMA_HIP(hipMalloc(&p, static_cast<size_t>(cap)));
    if (ptr_) {
      retired_.push_back(ptr_);
      retired_bytes_ += capacity_;
    }
    ptr_ = p;
    capacity_ = cap;
    captured_ = false;
  }
  static bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
    (void)hipGetLastError();   // the null stream while another one is captured
    return true;
  }
  void free_current() {
    if (ptr_) (void)hipFree(ptr_);
    ptr_ = nullptr;
    capacity_ = 0;
  }
  void release() {
    free_current();
    for (void* p : retired_) (void)hipFree(p);
    retired_.clear();
    retired_bytes_ = 0;
  }
  void* ptr_ = nullptr;
  int64_t capacity_ = 0;        // of ptr_
  bool captured_ = false;       // a captured call was given ptr_
  std::vector<void*> retired_;
  int64_t retired_bytes_ = 0;
};

}  // namespace anima
