// Scratch memory of a session (memory.h).
#include "memory.h"

namespace affon {

Workspace::~Workspace() {
  if (hipSetDevice(device_) != hipSuccess) return;
  if (ptr_ != nullptr) (void)hipFree(ptr_);
  for (void* p : retired_) (void)hipFree(p);
}

void* Workspace::get(size_t bytes) {
  if (bytes <= bytes_) return ptr_;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream_, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) return nullptr;
  // The old buffer stays allocated (retired) until the session ends: work
  // already enqueued, and graphs captured with its address, may still use it.
  if (ptr_ != nullptr) {
    retired_.push_back(ptr_);
    retired_bytes_ = bytes_;
  }
  ptr_ = nullptr;
  bytes_ = 0;
  // Grow at least twofold, so that retired buffers stay few.
  const size_t want = bytes > 2 * retired_bytes_ ? bytes : 2 * retired_bytes_;
  const size_t rounded = (want + (size_t(1) << 20) - 1) & ~((size_t(1) << 20) - 1);
  if (hipMalloc(&ptr_, rounded) != hipSuccess) {
    ptr_ = nullptr;
    (void)hipGetLastError();
    return nullptr;
  }
  // Not cleared: every launch writes what a later one reads, and a memset on the
  // null stream would invalidate captures that other streams are in.
  bytes_ = rounded;
  return ptr_;
}

}  // namespace affon
