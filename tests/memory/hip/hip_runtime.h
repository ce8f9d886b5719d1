// A stand-in for the HIP runtime, for CPU tests of memory.h: memory is host
// memory under a limit, a stream is captured when the test says so, and
// `device_busy` says whether work of any stream still runs, for which hipFree
// and hipDeviceSynchronize wait. The latter ends captures on all streams.
#pragma once

#include <cstdlib>
#include <cstring>
#include <map>
#include <stdexcept>
#include <string>

typedef int hipError_t;
typedef struct FakeStream* hipStream_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorNotReady = 600, hipErrorStreamCaptureUnsupported = 900 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 };

namespace fake {
inline std::map<void*, size_t> blocks;  // what hipMalloc gave and hipFree did not take
inline size_t used = 0, limit = size_t(1) << 40;
inline bool session_capturing = false, session_busy = false, device_busy = false, free_fails = false;
inline bool other_capturing = false, other_capture_broken = false;  // a capture on another stream
inline int frees_while_capturing = 0;
}  // namespace fake

inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMalloc(void** out, size_t bytes) {
  if (fake::used + bytes > fake::limit) return hipErrorOutOfMemory;
  *out = std::malloc(1);  // an address of its own
  fake::blocks[*out] = bytes;
  fake::used += bytes;
  return hipSuccess;
}
inline hipError_t hipFree(void* ptr) {
  const auto it = fake::blocks.find(ptr);
  if (it == fake::blocks.end()) throw std::logic_error("free of what is not allocated");
  if (fake::free_fails) return hipErrorStreamCaptureUnsupported;
  fake::frees_while_capturing += fake::session_capturing;
  fake::session_busy = fake::device_busy = false;
  fake::used -= it->second;
  fake::blocks.erase(it);  // its address is never used again, so that a second free shows
  return hipSuccess;
}
inline hipError_t hipMemset(void*, int, size_t) {  // on the null stream
  fake::other_capture_broken |= fake::other_capturing;
  return hipSuccess;
}
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status) {
  *status = fake::session_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
  if (fake::session_capturing) return hipErrorStreamCaptureUnsupported;
  fake::session_busy = false;
  return hipSuccess;
}
inline hipError_t hipStreamQuery(hipStream_t) { return fake::session_busy ? hipErrorNotReady : hipSuccess; }
inline hipError_t hipDeviceSynchronize() {
  fake::other_capture_broken |= fake::other_capturing;
  if (fake::session_capturing || fake::other_capturing) return hipErrorStreamCaptureUnsupported;
  fake::session_busy = fake::device_busy = false;
  return hipSuccess;
}
