// Device memory of a session: its allocations, and the scratch of its launches.
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace affon {

// Device scratch memory owned by a session and ordered by its stream.
// Buffers it outgrows are retired, not freed, until the session ends: a
// graph captured earlier keeps the old address in its kernel arguments and
// may still be replayed.
class Workspace {
 public:
  Workspace(int device, hipStream_t stream) : device_(device), stream_(stream) {}
  ~Workspace();
  Workspace(const Workspace&) = delete;
  Workspace& operator=(const Workspace&) = delete;
  // At least `bytes` of device memory, or nullptr when it cannot grow now
  // (the stream is being captured into a graph, or the allocation failed).
  void* get(size_t bytes);
  size_t retired() const { return retired_.size(); }
  std::mutex& mutex() { return mutex_; }

 private:
  std::mutex mutex_;
  int device_;
  hipStream_t stream_;
  void* ptr_ = nullptr;
  size_t bytes_ = 0;
  std::vector<void*> retired_;
  size_t retired_bytes_ = 0;  // size of the last retired buffer
};

// Where a launcher enqueues its work, and the scratch memory it may use for
// split-K partial sums: the session's workspace (grown on demand), or a
// fixed buffer of fixed_bytes (the no-allocation entry point), or none.
//
// A call that takes the workspace holds it until the call ends, so that the
// launches that fill and read it are enqueued with no other thread's between
// them; on the stream they then run in that order.
struct Launch {
  hipStream_t stream = nullptr;
  Workspace* workspace = nullptr;
  void* fixed = nullptr;
  size_t fixed_bytes = 0;
  // Set when a fixed buffer is too small for the launcher's plan; the
  // launcher then launches nothing and returns hipErrorOutOfMemory.
  mutable size_t fixed_short = 0;
  mutable std::unique_lock<std::mutex> held;

  bool can_split() const { return workspace != nullptr || fixed != nullptr; }
  // At least `bytes` of scratch, or nullptr (workspace: it cannot grow now;
  // fixed buffer: too small, recorded in fixed_short).
  void* scratch(size_t bytes) const {
    if (workspace != nullptr) {
      if (!held.owns_lock()) held = std::unique_lock<std::mutex>(workspace->mutex());
      return workspace->get(bytes);
    }
    if (fixed != nullptr && bytes <= fixed_bytes) return fixed;
    if (fixed != nullptr) fixed_short = bytes;
    return nullptr;
  }
};

// Device memory of a session. A freed block is kept for a later allocation of
// its size class instead of going back to the runtime: hipMalloc and hipFree
// cost tens of microseconds to milliseconds (a dequantize to 117 MB took 3.3
// ms in a loop for 36 us of kernel), and every free waited for the stream.
//
// What hipFree gave stays: memory is handed out again only when nothing
// anywhere on the device can still use it. A freed block waits in `resting`
// until the device has been idle at some moment after its free, whatever
// streams the caller used it on; blocks of one class are allocated anew
// until kRest of them rest, so that the wait (20 to 40 us beside other work)
// comes once for many frees.
// At most kKeepBytes are kept, blocks over kMostBytes not at all; the rest
// goes back to the runtime, as everything does when an allocation fails and
// when the session ends.
//
// A graph holds the addresses that its captured region used, and writes to
// them in every replay. What is allocated or freed while the session's stream
// is captured is therefore never handed out again, and is released when the
// session ends (as Workspace does with buffers it outgrew). While a capture
// lasts nothing goes back to the runtime.
//
// alloc and free may come from any thread (a caller's garbage collector
// frees from whichever thread it runs on): the mutex guards everything. Both
// may throw std::bad_alloc; a block is then where it was, or (alloc) returned.
class DeviceMemory {
 public:
  explicit DeviceMemory(hipStream_t stream) : stream_(stream) {}

  hipError_t alloc(size_t bytes, void** out) {
    size_t size = bytes <= kMostBytes ? size_class(bytes) : bytes;
    bool pooled = size <= kMostBytes;
    std::lock_guard<std::mutex> lock(mutex_);
    std::vector<void*>* ready = find_ready(size);
    if (ready == nullptr && worth_a_wait(size) && settle()) ready = find_ready(size);
    if (ready != nullptr) {
      *out = ready->back();
      ready->pop_back();
      kept_ -= size;
    } else {
      hipError_t e = hipMalloc(out, size);
      if (e != hipSuccess && kept_ > 0) {
        (void)hipGetLastError();
        give_back();
        e = hipMalloc(out, size);
      }
      if (e != hipSuccess && size > bytes && bytes > 0) {  // what the rounding up asks for may be too much
        (void)hipGetLastError();
        size = bytes;
        pooled = false;
        e = hipMalloc(out, size);
      }
      if (e != hipSuccess) {
        (void)hipGetLastError();
        *out = nullptr;
        return e;
      }
    }
    try {
      owned_.emplace(*out, Owned{size, pooled, capturing()});
    } catch (...) {
      (void)hipFree(*out);
      *out = nullptr;
      throw;
    }
    return hipSuccess;
  }

  // False when this session did not allocate ptr.
  bool free(void* ptr, hipError_t* status) {
    *status = hipSuccess;
    std::lock_guard<std::mutex> lock(mutex_);
    const auto it = owned_.find(ptr);
    if (it == owned_.end()) return false;
    const size_t size = it->second.size;
    if (it->second.captured || capturing()) {
      retired_.push_back(ptr);
      owned_.erase(it);
      return true;
    }
    if (it->second.pooled) {
      if (kept_ + size > kKeepBytes) give_back();
      if (kept_ + size <= kKeepBytes) {
        size_t& resting = resting_classes_[size];
        resting_.push_back({size, ptr});
        ++resting;
        kept_ += size;
        owned_.erase(it);
        return true;
      }
    }
    *status = hipStreamSynchronize(stream_);
    const hipError_t e = hipFree(ptr);
    if (*status == hipSuccess) *status = e;
    if (e != hipSuccess) retired_.push_back(ptr);  // released when the session ends
    owned_.erase(it);
    return true;
  }

  // Everything, live allocations too (the session's work has ended).
  void release_all() {
    std::lock_guard<std::mutex> lock(mutex_);
    free_all(resting_);
    for (auto& entry : ready_) free_all(entry.second);
    free_all(retired_);
    for (const auto& block : owned_) (void)hipFree(block.first);
    resting_classes_.clear();
    ready_.clear();
    owned_.clear();
    kept_ = 0;
  }

 private:
  static constexpr size_t kKeepBytes = size_t(1) << 30;
  static constexpr size_t kMostBytes = size_t(256) << 20;
  static constexpr size_t kLargeBytes = size_t(1) << 20;
  static constexpr size_t kRest = 64;

  // Sizes round up to eighths of a power of two, at least 256 bytes.
  static size_t size_class(size_t bytes) {
    size_t unit = 256;
    while (unit * 16 < bytes) unit *= 2;
    return (bytes + unit - 1) / unit * unit + (bytes == 0 ? unit : 0);
  }
  // The blocks of this class that can be handed out, if there are any.
  std::vector<void*>* find_ready(size_t size) {
    const auto it = ready_.find(size);
    return it == ready_.end() || it->second.empty() ? nullptr : &it->second;
  }
  bool capturing() const {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(stream_, &capture);
    if (e != hipSuccess) (void)hipGetLastError();
    return e != hipSuccess || capture != hipStreamCaptureStatusNone;
  }
  // Whether a resting block of this class is worth waiting for the device:
  // kRest of them rest (of a large class, half of what is kept), or the
  // session's own work is done, so that there is hardly anything to wait for,
  // and they are more than a few small ones (asking the device costs 1.3 us, as
  // an allocation of a word does; one of megabytes takes 20).
  bool worth_a_wait(size_t size) const {
    const auto it = resting_classes_.find(size);
    if (it == resting_classes_.end()) return false;
    if (it->second >= kRest || it->second * size >= kKeepBytes / 2) return true;
    if ((it->second < 8 && it->second * size < kLargeBytes) || capturing()) return false;
    const hipError_t e = hipStreamQuery(stream_);
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
  }
  // Waits for the device and makes the resting blocks ready; false (nothing
  // changed) where it cannot wait now, as while the stream is captured.
  bool settle() {
    if (capturing() || !wait_for_device()) return false;
    while (!resting_.empty()) {  // a block at a time: it is in one list, whatever throws
      const Block b = resting_.back();
      ready_[b.size].push_back(b.ptr);
      resting_.pop_back();
      --resting_classes_[b.size];
    }
    resting_classes_.clear();
    return true;
  }
  // Waits for all of the device's work, with blocks resting, by a hipFree: that
  // waits for every stream too, and hipDeviceSynchronize invalidates captures
  // that other streams are in. False where it could not wait. The session's own
  // work first, by a wait that polls: hipFree's costs 20 us more.
  bool wait_for_device() {
    if (hipStreamSynchronize(stream_) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    void* small = nullptr;
    const bool spare = hipMalloc(&small, 1) == hipSuccess;
    if (!spare) (void)hipGetLastError();  // no memory left: a resting block goes
    if (hipFree(spare ? small : resting_.back().ptr) != hipSuccess) {
      (void)hipGetLastError();
      if (spare) retired_.push_back(small);
      return false;
    }
    if (!spare) {
      --resting_classes_[resting_.back().size];
      kept_ -= resting_.back().size;
      resting_.pop_back();
    }
    return true;
  }
  // Returns every kept block to the runtime; none where the device cannot be
  // waited for now.
  void give_back() {
    if (capturing() || (!resting_.empty() && !settle())) return;
    for (auto& entry : ready_) free_all(entry.second);
    ready_.clear();
    kept_ = 0;
  }

  struct Block {
    size_t size;
    void* ptr;
  };
  struct Owned {
    size_t size;
    bool pooled;    // of a size class, kept when freed
    bool captured;  // allocated while the stream was captured
  };
  static void* address(const Block& b) { return b.ptr; }
  static void* address(void* ptr) { return ptr; }
  template <typename T>
  static void free_all(std::vector<T>& blocks) {
    for (const T& b : blocks) (void)hipFree(address(b));
    blocks.clear();
  }
  hipStream_t stream_;
  std::mutex mutex_;
  std::unordered_map<void*, Owned> owned_;  // handed out, by address
  std::map<size_t, std::vector<void*>> ready_;
  std::vector<Block> resting_;
  std::vector<void*> retired_;  // freed, but not to be used or released before the session ends
  std::unordered_map<size_t, size_t> resting_classes_;
  size_t kept_ = 0;  // bytes of ready_ and resting_
};

}  // namespace affon
