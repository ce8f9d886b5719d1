// DeviceMemory and Workspace against a stand-in HIP runtime. Run with the name of one check.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <new>
#include <set>
#include <thread>

#include "memory.h"

namespace {

// Allocations on the host until one fails (-1: none does).
int g_until_bad_alloc = -1;

constexpr size_t MiB = size_t(1) << 20;

#define CHECK(x)                                                   \
  do {                                                             \
    if (!(x)) {                                                    \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);          \
      std::exit(1);                                                \
    }                                                              \
  } while (0)

void* alloc(affon::DeviceMemory& m, size_t bytes) {
  void* p = nullptr;
  CHECK(m.alloc(bytes, &p) == hipSuccess && p != nullptr);
  CHECK(fake::blocks.at(p) >= bytes);
  return p;
}
void free(affon::DeviceMemory& m, void* p) {
  hipError_t e;
  CHECK(m.free(p, &e) && e == hipSuccess);
}
// Idle, what the session keeps is handed out: whether any of `ptrs` is, among many allocations.
bool comes_back(affon::DeviceMemory& m, const std::set<void*>& ptrs, size_t bytes) {
  for (int i = 0; i < 100; ++i)
    if (ptrs.count(alloc(m, bytes))) return true;
  return false;
}

void reuse() {
  affon::DeviceMemory m(nullptr);
  void* a = alloc(m, 5 * MiB);
  free(m, a);
  CHECK(alloc(m, 5 * MiB) == a);
  std::set<void*> small;
  for (int i = 0; i < 16; ++i) small.insert(alloc(m, 5000));
  for (void* p : small) free(m, p);
  CHECK(small.count(alloc(m, 5000)));
}

// A block freed while any stream works waits for the device to be idle.
void other_stream() {
  affon::DeviceMemory m(nullptr);
  void* a = alloc(m, 5 * MiB);
  fake::session_busy = fake::device_busy = true;
  free(m, a);
  CHECK(alloc(m, 5 * MiB) != a && fake::device_busy);  // the session works: no wait for one block
  fake::session_busy = false;  // only another stream works now
  CHECK(alloc(m, 5 * MiB) == a && !fake::device_busy);
}

// What a captured region allocates or frees stays aside until the session ends.
void capture(size_t bytes) {
  affon::DeviceMemory m(nullptr);
  void* before = alloc(m, bytes);
  void* kept = alloc(m, bytes);
  free(m, kept);
  fake::session_capturing = true;
  void *in = alloc(m, bytes), *out = alloc(m, bytes);
  free(m, in);      // as a captured Program's intermediate
  free(m, before);  // of before, used in the region
  CHECK(alloc(m, bytes) != in);
  CHECK(fake::frees_while_capturing == 0);
  fake::session_capturing = false;
  free(m, out);  // a captured output dropped later
  if (bytes <= 256 * MiB) CHECK(!comes_back(m, {in, out, before}, bytes));
  CHECK(fake::blocks.count(in) && fake::blocks.count(out) && fake::blocks.count(before));
  hipError_t e;
  CHECK(!m.free(in, &e));  // freed once
  m.release_all();
  CHECK(fake::blocks.empty());
}

// Nothing goes back to the runtime while the stream is captured, full pool or failing allocation.
void no_free_in_capture() {
  affon::DeviceMemory m(nullptr);
  std::set<void*> parked;
  for (int i = 0; i < 8; ++i) parked.insert(alloc(m, 100 * MiB));
  fake::session_busy = true;
  for (void* p : parked) free(m, p);
  fake::session_capturing = true;
  std::set<void*> live;
  for (int i = 0; i < 5; ++i) live.insert(alloc(m, 100 * MiB));
  for (void* p : live) free(m, p);
  fake::limit = fake::used;
  void* p = nullptr;
  CHECK(m.alloc(64 * MiB, &p) == hipErrorOutOfMemory && p == nullptr);
  CHECK(fake::frees_while_capturing == 0);
  fake::session_capturing = false;
  alloc(m, 64 * MiB);  // from what the parked blocks gave back
}

// The device cannot be waited for: kept blocks stay, and none is handed out.
void no_idle_moment() {
  affon::DeviceMemory m(nullptr);
  std::set<void*> ptrs;
  for (int i = 0; i < 20; ++i) ptrs.insert(alloc(m, 100 * MiB));
  fake::free_fails = true;
  hipError_t e;
  for (void* p : ptrs) CHECK(m.free(p, &e));
  for (int i = 0; i < 20; ++i) CHECK(!ptrs.count(alloc(m, 100 * MiB)));
  fake::free_fails = false;
  m.release_all();
  CHECK(fake::blocks.empty());
}

// Allocations, frees and reuse leave a capture on another stream alone.
void other_capture() {
  affon::DeviceMemory m(nullptr);
  fake::other_capturing = true;
  void* a = alloc(m, 5 * MiB);
  free(m, a);
  CHECK(alloc(m, 5 * MiB) == a);
  for (int i = 0; i < 30; ++i) free(m, alloc(m, 100 * MiB + 1000000 * i));
  CHECK(!fake::other_capture_broken);
}

void other_capture_scratch() {
  affon::Workspace w(0, nullptr);
  fake::other_capturing = true;
  CHECK(w.get(1000) != nullptr && w.get(10 * MiB) != nullptr && !fake::other_capture_broken);
}

// With no memory left even for a word, kept blocks still make room.
void full() {
  affon::DeviceMemory m(nullptr);
  std::set<void*> ptrs;
  for (int i = 0; i < 4; ++i) ptrs.insert(alloc(m, MiB));
  fake::session_busy = true;
  for (void* p : ptrs) free(m, p);
  fake::limit = fake::used;
  alloc(m, 3 * MiB);
}

// A size that fits only without rounding up is still given.
void exact_size() {
  affon::DeviceMemory m(nullptr);
  fake::limit = 17 * MiB + 4096;
  void* p = alloc(m, 17 * MiB + 1);
  free(m, p);
  CHECK(fake::used == 0);
  alloc(m, 17 * MiB + 2);
}

// Whichever allocation on the host fails, no block is lost, given twice or freed twice.
void host_memory_fails() {
  for (int n = 0; n < 60; ++n) {
    affon::DeviceMemory m(nullptr);
    std::set<void*> live;
    g_until_bad_alloc = n;
    for (int i = 0; i < 200; ++i) {
      try {
        if (i % 40 < 20) {
          void* p = nullptr;
          if (m.alloc(1000 + 300 * (i % 3), &p) == hipSuccess) {
            const int armed = g_until_bad_alloc;
            g_until_bad_alloc = -1;
            CHECK(live.insert(p).second && fake::blocks.count(p));
            g_until_bad_alloc = armed;
          }
        } else if (!live.empty()) {
          hipError_t e;
          void* p = *live.begin();
          CHECK(m.free(p, &e));
          live.erase(p);
        }
      } catch (const std::bad_alloc&) {
      }
    }
    g_until_bad_alloc = -1;
    m.release_all();
    CHECK(fake::blocks.empty());
  }
}

// A call's scratch is its own until the call ends, whichever threads call.
void scratch_between_threads() {
  affon::Workspace workspace(0, nullptr);
  std::atomic<bool> taken{false}, ended{false};
  std::thread first([&] {
    {
      affon::Launch l;
      l.workspace = &workspace;
      CHECK(l.scratch(1000) != nullptr && l.scratch(2000) != nullptr);  // taken twice by one call
      taken = true;
      std::this_thread::sleep_for(std::chrono::milliseconds(200));
      ended = true;
    }
  });
  while (!taken) std::this_thread::yield();
  affon::Launch l;
  l.workspace = &workspace;
  CHECK(l.scratch(1000) != nullptr);
  CHECK(ended);
  first.join();
}

}  // namespace

void* operator new(size_t bytes) {
  if (g_until_bad_alloc >= 0 && g_until_bad_alloc-- == 0) throw std::bad_alloc();
  return std::malloc(bytes);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int, char** argv) {
  const std::string name = argv[1];
  if (name == "reuse") reuse();
  else if (name == "other_stream") other_stream();
  else if (name == "capture") capture(5000);
  else if (name == "capture_large") capture(300 * MiB);
  else if (name == "no_free_in_capture") no_free_in_capture();
  else if (name == "no_idle_moment") no_idle_moment();
  else if (name == "other_capture") other_capture();
  else if (name == "other_capture_scratch") other_capture_scratch();
  else if (name == "full") full();
  else if (name == "exact_size") exact_size();
  else if (name == "scratch_between_threads") scratch_between_threads();
  else if (name == "host_memory_fails") host_memory_fails();
  else return 2;
  return 0;
}
