// devmem.h -- the engine's device memory: a cache of the trees' and builds'
// blocks, and the allocations that do not go through it.  Host code only.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include <map>
#include <mutex>
#include <unordered_map>

namespace hrt {

// Device memory of one context's trees and build scratch, kept for reuse when
// it is given back (a 128 MB hipMalloc takes 53 us and its hipFree 265 us, and
// a build has a dozen arrays: a million triangles loaded and committed took
// 10.3 ms, and 2.8 with this and the geometry expanded on the device), and
// pinned words for small readbacks (12 us with the wait, 21 us through pageable
// memory).  Safe with several threads.
//
// At most kMaxIdle bytes are kept idle, for blocks of up to a quarter less.
// They go back to the device when any allocation of the engine on it fails
// (here, device_malloc, stream_malloc), whichever context kept them, and at the
// end.  On a full list a block that was not taken again while kStale bytes came
// back makes room, so that a program whose sizes change finds its memory:
// scenes of 1 M triangles after some of 4 M are loaded in 3.7 ms and closed in
// none, with a list that keeps what it has in 4.3 and 2.2 for good.  Making room
// for every block would cost a program that needs more than kMaxIdle again and
// again: 16 M triangles loaded and closed 49.5 ms instead of 47.4.
class DevCache {
 public:
  explicit DevCache(int device);  // may throw std::bad_alloc
  DevCache(const DevCache&) = delete;
  DevCache& operator=(const DevCache&) = delete;
  ~DevCache();
  template <class T>
  hipError_t alloc(T** p, size_t bytes) {
    return alloc_bytes(reinterpret_cast<void**>(p), bytes);
  }
  // For memory that nothing on the device uses any more (null is fine).
  void free(void* p);
  // Waits for the whole device, whatever the caller's current one is.
  void wait();
  // Gives the idle blocks back; whether there were any.
  bool trim();
  // trim of every cache on the current device.
  static bool trim_device();
  // kPinnedWords words, or null when all are taken.
  static constexpr size_t kPinnedWords = 32;
  uint32_t* pinned_get();
  void pinned_put(uint32_t* w);

  static constexpr size_t kMaxIdle = size_t(1) << 30;
  static constexpr uint64_t kStale = 16 * uint64_t(kMaxIdle);

 private:
  static constexpr int kPinnedSlots = 16;
  hipError_t alloc_bytes(void** p, size_t bytes);
  bool note(void* p, size_t size);
  const int device_;
  std::mutex mu_;
  std::unordered_map<void*, size_t> live_;
  struct Idle {
    void* p;
    uint64_t order, since;  // since: given_back_ then
  };
  using IdleMap = std::multimap<size_t, Idle>;  // by size
  void* take(IdleMap::iterator it);
  IdleMap idle_;
  std::map<uint64_t, IdleMap::iterator> oldest_;  // the same blocks by `order`
  uint64_t order_ = 0, given_back_ = 0;           // blocks and bytes so far
  size_t idle_bytes_ = 0;
  uint32_t* pinned_ = nullptr;
  uint32_t pinned_taken_ = 0;  // a bit per slot
};

// hipMalloc and hipMallocAsync on the current device, tried again without the
// caches' idle blocks before they fail.  (Not while `stream` is captured: the
// blocks' hipFree would end the capture.)
hipError_t device_malloc_bytes(void** p, size_t bytes);
hipError_t stream_malloc_bytes(void** p, size_t bytes, hipStream_t stream);
template <class T>
hipError_t device_malloc(T** p, size_t bytes) {
  return device_malloc_bytes(reinterpret_cast<void**>(p), bytes);
}
template <class T>
hipError_t stream_malloc(T** p, size_t bytes, hipStream_t stream) {
  return stream_malloc_bytes(reinterpret_cast<void**>(p), bytes, stream);
}
// stream_malloc of `words` 32-bit words for each of *lanes lanes in whole
// groups; without the memory for a quarter as many each time, at least `least`.
hipError_t lane_malloc(uint32_t** p, uint64_t* lanes, uint64_t least, uint32_t group, size_t words,
                       hipStream_t stream);

}  // namespace hrt
