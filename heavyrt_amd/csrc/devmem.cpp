// devmem.cpp -- the device memory of devmem.h.
#include "devmem.h"

#include <algorithm>
#include <new>
#include <vector>

namespace hrt {

namespace {

// The caches alive, for trim_device; never destroyed (a cache may outlive
// static objects).
struct Registry {
  std::mutex mu;
  std::vector<DevCache*> caches;
};
Registry& registry() {
  static Registry* r = new Registry;
  return *r;
}

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

}  // namespace

DevCache::DevCache(int device) : device_(device) {
  std::lock_guard<std::mutex> lock(registry().mu);
  registry().caches.push_back(this);
}

DevCache::~DevCache() {
  {
    std::lock_guard<std::mutex> lock(registry().mu);
    std::vector<DevCache*>& c = registry().caches;
    c.erase(std::find(c.begin(), c.end(), this));
  }
  trim();
  if (pinned_) (void)hipHostFree(pinned_);
}

void DevCache::wait() {
  int current = device_;
  (void)hipGetDevice(&current);
  if (current != device_) (void)hipSetDevice(device_);
  (void)hipDeviceSynchronize();
  if (current != device_) (void)hipSetDevice(current);
}

bool DevCache::trim() {
  IdleMap idle;
  {
    std::lock_guard<std::mutex> lock(mu_);
    idle.swap(idle_);
    oldest_.clear();
    idle_bytes_ = 0;
  }
  for (auto& x : idle) (void)hipFree(x.second.p);
  return !idle.empty();
}

bool DevCache::trim_device() {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return false;
  bool any = false;
  std::lock_guard<std::mutex> lock(registry().mu);
  for (DevCache* c : registry().caches)
    if (c->device_ == device) any = c->trim() || any;
  return any;
}

hipError_t DevCache::alloc_bytes(void** p, size_t bytes) {
  // sizes in steps, so that a slightly different geometry finds its memory
  const size_t step = bytes < (size_t(1) << 16) ? size_t(1) << 12 : bytes < (size_t(1) << 20) ? size_t(1) << 16 : size_t(1) << 21;
  const size_t size = (std::max<size_t>(bytes, 1) + step - 1) / step * step;
  {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = idle_.lower_bound(size);
    if (it != idle_.end() && it->first <= size + size / 4) {
      if (!note(it->second.p, it->first)) return hipErrorOutOfMemory;
      *p = take(it);
      return hipSuccess;
    }
  }
  const hipError_t e = device_malloc_bytes(p, size);
  if (e != hipSuccess) {
    *p = nullptr;
    return e;
  }
  std::lock_guard<std::mutex> lock(mu_);
  if (note(*p, size)) return hipSuccess;
  (void)hipFree(*p);
  *p = nullptr;
  return hipErrorOutOfMemory;
}

// mu_ held; false: no host memory
bool DevCache::note(void* p, size_t size) {
  try {
    live_[p] = size;
  } catch (const std::bad_alloc&) {
    return false;
  }
  return true;
}

// mu_ held: the block, no longer idle
void* DevCache::take(IdleMap::iterator it) {
  void* p = it->second.p;
  idle_bytes_ -= it->first;
  oldest_.erase(it->second.order);
  idle_.erase(it);
  return p;
}

void DevCache::free(void* p) {
  if (!p) return;
  size_t size = 0;
  {
    std::lock_guard<std::mutex> lock(mu_);
    const auto it = live_.find(p);
    if (it == live_.end()) return;
    size = it->second;
    live_.erase(it);
    given_back_ += size;
  }
  // One block at a time: hipFree waits and must not hold the lock.
  while (size <= kMaxIdle) {
    void* old = nullptr;
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (idle_bytes_ + size <= kMaxIdle) {
        auto it = idle_.end();
        try {
          it = idle_.emplace(size, Idle{p, ++order_, given_back_});
          oldest_.emplace(order_, it);
        } catch (const std::bad_alloc&) {  // no host memory: given back below
          if (it != idle_.end()) idle_.erase(it);
          break;
        }
        idle_bytes_ += size;
        return;
      }
      const auto it = oldest_.begin()->second;
      if (given_back_ - it->second.since <= kStale) break;
      old = take(it);
    }
    (void)hipFree(old);
  }
  (void)hipFree(p);
}

uint32_t* DevCache::pinned_get() {
  std::lock_guard<std::mutex> lock(mu_);
  if (!pinned_ && hipHostMalloc(reinterpret_cast<void**>(&pinned_), 4 * kPinnedWords * kPinnedSlots,
                                hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    pinned_ = nullptr;
    return nullptr;
  }
  for (int k = 0; k < kPinnedSlots; k++) {
    if (pinned_taken_ & (1u << k)) continue;
    pinned_taken_ |= 1u << k;
    return pinned_ + k * kPinnedWords;
  }
  return nullptr;
}

void DevCache::pinned_put(uint32_t* w) {
  std::lock_guard<std::mutex> lock(mu_);
  pinned_taken_ &= ~(1u << (size_t(w - pinned_) / kPinnedWords));
}

hipError_t device_malloc_bytes(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory && DevCache::trim_device()) {
    (void)hipGetLastError();
    e = hipMalloc(p, bytes);
  }
  return e;
}

hipError_t stream_malloc_bytes(void** p, size_t bytes, hipStream_t stream) {
  hipError_t e = hipMallocAsync(p, bytes, stream);
  if (e == hipErrorOutOfMemory && !capturing(stream) && DevCache::trim_device()) {
    (void)hipGetLastError();
    e = hipMallocAsync(p, bytes, stream);
  }
  return e;
}

hipError_t lane_malloc(uint32_t** p, uint64_t* lanes, uint64_t least, uint32_t group, size_t words,
                       hipStream_t stream) {
  while (true) {
    const uint64_t whole = (*lanes + group - 1) / group * group;
    const hipError_t e = stream_malloc(p, sizeof(uint32_t) * whole * words, stream);
    if (e != hipErrorOutOfMemory || *lanes <= least) return e;
    (void)hipGetLastError();
    *lanes = std::max(*lanes / 4, least);
  }
}

}  // namespace hrt
