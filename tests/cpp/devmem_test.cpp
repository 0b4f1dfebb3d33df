// devmem.cpp on a device made of counters: the HIP calls it makes are defined
// here, with a capacity.  `devmem_test NAME` runs one scenario; the exit status
// is 0 when every check holds.
#include "devmem.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace {

constexpr size_t kMB = size_t(1) << 20;

struct Device {
  std::mutex mu;
  size_t capacity = size_t(1) << 40, used = 0;
  std::map<void*, size_t> blocks;
  int mallocs = 0, frees = 0, bad_frees = 0, current = 0;
  bool capturing = false;
  hipError_t take(void** p, size_t n) {
    std::lock_guard<std::mutex> lock(mu);
    mallocs++;
    if (used + n > capacity) return hipErrorOutOfMemory;
    *p = std::malloc(16);
    blocks[*p] = n;
    used += n;
    return hipSuccess;
  }
  hipError_t give(void* p) {
    std::lock_guard<std::mutex> lock(mu);
    const auto it = blocks.find(p);
    if (it == blocks.end()) {
      bad_frees++;
      return hipErrorInvalidValue;
    }
    frees++;
    used -= it->second;
    blocks.erase(it);
    std::free(p);
    return hipSuccess;
  }
} dev;

void check(bool ok, const char* what) {
  if (ok) return;
  std::fprintf(stderr, "failed: %s\n", what);
  std::exit(1);
}

}  // namespace

hipError_t hipMalloc(void** p, size_t n) { return dev.take(p, n); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return dev.take(p, n); }
hipError_t hipFree(void* p) { return dev.give(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = dev.current, hipSuccess; }
hipError_t hipSetDevice(int d) { return dev.current = d, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  *s = dev.capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}

namespace {

using hrt::DevCache;

// `n` blocks of `size`, given back to `mem`: idle there as far as it keeps them
void leave_idle(DevCache& mem, size_t size, int n) {
  std::vector<void*> p(n);
  for (void*& x : p) check(mem.alloc(&x, size) == hipSuccess, "alloc");
  for (void* x : p) mem.free(x);
}

void reuse() {
  DevCache mem(0);
  leave_idle(mem, 100 * kMB, 1);
  const int before = dev.mallocs;
  leave_idle(mem, 90 * kMB, 1);
  check(dev.mallocs == before, "a block up to a quarter larger is taken again");
  leave_idle(mem, 70 * kMB, 1);
  check(dev.mallocs == before + 1, "a larger one is not");
}

// A full list keeps what a program takes again and again, and gives back what
// none takes any more.
void reuse_after_the_sizes_change() {
  DevCache mem(0);
  const int rounds = int(DevCache::kStale / (200 * kMB)) + 2;
  leave_idle(mem, 10 * kMB, 110);
  check(dev.used <= DevCache::kMaxIdle, "no more than the bound stays");
  int before = dev.mallocs;
  for (int k = 0; k < 20; k++) leave_idle(mem, 10 * kMB, 110);
  check(dev.mallocs - before <= 20 * 8, "102 of 110 are taken again each time");
  for (int k = 0; k < rounds; k++) {
    leave_idle(mem, 50 * kMB, 4);
    check(dev.used <= DevCache::kMaxIdle, "the bound holds");
  }
  before = dev.mallocs;
  for (int k = 0; k < 20; k++) leave_idle(mem, 50 * kMB, 4);
  check(dev.mallocs == before, "the new size is taken again");
  leave_idle(mem, 10 * kMB, 70);
  check(dev.mallocs == before, "and what is left of the old one");
  leave_idle(mem, DevCache::kMaxIdle + kMB, 1);
  leave_idle(mem, 10 * kMB, 70);
  check(dev.mallocs == before + 1, "a block beyond the bound is not kept and costs the others nothing");
  check(dev.bad_frees == 0, "every block given back once");
}

// Allocations outside the cache get its idle memory, other contexts' too.
void others_get_the_idle_memory() {
  DevCache mem(0), second(0);
  leave_idle(mem, 100 * kMB, 4);
  leave_idle(second, 100 * kMB, 4);
  dev.capacity = dev.used + 10 * kMB;
  void* p = nullptr;
  check(hrt::device_malloc(&p, 700 * kMB) == hipSuccess, "device_malloc");
  check(dev.used == 700 * kMB, "nothing stays idle");
  check(hrt::device_malloc(&p, 700 * kMB) == hipErrorOutOfMemory, "what does not fit is refused");
  dev.capacity += 400 * kMB;
  leave_idle(second, 100 * kMB, 3);
  check(hrt::stream_malloc(&p, 350 * kMB, nullptr) == hipSuccess, "stream_malloc");
  dev.capacity += 200 * kMB;
  leave_idle(second, 100 * kMB, 1);
  check(mem.alloc(&p, 240 * kMB) == hipSuccess, "another context's cache");
}

void not_another_devices() {
  DevCache other(1);
  leave_idle(other, 100 * kMB, 1);
  dev.capacity = dev.used;
  void* p = nullptr;
  check(hrt::device_malloc(&p, kMB) == hipErrorOutOfMemory, "device 0 is full");
  check(dev.used == 100 * kMB, "device 1 keeps its own");
}

// A hipFree would end the capture.
void not_under_capture() {
  DevCache mem(0);
  leave_idle(mem, 100 * kMB, 1);
  dev.capacity = dev.used;
  dev.capturing = true;
  void* p = nullptr;
  check(hrt::stream_malloc(&p, kMB, nullptr) == hipErrorOutOfMemory, "refused");
  check(dev.frees == 0, "no hipFree");
}

void fewer_lanes_without_memory() {
  uint32_t* p = nullptr;
  uint64_t lanes = 1000;
  check(hrt::lane_malloc(&p, &lanes, 64, 64, 39, nullptr) == hipSuccess && lanes == 1000 && dev.used == 1024 * 156,
        "whole groups");
  hipFree(p);
  for (const uint64_t start : {uint64_t(1) << 22, uint64_t(3000001)}) {
    lanes = start;
    dev.capacity = (start / 16 + 64) * 156;
    check(hrt::lane_malloc(&p, &lanes, 65536, 64, 39, nullptr) == hipSuccess && lanes == start / 16, "a sixteenth");
    hipFree(p);
    lanes = start;
    dev.capacity = 65536 * 156 - 1;
    check(hrt::lane_malloc(&p, &lanes, 65536, 64, 39, nullptr) == hipErrorOutOfMemory && lanes == 65536, "the least");
  }
  lanes = 5000;
  check(hrt::lane_malloc(&p, &lanes, lanes, 64, 39000, nullptr) == hipErrorOutOfMemory && lanes == 5000, "all or none");
}

void threads() {
  DevCache mem(0);
  dev.capacity = 600 * kMB;
  std::vector<std::thread> t;
  for (int k = 0; k < 8; k++)
    t.emplace_back([&mem, k] {
      uint32_t* words = nullptr;
      for (int i = 0; i < 2000; i++) {
        void *a = nullptr, *b = nullptr;
        const hipError_t ea = mem.alloc(&a, size_t(1 + (i * 7 + k) % 30) * kMB);
        const hipError_t eb = hrt::device_malloc(&b, kMB);
        check(ea == hipSuccess && eb == hipSuccess && a != b, "eight threads' blocks fit");
        if (!words) words = mem.pinned_get();
        mem.free(a);
        hipFree(b);
        if (words && i % 3 == 0) mem.pinned_put(words), words = nullptr;
      }
    });
  for (std::thread& x : t) x.join();
  mem.trim();
  check(dev.used == 0 && dev.bad_frees == 0, "every block went back once");
}

void given_back_at_the_end() {
  {
    DevCache mem(0);
    leave_idle(mem, 100 * kMB, 5);
    check(dev.used > 0, "idle until then");
  }
  check(dev.used == 0, "with the cache");
}

}  // namespace

int main(int, char** argv) {
  const struct {
    const char* name;
    void (*fn)();
  } all[] = {{"reuse", reuse},
             {"reuse_after_the_sizes_change", reuse_after_the_sizes_change},
             {"others_get_the_idle_memory", others_get_the_idle_memory},
             {"not_another_devices", not_another_devices},
             {"not_under_capture", not_under_capture},
             {"fewer_lanes_without_memory", fewer_lanes_without_memory},
             {"threads", threads},
             {"given_back_at_the_end", given_back_at_the_end}};
  for (const auto& s : all)
    if (argv[1] && !std::strcmp(argv[1], s.name)) return s.fn(), 0;
  return 2;
}
