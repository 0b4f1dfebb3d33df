// refit.h -- bottom-up box refit of Karras trees (lbvh.cpp:443-489 computes
// the same boxes with 32 serial sweeps; here each internal node is merged
// once, by the second of its two children to arrive).
//
// Three launches, none of which needs device-scope ordering inside a kernel:
//
//   k_refit_chunks  one workgroup per kRefitLeaves consecutive leaves.  A node
//                   whose leaf range lies inside the chunk only ever sees
//                   arrivals from this workgroup, so its arrival counter is an
//                   LDS word (index = the node's position, which is an end of
//                   its range) and the acquire/release is workgroup-scoped.
//                   An arrival at a node whose range crosses the chunk's edge
//                   is appended to its group's list instead.
//   k_refit_climb<false>  one workgroup per kRefitGroup chunks climbs from its list;
//                   an arrival at a node that crosses the group's edge goes to
//                   the tree's list.
//   k_refit_climb<true>  one workgroup climbs from that (several groups only).
//
// On gfx950 a device-scope release writes back the issuing XCD's L2 and the
// matching acquire invalidates it; with thousands of chunk seams those
// flushes, not the arithmetic, would set the refit's time.  The kernel
// boundaries between the launches are the only device-wide synchronisation.
//
// What bounds it is latency: a climb is a chain of dependent fetches, and an
// append to a list an atomic on the list's word (7 to 12 ns each, one after
// the other).  With chunks of 4,096 leaves and one workgroup for all that left
// them, each an atomic, 300,000 triangles took 46 + 31 us, 1.07 M 55 + 64 and
// 4.2 M 352 + 366; now a workgroup appends once and the three passes take 17 +
// 22 + 18, 30 + 24 + 22 and 191 + 35 + 87.
//
// The leaf boxes are written into their parents' pairs by the leaf pass
// before these kernels run.  Each thread of k_refit_chunks owns kRefitPer
// consecutive leaves and walks them as a small state machine (arrive, then
// either stop or merge and climb), so lanes stay busy instead of idling
// while a few of them climb.
#pragma once

#include "hrt_device.h"

namespace hrt {

constexpr uint32_t kRefitLeaves = 512;     // leaves per workgroup in k_refit_chunks
constexpr uint32_t kRefitGroup = 32;       // chunks per workgroup in k_refit_climb<false>
constexpr uint32_t kRefitThreads = 256;
constexpr uint32_t kRefitPer = kRefitLeaves / kRefitThreads;
constexpr uint32_t kRefitTopsThreads = 1024;
constexpr uint32_t kNoNode = 0xFFFFFFFFu;

// Internal nodes on one root-to-leaf path of a Karras tree over unique 30-bit
// codes: each level lengthens the common prefix, so at most 30; a chunk edge
// inside a tree is crossed by at most that many nodes, each of which takes
// at most two entries from below.
constexpr uint32_t kTopsPerEdge = 64;

// A group's list, and the groups of a tree of at most n leaves; the lists of
// all groups and then the tree's.
constexpr uint32_t kGroupCap = kTopsPerEdge * (kRefitGroup + 2);
inline uint32_t refit_chunks(uint64_t n) { return uint32_t((n + kRefitLeaves - 1) / kRefitLeaves); }
inline uint32_t refit_groups(uint64_t n) { return (refit_chunks(n) + kRefitGroup - 1) / kRefitGroup; }
inline uint32_t refit_top_cap(uint64_t n) { return kTopsPerEdge * (refit_groups(n) + 2); }
inline size_t refit_list_words(uint64_t n) { return size_t(refit_groups(n)) * kGroupCap + refit_top_cap(n); }

// Scene of element i: the last s with off[s] <= i (off holds S + 1 prefix
// sums; empty scenes are skipped because their offset equals the next one).
__device__ inline uint32_t seg_of(const uint32_t* __restrict__ off, uint32_t S, uint32_t i) {
  uint32_t lo = 0, hi = S;  // answer in [lo, hi)
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (off[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// seg_of for an index that grows with the lane (thread-per-element kernels):
// one search for the wave's first active lane, which the compiler keeps in
// scalar registers and the scalar cache, then a short walk per lane (a
// wave's elements span one or a few segments).
__device__ inline uint32_t seg_of_wave(const uint32_t* __restrict__ off, uint32_t S, uint32_t i) {
  uint32_t s = seg_of(off, S, __builtin_amdgcn_readfirstlane(i));
  while (s + 1 < S && off[s + 1] <= i) s++;
  return s;
}

// A tree's place in the (possibly concatenated) arrays: its index, its first
// and end global leaf, its first pair.  Leaves, parent_leaf and node ranges
// use global leaf numbers; pairs and parent_int are indexed pb + local node.
struct TreeLoc {
  uint32_t s, lb, le, pb;
};

// S trees side by side: leaf_off and tops_off hold S + 1 prefix sums,
// pair_off S + 1 first pairs.
struct ManyTrees {
  const uint32_t* leaf_off;
  const uint32_t* pair_off;
  const uint32_t* tops_off;
  uint32_t S;
  __device__ uint32_t leaves() const { return leaf_off[S]; }
  __device__ TreeLoc tree(uint32_t s) const { return {s, leaf_off[s], leaf_off[s + 1], pair_off[s]}; }
  __device__ TreeLoc find(uint32_t m) const { return tree(seg_of(leaf_off, S, m)); }
  // leaves are walked in increasing order: step to the tree holding m
  __device__ TreeLoc advance(TreeLoc t, uint32_t m) const {
    while (m >= t.le) t = tree(t.s + 1);
    return t;
  }
  __device__ uint32_t tops_base(uint32_t s) const { return tops_off[s]; }
  __device__ uint32_t tops_cap(uint32_t s) const { return tops_off[s + 1] - tops_off[s]; }
};

// Second arrival at pair p: the union of its two child boxes becomes p's box
// in its parent's pair, whose entry (pair << 1 | side) is pp.
__device__ inline void refit_merge_into(NodePair* pairs, uint32_t p, uint32_t pp) {
  const uint32_t* pw = reinterpret_cast<const uint32_t*>(pairs + p);
  const float3 l0 = make_float3(__uint_as_float(pw[0]), __uint_as_float(pw[1]), __uint_as_float(pw[2]));
  const float3 h0 = make_float3(__uint_as_float(pw[4]), __uint_as_float(pw[5]), __uint_as_float(pw[6]));
  const float3 l1 = make_float3(__uint_as_float(pw[8]), __uint_as_float(pw[9]), __uint_as_float(pw[10]));
  const float3 h1 = make_float3(__uint_as_float(pw[12]), __uint_as_float(pw[13]), __uint_as_float(pw[14]));
  const float3 ul = make_float3(fminf(l0.x, l1.x), fminf(l0.y, l1.y), fminf(l0.z, l1.z));
  const float3 uh = make_float3(fmaxf(h0.x, h1.x), fmaxf(h0.y, h1.y), fmaxf(h0.z, h1.z));
  store_box(pairs, pp >> 1, pp & 1u, ul, uh);
}

// Pass 1.  lists: kGroupCap pair indices per group; counts: per group and then
// the tree's, zero on entry; err[0] is set when a list would overflow (it
// cannot for trees over unique 30-bit codes).
static __global__ __launch_bounds__(kRefitThreads) void k_refit_chunks(const uint32_t* __restrict__ leaves, NodePair* pairs,
                                                                const uint32_t* __restrict__ parent_int,
                                                                const uint32_t* __restrict__ parent_leaf,
                                                                const uint2* __restrict__ range,
                                                                uint32_t* __restrict__ lists,
                                                                uint32_t* __restrict__ counts,
                                                                uint32_t* __restrict__ err) {
  __shared__ uint32_t arrived[kRefitLeaves];
  __shared__ uint32_t left[2 * kTopsPerEdge];  // arrivals that left the chunk (two edges)
  __shared__ uint32_t nleft, base;
  for (uint32_t k = threadIdx.x; k < kRefitLeaves; k += kRefitThreads) arrived[k] = 0u;
  if (threadIdx.x == 0) nleft = 0u;
  __syncthreads();
  const uint32_t total = *leaves;
  const uint32_t chunk_lo = blockIdx.x * kRefitLeaves, group = blockIdx.x / kRefitGroup;
  if (chunk_lo >= total || total == 1u) return;  // (a one-leaf tree has no internal node)
  const uint32_t chunk_hi = min(chunk_lo + kRefitLeaves, total) - 1u;
  uint32_t m = chunk_lo + threadIdx.x * kRefitPer;
  const uint32_t m_end = min(m + kRefitPer, chunk_hi + 1u);
  // p: pair of the next arrival; r, pp: its leaf range and its own parent
  // entry, loaded together one step ahead
  uint32_t p = kNoNode, pp = 0u;
  uint2 r = make_uint2(0u, 0u);
  auto next_leaf = [&]() {
    p = kNoNode;
    if (m < m_end) {
      p = parent_leaf[m] >> 1;
      r = range[p];
      pp = parent_int[p];  // unused (and unwritten) for the root
    }
  };
  next_leaf();
  while (p != kNoNode) {
    bool climb = false;
    if ((r.x < chunk_lo) | (r.y > chunk_hi)) {
      const uint32_t k = atomicAdd(&nleft, 1u);
      if (k < 2 * kTopsPerEdge) left[k] = p;
    } else {
      // releases this thread's box store into pair p, acquires the sibling's
      const uint32_t old =
          __hip_atomic_fetch_add(&arrived[p - chunk_lo], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
      climb = old != 0u && p != 0u;  // the root's own box is not stored
    }
    if (climb) {
      const uint32_t q = pp >> 1;
      const uint2 rq = range[q];
      const uint32_t pq = parent_int[q];
      refit_merge_into(pairs, p, pp);
      p = q;
      r = rq;
      pp = pq;
    } else {
      m++;
      next_leaf();
    }
  }
  __syncthreads();
  const uint32_t n = min(nleft, 2 * kTopsPerEdge);
  if (threadIdx.x == 0) {
    base = __hip_atomic_fetch_add(&counts[group], n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (nleft > n || base + n > kGroupCap) __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < n; k += kRefitThreads)
    if (base + k < kGroupCap) lists[group * kGroupCap + base + k] = left[k];
}

// Passes 2 (a workgroup per group, kTop false) and 3 (one workgroup for the
// tree).  arrive: per-pair counters, zero before pass 2.
template <bool kTop>
__global__ __launch_bounds__(kRefitTopsThreads) void k_refit_climb(NodePair* pairs,
                                                                   const uint32_t* __restrict__ parent_int,
                                                                   const uint2* __restrict__ range,
                                                                   uint32_t* __restrict__ lists,
                                                                   uint32_t* __restrict__ counts, uint32_t groups,
                                                                   uint32_t top_cap, uint32_t* arrive,
                                                                   uint32_t* __restrict__ err) {
  uint32_t* top = lists + size_t(groups) * kGroupCap;
  const uint32_t group = kTop ? groups : blockIdx.x;
  const uint32_t* list = kTop ? top : lists + size_t(group) * kGroupCap;
  const uint32_t n = min(counts[group], kTop ? top_cap : kGroupCap);
  const uint32_t lo = group * kRefitLeaves * kRefitGroup, hi = lo + kRefitLeaves * kRefitGroup - 1u;
  uint32_t i = threadIdx.x;
  uint32_t p = i < n ? list[i] : kNoNode;
  // r, pp: p's leaf range and parent entry (unwritten for the root), one step ahead
  uint2 r = make_uint2(0u, 0u);
  uint32_t pp = 0u;
  auto fetch = [&](uint32_t k) {
    if (!kTop) r = range[k];
    pp = parent_int[k];
  };
  if (p != kNoNode) fetch(p);
  while (p != kNoNode) {
    bool climb = false;
    if (!kTop && groups > 1u && ((r.x < lo) | (r.y > hi))) {
      const uint32_t k = __hip_atomic_fetch_add(&counts[groups], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (k < top_cap) top[k] = p;
      else __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      const uint32_t old = __hip_atomic_fetch_add(&arrive[p], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
      climb = old != 0u && p != 0u;
    }
    if (climb) {
      const uint32_t q = p, into = pp;
      p = pp >> 1;
      fetch(p);
      refit_merge_into(pairs, q, into);
    } else {
      i += kRefitTopsThreads;
      p = i < n ? list[i] : kNoNode;
      if (p != kNoNode) fetch(p);
    }
  }
}

// The three passes over a tree of at most n leaves; arrive has n words, counts
// refit_groups(n) + 1, all zero.
static inline hipError_t refit_boxes(const uint32_t* leaves, uint64_t n, NodePair* pairs, const uint32_t* parent_int,
                              const uint32_t* parent_leaf, const uint2* range, uint32_t* lists, uint32_t* counts,
                              uint32_t* arrive, uint32_t* err, hipStream_t s) {
  const uint32_t groups = refit_groups(n);
  k_refit_chunks<<<refit_chunks(n), kRefitThreads, 0, s>>>(leaves, pairs, parent_int, parent_leaf, range, lists, counts,
                                                          err);
  k_refit_climb<false><<<groups, kRefitTopsThreads, 0, s>>>(pairs, parent_int, range, lists, counts, groups,
                                                            refit_top_cap(n), arrive, err);
  if (groups > 1)
    k_refit_climb<true><<<1, kRefitTopsThreads, 0, s>>>(pairs, parent_int, range, lists, counts, groups,
                                                        refit_top_cap(n), arrive, err);
  return hipGetLastError();
}

}  // namespace hrt
