// trace.hip -- BVH2 nearest-hit / any-hit traversal for gfx950.
//
// Semantics follow BVH2CommonRT::BVH2TraverseC32 (core/BVH2CommonRT.cpp:49-141)
// step for step: start at the root's children, test both boxes of a pair,
// descend into the nearer hit child (the left one on equal entry distance,
// :106) and defer the other, intersect every triangle of a leaf with the
// reference's Moller-Trumbore (first strictly closer hit wins, :37), pop when
// a leaf is done or both children miss.  Box culling uses the current hit
// distance (:97-98).  A ray whose tFar is <= 0 is an any-hit query with
// tFar = -w that stops at its first hit (BVH4HalfRT.cpp:260-262, 82).
//
// Layout: NodePair (64 B, both children of one internal node) and TriPre
// (48 B, A / B-A / C-A / original id), both in HBM, and WideNode (128 B, two
// levels) for the four-lane walk; the stack of deferred children lives in LDS,
// interleaved by lane or ray (walk2.h).
//
// Execution: a persistent wave64 kernel.  Each wave keeps 64 rays in flight;
// when enough lanes have finished, the wave counts its idle lanes with one
// ballot, takes that many consecutive ray indices from a global queue with a
// single atomic and refills exactly those lanes (ballot-based compaction), so
// long rays never hold a wave of finished lanes.
//
// Nearest-hit keeps the reference's exact order: a lane that reaches a leaf
// intersects it before it tests any further node.  Any-hit only has to decide
// whether some triangle is hit, which does not depend on the order, so it
// traverses speculatively (Aila & Laine, "Understanding the Efficiency of Ray
// Traversal on GPUs", HPG 2009): a lane that has found a leaf parks it and
// keeps descending until all but a few lanes of the wave hold a leaf, then
// those lanes intersect their leaves together.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "eye.h"
#include "hrt_internal.h"
#include "walk2.h"

namespace hrt {
namespace {

constexpr int kWave = 64;
constexpr int kWavesPerBlock = 1;
constexpr int kTraceBlock = kWave * kWavesPerBlock;
static_assert(kWavesPerBlock == 1, "RayPool counts workgroups");
constexpr int kRefillAt = 16;  // refill when at least this many lanes are idle
constexpr uint32_t kClaim = 128;  // ray indices a wave claims from the queue at once
// One-ray-per-lane kernel: stack entries per lane in LDS.  With 16 (16 KB
// per 256-thread block) LDS allows 8 waves per SIMD and deeper entries, up to
// kWalkDepth, go to a per-lane global spill area; with kWalkDepth nothing
// spills but LDS allows 4 waves per SIMD.  The launcher takes the full LDS
// stack when its whole grid is resident at once (a small batch gains nothing
// from more waves and would pay for the spills), the short one otherwise.
constexpr int kSimpleLds = 16;
// Speculative any-hit leaves the node loop for the leaf phase once this many
// lanes or fewer still look for a leaf (and some lane holds one).
constexpr uint32_t kLeafPhaseAt = 8;

struct HitOutFull {  // CRT_Hit (CrossRT.h:20-27)
  float t;
  uint32_t prim, inst, geom;
  float coords[4];
};

__global__ void k_reset_counter(uint32_t* c) { *c = 0u; }

// Where a nearest-hit kernel's rays come from and its hits go.
//   RayBatch   rays and hit records of a batch in HBM
//   EyeFrame   a frame of hrt_eye_render: rays made in registers, the pixel's
//              colour written (0 on a miss, else palette[primId % size]).  One
//              launch instead of rays, trace and colours with 40 bytes a pixel
//              through a buffer allocated per frame: 512x512 frames of sphere,
//              hills with boxes and soup (100,000 triangles) 134, 253 and 308
//              us before the one-fetch walk, 87, 150 and 246 now; 64x64 109,
//              160 and 200, now 57, 86 and 105.
struct RayBatch {
  const Ray* __restrict__ rays;
  void* __restrict__ out;
  int format;
  uint2 ids;
  __device__ Ray ray(uint64_t i) const { return rays[i]; }
  __device__ void put(uint64_t i, const HitRec& h) const {
    if (format == kHitCompact) {
      static_cast<uint2*>(out)[i] = make_uint2(__float_as_uint(h.t), h.prim);
      return;
    }
    const bool hit = h.prim != kInvalid;
    float4* o4 = reinterpret_cast<float4*>(static_cast<HitOutFull*>(out) + i);
    o4[0] = make_float4(h.t, __uint_as_float(h.prim), __uint_as_float(hit ? ids.x : kInvalid),
                        __uint_as_float(hit ? ids.y : kInvalid));
    o4[1] = make_float4(h.u, h.v, 0.0f, 0.0f);
  }
};

struct EyeFrame {
  EyeCamera cam;
  EyePalette pal;
  uint32_t width, height;
  uint32_t* __restrict__ color;
  uint32_t group;  // rays per workgroup of the kernel
  __device__ uint2 pixel(uint32_t i) const { return xcd_stripe_pixel(i, width, height, group); }
  __device__ Ray ray(uint64_t i) const { return eye_ray(cam, pixel(uint32_t(i)), width, height); }
  __device__ void put(uint64_t i, const HitRec& h) const {
    const uint2 px = pixel(uint32_t(i));
    color[px.y * width + px.x] = h.prim == kInvalid ? 0u : pal.c[h.prim % pal.n];
  }
};

// The reference's order, one ray per lane (no refill): nearest hits, and the
// counting variant, whose counters are the reference's.
template <bool kForceAny, bool kStats, int kLds, class Tri, class Io>
__global__ __launch_bounds__(256) void k_trace_simple(const NodePair* __restrict__ pairs,
                                                      const TriPre* __restrict__ tris, Io io, uint64_t n,
                                                      uint32_t* __restrict__ stats, uint32_t* __restrict__ spill) {
  __shared__ uint32_t stack_mem[kLds * 256];
  const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  std::conditional_t<kLds == kWalkDepth, LdsStack<256>, ShortStack<kLds, 256>> stk = [&] {
    if constexpr (kLds == kWalkDepth) return LdsStack<256>(stack_mem + threadIdx.x);
    else return ShortStack<kLds, 256>{stack_mem + threadIdx.x, spill + i, gridDim.x * 256u};
  }();
  const Ray r = io.ray(i);
  const float3 o = make_float3(r.pos_near.x, r.pos_near.y, r.pos_near.z);
  const float3 d = make_float3(r.dir_far.x, r.dir_far.y, r.dir_far.z);
  const float tnear = r.pos_near.w;
  const bool any = kForceAny || (r.dir_far.w <= 0.0f);
  const float tfar = kForceAny ? fabsf(r.dir_far.w) : (any ? -r.dir_far.w : r.dir_far.w);
  const float3 inv = safe_inverse(d);
  const Tri tt(o, d);
  HitRec h;
  h.t = tfar;
  h.prim = kInvalid;
  h.u = 0.0f;
  h.v = 0.0f;
  uint32_t npairs = 0, ntests = 0;
  int top = 1;
  uint32_t cur = 0;
  stk.put(0, kInvalid, true);
  while (cur != kInvalid) {
    if (kStats) {
      npairs += (cur & kLeafBit) == 0;
      ntests += (cur & kLeafBit) != 0 && leaf_count(cur) != 0;
    }
    const bool leaf_done = walk_step(pairs, tris, tt, o, d, inv, tnear, h.t, stk, top, cur,
                                     [&h](float t, float u, float v, uint32_t prim) {
                                       if (t < h.t) h = HitRec{t, prim, u, v};
                                     });
    if (any && leaf_done && h.prim != kInvalid) break;
  }
  if (kStats) {
    stats[2 * i + 0] = npairs;
    stats[2 * i + 1] = ntests;
  }
  if constexpr (kForceAny) static_cast<uint8_t*>(io.out)[i] = (h.prim != kInvalid) ? 1 : 0;
  else io.put(i, h);
}

// Nearest hits in the reference's order, four lanes per ray (walk_quad_step),
// kQuadRays rays per workgroup.  On a tree whose WideNodes may not be walked
// the four lanes walk its pairs alike.
constexpr uint32_t kQuadRays = 64;
template <class Tri, class Io>
__global__ __launch_bounds__(256) void k_trace_quad(WalkNodes nodes, const TriPre* __restrict__ tris, Io io,
                                                    uint64_t n) {
  __shared__ uint32_t stack_mem[kWalkDepth * kQuadRays];
  const uint32_t l = threadIdx.x & 3u, q = threadIdx.x >> 2;
  const uint64_t i = uint64_t(blockIdx.x) * kQuadRays + q;
  if (i >= n) return;
  const LdsStack<int(kQuadRays)> stk(stack_mem + q);
  const Ray r = io.ray(i);
  const float3 o = make_float3(r.pos_near.x, r.pos_near.y, r.pos_near.z);
  const float3 d = make_float3(r.dir_far.x, r.dir_far.y, r.dir_far.z);
  const float tnear = r.pos_near.w;
  const bool any = r.dir_far.w <= 0.0f;
  const float3 inv = safe_inverse(d);
  const Tri tt(o, d);
  HitRec h{any ? -r.dir_far.w : r.dir_far.w, kInvalid, 0.0f, 0.0f};
  int top = 1;
  uint32_t cur = 0;
  stk.put(0, kInvalid, true);
  if (*nodes.differ == 0u) {
    while (cur != kInvalid) {
      const bool leaf_done = walk_quad_step(nodes.wide, tris, tt, l, o, d, inv, tnear, stk, top, cur, h);
      if (any && leaf_done && h.prim != kInvalid) break;
    }
  } else {
    while (cur != kInvalid) {
      const bool leaf_done = walk_step(nodes.pairs, tris, tt, o, d, inv, tnear, h.t, stk, top, cur,
                                       [&h](float t, float u, float v, uint32_t prim) {
                                         if (t < h.t) h = HitRec{t, prim, u, v};
                                       });
      if (any && leaf_done && h.prim != kInvalid) break;
    }
  }
  if (l == 0) io.put(i, h);
}

// Persistent wave64 traversal with ballot-based refill.
//   kForceAny: every ray is an any-hit query (hrt_trace_any)
//   kSpec:     speculative while-while traversal (any-hit only)
template <bool kForceAny, bool kSpec, class Tri = MtTest>
__global__ __launch_bounds__(kTraceBlock) void k_trace_persistent(const NodePair* __restrict__ pairs,
                                                                  const TriPre* __restrict__ tris,
                                                                  const Ray* __restrict__ rays, uint64_t n,
                                                                  void* out, int format, uint2 ids,
                                                                  uint32_t* __restrict__ queue,
                                                                  uint32_t* __restrict__ spill) {
  __shared__ uint32_t stack_mem[kShortStack * kTraceBlock];
  const uint32_t lanes = gridDim.x * kTraceBlock;
  const ShortStack<kShortStack, kTraceBlock> stk{stack_mem + threadIdx.x,
                                                 spill + blockIdx.x * kTraceBlock + threadIdx.x, lanes};

  // per-lane ray state
  bool active = false;
  uint64_t rid = 0;
  float3 o = make_float3(0.f, 0.f, 0.f), d = o, inv = o;
  float tnear = 0.f;
  bool any = kForceAny;
  Tri tt;
  HitRec h;
  h.t = 0.f;
  h.prim = kInvalid;
  h.u = h.v = 0.f;
  int top = 0;          // entries on the stack
  uint32_t cur = kInvalid;   // node pair to test next, a leaf, or kInvalid
  uint32_t leaf = 0;    // parked leaf (speculative any-hit), 0 = none
  RayPool pool(blockIdx.x, gridDim.x, n);  // ray indices claimed by this wave

  while (true) {
    // ---- refill idle lanes from the global queue -------------------------
    const uint64_t idle = __ballot(!active);
    const uint32_t nidle = __popcll(idle);
    if (!pool.drained() && (nidle >= kRefillAt || nidle == kWave)) {
      const uint64_t idx = pool.take<kClaim>(nidle, lanes_below(idle), queue, n);
      if (!active) {
        if (idx < n) {
          rid = idx;
          const Ray r = rays[idx];
          o = make_float3(r.pos_near.x, r.pos_near.y, r.pos_near.z);
          d = make_float3(r.dir_far.x, r.dir_far.y, r.dir_far.z);
          tnear = r.pos_near.w;
          any = kForceAny || (r.dir_far.w <= 0.0f);
          h.t = kForceAny ? fabsf(r.dir_far.w) : (any ? -r.dir_far.w : r.dir_far.w);
          h.prim = kInvalid;
          h.u = h.v = 0.f;
          inv = safe_inverse(d);
          tt = Tri(o, d);
          top = 0;
          cur = 0;
          leaf = 0;
          active = true;
        }
      }
    }
    if (__ballot(active) == 0) break;

    // ---- traverse until enough lanes are idle -----------------------------
    while (true) {
      bool done = false;
      if (kSpec) {
        // inner phase: lanes without a parked leaf search for one; lanes
        // holding one keep descending while their next node is internal
        while (true) {
          // park a leaf reached in `cur` (at most one per lane)
          if (active && leaf == 0 && (cur & kLeafBit) != 0 && cur != kInvalid) {
            leaf = cur;
            cur = (top > 0) ? stk.pop(top) : kInvalid;
          }
          const bool searching = active && leaf == 0 && (cur & kLeafBit) == 0;
          const uint32_t nsearch = __popcll(__ballot(searching));
          if (nsearch == 0 || (nsearch <= kLeafPhaseAt && __any(leaf != 0))) break;
          if (active && (cur & kLeafBit) == 0) {
            const float4* pp = reinterpret_cast<const float4*>(pairs + cur);
            const float4 lmin = pp[0], lmax = pp[1], rmin = pp[2], rmax = pp[3];
            const float2 t0 = tt.box(o, inv, lmin.x, lmin.y, lmin.z, lmax.x, lmax.y, lmax.z);
            const float2 t1 = tt.box(o, inv, rmin.x, rmin.y, rmin.z, rmax.x, rmax.y, rmax.z);
            const bool h0 = (t0.x <= t0.y) && (t0.y >= tnear) && (t0.x <= h.t);
            const bool h1 = (t1.x <= t1.y) && (t1.y >= tnear) && (t1.x <= h.t);
            const uint32_t c0 = __float_as_uint(lmin.w), c1 = __float_as_uint(rmin.w);
            if (h0 && h1) {
              const bool left_first = t0.x <= t1.x;
              cur = left_first ? c0 : c1;
              stk.push(top, left_first ? c1 : c0);
            } else if (h0 || h1) {
              cur = h0 ? c0 : c1;
            } else {
              cur = (top > 0) ? stk.pop(top) : kInvalid;
            }
          }
        }
        // leaf phase
        if (active && leaf != 0) {
          const uint32_t s = leaf_start(leaf), c = leaf_count(leaf);
          for (uint32_t k = s; k < s + c; k++) {
            if (tri_hit_before(tt, o, d, tnear, tris[k], h.t)) {  // any-hit: the first hit decides
              h.prim = 0u;
              break;
            }
          }
          leaf = 0;
        }
        done = active && (h.prim != kInvalid || (leaf == 0 && cur == kInvalid));
      } else {
        // one step in the reference's order: a pair or a leaf
        if (active) {
          if ((cur & kLeafBit) == 0) {
            const float4* pp = reinterpret_cast<const float4*>(pairs + cur);
            const float4 lmin = pp[0], lmax = pp[1], rmin = pp[2], rmax = pp[3];
            const float2 t0 = tt.box(o, inv, lmin.x, lmin.y, lmin.z, lmax.x, lmax.y, lmax.z);
            const float2 t1 = tt.box(o, inv, rmin.x, rmin.y, rmin.z, rmax.x, rmax.y, rmax.z);
            const bool h0 = (t0.x <= t0.y) && (t0.y >= tnear) && (t0.x <= h.t);
            const bool h1 = (t1.x <= t1.y) && (t1.y >= tnear) && (t1.x <= h.t);
            const uint32_t c0 = __float_as_uint(lmin.w), c1 = __float_as_uint(rmin.w);
            if (h0 && h1) {
              const bool left_first = t0.x <= t1.x;
              cur = left_first ? c0 : c1;
              stk.push(top, left_first ? c1 : c0);
            } else if (h0 || h1) {
              cur = h0 ? c0 : c1;
            } else {
              cur = (top > 0) ? stk.pop(top) : kInvalid;
            }
          } else if (cur != kInvalid) {
            const uint32_t s = leaf_start(cur), c = leaf_count(cur);
            for (uint32_t k = s; k < s + c; k++) tri_test(tt, o, d, tnear, tris[k], h);
            cur = (top > 0) ? stk.pop(top) : kInvalid;
          }
          done = (cur == kInvalid) || (any && h.prim != kInvalid);
        }
      }
      if (done) {
        if (kForceAny) {
          static_cast<uint8_t*>(out)[rid] = (h.prim != kInvalid) ? 1 : 0;
        } else if (format == kHitCompact) {
          static_cast<uint2*>(out)[rid] = make_uint2(__float_as_uint(h.t), h.prim);
        } else {
          const bool hit = h.prim != kInvalid;
          float4* o4 = reinterpret_cast<float4*>(static_cast<HitOutFull*>(out) + rid);
          o4[0] = make_float4(h.t, __uint_as_float(h.prim), __uint_as_float(hit ? ids.x : kInvalid),
                              __uint_as_float(hit ? ids.y : kInvalid));
          o4[1] = make_float4(h.u, h.v, 0.0f, 0.0f);
        }
        active = false;
      }
      const uint32_t nact = __popcll(__ballot(active));
      if (nact == 0 || (!pool.drained() && kWave - nact >= kRefillAt)) break;
    }
  }
}

template <bool kAny, bool kSpec, class Tri>
hipError_t launch_persistent(const Blas& b, const TraceArgs& a, hipStream_t stream) {
  const void* kfn = reinterpret_cast<const void*>(&k_trace_persistent<kAny, kSpec, Tri>);
  uint64_t want = (a.n + kTraceBlock - 1) / kTraceBlock;
  constexpr size_t kLaneWords = kStackDepth - kShortStack;
  uint64_t cap = resident_grid(kfn, kTraceBlock);
  if (a.workspace) cap = std::min<uint64_t>(cap, (a.workspace_words - 64) / (kTraceBlock * kLaneWords));
  const int grid = int(std::max<uint64_t>(1, std::min<uint64_t>(want, cap)));
  // queue counter + spill area for stack entries beyond the LDS part
  const size_t spill_words = size_t(grid) * kTraceBlock * kLaneWords;
  uint32_t* buf = a.workspace;
  hipError_t e = hipSuccess;
  if (!buf && (e = stream_malloc(&buf, sizeof(uint32_t) * (64 + spill_words), stream)) != hipSuccess) return e;
  k_reset_counter<<<1, 1, 0, stream>>>(buf);
  k_trace_persistent<kAny, kSpec, Tri><<<grid, kTraceBlock, 0, stream>>>(
      b.pairs, tri_records<Tri>(b), a.rays, a.n, a.out, a.format, make_uint2(a.inst_id, a.geom_id), buf, buf + 64);
  e = hipGetLastError();
  hipError_t f = a.workspace ? hipSuccess : hipFreeAsync(buf, stream);
  return e != hipSuccess ? e : f;
}

// Nearest hits of n rays in the reference's order.  Four lanes per ray while
// that fills at most half of the chip's waves (65,536 rays): the launch then lasts as long as its longest walks, which are shorter this
// way.  us a call on soup (400,000 triangles), hills with boxes (500,000) and
// sphere (80,000), random rays / camera, four lanes and one: 1,000 rays 121
// and 150 / 83 and 103, 74 and 98; 65,000 rays 202 and 229 / 107 and 145, 93
// and 113; 130,000 rays (every wave resident) 315 and 264 / 113 and 169, 87
// and 92; 262,000 rays 471 and 387 / 168 and 200.
template <class Tri, class Io>
hipError_t trace_nearest(const Blas& b, const Io& io, uint64_t n, hipStream_t stream) {
  const TriPre* tris = tri_records<Tri>(b);
  const WalkNodes nodes = walk_nodes(b);
  const uint64_t quads = (n + kQuadRays - 1) / kQuadRays;
  if (nodes.wide && 2 * quads <= resident_grid(reinterpret_cast<const void*>(&k_trace_quad<Tri, Io>), 256)) {
    Io qio = io;
    if constexpr (std::is_same<Io, EyeFrame>::value) qio.group = kQuadRays;
    k_trace_quad<Tri, Io><<<uint32_t(quads), 256, 0, stream>>>(nodes, tris, qio, n);
    return hipGetLastError();
  }
  // One ray per lane (rays that arrive in screen order stay coherent within a
  // wave, which a refilling kernel gives up).
  const uint32_t blocks = uint32_t((n + 255) / 256);
  if (blocks <= resident_grid(reinterpret_cast<const void*>(&k_trace_simple<false, false, kWalkDepth, Tri, Io>), 256)) {
    k_trace_simple<false, false, kWalkDepth, Tri, Io><<<blocks, 256, 0, stream>>>(b.pairs, tris, io, n, nullptr,
                                                                                  nullptr);
    return hipGetLastError();
  }
  uint32_t* spill = nullptr;
  hipError_t e = stream_malloc(&spill, sizeof(uint32_t) * size_t(blocks) * 256 * (kWalkDepth - kSimpleLds), stream);
  if (e != hipSuccess) return e;
  k_trace_simple<false, false, kSimpleLds, Tri, Io><<<blocks, 256, 0, stream>>>(b.pairs, tris, io, n, nullptr, spill);
  e = hipGetLastError();
  const hipError_t f = hipFreeAsync(spill, stream);
  return e != hipSuccess ? e : f;
}

template <class Tri>
hipError_t trace_blas_with(const Blas& b, const TraceArgs& a, hipStream_t stream) {
  if (a.anyhit && !a.stats) return launch_persistent<true, true, Tri>(b, a, stream);
  const RayBatch io{a.rays, a.out, a.format, make_uint2(a.inst_id, a.geom_id)};
  if (!a.stats) return trace_nearest<Tri>(b, io, a.n, stream);
  // the counting variant, on the pairs
  const TriPre* tris = tri_records<Tri>(b);
  const uint32_t blocks = uint32_t((a.n + 255) / 256);
  if (a.anyhit)
    k_trace_simple<true, true, kWalkDepth, Tri><<<blocks, 256, 0, stream>>>(b.pairs, tris, io, a.n, a.stats, nullptr);
  else
    k_trace_simple<false, true, kWalkDepth, Tri><<<blocks, 256, 0, stream>>>(b.pairs, tris, io, a.n, a.stats, nullptr);
  return hipGetLastError();
}

}  // namespace

void warm_bvh2_any_hit_launchers() {
  (void)resident_grid(reinterpret_cast<const void*>(&k_trace_persistent<true, true, MtTest>), kTraceBlock);
  (void)resident_grid(reinterpret_cast<const void*>(&k_trace_persistent<true, true, WtTest>), kTraceBlock);
}

uint32_t resident_grid(const void* kernel, int block) {
  struct Entry {
    int dev;
    const void* kernel;
    int block;
    uint32_t grid;
  };
  static std::mutex mu;
  static std::vector<Entry> cache;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 1024;
  {
    std::lock_guard<std::mutex> lock(mu);
    for (const Entry& e : cache)
      if (e.dev == dev && e.kernel == kernel && e.block == block) return e.grid;
  }
  int cus = 0, per_cu = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess || per_cu <= 0)
    per_cu = 1;
  const uint32_t grid = uint32_t(cus) * uint32_t(per_cu);
  std::lock_guard<std::mutex> lock(mu);
  cache.push_back(Entry{dev, kernel, block, grid});
  return grid;
}

hipError_t eye_frame(const Blas& b, bool watertight, const EyeCamera& cam, uint32_t width, uint32_t height,
                     const EyePalette& pal, uint32_t* out_color, hipStream_t stream) {
  const uint64_t n = uint64_t(width) * height;
  if (n == 0) return hipSuccess;
  if (watertight && !b.tris_wt) return hipErrorInvalidValue;
  const EyeFrame io{cam, pal, width, height, out_color, 256u};
  return watertight ? trace_nearest<WtTest>(b, io, n, stream) : trace_nearest<MtTest>(b, io, n, stream);
}

hipError_t trace_blas(const Blas& b, const TraceArgs& a, hipStream_t stream) {
  if (a.n == 0) return hipSuccess;
  if (a.watertight) {
    if (!b.tris_wt) return hipErrorInvalidValue;
    return trace_blas_with<WtTest>(b, a, stream);
  }
  return trace_blas_with<MtTest>(b, a, stream);
}

}  // namespace hrt
