// trace_tlas.hip -- two-level (instanced) nearest-hit / any-hit traversal.
//
// Semantics follow BVH2CommonRT::RayQuery_NearestHit (core/BVH2CommonRT.cpp:
// 228-279): the ray is tested against the top-level tree over instance boxes;
// for every instance it reaches, the ray is moved into object space with the
// instance's inverse matrix (matmul4x3 / matmul3x3, raytrace_common.h:82-90;
// the direction is not renormalised, so t stays a world-space distance) and
// the object's BVH2 is walked exactly as the single-instance kernel walks it,
// carrying the running hit between instances.  Two deliberate differences
// from the reference:
//   * the reference collects instance leaves first (at most LBVH_MAXHITS =
//     32 of them, BVH2CommonRT.cpp:213-221) and uses a placeholder entry
//     distance; here the walk is interleaved, culls with the running hit
//     distance and has no limit on the number of instances a ray meets;
//   * on equal t across instances the smaller instance id wins, so the
//     answer does not depend on the shape of the top-level tree.
//
// Layout: the top-level tree is NodePair pairs over instance boxes (the same
// builder as the BLAS, fed with boxes), leaves index an InstDev array in leaf
// order (80 B each: inverse rows, the object's pairs and triangles, ids).
//
// Execution: a persistent wave64 kernel with ballot-based refill, one node
// pair, one triangle or one instance per lane per step (walk2.h), and a
// per-lane stack of kTwoLevelDepth entries: 16 in LDS, the rest in a per-lane
// global spill area.  That covers the deepest possible walk: the pending
// entries of the top-level tree and of one object's tree (at most kStackDepth
// each), the entry that ends the walk and the one that ends an object's.
// Bound by waits for fetches: 480,000 camera rays over 2,001 instances took
// 495 us with a pair and then a whole leaf per step, 426 with one fetch.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "hrt_internal.h"
#include "walk2.h"

namespace hrt {
namespace {

constexpr int kWave = 64;
constexpr int kBlock = kWave;
constexpr int kRefillAt = 16;
constexpr uint32_t kClaim = 128;  // ray indices a wave claims from the queue at once
constexpr int kTwoLevelDepth = 2 * kStackDepth + 3;
// Stack entry under an object's walk: the instance is done when it is popped.
// (No leaf has this value: its triangles would lie past the 24-bit range.)
constexpr uint32_t kInstanceDone = kInvalid - 1u;

__global__ void k_reset_counter(uint32_t* c) { *c = 0u; }

template <bool kForceAny, bool kStats>
__global__ __launch_bounds__(kBlock) void k_trace_two_level(const NodePair* __restrict__ tlas,
                                                            const InstDev* __restrict__ inst,
                                                            const Ray* __restrict__ rays, uint64_t n, void* out,
                                                            int format, uint32_t* __restrict__ stats,
                                                            uint32_t* __restrict__ queue,
                                                            uint32_t* __restrict__ spill) {
  __shared__ uint32_t stack_mem[kShortStack * kBlock];
  const uint32_t lanes = gridDim.x * kBlock;
  const ShortStack<kShortStack, kBlock> stk{stack_mem + threadIdx.x, spill + blockIdx.x * kBlock + threadIdx.x,
                                             lanes};

  bool active = false;
  uint64_t rid = 0;
  float3 wo = make_float3(0.f, 0.f, 0.f), wd = wo, winv = wo;  // world-space ray
  float3 o = wo, d = wo, inv = wo;                               // ray in the current tree's space
  float tnear = 0.f;
  bool any = kForceAny;
  HitRec h;
  h.t = 0.f;
  h.prim = kInvalid;
  h.u = h.v = 0.f;
  uint32_t h_inst = kInvalid, h_geom = kInvalid;
  const NodePair* P = tlas;  // tree being walked
  const TriPre* T = nullptr;
  bool in_blas = false;
  int top = 0;
  uint32_t k = 0, kend = 0;  // instances of the current top-level leaf
  uint32_t cur_inst = 0, cur_geom = 0;
  uint32_t cur = kInvalid;
  uint32_t npairs = 0, ntests = 0;
  RayPool pool(blockIdx.x, gridDim.x, n);  // ray indices claimed by this wave

  auto enter = [&](uint32_t slot) {
    const InstDev* I = inst + slot;
    const float4 r0 = I->inv_row[0], r1 = I->inv_row[1], r2 = I->inv_row[2];
    o = xform_point(r0, r1, r2, wo);
    d = xform_dir(r0, r1, r2, wd);
    inv = safe_inverse(d);
    P = I->pairs;
    T = I->tris;
    cur_inst = I->inst;
    cur_geom = I->geom;
    in_blas = true;
    stk.put(top, kInstanceDone, true);
    top++;
    cur = 0;
  };
  auto pop = [&]() { cur = stk.pop(top); };

  while (true) {
    const uint64_t idle = __ballot(!active);
    const uint32_t nidle = __popcll(idle);
    if (!pool.drained() && (nidle >= kRefillAt || nidle == kWave)) {
      const uint64_t idx = pool.take<kClaim>(nidle, lanes_below(idle), queue, n);
      if (!active) {
        if (idx < n) {
          rid = idx;
          const Ray r = rays[idx];
          wo = make_float3(r.pos_near.x, r.pos_near.y, r.pos_near.z);
          wd = make_float3(r.dir_far.x, r.dir_far.y, r.dir_far.z);
          winv = safe_inverse(wd);
          o = wo;
          d = wd;
          inv = winv;
          tnear = r.pos_near.w;
          any = kForceAny || (r.dir_far.w <= 0.0f);
          h.t = kForceAny ? fabsf(r.dir_far.w) : (any ? -r.dir_far.w : r.dir_far.w);
          h.prim = kInvalid;
          h.u = h.v = 0.f;
          h_inst = h_geom = kInvalid;
          P = tlas;
          in_blas = false;
          stk.put(0, kInvalid, true);
          top = 1;
          k = kend = 0;
          cur = 0;
          npairs = ntests = 0;
          active = true;
        }
      }
    }
    if (__ballot(active) == 0) break;

    while (true) {
      bool done = false;
      if (active) {
        bool leaf_done = false;
        if (in_blas || (cur & kLeafBit) == 0) {
          if (kStats) {
            npairs += (cur & kLeafBit) == 0;
            ntests += (cur & kLeafBit) != 0 && leaf_count(cur) != 0;
          }
          // inside one instance the first strictly closer hit wins; at equal
          // t an instance with a smaller id replaces one with a larger id
          leaf_done = walk_step(P, T, MtTest(), o, d, inv, tnear, h.t, stk, top, cur,
                                [&](float t, float u, float v, uint32_t prim) {
                                  if (t < h.t || (t == h.t && h.prim != kInvalid && cur_inst < h_inst)) {
                                    h = HitRec{t, prim, u, v};
                                    h_inst = cur_inst;
                                    h_geom = cur_geom;
                                  }
                                });
        } else {
          const uint32_t s = leaf_start(cur), c = leaf_count(cur);
          if (c > 0) {
            k = s;
            kend = s + c;
            enter(k);
          } else {
            pop();
          }
        }
        if (cur == kInstanceDone) {  // the next instance of the leaf, or on with the top-level tree
          if (++k < kend) {
            enter(k);
          } else {
            in_blas = false;
            P = tlas;
            o = wo;
            d = wd;
            inv = winv;
            pop();
          }
        }
        done = (cur == kInvalid) || (any && leaf_done && h.prim != kInvalid);
      }
      if (done) {
        const bool hit = h.prim != kInvalid;
        if (kStats) {
          stats[2 * rid + 0] = npairs;
          stats[2 * rid + 1] = ntests;
        }
        if (kForceAny) {
          static_cast<uint8_t*>(out)[rid] = hit ? 1 : 0;
        } else if (format == kHitCompact) {
          static_cast<uint2*>(out)[rid] = make_uint2(__float_as_uint(h.t), h.prim);
        } else {
          float4* o4 = reinterpret_cast<float4*>(static_cast<char*>(out) + 32 * rid);
          o4[0] = make_float4(h.t, __uint_as_float(h.prim), __uint_as_float(hit ? h_inst : kInvalid),
                              __uint_as_float(hit ? h_geom : kInvalid));
          o4[1] = make_float4(h.u, h.v, 0.0f, 0.0f);
        }
        active = false;
      }
      const uint32_t nact = __popcll(__ballot(active));
      if (nact == 0 || (!pool.drained() && kWave - nact >= kRefillAt)) break;
    }
  }
}

// Misses for every ray of a scene without instances.
__global__ __launch_bounds__(256) void k_misses(const Ray* __restrict__ rays, uint64_t n, void* out, int format,
                                                int force_any, uint32_t* __restrict__ stats) {
  const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  if (stats) {
    stats[2 * i + 0] = 0u;
    stats[2 * i + 1] = 0u;
  }
  if (force_any) {
    static_cast<uint8_t*>(out)[i] = 0;
    return;
  }
  const float w = rays[i].dir_far.w;
  const float t = (w <= 0.0f) ? -w : w;
  if (format == kHitCompact) {
    static_cast<uint2*>(out)[i] = make_uint2(__float_as_uint(t), kInvalid);
  } else {
    float4* o4 = reinterpret_cast<float4*>(static_cast<char*>(out) + 32 * i);
    o4[0] = make_float4(t, __uint_as_float(kInvalid), __uint_as_float(kInvalid), __uint_as_float(kInvalid));
    o4[1] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

template <bool kAny, bool kStats>
hipError_t launch(const Blas& tlas, const InstDev* inst, const TraceArgs& a, hipStream_t stream) {
  const void* kfn = reinterpret_cast<const void*>(&k_trace_two_level<kAny, kStats>);
  const uint64_t want = (a.n + kBlock - 1) / kBlock;
  const int grid = int(std::min<uint64_t>(want, uint64_t(resident_grid(kfn, kBlock))));
  const size_t spill_words = size_t(grid) * kBlock * (kTwoLevelDepth - kShortStack);
  uint32_t* buf = nullptr;
  hipError_t e = stream_malloc(&buf, sizeof(uint32_t) * (64 + spill_words), stream);
  if (e != hipSuccess) return e;
  k_reset_counter<<<1, 1, 0, stream>>>(buf);
  k_trace_two_level<kAny, kStats><<<grid, kBlock, 0, stream>>>(tlas.pairs, inst, a.rays, a.n, a.out, a.format,
                                                               a.stats, buf, buf + 64);
  e = hipGetLastError();
  hipError_t f = hipFreeAsync(buf, stream);
  return e != hipSuccess ? e : f;
}

}  // namespace

hipError_t trace_two_level(const Blas& tlas, const InstDev* inst, const TraceArgs& a, hipStream_t stream) {
  if (a.n == 0) return hipSuccess;
  if (tlas.ntris == 0 || !inst) {
    const uint32_t blocks = uint32_t((a.n + 255) / 256);
    k_misses<<<blocks, 256, 0, stream>>>(a.rays, a.n, a.out, a.format, a.anyhit, a.stats);
    return hipGetLastError();
  }
  if (a.anyhit) return a.stats ? launch<true, true>(tlas, inst, a, stream) : launch<true, false>(tlas, inst, a, stream);
  return a.stats ? launch<false, true>(tlas, inst, a, stream) : launch<false, false>(tlas, inst, a, stream);
}

}  // namespace hrt
