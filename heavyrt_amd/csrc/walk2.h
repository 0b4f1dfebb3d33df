// walk2.h -- one step of a nearest-hit walk in the reference's BVH2 order,
// shared by the nearest-hit kernels.
//
// A lane's place in the walk is one reference: an internal node, or what is
// left of a leaf (kLeafBit, triangles left, next triangle).  What bounds these
// walks differs with the size of the launch, so there are two forms.
//
// walk_step: a ray per lane, on node pairs, for launches that fill the chip.
// Those are bound by the texture addresser (a lane's four 16-byte loads from a
// line of its own take a cycle each: 82 % busy on a million bounced rays) and
// by VALU issue (78 %).  A step tests one pair or ONE triangle, and both kinds
// of lanes fetch before the code splits; with a leaf loop a wave whose lanes
// are at different places waits for a pair and then again for every triangle
// of its longest leaf.  Waits per 64-ray wave, counted in lock step on the CPU
// (pair and leaf loop / pair or triangle a step): 1024x1024 primaries over the
// 1.07 M-triangle scene 152 / 106; incoherent rays in a 500,000-triangle soup
// 444 / 266.
//
// walk_quad_step: a ray per four lanes, on WideNodes, for launches that leave
// the chip idle.  Those last as long as their longest walk, a chain of steps
// of one fetch and its arithmetic each.  A step takes two levels: lane l holds
// the box of grandchild l, the children's boxes are unions over lane pairs,
// and the four lanes' fetches are one coalesced 128-byte record, so a step is
// 2 loads and about a third of the instructions of two pair steps.
#pragma once

#include <hip/hip_runtime.h>

#include "hrt_device.h"
#include "quad.h"

namespace hrt {

__device__ inline bool walk_hit(float t0, float t1, float tnear, float tmax) {
  return bool(int(t0 <= t1) & int(t1 >= tnear) & int(t0 <= tmax));  // no branches
}

// One step of a lane at `cur` (not kInvalid): the pair's or the triangle's
// test, then the next reference in the reference's order -- the nearer hit
// child (the left one on equal entry distance, BVH2CommonRT.cpp:97-110) with
// the other one deferred, the leaf's next triangle, or the deferred entry on
// top of the stack.  The stack's entry 0 is kInvalid, so a walk that runs out
// of entries ends by itself; the top entry is read before it is known to be
// needed and the deferred child is stored whether or not it counts (a slot at
// top holds nothing), which leaves no branch but the one between pairs and
// triangles.  accept(t, u, v, prim) is the hit rule.  Returns true for a lane
// that has just finished a leaf.
// The empty asm statements keep each side's loads together before its
// arithmetic (the compiler sinks them to their first uses otherwise).
template <class Tri, class Stack, class Accept>
__device__ inline bool walk_step(const NodePair* __restrict__ P, const TriPre* __restrict__ T, const Tri& tt, float3 o,
                                 float3 d, float3 inv, float tnear, float tmax, const Stack& stk, int& top,
                                 uint32_t& cur, Accept&& accept) {
  const bool leaf = int32_t(cur) < 0;
  // indices are below 2^24, so the offset fits 32 bits
  const uint32_t off = __umul24(cur & kStartMask, leaf ? uint32_t(sizeof(TriPre)) : uint32_t(sizeof(NodePair)));
  const char* p = (leaf ? reinterpret_cast<const char*>(T) : reinterpret_cast<const char*>(P)) + off;
  walk_f4 q0 = *reinterpret_cast<const walk_f4*>(p);
  walk_f4 q1 = *reinterpret_cast<const walk_f4*>(p + 16);
  walk_f4 q2 = *reinterpret_cast<const walk_f4*>(p + 32);
  const uint32_t peeked = stk.peek(top);
  bool pop;
  if (!leaf) {
    walk_f4 q3 = *reinterpret_cast<const walk_f4*>(p + 48);
    asm volatile("" : "+v"(q0), "+v"(q1), "+v"(q2), "+v"(q3));
    const float2 t0 = tt.box(o, inv, q0.x, q0.y, q0.z, q1.x, q1.y, q1.z);
    const float2 t1 = tt.box(o, inv, q2.x, q2.y, q2.z, q3.x, q3.y, q3.z);
    const bool h0 = walk_hit(t0.x, t0.y, tnear, tmax), h1 = walk_hit(t1.x, t1.y, tnear, tmax);
    const uint32_t c0 = __float_as_uint(q0.w), c1 = __float_as_uint(q2.w);
    const bool both = h0 && h1, left = h0 && !(h1 && t1.x < t0.x);
    stk.put(top, left ? c1 : c0, both);
    cur = left ? c0 : c1;
    top += int(both);
    pop = !h0 && !h1;
  } else {
    asm volatile("" : "+v"(q0), "+v"(q1), "+v"(q2));
    float t, u, v;
    if (tt.eval(o, d, tnear, walk_triangle(q0, q1, q2), t, u, v) && leaf_count(cur) != 0u)
      accept(t, u, v, __float_as_uint(q0.w));
    pop = leaf_count(cur) <= 1u;
    cur = cur - (1u << 24) + 1u;
  }
  if (pop) {
    cur = stk.pop_peeked(top, peeked);
    top--;
  }
  return leaf && pop;
}

// Entry and exit of the union of this lane's box and lane ^ 1's, from their
// distances per axis.  In asm because the compiler quiets (v_max x, x) every
// operand that comes through DPP or asm, 14 instructions more; a DPP source
// must be two wait states old (s_nop 1).
__device__ inline void quad_union(float nx, float ny, float nz, float fx, float fy, float fz, float& entry,
                                  float& exit) {
  float t0, t1, t2;
  asm("s_nop 1\n\t"
      "v_min_f32_dpp %2, %5, %5 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_min_f32_dpp %3, %6, %6 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_min_f32_dpp %4, %7, %7 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_max3_f32 %0, %2, %3, %4\n\t"
      "v_max_f32_dpp %2, %8, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_max_f32_dpp %3, %9, %9 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_max_f32_dpp %4, %10, %10 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_min3_f32 %1, %2, %3, %4"
      : "=&v"(entry), "=&v"(exit), "=&v"(t0), "=&v"(t1), "=&v"(t2)
      : "v"(nx), "v"(ny), "v"(nz), "v"(fx), "v"(fy), "v"(fz));
}

// One step of four lanes (lane & 3 = l) that hold one ray's state alike: two
// levels of the walk, or up to four triangles of a leaf.  The distances to a
// child's planes are the least (entry) and greatest (exit) of its children's,
// exactly, because rounding is monotonic; k_wide_nodes finds the trees where a
// stored child box is not the union of its children's, and they are walked on
// their pairs.  Both levels use the same hit distance, as the reference's two
// steps do, since no triangle lies between them.  Returns true when the ray
// has just finished a leaf.
template <class Tri, class Stack>
__device__ inline bool walk_quad_step(const WideNode* __restrict__ W, const TriPre* __restrict__ T, const Tri& tt,
                                      uint32_t l, float3 o, float3 d, float3 inv, float tnear, const Stack& stk,
                                      int& top, uint32_t& cur, HitRec& h) {
  const uint32_t popped = stk.pop_peeked(top, stk.peek(top));
  if (int32_t(cur) >= 0) {
    const walk_f4* p = reinterpret_cast<const walk_f4*>(W + cur) + 2 * l;
    walk_f4 lo = p[0], hi = p[1];
    asm volatile("" : "+v"(lo), "+v"(hi));
    float a, b, ca, cb;  // entry and exit of this lane's grandchild and of its child
    if constexpr (Tri::kRobustBoxes) {
      // a parallel axis is decided by the planes, not by distances: the
      // child's box itself is needed
      const float2 t = tt.box(o, inv, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z);
      const float2 c = tt.box(o, inv, fminf(lo.x, quad_x1(lo.x)), fminf(lo.y, quad_x1(lo.y)),
                              fminf(lo.z, quad_x1(lo.z)), fmaxf(hi.x, quad_x1(hi.x)), fmaxf(hi.y, quad_x1(hi.y)),
                              fmaxf(hi.z, quad_x1(hi.z)));
      a = t.x, b = t.y, ca = c.x, cb = c.y;
    } else {
      // the slab test (hrt_device.h), its per-axis distances kept for the unions
      const float x0 = inv.x * (lo.x - o.x), x1 = inv.x * (hi.x - o.x);
      const float y0 = inv.y * (lo.y - o.y), y1 = inv.y * (hi.y - o.y);
      const float z0 = inv.z * (lo.z - o.z), z1 = inv.z * (hi.z - o.z);
      const float nx = fminf(x0, x1), fx = fmaxf(x0, x1);
      const float ny = fminf(y0, y1), fy = fmaxf(y0, y1);
      const float nz = fminf(z0, z1), fz = fmaxf(z0, z1);
      a = fmaxf(fmaxf(nx, ny), nz);
      b = fminf(fminf(fx, fy), fz);
      quad_union(nx, ny, nz, fx, fy, fz, ca, cb);
    }
    const uint32_t ref = __float_as_uint(lo.w), child = __float_as_uint(hi.w);
    // the children: the nearer one is walked, the left one on equal entry
    // (an entry of NaN stands for a miss: it compares false)
    const float kMiss = __builtin_nanf("");
    const bool hc = walk_hit(ca, cb, tnear, h.t);
    const float e = hc ? ca : kMiss, oe = quad_x2(e);
    const bool nearer = hc & !((oe < e) | ((oe == e) & ((l & 2u) != 0u)));
    // the nearer child's children, likewise
    const bool hg = nearer & (ref != kInvalid) & walk_hit(a, b, tnear, h.t);
    const float eg = hg ? a : kMiss, og = quad_x1(eg);
    const bool first = hg & !((og < eg) | ((og == eg) & ((l & 1u) != 0u)));
    // references are never 0: the root is nobody's child, a leaf has kLeafBit
    const uint32_t next = quad_or(first ? ref : 0u);
    const uint32_t far_grand = quad_or((hg & !first) ? ref : 0u);
    uint32_t far_child = (hc & !nearer) ? child : 0u;
    far_child |= quad_x2(far_child);
    const bool on = next != 0u, deferred = far_child != 0u, deferred2 = far_grand != 0u;
    cur = on ? next : (deferred ? far_child : popped);
    stk.put(top, far_child, on & deferred);
    top += int(on & deferred);
    stk.put(top, far_grand, deferred2);
    top += int(deferred2) - int(!(on | deferred));
    return false;
  }
  const uint32_t count = leaf_count(cur);
  quad_triangles(T, l, leaf_start(cur), count, tt, o, d, tnear, h,
                 [](float t, uint32_t, const HitRec& h0) { return t < h0.t; });
  const bool last = count <= 4u;
  cur = last ? popped : cur - (4u << 24) + 4u;
  top -= int(last);
  return last;
}

}  // namespace hrt
