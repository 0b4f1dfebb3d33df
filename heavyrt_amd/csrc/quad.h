// quad.h -- what the kernels share that give one ray to four lanes: exchanges
// within a group of four lanes (lane & 3 = l) and the test of up to four
// triangles of a leaf at once.  The four lanes hold their ray's state alike, so
// a group is active or idle as a whole and every exchange reads active lanes.
#pragma once

#include <hip/hip_runtime.h>

#include "hrt_device.h"

namespace hrt {

typedef float walk_f4 __attribute__((ext_vector_type(4)));

__device__ inline TriPre walk_triangle(walk_f4 q0, walk_f4 q1, walk_f4 q2) {
  return TriPre{make_float4(q0.x, q0.y, q0.z, q0.w), make_float4(q1.x, q1.y, q1.z, 0.0f),
                make_float4(q2.x, q2.y, q2.z, 0.0f)};
}

// DPP quad_perm controls: lane i of the group reads the lane at place i.
constexpr int quad_perm(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }
template <int kPerm>
__device__ inline uint32_t quad_read(uint32_t v) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), kPerm, 0xF, 0xF, true));
}
template <int kPerm>
__device__ inline float quad_read(float v) {
  return __uint_as_float(quad_read<kPerm>(__float_as_uint(v)));
}
// The value of lane l ^ 1, of lane l ^ 2, and the four lanes' values or-ed.
template <class V>
__device__ inline V quad_x1(V v) { return quad_read<quad_perm(1, 0, 3, 2)>(v); }
template <class V>
__device__ inline V quad_x2(V v) { return quad_read<quad_perm(2, 3, 0, 1)>(v); }
__device__ inline uint32_t quad_or(uint32_t v) {
  v |= quad_x1(v);
  return v | quad_x2(v);
}

// Lane l tests triangle start + l of a leaf with `count` triangles left (lanes
// past the fourth wait for the next call).  accept(t, prim, h) filters the
// candidates against the hit so far; the lowest lane of the nearest ones
// becomes the hit (kFirst: the lowest lane of all of them), which is what
// testing them one after the other leaves.  Returns whether one did.
template <bool kFirst = false, bool kPrimTies = false, class Tri, class Accept>
__device__ inline bool quad_triangles(const TriPre* __restrict__ T, uint32_t l, uint32_t start, uint32_t count,
                                      const Tri& tt, float3 o, float3 d, float tnear, HitRec& h, Accept&& accept) {
  float t = 0.0f, u = 0.0f, v = 0.0f;
  uint32_t prim = kInvalid;
  if (l < count) {
    const walk_f4* p = reinterpret_cast<const walk_f4*>(T + start + l);
    walk_f4 q0 = p[0], q1 = p[1], q2 = p[2];
    asm volatile("" : "+v"(q0), "+v"(q1), "+v"(q2));
    if (tt.eval(o, d, tnear, walk_triangle(q0, q1, q2), t, u, v) && accept(t, __float_as_uint(q0.w), h))
      prim = __float_as_uint(q0.w);
  }
  uint32_t w;  // the lanes that could be the hit
  if constexpr (kFirst) {
    w = quad_or(prim != kInvalid ? 1u << l : 0u);
  } else {
    const float tc = prim != kInvalid ? t : __builtin_inff();
    float m = fminf(tc, quad_x1(tc));
    m = fminf(m, quad_x2(m));
    uint32_t near = prim != kInvalid && tc == m ? prim : kInvalid;
    if constexpr (kPrimTies) {  // the smallest id of the nearest ones
      uint32_t least = near < quad_x1(near) ? near : quad_x1(near);
      least = least < quad_x2(least) ? least : quad_x2(least);
      if (near != least) near = kInvalid;
    }
    w = quad_or(near != kInvalid ? 1u << l : 0u);
  }
  if (w == 0u) return false;
  const bool mine = (w & (0u - w)) == (1u << l);
  h.t = __uint_as_float(quad_or(mine ? __float_as_uint(t) : 0u));  // not the minimum: +0 and -0 are equal
  h.prim = quad_or(mine ? prim : 0u);
  h.u = __uint_as_float(quad_or(mine ? __float_as_uint(u) : 0u));
  h.v = __uint_as_float(quad_or(mine ? __float_as_uint(v) : 0u));
  return true;
}

}  // namespace hrt
