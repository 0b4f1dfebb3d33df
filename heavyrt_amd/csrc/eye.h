// eye.h -- eye rays of a pinhole camera, shared by the kernel that writes them
// to HBM (eye.hip) and the nearest-hit kernels that make them in registers
// (trace.hip).  Both call the same functions, so a ray made in either place is
// the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>

#include "hrt_internal.h"

namespace hrt {

// Thread tid -> pixel: the inverse of SuperBlockIndex2DOpt for a width that
// is a multiple of 8.
__device__ inline uint2 superblock_pixel(uint32_t tid, uint32_t width) {
  const uint32_t wblocks_h = width >> 3;
  const uint32_t sb = tid >> 6, in_h = (tid >> 4) & 3u, in_b = tid & 15u;
  const uint32_t bx = (sb % wblocks_h) * 2u + (in_h & 1u);
  const uint32_t by = (sb / wblocks_h) * 2u + (in_h >> 1);
  return make_uint2(bx * 4u + (in_b & 3u), by * 4u + (in_b >> 2));
}

// Thread tid -> pixel in XCD stripes: the nearest-hit kernels run rays
// [group b, group b + group) as workgroup b, which the dispatcher hands to XCD
// b mod 8, so ray tid is given a pixel of the rows r with (r / 4) mod 8 equal
// to that XCD (4-row stripes, row order within each XCD's share).  Each XCD's
// L2 then serves one eighth of the screen while the stripes keep every XCD's
// share spread over the whole frame (contiguous eighths leave some XCDs the
// costly regions).  For a height that is a multiple of 32 and a width that
// is a multiple of group / 4 (each XCD's share is then a whole number of
// workgroups); rows otherwise.  A permutation of the pixels either way.
constexpr uint32_t kTraceGroup = 256;  // lanes per workgroup of the nearest-hit kernel
constexpr uint32_t kStripeRows = 4;
__device__ inline uint2 xcd_stripe_pixel(uint32_t tid, uint32_t width, uint32_t height, uint32_t group = kTraceGroup) {
  if (height % (kStripeRows * kXcds) != 0 || width % (group / kStripeRows) != 0)
    return make_uint2(tid % width, tid / width);
  const uint32_t b = tid / group, x = b % kXcds;
  const uint32_t k = (b / kXcds) * group + tid % group;  // place in XCD x's share
  const uint32_t rk = k / width;
  const uint32_t row = (rk / kStripeRows) * (kStripeRows * kXcds) + x * kStripeRows + rk % kStripeRows;
  return make_uint2(k % width, row);
}

// Thread tid -> pixel in superblock order, or in XCD stripes (kStripes).
template <bool kStripes>
__device__ inline uint2 thread_pixel(uint32_t tid, uint32_t width, uint32_t height) {
  return kStripes ? xcd_stripe_pixel(tid, width, height) : superblock_pixel(tid, width);
}

// LiteMath float4x4 * float4 with a column-major matrix: each row's four
// products summed left to right.
__device__ inline float4 mat_vec(const EyeCamera::Mat& m, float4 v) {
  const float* a = m.m;
  return make_float4(a[0] * v.x + a[4] * v.y + a[8] * v.z + a[12] * v.w,
                     a[1] * v.x + a[5] * v.y + a[9] * v.z + a[13] * v.w,
                     a[2] * v.x + a[6] * v.y + a[10] * v.z + a[14] * v.w,
                     a[3] * v.x + a[7] * v.y + a[11] * v.z + a[15] * v.w);
}

// normalize(u) = u / length(u), length = sqrt(dot(u, u))
__device__ inline float3 normalize3(float3 u) {
  const float len = sqrtf(u.x * u.x + u.y * u.y + u.z * u.z);
  return make_float3(u.x / len, u.y / len, u.z / len);
}

// EyeRayDirNormalized and transform_ray3f for the centre of pixel px.
__device__ inline Ray eye_ray(const EyeCamera& cam, uint2 px, uint32_t width, uint32_t height) {
  const float x = (float(px.x) + 0.5f) / float(width);
  const float y = (float(px.y) + 0.5f) / float(height);
  // EyeRayDirNormalized
  float4 pos = make_float4(2.0f * x - 1.0f, -2.0f * y + 1.0f, 0.0f, 1.0f);
  pos = mat_vec(cam.proj_inv, pos);
  const float w = pos.w;
  pos = make_float4(pos.x / w, pos.y / w, pos.z / w, pos.w / w);
  float3 dir = normalize3(make_float3(pos.x, pos.y, pos.z));
  // transform_ray3f from the camera origin
  const float3 o = make_float3(0.0f, 0.0f, 0.0f);
  const float4 p1 = mat_vec(cam.world_view_inv, make_float4(o.x, o.y, o.z, 1.0f));
  const float3 o2 = make_float3(o.x + 100.0f * dir.x, o.y + 100.0f * dir.y, o.z + 100.0f * dir.z);
  const float4 p2 = mat_vec(cam.world_view_inv, make_float4(o2.x, o2.y, o2.z, 1.0f));
  dir = normalize3(make_float3(p2.x - p1.x, p2.y - p1.y, p2.z - p1.z));
  Ray r;
  r.pos_near = make_float4(p1.x, p1.y, p1.z, 0.0f);
  r.dir_far = make_float4(dir.x, dir.y, dir.z, FLT_MAX);
  return r;
}

}  // namespace hrt
