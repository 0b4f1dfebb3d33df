// eye.hip -- the 01_eye_rays renderer's ray generation and colouring on the
// device.
//
// The reference renders one pixel per call (EyeRayCaster::CastRaySingle,
// examples/01_eye_rays/eye_ray.cpp:13-24): thread tid reads its pixel from
// m_packedXY, which kernel_PackXY (eye_ray.cpp:133-138) fills in
// SuperBlockIndex2DOpt order (eye_ray.cpp:114-131: 4x4 pixel blocks, 2x2
// blocks per 8x8 superblock, superblocks row by row), builds its ray with
// EyeRayDirNormalized + transform_ray3f (eye_ray.cpp:26-47,
// render_common.h:6-36) and colours the pixel from the hit's primId
// (eye_ray.cpp:50-75).  Here one lane makes one ray directly in HBM, in that
// same order for hrt_eye_make_rays (64 consecutive rays are one 8x8
// superblock).  The whole frame on the device (hrt_eye_render) only owes the
// image, so it makes, traces and colours its rays in the order that traces
// fastest: XCD stripes (xcd_stripe_pixel).  On the 512x512 eye frame the
// trace took 0.126 ms that way, 0.145 in row order, 0.164 in superblocks.  On
// a BVH2 the frame is one launch (trace.hip, EyeFrame); the kernels below are
// its parts for the other trees.
#include <hip/hip_runtime.h>

#include "eye.h"

namespace hrt {
namespace {

constexpr int kBlock = 256;

template <bool kStripes>
__global__ __launch_bounds__(kBlock) void k_eye_rays(EyeCamera cam, uint32_t width, uint32_t height,
                                                     Ray* __restrict__ out, uint32_t* __restrict__ packed_xy) {
  const uint32_t tid = blockIdx.x * kBlock + threadIdx.x;
  if (tid >= width * height) return;
  const uint2 px = thread_pixel<kStripes>(tid, width, height);
  out[tid] = eye_ray(cam, px, width, height);
  if (packed_xy) packed_xy[tid] = (px.y << 16) | px.x;
}

// out_color[y * width + x] = 0 on a miss, else palette[primId % size]
template <bool kStripes>
__global__ __launch_bounds__(kBlock) void k_eye_colors(const uint2* __restrict__ hits, uint32_t width,
                                                       uint32_t height, EyePalette pal,
                                                       uint32_t* __restrict__ out_color) {
  const uint32_t tid = blockIdx.x * kBlock + threadIdx.x;
  if (tid >= width * height) return;
  const uint2 px = thread_pixel<kStripes>(tid, width, height);
  const uint32_t prim = hits[tid].y;
  out_color[px.y * width + px.x] = prim == 0xFFFFFFFFu ? 0u : pal.c[prim % pal.n];
}

// The 02_rtao frame's colour (RTAO::kernel_AO2Color and floatToGrayRGBA,
// examples/02_rtao/rtao.cpp:15-24, 62-72): 0 where the eye ray missed, else
// the occluded fraction of the pixel's spp AO rays, raised to `power`,
// clamped to [0, 1] and truncated to a gray level with alpha 255.
__global__ __launch_bounds__(kBlock) void k_ao_colors(const uint2* __restrict__ hits,
                                                      const uint8_t* __restrict__ occluded, uint32_t width,
                                                      uint32_t height, uint32_t spp, float power,
                                                      uint32_t* __restrict__ out_color) {
  const uint32_t tid = blockIdx.x * kBlock + threadIdx.x;
  if (tid >= width * height) return;
  const uint2 px = superblock_pixel(tid, width);
  uint32_t c = 0u;
  if (hits[tid].y != 0xFFFFFFFFu) {
    uint32_t count = 0;
    for (uint32_t k = 0; k < spp; k++) count += occluded[uint64_t(tid) * spp + k] ? 1u : 0u;
    float v = float(count) * (1.0f / float(spp));
    if (power != 1.0f) v = powf(v, power);
    const uint32_t g = uint32_t(fminf(fmaxf(v, 0.0f), 1.0f) * 255.0f);
    c = g | (g << 8) | (g << 16) | (255u << 24);
  }
  out_color[px.y * width + px.x] = c;
}

}  // namespace

hipError_t ao_colors(const void* hits_compact, const uint8_t* occluded, uint32_t width, uint32_t height,
                     uint32_t spp, float power, uint32_t* out_color, hipStream_t stream) {
  const uint64_t n = uint64_t(width) * height;
  if (n == 0) return hipSuccess;
  k_ao_colors<<<uint32_t((n + kBlock - 1) / kBlock), kBlock, 0, stream>>>(
      static_cast<const uint2*>(hits_compact), occluded, width, height, spp, power, out_color);
  return hipGetLastError();
}

hipError_t eye_make_rays(const EyeCamera& cam, uint32_t width, uint32_t height, Ray* out, uint32_t* packed_xy,
                         hipStream_t stream, bool stripes) {
  const uint64_t n = uint64_t(width) * height;
  if (n == 0) return hipSuccess;
  const uint32_t blocks = uint32_t((n + kBlock - 1) / kBlock);
  if (stripes) k_eye_rays<true><<<blocks, kBlock, 0, stream>>>(cam, width, height, out, packed_xy);
  else k_eye_rays<false><<<blocks, kBlock, 0, stream>>>(cam, width, height, out, packed_xy);
  return hipGetLastError();
}

hipError_t eye_colors(const void* hits_compact, uint32_t width, uint32_t height, const EyePalette& pal,
                      uint32_t* out_color, hipStream_t stream, bool stripes) {
  const uint64_t n = uint64_t(width) * height;
  if (n == 0) return hipSuccess;
  const uint32_t blocks = uint32_t((n + kBlock - 1) / kBlock);
  const uint2* hits = static_cast<const uint2*>(hits_compact);
  if (stripes) k_eye_colors<true><<<blocks, kBlock, 0, stream>>>(hits, width, height, pal, out_color);
  else k_eye_colors<false><<<blocks, kBlock, 0, stream>>>(hits, width, height, pal, out_color);
  return hipGetLastError();
}

}  // namespace hrt
