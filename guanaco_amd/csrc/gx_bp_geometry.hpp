// Geometry and staging helpers shared by the backprojection kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace gx {

// Per-tilt tables are read through the constant address space: uniform
// indices become scalar loads, independent of the workgroup barriers.
typedef const __attribute__((address_space(4))) float kfloat;
typedef const __attribute__((address_space(4))) int kint;

__device__ __forceinline__ float4 kload(const float4 *p, size_t i) {
  kfloat *q = (kfloat *)p + 4 * i;
  return make_float4(q[0], q[1], q[2], q[3]);
}
__device__ __forceinline__ int2 kload(const int2 *p, size_t i) {
  kint *q = (kint *)p + 2 * i;
  return make_int2(q[0], q[1]);
}
__device__ __forceinline__ float kload(const float *p, size_t i) {
  return ((kfloat *)p)[i];
}

// reconstructor.cpp:56-58: half-integer voxel centres (exact in float).
__device__ __forceinline__ float voxel_coord(int i, int n) {
  return (float)((double)i - 0.5 * (double)n + 0.5);
}

// reconstructor.cpp:59-60,76-79: detector position p = x c - z s + offset,
// i0 = floor(p - 0.5), t = (p - 0.5) - i0. EXACT: the reference's operation
// order; otherwise cf.z already holds offset - 1/2 and p is two fused
// multiply-adds.
template <bool EXACT>
__device__ __forceinline__ int tap_index(float x, float z, float4 cf,
                                         float &tt) {
  float p;
  if constexpr (EXACT) {
    p = x * cf.x - z * cf.y + cf.z;
    p = p - 0.5f;
  } else {
    p = fmaf(x, cf.x, fmaf(-z, cf.y, cf.z));
  }
  const float fi = floorf(p);
  tt = p - fi;
  return (int)fi;
}

// reconstructor.cpp:66-73: slab k = clamp(floor(h * dscale + doffset + 0.5)),
// h = -x s - z c. floor((double)d + 0.5) without FP64: round half to even,
// then move exact ties up.
__device__ __forceinline__ float slab_coord(float x, float z, float4 cf,
                                            float dscale, float doffset) {
  const float h = -x * cf.y - z * cf.x;
  return h * dscale + doffset;
}
__device__ __forceinline__ int slab_of(float x, float z, float4 cf,
                                       float dscale, float doffset, int ndf) {
  const float d = slab_coord(x, z, cf, dscale, doffset);
  float n = rintf(d);
  if (d - n == 0.5f) n += 1.0f;
  return min(max((int)n, 0), ndf - 1);
}

// One 16-byte raw buffer load per lane, written to LDS at dst + 16 lane
// instead of to registers (M0 holds dst). Out-of-range offsets write zeros.
__device__ __forceinline__ void load_to_lds16(__amdgpu_buffer_rsrc_t rs,
                                              uint4 *dst, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      rs, (__attribute__((address_space(3))) void *)dst, 16, off, 0, 0, 0);
}

// The same with 4 bytes per lane, written at dst + 4 lane.
__device__ __forceinline__ void load_to_lds4(__amdgpu_buffer_rsrc_t rs,
                                             uint4 *dst, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      rs, (__attribute__((address_space(3))) void *)dst, 4, off, 0, 0, 0);
}

}  // namespace gx
