// wave_ops.h -- device helpers shared by the kernels: 64-lane reductions by
// DPP lane moves, single-instruction floor, the XCD-aware block order, and
// correctly rounded sqrt / division without the compiler's special cases.
#pragma once

#include <hip/hip_runtime.h>

namespace fct {

// Lane move; rows outside ROW_MASK are left unspecified (the reductions
// below only read lane 63, whose inputs are always in enabled rows).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp(int v) {
  return __builtin_amdgcn_mov_dpp(v, CTRL, ROW_MASK, 0xF, true);
}

// Order-preserving map of a float's bits to a signed int (negative floats get
// their magnitude bits flipped); the map is its own inverse.  Integer min /
// max fuse with the DPP lane moves, one instruction per step.
__device__ __forceinline__ int fkey(float x) {
  const int b = __float_as_int(x);
  return b ^ ((b >> 31) & 0x7FFFFFFF);
}
__device__ __forceinline__ float fkey_inv(int k) {
  return __int_as_float(k ^ ((k >> 31) & 0x7FFFFFFF));
}

// Wave-wide min / max (all 64 lanes must be active), result uniform.
__device__ __forceinline__ int wave_min_i(int v) {
  v = min(v, dpp<0xB1, 0xF>(v));    // quad_perm [1,0,3,2]
  v = min(v, dpp<0x4E, 0xF>(v));    // quad_perm [2,3,0,1]
  v = min(v, dpp<0x141, 0xF>(v));   // row_half_mirror
  v = min(v, dpp<0x140, 0xF>(v));   // row_mirror
  v = min(v, dpp<0x142, 0xA>(v));   // row_bcast:15
  v = min(v, dpp<0x143, 0xC>(v));   // row_bcast:31
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max_i(int v) {
  v = max(v, dpp<0xB1, 0xF>(v));
  v = max(v, dpp<0x4E, 0xF>(v));
  v = max(v, dpp<0x141, 0xF>(v));
  v = max(v, dpp<0x140, 0xF>(v));
  v = max(v, dpp<0x142, 0xA>(v));
  v = max(v, dpp<0x143, 0xC>(v));
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ float wave_min(float x) { return fkey_inv(wave_min_i(fkey(x))); }
__device__ __forceinline__ float wave_max(float x) { return fkey_inv(wave_max_i(fkey(x))); }

// Logical block of launch block b out of nb, such that each XCD (block b
// runs on XCD b % 8) takes one contiguous range of logical blocks.
__device__ __forceinline__ int xcd_block(int b, int nb) {
  const int x = b & 7, i = b >> 3;
  const int q = nb >> 3, r = nb & 7;
  return x * q + min(x, r) + i;
}

// Read-only table entry at a wave-uniform address, loaded through the
// constant address space so it becomes a scalar load into SGPRs even where
// the kernel also stores to global memory (the persistent batch loop).
template <class T>
__device__ __forceinline__ T ld_uniform(const T* p) {
  return *(const __attribute__((address_space(4))) T*)p;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ld_uniform4(const float4* p) {
  const f32x4 v = *(const __attribute__((address_space(4))) f32x4*)p;
  return make_float4(v.x, v.y, v.z, v.w);
}

// floor(x) as an int in one instruction (hipcc emits v_floor + v_cvt for
// (int)floorf(x)); same value for every finite x in int range.
__device__ __forceinline__ int floor_int(float x) {
  int r;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// sqrt(x) correctly rounded, as sqrtf, for x >= 2^-96 (R^2 - p^2 is of the
// order of R^2): the hardware square root (within 1 ulp) moved to
// its neighbour below or above when the residual x - s' s of that neighbour
// says the true root lies beyond it.  sqrtf's expansion adds a rescaling of
// tiny inputs and the zero / infinity cases, which cannot occur here.
__device__ __forceinline__ float sqrt_rn_large(float x) {
  const float s = __builtin_amdgcn_sqrtf(x);
  const float sdn = __int_as_float(__float_as_int(s) - 1);
  const float sup = __int_as_float(__float_as_int(s) + 1);
  float r = fmaf(-sdn, s, x) <= 0.0f ? sdn : s;
  r = fmaf(-sup, s, x) > 0.0f ? sup : r;
  return r;
}

// n / d correctly rounded, as the IEEE division, for operands far from the
// range limits (here n = hr < 2^15 and d = lt, a cone length of millimetres
// times tan(cone / 2)): the hardware reciprocal refined once, the quotient
// corrected twice by its exact residual -- the division's own sequence
// without its operand scaling and special-case fix-up, identities for such
// operands.
__device__ __forceinline__ float div_rn_normal(float n, float d) {
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  float q = n * r;
  q = fmaf(fmaf(-d, q, n), r, q);
  return fmaf(fmaf(-d, q, n), r, q);
}

}  // namespace fct
