/*
 * fno_device.h -- device helpers shared by the pass surrogate's kernels:
 * BF16 rounding, matrix-core operand types, GELU and its derivative.
 */
#ifndef MPC_FNO_DEVICE_H
#define MPC_FNO_DEVICE_H

#include <hip/hip_runtime.h>
#include <cmath>
#include "gelu_poly.h"

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

/* FP32 -> BF16, round to nearest even (v_cvt_pk_bf16_f32) */
__device__ __forceinline__ short to_bf16(float f) { return __builtin_bit_cast(short, (__bf16)f); }
__device__ __forceinline__ int bf16_pair(float lo, float hi) {
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    v2 p;
    p.x = (__bf16)lo;
    p.y = (__bf16)hi;
    return __builtin_bit_cast(int, p);
}
__device__ __forceinline__ float bf16_round(float x) { return (float)(__bf16)x; }
__device__ __forceinline__ bf16x8 bf16_octet(const float (&v)[8]) {
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (__bf16)v[j];
    return o;
}

/*
 * The training path's GELU.  The gradients of the high modes lie near the
 * BF16 operands' rounding noise, where one activation in 1e5 rounding the
 * other way moves them by 4e-3 (measured with another form), so its bits
 * stay as they are.
 */
__device__ __forceinline__ float gelu(float x) {
    return 0.5f * x * (1.f + erff(x * 0.70710678118654752f));
}
/*
 * The inference path's GELU(x) = max(x, 0) - |x| / 2 erfc(|x| / sqrt 2), with erfc(a / sqrt 2)
 * = 2^(-a M(a)) and M a polynomial (gelu_poly.h): no cancellation at negative x,
 * and its error is no larger than that of 0.5 x (1 + erff(x / sqrt 2)) over any
 * range of |x| (measured on the device in |x| / 2: at 0 < x < 0.1 3.1e-8 rms
 * against 4.3e-8, at 1 < x < 2 4.5e-8 against 6.5e-8, largest anywhere 1.3e-7
 * against 2.4e-7).  Takes about half the instructions: erff evaluates both of
 * its ranges in a mixed wave.
 * The clamp keeps +inf: there the power is 0 and inf * 0 would be NaN.  NaN stays NaN.
 */
__device__ __forceinline__ float gelu_fast(float x) {
    const float a = fabsf(x);
    const float e = __builtin_amdgcn_exp2f(-a * gelu_poly(a));
    return fmaf(-__builtin_amdgcn_fmed3f(0.5f * a, 0.f, 64.f), e, __builtin_amdgcn_fmed3f(x, 0.f, INFINITY));
}
/*
 * Buffer accesses: a wave-uniform base, a per-lane byte offset in one VGPR
 * and a wave-uniform byte offset in an SGPR, so rows at a constant stride need
 * no vector address arithmetic.  Word 3 of the descriptor: raw 32-bit
 * elements.  Offsets stay below 2^32 - 1 and inside the array the base points
 * into (the callers check sizes on the host).
 */
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t buf_of(const float *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, 0xffffffffu, 0x00020000);
}
__device__ __forceinline__ float buf_ld(rsrc_t r, unsigned lane_off, unsigned off) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, lane_off, off, 0));
}
__device__ __forceinline__ float2 buf_ld2(rsrc_t r, unsigned lane_off, unsigned off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, off, 0);
    return make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
}
__device__ __forceinline__ float4 buf_ld4(rsrc_t r, unsigned lane_off, unsigned off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0);
    return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}
__device__ __forceinline__ void buf_st(rsrc_t r, unsigned lane_off, unsigned off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, lane_off, off, 0);
}
__device__ __forceinline__ float gelu_d(float x) {
    return 0.5f * (1.f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

} // namespace

#endif
