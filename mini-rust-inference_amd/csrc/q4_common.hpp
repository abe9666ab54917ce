// q4_common.hpp — the exact bf16 forms of f32 activations and Q4_0 quants
// that the matrix-core kernels of matmul_q4_0_dequant multiply.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace mri {

// An f32 value is exactly the sum of three bf16 values: its leading 8
// significand bits, the next 8 and the last 8, each cut off (not rounded)
// from what the ones before leave, down to 2^-133, a bf16's last bit.  cut() is
// the part a bf16 holds; top16() stores the parts of two values as a bf16 pair
// (a low, b high).  rest() is 2^64 times what the three leave of a value (its
// bits below 2^-133), rest_scale() the block scale that undoes the factor.
__device__ inline float q4_cut(float v) {
    return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u);
}
__device__ inline unsigned q4_top16(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ inline float q4_rest(float v) {
    v -= q4_cut(v);
    v -= q4_cut(v);
    return (v - q4_cut(v)) * 0x1p64f;
}
__device__ inline float q4_rest_scale(float d) {
    return fabsf(d) < INFINITY ? d * 0x1p-64f : 0.0f;
}

// The quant (nibble - 8) of the nibble at bit P <= 12 of w, exactly: the
// nibble placed in the significand of 2^(23 - P) counts units of 1.
template <int P>
__device__ inline float q4_quant(unsigned w) {
    constexpr unsigned one = (unsigned)(127 + 23 - P) << 23;
    constexpr float base = (float)(1u << (23 - P)) + 8.0f;
    return __uint_as_float((w & (0xFu << P)) | one) - base;
}
// The eight quants of four bytes: l[i] of the low nibble of byte i, h[i] of
// the high one.
__device__ inline void q4_quants(unsigned w, float (&l)[4], float (&h)[4]) {
    const unsigned v = w >> 16;
    l[0] = q4_quant<0>(w), h[0] = q4_quant<4>(w), l[1] = q4_quant<8>(w), h[1] = q4_quant<12>(w);
    l[2] = q4_quant<0>(v), h[2] = q4_quant<4>(v), l[3] = q4_quant<8>(v), h[3] = q4_quant<12>(v);
}

// Workgroups of one launch, a multiple of 8: HIP takes fewer than 2^32 threads
// in a grid dimension, which 2^27 channels exceed.  More take more launches.
inline size_t q4_max_grid(size_t threads) { return 0xFFFFFFFFull / threads / 8 * 8; }

}  // namespace mri
