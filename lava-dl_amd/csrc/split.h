// A float32 as the sum of three bfloat16 numbers, the operands of v_mfma_f32_16x16x32_bf16: each part is the rounding
// to nearest of what the parts before it leave (|second| <= 2^-9, |third| <= 2^-18 of the value, what the three leave
// out <= 2^-27).  The products of parts are exact in float32; of two split factors the products part i x part j with
// i + j <= 2 are taken, what is left out is below 2^-26 of the product.
//   A value that is not finite leaves a NaN (so does a finite one beyond the largest bfloat16, 3.3895e38): callers
// either treat it (conv.hip) or recognise a result that is not finite and compute it again in float32 (synapse_walk.hip,
// synapse_wgrad_walk.hip).
//   Parts below the smallest normal number are lost: a value under 3e-33 enters with an absolute error of 1e-38.  Every
// float32 is a multiple of 2^-149, and so is what its parts leave: multiplied by kSplitScale first (exact), every part of
// every value is zero or a normal number.  These two scale both operands; values from 1e31 on then overflow, like
// values that are not finite.
#pragma once
#include <hip/hip_runtime.h>

namespace slayer {

constexpr float kSplitScale = 0x1p24f;
constexpr float kSplitProductScale = 0x1p-48f;      // what takes the scale out of a product

typedef __bf16 split_bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 split_bf8 __attribute__((ext_vector_type(8)));
typedef float split_f2 __attribute__((ext_vector_type(2)));
typedef float split_f4 __attribute__((ext_vector_type(4)));

// two floats rounded to bfloat16 in one dword
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(split_f2{a, b}, split_bf2));
}
// ... and a and b become what the rounding left
__device__ __forceinline__ unsigned round_pair(float& a, float& b) {
    const split_bf2 h = __builtin_convertvector(split_f2{a, b}, split_bf2);
    const split_f2 back = __builtin_convertvector(h, split_f2);
    a -= back.x;
    b -= back.y;
    return __builtin_bit_cast(unsigned, h);
}
// Eight floats (the k of one lane) as one operand of the instruction: rounded; what that rounding leaves; both.
__device__ __forceinline__ uint4 bf16_eight(const float (&v)[8]) {
    return make_uint4(bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3]), bf16_pair(v[4], v[5]), bf16_pair(v[6], v[7]));
}
__device__ __forceinline__ void leave_eight(float (&v)[8], uint4 rounded) {
    const unsigned pair[4] = {rounded.x, rounded.y, rounded.z, rounded.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] -= __uint_as_float(pair[i] << 16);
        v[2 * i + 1] -= __uint_as_float(pair[i] & 0xffff0000u);
    }
}
__device__ __forceinline__ uint4 round_eight(float (&v)[8]) {
    const uint4 r = bf16_eight(v);
    leave_eight(v, r);
    return r;
}
__device__ __forceinline__ split_f4 mfma_bf16(uint4 a, uint4 b, split_f4 d) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(split_bf8, a), __builtin_bit_cast(split_bf8, b), d, 0, 0, 0);
}

}  // namespace slayer
