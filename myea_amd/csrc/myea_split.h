// myea_split.h — an FP32 number as the sum of three BF16 numbers: what the kernels that multiply on the BF16 matrix cores share.
// myea_gemm.hip says which products are formed and what that leaves of the error.
//
// Range.  BF16 has FP32's exponents but 8 bits: the third number of an operand below 2^-110 would fall among the subnormals and lose
// bits (3.5e-5 of an operand of 2^-120, all of one below 2^-134).  So an operand is split as x * 2^24: the last bit of the smallest
// FP32 subnormal becomes 2^-125, a normal number, and the sum is exact for every x below 2^103.  The sums of products come out times
// 2^48 and go through unscaled() before anything else is done with them.  Larger operands and sums beyond 2^79 leave an infinity
// or a NaN, and whoever finds one computes the sum again in FP32.  The two multiplications are 2 of the 13 vector instructions a pair
// takes.
#pragma once

#include <hip/hip_runtime.h>

namespace myea {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));   // a 16-byte load from any element's address

// the smaller five of the six products a_x b_y, in this order; hi hi has an accumulator of its own
constexpr int kSmallA[5] = {0, 2, 1, 0, 1}, kSmallB[5] = {2, 0, 1, 1, 0};

constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

// an accumulator of products of two split operands -> the sum itself
__device__ __forceinline__ float unscaled(float sum) { return sum * kSplitUnscale; }

// two FP32 numbers -> the two BF16 numbers of each plane, packed
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned &hi, unsigned &mid, unsigned &lo)
{
    x0 *= kSplitScale; x1 *= kSplitScale;
    hi = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){x0, x1}, bf16x2));
    const float r0 = x0 - __uint_as_float(hi << 16), r1 = x1 - __uint_as_float(hi & 0xffff0000u);
    mid = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){r0, r1}, bf16x2));
    const float q0 = r0 - __uint_as_float(mid << 16), q1 = r1 - __uint_as_float(mid & 0xffff0000u);
    lo = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){q0, q1}, bf16x2));
}

// eight consecutive k's of a lane -> its fragment of each plane
__device__ __forceinline__ void split_eight(const float (&x)[8], bf16x8 (&planes)[3])
{
    u32x4 hi, mid, lo;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        unsigned h, m, l;
        split_pair(x[2 * e], x[2 * e + 1], h, m, l);
        hi[e] = h; mid[e] = m; lo[e] = l;
    }
    planes[0] = __builtin_bit_cast(bf16x8, hi); planes[1] = __builtin_bit_cast(bf16x8, mid); planes[2] = __builtin_bit_cast(bf16x8, lo);
}

// Eight k's of one row of an operand, from k on, straight from memory; zeros from K on.
template <bool KC>
__device__ __forceinline__ void load_eight(float (&x)[8], const float *at, long ld, int k, int K)
{
    if (k + 8 <= K) {
        if (KC) {
            *reinterpret_cast<f32x4 *>(x) = *reinterpret_cast<const f32x4_any *>(at);
            *reinterpret_cast<f32x4 *>(x + 4) = *reinterpret_cast<const f32x4_any *>(at + 4);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = at[e * ld];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            x[e] = 0.f;
            if (k + e < K) x[e] = at[KC ? (long)e : e * ld];
        }
    }
}

}  // namespace myea
