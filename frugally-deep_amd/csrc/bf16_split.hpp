// fp32 values as sums of three bf16 values, for products on the bf16 matrix instructions.
#pragma once
#include "common.hpp"

namespace fdx {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t bf16_pair(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2 { a, b }), bf16x2));
}
// Operands are multiplied by 2^16 before they are split and sums of products by 2^-32 behind the products, both exact: the last
// bit of the smallest fp32 value is then bf16's smallest subnormal, 2^-133, and no operand loses bits (without it the bits below
// 2^-133 went: 2^-122 was held to 1.4e-4, fp32 subnormals not at all).  Operands from 2^112 and sums from 2^96 on become infinite
// and take the way of those.  One vector instruction a value, 6.5 with it: 8192 x 2048 x 512 87.0 -> 88.5 us,
// 8192 x 512 x 2048 86.7 -> 90.6 (what a remainder leaves as a dot product of the pair, 4.5 instructions, was slower beside MFMAs:
// 94.1 and 94.9).
constexpr float kSplitUp = 65536.f, kSplitDown = 1.f / 65536.f / 65536.f;
// Two floats as three pairs of bf16 that add up to them exactly.
__device__ __forceinline__ void split3(float a, float b, uint32_t& p0, uint32_t& p1, uint32_t& p2)
{
    p0 = bf16_pair(a, b);
    a -= __builtin_bit_cast(float, p0 << 16);
    b -= __builtin_bit_cast(float, p0 & 0xffff0000u);
    p1 = bf16_pair(a, b);
    a -= __builtin_bit_cast(float, p1 << 16);
    b -= __builtin_bit_cast(float, p1 & 0xffff0000u);
    p2 = bf16_pair(a, b);
}
// Eight floats, times kSplitUp, as one MFMA operand per plane.
__device__ __forceinline__ void split3x8(const float (&x)[8], u32x4 (&planes)[3])
{
    uint32_t w[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        split3(x[2 * i] * kSplitUp, x[2 * i + 1] * kSplitUp, w[0][i], w[1][i], w[2][i]);
#pragma unroll
    for (int q = 0; q < 3; ++q)
        planes[q] = u32x4 { w[q][0], w[q][1], w[q][2], w[q][3] };
}

} // namespace fdx
