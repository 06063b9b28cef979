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
// Two floats as three pairs of bf16 that add up to them exactly (below 2^-110 the last bits fall under bf16's subnormals).
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
// Eight floats as one MFMA operand per plane.
__device__ __forceinline__ void split3x8(const float (&x)[8], u32x4 (&planes)[3])
{
    uint32_t w[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        split3(x[2 * i], x[2 * i + 1], w[0][i], w[1][i], w[2][i]);
#pragma unroll
    for (int q = 0; q < 3; ++q)
        planes[q] = u32x4 { w[q][0], w[q][1], w[q][2], w[q][3] };
}

} // namespace fdx
