// Products of 32-bit floats on the bf16 matrix cores, for masks and matrices dense enough to be computed as dense tiles.
//
// A float is the sum of three bf16 (8 + 8 + 8 significand bits, each rounded to nearest: nothing is left), and a product of two
// floats is six of the nine products of the parts; the three left out come to 2^-24 of it at most, as a rule to 2^-27. The matrix cores
// add up bf16 products in 32 bits and do 16 times the multiplications per clock that they do in fp32: six for one is still 2.7 times
// the fp32 rate.
// Errors against 64 bits, operands of normal distribution, the sums' order as in the kernels: dot products of 32 / 64 / 128
// 3.8e-8 / 4.3e-8 / 5.2e-8, eight chains of fp32 fma 6.2e-8 / 7.2e-8 / 8.8e-8 (2.5e-8: rounded once).
// What the parts cannot hold: an infinity, a NaN or a value that rounds to infinity in bf16 makes the result NaN or infinite, and the
// last part of a nonzero value below 2^-109 would be below bf16's smallest, which loses up to 2^-134 of it. The kernels compute
// results that are not finite, and those that are not large against what such values can lose, from the floats themselves.
#pragma once

#include "common.hpp"

namespace dlspm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct Parts { bf16x8 hi, mid, lo; };

// the eight floats x[0 ... 7] of a lane. Two at a time: the conversion makes two, and what it rounds them to are the halves of its
// result (seven instructions a float with the look for values too small). The least of 2 |x| - 1 as an integer (x == 0: the largest)
// goes to `least`.
constexpr unsigned kTooSmall = (18u << 24) - 1;  // `least` below this: a nonzero value below 2^-109
__device__ __forceinline__ Parts split_parts(const float* x, unsigned& least)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    auto round2 = [](float a, float b) { return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2)); };
    u4 hi, mid, lo;
    least = ~0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = x[2 * i], b = x[2 * i + 1];
        hi[i] = round2(a, b);
        const float ra = a - __uint_as_float(hi[i] << 16), rb = b - __uint_as_float(hi[i] & 0xffff0000u);
        mid[i] = round2(ra, rb);
        lo[i] = round2(ra - __uint_as_float(mid[i] << 16), rb - __uint_as_float(mid[i] & 0xffff0000u));
        least = min(min(least, (__float_as_uint(a) << 1) - 1u), (__float_as_uint(b) << 1) - 1u);
    }
    return Parts{__builtin_bit_cast(bf16x8, hi), __builtin_bit_cast(bf16x8, mid), __builtin_bit_cast(bf16x8, lo)};
}
// ... and the lanes with a value that is too small among those of `few`
__device__ __forceinline__ Parts split_parts(const float* x, unsigned long long& few)
{
    unsigned least;
    const Parts p = split_parts(x, least);
    few |= __ballot(least < kTooSmall);
    return p;
}

// 32 x 32 results, sixteen products each: lane l holds row l % 32 of `a` and of `b`, elements 8 (l / 32) ... + 7; element r of the
// sum is row 8 (r / 4) + 4 (l / 32) + r % 4 of a and row l % 32 of b
__device__ __forceinline__ f32x16 mfma(const bf16x8& a, const bf16x8& b, const f32x16& c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

}  // namespace dlspm
