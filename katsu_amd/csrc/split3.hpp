// split3.hpp -- float32 products on the bf16 matrix cores: each operand is
// written as the sum of three bf16 values, and a product as six of bf16 ones.
//
//   2^16 x = x0 + x1 + x2,  x0 = bf16(2^16 x), x1 = bf16(2^16 x - x0), x2 = the rest
//
// (round to nearest).  A bf16 has 8 significant bits and the exponents of
// float32, so |x1| <= 2^-9 |x0|, |x2| <= 2^-18 |x0|, both differences are exact
// and nothing is left after x2: the split loses no bit of x.  The factor keeps
// that so for the smallest x: a bf16 ends at 2^-133, a float32 at 2^-149, and
// without it operands below 2^-109 (1.5e-33) lost bits, those below 2^-134 all
// of them.  Sums are multiplied by 2^-32, which is exact above 2^-126.
// Operands of 2^112 and sums of 2^96 overflow in turn, and take the
// way of the non-finite ones below.
//
// Of the nine products the kernels form six,
//
//   x0 y0 + (x0 y1 + x1 y0) + (x1 y1 + x0 y2 + x2 y0),
//
// each exact in float32; the three left out sum to at most 2^-26 |x y|, a
// quarter of the rounding of one float32 product.
//
// v_mfma_f32_32x32x16_bf16 does 16x the FLOP per cycle of the float32
// v_mfma_f32_16x16x4_f32, so six of them do the work of the float32 pipe in
// 6/16 of its time: 333 TFLOP/s of float32 products at the 2.0 PFLOP/s that
// a loop of nothing else reached, against 135-143 on the float32 pipe.
//
// Accumulation.  The instruction adds its 16 products to the accumulator
// aligned to the largest term and keeps 2 bits below the accumulator's last
// one (measured: 1 + 32 * 2^-26 is exact, 1 + 32 * 2^-27 is 1): a long sum
// would lose the tails of terms of one sign.  The kernels therefore sum short
// runs from zero (128 k of a GEMM, at most 9 steps or 144 products of a
// convolution, 64 pixels of a filter gradient) and add each run to a float32
// total with an ordinary addition, so that terms and accumulator stay near in
// size.
//
// Non-finite values: Inf - Inf in the split, or a value that overflows when it
// is scaled or rounded to bf16, makes the sum NaN or Inf; a finite sum holds
// finite products only.  Every kernel tests its sums and computes non-finite
// ones again in float32.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace katsu {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 0x1p16f;     // of an operand
constexpr float kSplitUnscale = 0x1p-32f;  // of a sum

// Eight floats as three vectors of eight bf16: 13 vector instructions a pair.
// (The differences as two-term bf16 products on the packed pair are exact too
// and take 4 fewer, but run slower beside the matrix instructions: 4096^3 in 687
// against 632 us, both without the two that scale; 647 with them.)
__device__ __forceinline__ void split3(const float (&x)[8], uintx4 (&p)[3]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = kSplitScale * x[2 * i], b = kSplitScale * x[2 * i + 1];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const uint32_t h =
                __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{a, b}, bf16x2));
            p[q][i] = h;
            if (q < 2) {
                a -= __builtin_bit_cast(float, h << 16);
                b -= __builtin_bit_cast(float, h & 0xffff0000u);
            }
        }
    }
}

// The six products, smallest first.
constexpr int kSplitA[6] = {2, 0, 1, 1, 0, 0};
constexpr int kSplitB[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ floatx16 mfma32(uintx4 a, uintx4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

}  // namespace katsu
