// bf16x3.h -- f32 values as three bf16 pieces, for products on the bf16 matrix
// cores (gemm_bf16x3.hip, flash_attention.hip).
//
// x = x1 + x2 + x3 with x1 = bf16(x), x2 = bf16(x - x1), x3 = bf16(x - x1 - x2),
// each rounded to nearest: 3 x 8 bits hold f32's 24 exactly, as long as the
// last piece is no subnormal and the first does not round to infinity (the split
// of f32 into three bf16 is Henry, Tang and Heinecke's, "Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", 2019).
// A product x y keeps x1y1 + (x1y2 + x2y1) + (x2y2 + x1y3 + x3y1).  With |x1| >= 1,
// |x2| <= 2^-8 and |x3| <= 2^-17, so the three left out are at most 2^-24 |x y|
// together, one half of an f32 unit in the last place, which x = y = 1 + 2^-8 -
// 2^-17 reaches, always with the same sign; over random data they are a tenth of
// that.
#pragma once

#include <hip/hip_runtime.h>

namespace clove {
namespace k {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

// Operands are split as 2^24 x.  A value's lowest bit is 2^-149 or more, so no
// piece is then a bf16 subnormal, and a product of operands, 2^48 times larger,
// is normal wherever f32 holds it at all; the factor comes off the sums at the
// end, exactly (or with the one rounding of a subnormal result).  |x| of 2^103
// and sums of 2^79 overflow instead: those, infinities and NaN end as a sum that
// is not finite, which is where a kernel takes the f32 values instead.
constexpr float kPieceScale = 0x1p24f, kPieceUnscale = 0x1p-24f, kSumUnscale = 0x1p-48f;

// The six products, smallest first: piece of the first operand, of the second.
constexpr int kPieceA[6] = {2, 0, 1, 1, 0, 0}, kPieceB[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f2){a, b}, bf2));
}

// Two floats, times 2^24 with SCALE, as one dword of each of the three pieces.
// FUSED takes the first remainder as an FMA of the unscaled value, which frees
// its register earlier but is a longer instruction (the same value).
template <bool SCALE, bool FUSED = false>
__device__ __forceinline__ void split_pair(float a, float b, unsigned *p1, unsigned *p2,
                                           unsigned *p3) {
#pragma clang fp contract(off)
    const float sa = SCALE ? a * kPieceScale : a, sb = SCALE ? b * kPieceScale : b;
    const unsigned h = bf16_pair(sa, sb);
    const auto rest = [](float x, float scaled, unsigned bits) {
        return SCALE && FUSED ? __builtin_fmaf(x, kPieceScale, -__uint_as_float(bits))
                              : scaled - __uint_as_float(bits);
    };
    const float ra = rest(a, sa, h << 16), rb = rest(b, sb, h & 0xffff0000u);
    const unsigned m = bf16_pair(ra, rb);
    *p1 = h;
    *p2 = m;
    *p3 = bf16_pair(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
}

// LDS contents are published by a wait for this wave's LDS operations and a
// bare barrier: __syncthreads() would also wait for the slab in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace k
}  // namespace clove
