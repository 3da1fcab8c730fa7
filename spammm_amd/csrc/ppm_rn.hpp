// ppm_rn.hpp — correctly rounded FP32 reciprocal, quotient and square root of operands in the middle of
// the exponent range.
//
// The compiler's IEEE forms scale their operands for the ends of the range and fix up specials: 11
// instructions for a / b or 1 / x, 16 for sqrtf, most of them dependent.  Without those cases gfx950's
// v_rcp_f32 and v_rsq_f32 (1 ulp) need one FMA correction each: 3 instructions for 1 / x, 6 for a / b,
// 5 for a square root, with the same bits.  Checked on the card against the IEEE forms: rcp_rn and
// sqrt_rn on every mantissa at exponents -60..61 (both parities); div_rn on 512 numerators for every
// mantissa of the divisor (its last step rounds correctly when y = RN(1/b): P. Markstein, "Computation
// of elementary functions on the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 111 (1990)).
#pragma once

#include <hip/hip_runtime.h>

namespace ppm {

// 1 / x, 2^-100 <= |x| <= 2^100.
__device__ __forceinline__ float rcp_rn(float x) {
    const float y = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, y, 1.0f), y, y);
}

// a / b, 2^-60 <= |b| <= 2^60 and a = 0 or 2^-94 <= |a| <= 2^62 (the remainder below is then exact).
__device__ __forceinline__ float div_rn(float a, float b) {
    const float y = rcp_rn(b);
    const float q = a * y;
    return fmaf(fmaf(-b, q, a), y, q);
}

// sqrt(x), x = 0 or 2^-100 <= x <= 2^100.  ZERO: x may be 0.
template <bool ZERO = false>
__device__ __forceinline__ float sqrt_rn(float x) {
    const float y = __builtin_amdgcn_rsqf(ZERO ? fmaxf(x, 0x1p-100f) : x);
    const float s = x * y;
    return fmaf(fmaf(-s, s, x), 0.5f * y, s);
}

}  // namespace ppm
