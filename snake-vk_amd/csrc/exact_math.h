// Square root, reciprocal and quotient rounded as IEEE arithmetic rounds them, for
// operands of ordinary size.  The general forms take about 10 instructions for a
// quotient and 16 for a root, most of them on the half-rate pipe (V_DIV_SCALE,
// V_DIV_FIXUP, the compares and selects of sqrtf); without the scaling that these
// ranges do not need it is 6 and 5, all but one at the full rate.  Shading is bound
// by instruction issue wherever its surfaces are cached (ReSTIR's resampling, path
// tails of small scenes); a range test on the operands picks the form.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace snkpt {

// a where the mask's bits are set, else b.  V_BITOP3 issues in 2 cycles per wave
// beside the other pipe; V_CNDMASK takes 4, and a run of them on one VCC measured
// 15-22 cycles each (the near / far choice and the axis permutation are such runs).
__device__ __forceinline__ uint32_t bit_sel(uint32_t a, uint32_t b, uint32_t m) {
    return __builtin_amdgcn_bitop3_b32(a, b, m, 0xE4);
}

// 2^-100 <= x < 2^100 (false for negative numbers and NaN), in one compare.
__device__ __forceinline__ bool exact_range(float x) { return __float_as_uint(x) - 0x0D800000u < 0x64000000u; }

// 1 / d and x / d for 2^-100 <= |d| < 2^100, |x| >= 2^-100 and 2^-60 <= |x / d| <=
// 2^60: one Newton step on V_RCP_F32 gave the correctly rounded reciprocal for each
// of the 2^23 mantissas, and Markstein's correction then rounds the quotient
// correctly (no off result in 4e9 random pairs over those exponents).  A smaller x
// may come out one unit in the last place off; x = -0 gives +0.
__device__ __forceinline__ float rcp_exact(float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    return fmaf(fmaf(-d, r, 1.0f), r, r);
}
__device__ __forceinline__ float div_exact(float x, float d, float r) {
    const float q = x * r;
    return fmaf(fmaf(-q, d, x), r, q);
}
__device__ __forceinline__ float div_exact(float x, float d) { return div_exact(x, d, rcp_exact(d)); }
// div_exact that keeps the sign of a zero x (d > 0)
__device__ __forceinline__ float div_signed(float x, float d, float r) {
    return __uint_as_float(bit_sel(__float_as_uint(div_exact(x, d, r)), __float_as_uint(x), 0x7FFFFFFFu));
}

// sqrt(x) for exact_range(x): V_RSQ_F32 and the residual's correction.  All 2^23
// mantissas of an even and an odd exponent matched sqrtf (the other exponents are
// these scaled by powers of 4; thirteen more were tried).
__device__ __forceinline__ float sqrt_exact(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float g = x * y;
    return fmaf(fmaf(-g, g, x), 0.5f * y, g);
}

}  // namespace snkpt
