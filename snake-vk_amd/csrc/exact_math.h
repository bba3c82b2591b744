// Square root, reciprocal and quotient rounded as IEEE arithmetic rounds them, for
// operands of ordinary size; callers test the operands and give the rest to the
// general forms, so that the result is the general form's for every operand.  The
// general forms take about 10 instructions for a quotient and 16 for a root, most of
// them on the half-rate pipe (V_DIV_SCALE, V_DIV_FIXUP, the compares and selects of
// sqrtf); without the scaling that these ranges do not need it is 6 and 5, all but one
// at the full rate.  That pays for roots, normalisations and ReSTIR's targets (bound by
// instruction issue).  In the path kernels' BRDF the tests take back what the short
// quotients save: with both, 1,627 us for the 1.02M-triangle frame and 1,009 for the
// G-buffer room (1920x1080), with general quotients 1,566 and 981.
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

// Whether every test holds, without a branch between them (with && the path kernels
// spilled twice as many registers).
template <class... B>
__device__ __forceinline__ bool every(B... b) {
    return (... & b);
}

// 2^-100 <= x < 2^100 (false for negative numbers and NaN), in one compare.
__device__ __forceinline__ bool exact_range(float x) { return __float_as_uint(x) - 0x0D800000u < 0x64000000u; }

// 2^-60 <= x < 2^60 (false for zero, negative numbers and NaN), in one compare: what
// both operands of a quotient are tested for, so that it is neither denormal nor infinite.
__device__ __forceinline__ bool short_range(float x) { return __float_as_uint(x) - 0x21800000u < 0x3C000000u; }
// Each of x, y and z is zero or at least 2^-74 in size.
__device__ __forceinline__ bool short_or_zero(float x, float y, float z) {
    const uint32_t a = (__float_as_uint(x) << 1) - 1u, b = (__float_as_uint(y) << 1) - 1u,
                   c = (__float_as_uint(z) << 1) - 1u;
    const uint32_t ab = a < b ? a : b;
    return (ab < c ? ab : c) >= (0x1A800000u << 1) - 1u;
}

// 1 / d for 2^-100 <= |d| < 2^100: one Newton step on V_RCP_F32 gives the correctly
// rounded reciprocal for each of the 2^23 mantissas (the exponent only scales it).
// x / d for such a d, x = 0 or |x| >= 2^-100, and 2^-125 <= |x / d| < 2^125: the
// estimate is a normal number and the residual x - q d is a multiple of 2^-147 of at
// most 24 bits, hence exact, so that Markstein's correction with a correctly rounded
// reciprocal rounds the quotient correctly.  A zero x gives +0.
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
