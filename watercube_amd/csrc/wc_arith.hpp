// wc_arith.hpp -- short forms of division, reciprocal and square root with the bits of the IEEE operations, and the
// operand ranges that they hold in.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wc {

// Correctly rounded a / b from y = RN(1 / b): q0 = RN(a y), r = a - b q0 (exact), RN(q0 + r y)
// (Markstein's theorem).  Equal to the IEEE quotient, except that a = -0 gives +0, when b and y
// are normal and a is 0 or at least 2^-100 in magnitude with a normal quotient, so that no step
// underflows or overflows.  The force pass uses it only on steps whose operands the density pass
// found in that range (div_operand); then three quotients share one division.
__device__ __forceinline__ float quot(float a, float b, float y) {
    const float q0 = a * y;
    const float r = fmaf(-b, q0, a);
    return fmaf(r, y, q0);
}

// True for 0 and for 2^-40 <= |x| <= 2^40 (false for NaN and infinity).  Sums and differences of
// two such values are 0 or at least 2^-63 and at most 2^41 in magnitude, which keeps every
// quotient of the force pass inside the range where quot() is exact.
__device__ __forceinline__ bool div_operand(float x) {
    const uint32_t u = __float_as_uint(x) & 0x7fffffffu;
    return u == 0u || u - 0x2b800000u <= 0x53800000u - 0x2b800000u;
}

// Correctly rounded square root and reciprocal in five and three instructions, of the tile passes.
// tests/test_short_arithmetic.py compares both with sqrtf and 1 / x for every float in [2^-96, 2^60).
// x = 0 gives 0 (the clamped estimate keeps infinity out), NaN stays NaN.
__device__ __forceinline__ float sqrt_in_range(float x) {
    const float y = __builtin_amdgcn_rsqf(fmaxf(x, 0x1p-96f));
    const float s = x * y;
    return fmaf(fmaf(-s, s, x), 0.5f * y, s);
}
__device__ __forceinline__ float rcp_in_range(float x) {
    const float y = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, y, 1.0f), y, y);
}

// The tile passes' positions: those of 0 or of [2^-20, 2^20] in magnitude differ by 0 or at least 2^-43, so their
// squared distances are 0 or in sqrt_in_range's range.
__device__ __forceinline__ bool pos_operand(float x) {
    const uint32_t u = __float_as_uint(x) & 0x7fffffffu;
    return u == 0u || u - 0x35800000u <= 0x49800000u - 0x35800000u;
}

}  // namespace wc
