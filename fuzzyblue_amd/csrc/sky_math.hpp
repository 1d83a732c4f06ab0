// sky_math.hpp — quotients and square roots of the sky lookups: the bits of
// the IEEE operations in fewer instructions than the compiler's expansions.
//
// They rest on the hardware's v_rcp_f32 and v_rsq_f32: rcp_nr is the correctly
// rounded reciprocal for every denominator and sqrt_nr the correctly rounded
// root for every argument, both checked over all binary32 values
// (sky_math_check.hip), and Markstein's correction of a quotient with a
// correctly rounded reciprocal is the correctly rounded quotient.
//
// A wavefront with a lane outside a quotient's ranges takes the compiler's
// division (a wave-uniform branch; the empty asm statement keeps the compiler
// from evaluating it unconditionally and selecting), which has the same bits,
// so a lane's result does not depend on the others'.
#pragma once

#include "atmo_device.hpp"

namespace fbk {

// 1 / b for 2^-100 < |b| < 2^100.
__device__ __forceinline__ float rcp_nr(float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    return fmaf(fmaf(-b, y, 1.0f), y, y);
}
// a / b for such b and a 0 or of at least 2^-80, where the quotient is normal
// -- 9 instruction slots, the compiler's division about 16.  (A smaller
// numerator's quotient may be an ulp off.)
__device__ __forceinline__ float div_nr(float a, float b) {
    return div_markstein(a, b, rcp_nr(b));
}
// Whether |x| is outside [lo, hi] (or NaN).
__device__ __forceinline__ bool outside(float x, float lo, float hi) {
    return __builtin_amdgcn_fmed3f(fabsf(x), lo, hi) != fabsf(x);
}
// Denominators and numerators (other than 0) that div_nr divides exactly in
// any combination.
__device__ __forceinline__ bool extreme_den(float b) { return outside(b, 0x1p-60f, 0x1p40f); }
__device__ __forceinline__ bool extreme_num(float a) { return outside(a, 0x1p-80f, 0x1p60f); }
// a / b for any operands (but for the sign of a zero quotient).
__device__ __forceinline__ float div_any(float a, float b) {
    float d = div_nr(a, b);
    if (__builtin_amdgcn_ballot_w64(extreme_den(b) || (extreme_num(a) && a != 0.0f))) {
        asm volatile("");
        d = a / b;
    }
    return d;
}
// (s a) / b per channel, by one reciprocal.
__device__ __forceinline__ float3 scale_div_any(float3 a, float s, float b) {
    const float3 n = make_float3(a.x * s, a.y * s, a.z * s);
    const float y = rcp_nr(b);
    float3 d = make_float3(div_markstein(n.x, b, y), div_markstein(n.y, b, y),
                           div_markstein(n.z, b, y));
    const float lo = fminf(fminf(fabsf(n.x), fabsf(n.y)), fabsf(n.z)),
                hi = fmaxf(fmaxf(fabsf(n.x), fabsf(n.y)), fabsf(n.z));
    if (__builtin_amdgcn_ballot_w64(extreme_den(b) ||
                                    ((lo < 0x1p-80f || hi > 0x1p60f) && s != 0.0f))) {
        asm volatile("");
        d = make_float3(n.x / b, n.y / b, n.z / b);
    }
    return d;
}
// sqrt(max(x, 0)) for any x: the hardware's reciprocal square root and one
// correction with the exact residual, of an argument scaled up where that
// would be subnormal.  No branch, so that a lookup's other chains overlap it
// (with one for small arguments 22 frames of 28,469 pixels took 43.5 us, not
// 41.7); 16 slots, the compiler's root about 23.
__device__ __forceinline__ float sqrt_nr(float x) {
    x = fmaxf(x, 0.0f);
    const bool small = x < 0x1p-60f;
    const float xs = x * (small ? 0x1p96f : 1.0f);
    const float y = __builtin_amdgcn_rsqf(xs), g = xs * y;
    const float root = fmaf(fmaf(-g, g, xs), 0.5f * y, g) * (small ? 0x1p-48f : 1.0f);
    constexpr int kZeroOrInf = 0x260;
    return __builtin_amdgcn_classf(x, kZeroOrInf) ? x : root;
}

}  // namespace fbk
