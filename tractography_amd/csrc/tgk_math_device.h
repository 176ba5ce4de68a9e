// tgk_math_device.h -- the elementary functions of tgk_math.h for the device:
// the same operations on the same operands, so the same bits, with the cases
// chosen by selects instead of branches.
//
// A wavefront nearly always holds lanes on both sides of a test such as
// "|x| <= 1/2" or the quadrant of an angle, so a branch there runs both sides
// anyway and adds the scalar instructions that mask and restore the lanes:
// the plain SH45 Transport step had 110 such regions and 740 scalar
// instructions beside 1940 vector ones, and has 51, 380 and 1650 this way.
// Arguments that no lane has on an ordinary step (infinities, zeros of atan2,
// sines beyond 2^20) are left to tgk_math.h behind one branch. 32^3 SH45
// Transport, 10k seeds (a chain of up to 3000 steps, one wavefront to a
// SIMD): 20.3 -> 15.9 ms per call; 145 x 174 x 145 SH45 Diffusion, 1M seeds:
// 74.5 -> 66.4 ms; 64 candidates of a Probabilistic step, 300k seeds: 51.9 ->
// 38.5 ms.
//
// Include only from translation units compiled with -ffp-contract=off.
#pragma once

#include <hip/hip_runtime.h>

#include "tgk_math.h"

namespace tgk {
namespace dm {

__device__ __forceinline__ float flip_sign(float x, bool flip)
{
    return tgk_as_f32(tgk_as_u32(x) ^ (flip ? 0x80000000u : 0u));
}

// tgk_sincosf for |x| <= 2^20 (NaN gives NaN).
__device__ __forceinline__ void sincosf_small(float x, float *s, float *c)
{
    const float k = rintf(x * TGK_TWO_OVER_PI);
    float r = fmaf(-k, TGK_PIO2_1, x);
    r = fmaf(-k, TGK_PIO2_2, r);
    r = fmaf(-k, TGK_PIO2_3, r);
    const float w = r * r;

    float ps = fmaf(w, 2.832745849e-06f, -1.985307608e-04f);
    ps = fmaf(w, ps, 8.333379403e-03f);
    ps = fmaf(w, ps, -1.666666716e-01f);
    const float sr = fmaf(r * w, ps, r);

    float pc = fmaf(w, -2.888124584e-07f, 2.482202217e-05f);
    pc = fmaf(w, pc, -1.388898003e-03f);
    pc = fmaf(w, pc, 4.166666791e-02f);
    pc = fmaf(w, pc, -5.000000000e-01f);
    const float cr = fmaf(w, pc, 1.0f);

    // The quadrant k mod 4: odd ones swap sine and cosine; the sine is
    // negated in 2 and 3, the cosine in 1 and 2.
    const uint32_t q = (uint32_t)(int)k;
    const bool odd = (q & 1u) != 0;
    const float a = odd ? cr : sr, b = odd ? sr : cr;
    *s = tgk_as_f32(tgk_as_u32(a) ^ ((q & 2u) << 30));
    *c = tgk_as_f32(tgk_as_u32(b) ^ (((q + 1u) & 2u) << 30));
}

__device__ __forceinline__ void sincosf(float x, float *s, float *c)
{
    if (!(fabsf(x) <= 1048576.0f))
        x = fabsf(x) < tgk_inf() ? (float)fmod((double)x, TGK_TWO_PI_D) : x - x;
    sincosf_small(x, s, c);
}

// tgk_cosf for |x| <= 2^20.
__device__ __forceinline__ float cosf_small(float x)
{
    float s, c;
    sincosf_small(x, &s, &c);
    return c;
}

__device__ __forceinline__ float atan2f(float y, float x)
{
    const float ax = fabsf(x), ay = fabsf(y);
    const bool swap = ay > ax;
    const float num = swap ? ax : ay, den = swap ? ay : ax;
    // NaN, an infinity (or a sum that reaches it) or a zero.
    if (!(ax + ay < tgk_inf()) || num == 0.0f)
        return tgk_atan2f(y, x);
    const float a = num / den;
    const bool reduced = a > 0.41421356f;
    const float b = (num - den) / (num + den);
    const float at = tgk_atan_kernel(reduced ? b : a);
    const bool left = tgk_signbitf(x) != 0;
    // K by octant (tgk_atan2f): pi/4 or 3 pi/4 where reduced, else pi/2
    // where swapped, else 0 or pi; pi/2 - angle and pi - angle each negate.
    const float hi = reduced ? (left ? TGK_3PIO4_HI : TGK_PIO4_HI) : swap ? TGK_PIO2_HI : left ? TGK_PI_HI : 0.0f;
    const float lo = reduced ? (left ? TGK_3PIO4_LO : TGK_PIO4_LO) : swap ? TGK_PIO2_LO : left ? TGK_PI_LO : 0.0f;
    return tgk_copysignf(hi + (flip_sign(at, swap != left) + lo), y);
}

__device__ __forceinline__ float acosf(float x)
{
    const float ax = fabsf(x);
    const bool small = ax <= 0.5f;
    const float z = (1.0f - ax) * 0.5f;
    const float w = small ? x * x : z;
    float p = fmaf(w, 3.770212084e-02f, 1.431217324e-02f);
    p = fmaf(w, p, 3.183952346e-02f);
    p = fmaf(w, p, 4.451335222e-02f);
    p = fmaf(w, p, 7.500521839e-02f);
    p = fmaf(w, p, 1.666665971e-01f);
    const float s = sqrtf(z);
    const float v = small ? x : s;
    const float u = v * w;
    const float as = 2.0f * fmaf(u, p, s);
    const float central = TGK_PIO2_HI - (x + fmaf(u, p, -TGK_PIO2_LO));
    const float outer = x > 0.0f ? as : TGK_PI_HI - (as - TGK_PI_LO);
    const float r = small ? central : outer;
    return ax <= 1.0f ? r : __builtin_nanf("");
}

__device__ __forceinline__ float expf(float x)
{
    const float xc = fminf(fmaxf(x, -104.0f), 89.0f);
    const float k = rintf(xc * TGK_LOG2E);
    float r = fmaf(-k, TGK_LN2_HI, xc);
    r = fmaf(-k, TGK_LN2_LO, r);
    float p = fmaf(r, 1.974024926e-04f, 1.393507817e-03f);
    p = fmaf(r, p, 8.333570324e-03f);
    p = fmaf(r, p, 4.166646302e-02f);
    p = fmaf(r, p, 1.666666567e-01f);
    p = fmaf(r, p, 5.000000000e-01f);
    const float e = fmaf(r * r, p, r) + 1.0f;
    // One rounding where the result is subnormal, infinity past the range.
    const float v = __builtin_ldexpf(e, (int)k);
    const float bounded = x > 89.0f ? tgk_inf() : x < -104.0f ? 0.0f : v;
    return x != x ? x : bounded;
}

// n / d, correctly rounded, where neither operand nor quotient comes near the
// ends of the exponent range: Newton's step on the approximate reciprocal, then
// the quotient corrected twice by its residual, each exact in a fused operation
// (P. Markstein, IBM J. Res. Dev. 34, 1990). logf_normal's quotients depend on
// the argument's 2^23 mantissas alone; tests compare all of them.
__device__ __forceinline__ float divide_inner(float n, float d)
{
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    float q = n * r;
    q = fmaf(fmaf(-d, q, n), r, q);
    return fmaf(fmaf(-d, q, n), r, q);
}

// x / 100, correctly rounded, for 0 and 2^-32 <= x <= 64: the quotient by the
// rounded 1/100, corrected by its residual (Markstein, as above). Scaling by
// powers of two changes no rounding here, so one binade stands for all; tests
// go through it.
__device__ __forceinline__ float divide_100(float x)
{
    const float q = x * 0.01f;
    return fmaf(fmaf(-100.0f, q, x), 0.01f, q);
}

// tgk_logf for normal positive finite x.
__device__ __forceinline__ float logf_normal(float x)
{
    const uint32_t ix = tgk_as_u32(x);
    const uint32_t mb = (ix & 0x007fffffu) | 0x3f800000u;
    const bool upper = mb > 0x3fb504f3u;
    const int e = (int)(ix >> 23) - (upper ? 126 : 127);
    const float f = tgk_as_f32(upper ? mb - 0x00800000u : mb) - 1.0f;
    const float s = divide_inner(f, 2.0f + f);
    const float w = s * s;
    float p = fmaf(w, 2.428623587e-01f, 2.849848568e-01f);
    p = fmaf(w, p, 4.000097513e-01f);
    p = fmaf(w, p, 6.666666269e-01f);
    const float correction = s * fmaf(-w, p, f);
    const float ef = (float)e;
    return fmaf(ef, TGK_LN2_HI, f - fmaf(-ef, TGK_LN2_LO, correction));
}

// log(1 + exp(x)) / 100 for x < 30, as tgk_logf(1 + tgk_expf(x)) / 100
// rounds it: below -20 the sum rounds to 1, whatever the exponential.
__device__ __forceinline__ float log1pexp_100(float x)
{
    const float xc = fmaxf(x, -20.0f);
    const float k = rintf(xc * TGK_LOG2E);
    float r = fmaf(-k, TGK_LN2_HI, xc);
    r = fmaf(-k, TGK_LN2_LO, r);
    float p = fmaf(r, 1.974024926e-04f, 1.393507817e-03f);
    p = fmaf(r, p, 8.333570324e-03f);
    p = fmaf(r, p, 4.166646302e-02f);
    p = fmaf(r, p, 1.666666567e-01f);
    p = fmaf(r, p, 5.000000000e-01f);
    const float e = fmaf(r * r, p, r) + 1.0f;
    return divide_100(logf_normal(1.0f + __builtin_ldexpf(e, (int)k)));
}

__device__ __forceinline__ float logf(float x)
{
    if (!(x >= 1.17549435e-38f && x < tgk_inf()))
        return tgk_logf(x);
    return logf_normal(x);
}

}  // namespace dm
}  // namespace tgk
