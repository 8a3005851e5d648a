// Short forms of the functions that the onboard control kernel spends its
// instructions on.  The kernel is a chain of scalar code with one or two
// waves on a SIMD: a wave issues one instruction every 4 to 5 cycles (8 and 16
// for a single and a double reciprocal, 8 more for a compare whose mask the
// next instruction selects with), dependent or not, so the kernel's time is
// its instruction count, scalar moves and waits for hazards included.  The
// library's functions spend theirs on arguments that cannot occur here, and
// on branches around them.
//
// The leading terms are in double, which issues at the rate of single, and
// the polynomials' tails, which are at most a tenth of the result, in single
// (their coefficients are literals of the instruction; a double coefficient
// takes two scalar moves), except where an ulp can flip a sign (atan2).  None
// is further from 64 bits than the library function it stands for: worst
// errors are 0.5 ulp of a float (quotients, roots, atan2, directions) to 0.8
// (cosine, tangent), where the single-precision library's are 0.5 to 3.5
// (tests/csrc/check_onboard_math.hip).  Polynomials interpolate the power
// series' tails at Chebyshev nodes (coefficients computed with 60 digits).
//
// TAME: the wave's inputs are finite and below kTameMax in magnitude, so no
// value of the chain is infinite or NaN and no angle is large.  The other
// form takes any float and has the library's limits.  For tame arguments
// both forms perform the same operations and give the same bits, so a
// result never depends on which form its wave took.
#pragma once

#include <hip/hip_runtime.h>

namespace onboard_math {

constexpr float kTameMax = 1.0e4f;

// The least positive float: an operand of max that turns an exact zero into
// something that can be divided by.
__device__ __forceinline__ float above_zero(float x) {
    return __builtin_fmaxf(x, __builtin_bit_cast(float, 1u));
}

// 1 / y within 2^-48 (the hardware value, 2^-24, refined once) or 2^-52 (by
// the cubic iteration, one operation more).  For y not 0, infinite or NaN.
__device__ __forceinline__ double recip48(double y) {
    const double r = __builtin_amdgcn_rcp(y);
    return __builtin_fma(__builtin_fma(-y, r, 1.0), r, r);
}
__device__ __forceinline__ double recip52(double y) {
    const double r = __builtin_amdgcn_rcp(y), e = __builtin_fma(-y, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// 1 / sqrt(x) within 2^-47 (the hardware value, 2^-24, refined once) or 2^-52,
// for positive normal x.
__device__ __forceinline__ double rsqrt47(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    return __builtin_fma(r * 0.5, __builtin_fma(-x * r, r, 1.0), r);
}
__device__ __forceinline__ double rsqrt52(double x) {
    const double r = __builtin_amdgcn_rsq(x), e = __builtin_fma(-x * r, r, 1.0);
    return __builtin_fma(r * e, __builtin_fma(e, 0.375, 0.5), r);
}

// The IEEE quotient x / y for y not 0: the product of x and the reciprocal is
// within 1.5 2^-52 of x / y, and no quotient of two floats lies closer than
// 2^-49 to a rounding boundary.
template <bool TAME>
__device__ __forceinline__ float quotient(float x, float y) {
    const float q = (float)((double)x * recip52((double)y));
    if constexpr (TAME) return q;
    const bool limit = !(__builtin_fabsf(y) < __builtin_huge_valf());
    const float l = x / y;
    return limit ? l : q;
}

// The IEEE quotients by one divisor y > 0 (infinity included: quotients 0).
struct Divisor {
    double r;
    __device__ __forceinline__ explicit Divisor(float y)
        : r(recip52(__builtin_fmin((double)y, 1.0e300))) {}
    __device__ __forceinline__ float operator()(float x) const { return (float)((double)x * r); }
};

// The IEEE square root, x >= 0: within 1.5 2^-52 before its rounding, and no
// root of a float lies closer than 2^-51 to a rounding boundary.
template <bool TAME>
__device__ __forceinline__ float square_root(float x) {
    const float s = (float)((double)x * rsqrt52((double)above_zero(x)));
    if constexpr (TAME) return s;
    const bool limit = !(x < __builtin_huge_valf());
    return limit ? x : s;  // infinity or NaN
}

// |x| or 2^-500: what a sum of squares takes in place of an exact zero, so that
// it can be divided by; it is far below the least float's share.
__device__ __forceinline__ double above_tiny(float x) {
    return __builtin_fmax((double)__builtin_fabsf(x), 0x1p-500);
}

// sqrt(x^2 + y^2).
template <bool TAME>
__device__ __forceinline__ float hypotenuse(float xf, float yf) {
    const double x = above_tiny(xf), y = yf;
    const double h2 = __builtin_fma(y, y, x * x);
    const float h = (float)(h2 * rsqrt47(h2));
    if constexpr (TAME) return h;
    const bool limit = !(__builtin_fabsf(xf) + __builtin_fabsf(yf) < __builtin_huge_valf());
    if (__builtin_amdgcn_ballot_w64(limit)) return limit ? hypotf(xf, yf) : h;
    return h;
}

// atan2 of any two floats, as one rounding of a double value within 2^-51: the
// angles reach wrap_angle's discontinuity, where the side that an angle rounds
// to decides the sign of the wrapped difference.  The smaller magnitude over
// the larger, brought below tan(pi/8) by the addition theorem ((z - 1) / (z +
// 1), plus pi/4), an odd polynomial, and a whole number of pi/4.  The
// polynomial is the interpolant of (atan q - q) / q^3 in t = q^2 at 11
// Chebyshev nodes of [0, 1.0001 tan^2(pi/8)], within 2^-56 of q.  With 8 terms
// in single it was up to 0.85 ulp off, and the difference of two angles half a
// turn apart changed sign for one pair of small integers in 350.
template <bool TAME>
__device__ __forceinline__ float atan2_float(float yf, float xf) {
    const float ay = __builtin_fabsf(yf), ax = __builtin_fabsf(xf);
    const float hf = above_zero(__builtin_fmaxf(ay, ax)), lf = __builtin_fminf(ay, ax);
    const bool upper = lf > hf * 0x1.a82799p-2f;  // tan(pi/8)
    const bool steep = ay > ax, back = __builtin_signbit(xf);
    const double h = hf, l = lf;
    const double diff = l - h, sum = l + h;
    const double num = upper ? diff : l, den = upper ? sum : h;
    const double r = recip48(den);
    double q = num * r;
    q = __builtin_fma(__builtin_fma(-den, q, num), r, q);
    const double t = q * q;
    double p = __builtin_fma(t, -0x1.3a2b7a07caea9p-6, 0x1.41603647c7a7cp-5);
    p = __builtin_fma(t, p, -0x1.a098bb6ba4941p-5);
    p = __builtin_fma(t, p, 0x1.dfe61e80903d2p-5);
    p = __builtin_fma(t, p, -0x1.10fa75382537fp-4);
    p = __builtin_fma(t, p, 0x1.3b1262d95579ep-4);
    p = __builtin_fma(t, p, -0x1.745d0b26b83e7p-4);
    p = __builtin_fma(t, p, 0x1.c71c7185314cbp-4);
    p = __builtin_fma(t, p, -0x1.24924924360cbp-3);
    p = __builtin_fma(t, p, 0x1.999999999934ap-3);
    p = __builtin_fma(t, p, -0x1.5555555555555p-2);
    const double v = __builtin_fma(q * t, p, q);
    // Quarter turns: pi/4 for the upper octant, then reflected at pi/4 and
    // at pi/2.
    float k = upper ? 1.0f : 0.0f;
    k = steep ? 2.0f - k : k;
    k = back ? 4.0f - k : k;
    const double w = steep != back ? -v : v;
    const float f = __builtin_copysignf((float)__builtin_fma((double)k, 0x1.921fb54442d18p-1, w), yf);
    if constexpr (TAME) return f;
    const bool limit = !(ay + ax < __builtin_huge_valf());
    if (__builtin_amdgcn_ballot_w64(limit))
        return limit ? (float)atan2((double)yf, (double)xf) : f;
    return f;
}

// Sine and cosine of the angle atan2(y, x) of two finite floats, from its
// components: y and x over the hypotenuse.  y = x = 0 gives atan2's angles
// (0 and pi by the sign of x).
struct Direction {
    float s, c;
};
__device__ __forceinline__ Direction direction(float yf, float xf) {
    const double y = yf, x = __builtin_copysign(above_tiny(xf), (double)xf);
    const double r = rsqrt47(__builtin_fma(y, y, x * x));
    return Direction{(float)(y * r), (float)(x * r)};
}

// atanh(x) for |x| <= 0.9999 (NaN gives NaN): half the logarithm of
// (1 + x) / (1 - x) = 2^k m with m near 1, as k ln 2 / 2 + atanh(s),
// s = (m - 1) / (m + 1) = ((1 - 2^k) + x (1 + 2^k)) / ((1 + 2^k) + x (1 - 2^k)),
// which is x for k = 0.  k comes from a single-precision estimate, so m stays
// within 2^(1/2) (1 + 2^-20) and the tail's polynomial covers s^2 <= 0.0296.
__device__ __forceinline__ float atanh_float(float xf) {
    const double x = xf;
    const float k = __builtin_rintf(
        __builtin_amdgcn_logf((1.0f + xf) * __builtin_amdgcn_rcpf(1.0f - xf)));
    const double p = __builtin_amdgcn_ldexp(1.0, (int)k);
    const double minus = 1.0 - p, plus = 1.0 + p;
    const double num = __builtin_fma(x, plus, minus), den = __builtin_fma(x, minus, plus);
    const double s = num * recip48(den);
    const float sf = (float)s, t = sf * sf;
    float c = __builtin_fmaf(t, 0x1.ddf01984cfbd1p-4f, 0x1.245ba6a054aeep-3f);
    c = __builtin_fmaf(t, c, 0x1.9999ecc082d44p-3f);
    c = __builtin_fmaf(t, c, 0x1.5555554b7afc8p-2f);
    const double v = s + (double)(sf * t * c);
    // The numerator's 1 - 2^k turns a -0 into +0: the sign is x's.
    return __builtin_copysignf((float)__builtin_fma((double)k, 0x1.62e42fefa39efp-2, v), xf);
}

// Sine and cosine tails over |r| <= pi/4: sin r = r + r t S(t), cos r =
// 1 - t/2 + t^2 C(t), t = r^2.
__device__ __forceinline__ float sin_tail(float r, float t) {
    float p = __builtin_fmaf(t, 0x1.6dbb0d6f050edp-19f, -0x1.a0139e5f4ae7ap-13f);
    p = __builtin_fmaf(t, p, 0x1.11110de85ad69p-7f);
    p = __builtin_fmaf(t, p, -0x1.555555545b3adp-3f);
    return r * t * p;
}
__device__ __forceinline__ float cos_tail(float t) {
    float p = __builtin_fmaf(t, -0x1.252250d29fd3ep-22f, 0x1.a015be5836519p-16f);
    p = __builtin_fmaf(t, p, -0x1.6c16bf50588e4p-10f);
    p = __builtin_fmaf(t, p, 0x1.5555555501defp-5f);
    return t * t * p;
}

// cos(x): the remainder of x by pi/2 (two terms, so that it is exact to 2^-52 of
// itself near the zeros of the cosine up to kTameMax) and the quadrant's
// function of it.
template <bool TAME>
__device__ __forceinline__ float cos_float(float xf) {
    const double x = xf;
    const double n = __builtin_rint(x * 0x1.45f306dc9c883p-1);  // 2 / pi
    const double r =
        __builtin_fma(n, -0x1.1a62633145c07p-54, __builtin_fma(n, -0x1.921fb54442d18p+0, x));
    const int quadrant = (int)n;
    const double t = r * r;
    const float tf = (float)t;
    const float c = (float)(__builtin_fma(t, -0.5, 1.0) + (double)cos_tail(tf));
    const float s = (float)(r + (double)sin_tail((float)r, tf));
    // cos(r + n pi/2) = c, -s, -c, s for n = 0, 1, 2, 3 (mod 4).
    const float v = (quadrant & 1) ? s : c;
    const unsigned flip = ((unsigned)(quadrant + 1) << 30) & 0x80000000u;
    const float f = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) ^ flip);
    if constexpr (TAME) return f;
    const bool far = !(__builtin_fabsf(xf) < kTameMax);
    if (__builtin_amdgcn_ballot_w64(far)) return far ? cosf(xf) : f;
    return f;
}

// sin(p h) for h in [0, 1] and the float p nearest to pi: 1 - 2 sin^2 of half
// the distance of p h to pi/2, which is at most pi/4.
__device__ __forceinline__ float sin_half_turn(float h) {
    const double a = __builtin_fma((double)h, 0x1.921fb6p+0, -0x1.921fb54442d18p-1);
    const float af = (float)a;
    const double s = a + (double)sin_tail(af, af * af);
    return (float)__builtin_fma(s * -2.0, s, 1.0);
}

// cos(asin s) cos(asin t) for |s|, |t| <= 0.9: one square root of the product
// of the two squared cosines.
__device__ __forceinline__ float cosine_product(float sf, float tf) {
    const double s = sf, t = tf;
    const double p = __builtin_fma(-s, s, 1.0) * __builtin_fma(-t, t, 1.0);
    return (float)(p * rsqrt47(p));
}

// tan(x) for |x| <= 0.75.
__device__ __forceinline__ float tan_float(float xf) {
    const double x = xf, t = x * x;
    const float tf = (float)t;
    const double c = __builtin_fma(t, -0.5, 1.0) + (double)cos_tail(tf);
    const double s = x + (double)sin_tail(xf, tf);
    return (float)(s * recip48(c));
}

// atan2(sin(d), cos(d)): d less its whole turns.  d is a float, so it never
// lies on the discontinuity, and the nearest multiple of 2 pi decides its
// side as the signs of sin(d) and cos(d) do.
template <bool TAME>
__device__ __forceinline__ float wrap_angle(float d) {
    const double x = d;
    const double n = __builtin_rint(x * 0x1.45f306dc9c882p-3);  // 1 / (2 pi)
    const float w = (float)__builtin_fma(n, -0x1.921fb54442d18p+2, x);
    if constexpr (TAME) return w;
    const bool far = !(__builtin_fabsf(d) < 2.0f * kTameMax);
    if (__builtin_amdgcn_ballot_w64(far)) {
        float s, c;
        sincosf(d, &s, &c);
        return far ? atan2f(s, c) : w;
    }
    return w;
}

}  // namespace onboard_math
