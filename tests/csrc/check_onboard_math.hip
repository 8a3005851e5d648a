// GPU check of turbinator_c_amd/csrc/onboard_math.h against the host's double
// (and long double) functions on arguments of the ranges each is stated for,
// with exact angles, zeros, infinities and NaN among them.
// Prints one line per function: "<name> <arguments> <worst error in ulp of a
// float> <arguments whose two forms differ> <limit arguments that differ from
// the library function>", and exits 0 when the run itself succeeded.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

#include "../../turbinator_c_amd/csrc/onboard_math.h"

namespace om = onboard_math;

enum { QUOTIENT, DIVISOR, ROOT, HYPOT, ATAN2, DIR_S, DIR_C, ATANH, COS, SIN_PI, TAN, WRAP, COS2, KINDS };
static const char *const kNames[KINDS] = {"quotient", "divisor", "square_root", "hypotenuse",
                                          "atan2", "direction_s", "direction_c", "atanh", "cos",
                                          "sin_half_turn", "tan", "wrap", "cosine_product"};

template <bool TAME>
__device__ float eval(int kind, float a, float b) {
    switch (kind) {
    case QUOTIENT: return om::quotient<TAME>(a, b);
    case DIVISOR: return om::Divisor(b)(a);
    case ROOT: return om::square_root<TAME>(a);
    case HYPOT: return om::hypotenuse<TAME>(a, b);
    case ATAN2: return om::atan2_float<TAME>(a, b);
    case DIR_S: return om::direction(a, b).s;
    case DIR_C: return om::direction(a, b).c;
    case ATANH: return om::atanh_float(a);
    case COS: return om::cos_float<TAME>(a);
    case SIN_PI: return om::sin_half_turn(a);
    case TAN: return om::tan_float(a);
    case COS2: return om::cosine_product(a, b);
    default: return om::wrap_angle<TAME>(a);
    }
}

__global__ void run(int kind, const float *a, const float *b, float *tame, float *any, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        tame[i] = eval<true>(kind, a[i], b[i]);
        any[i] = eval<false>(kind, a[i], b[i]);
    }
}

#define CHECK(call)                                                  \
    do {                                                             \
        hipError_t e_ = (call);                                      \
        if (e_ != hipSuccess) {                                      \
            printf("%s failed: %s\n", #call, hipGetErrorString(e_)); \
            return 1;                                                \
        }                                                            \
    } while (0)

static uint64_t rng = 0x9e3779b97f4a7c15ull;
static uint32_t next32(void) {  // xorshift64*
    rng ^= rng >> 12;
    rng ^= rng << 25;
    rng ^= rng >> 27;
    return (uint32_t)((rng * 2685821657736338717ull) >> 32);
}
static uint64_t hard_rng = 0x2545f4914f6cdd1dull;  // its own: the other arguments stay
static uint32_t hard32(void) {
    const uint64_t kept = rng;
    rng = hard_rng;
    const uint32_t v = next32();
    hard_rng = rng;
    rng = kept;
    return v;
}
static float unit(void) { return (float)(next32() >> 8) / 16777216.0f; }
static float sign(void) { return next32() & 1 ? -1.0f : 1.0f; }
// Log-uniform magnitude in [2^lo, 2^hi), random sign.
static float spread(int lo, int hi) { return sign() * ldexpf(1.0f + unit(), lo + (int)(next32() % (unsigned)(hi - lo))); }

// x, y whose quotient lies within 2^-47 of a rounding boundary: x 2^25 = +-1
// (mod y), so that x / y is 1 / (2^25 y) beside an odd multiple of 2^-25.
static void hard_quotient(float *x, float *y) {
    for (;;) {
        const uint64_t d = (1u << 23) | (hard32() >> 9) | 1u;
        uint64_t inv = 1, base = (d + 1) / 2;  // 1 / 2 (mod y), to the 25th power
        for (int e = 25; e; e >>= 1) {
            if (e & 1) inv = inv * base % d;
            base = base * base % d;
        }
        const uint64_t n = hard32() & 1 ? inv : d - inv;
        if (2 * n < d) continue;  // the quotient is to lie in [1/2, 1)
        *x = (float)n;
        *y = (float)d;
        return;
    }
}
// x = m^2 - s with an odd 25-bit m and a small s: its root lies within |s| 2^-49
// of a rounding boundary.  s = 1 (mod 8) has a square root modulo 2^26.
static float hard_square(void) {
    const int64_t s = 8 * ((int64_t)(hard32() % 64) - 32) + 1;
    int64_t m = 1;
    for (int b = 3; b < 26; ++b)
        if ((m * m - s) & ((int64_t)1 << b)) m += (int64_t)1 << (b - 1);
    m &= (1 << 26) - 1;
    if (m >= 1 << 25) m = (1 << 26) - m;
    if (m < 1 << 24) m = (1 << 25) - m;
    return (float)(m * m - s);
}

static const long double kTwoPi = 6.283185307179586476925286766559005768L;

static long double truth(int kind, float a, float b) {
    switch (kind) {
    case QUOTIENT:
    case DIVISOR: return (long double)a / b;
    case ROOT: return sqrtl(a);
    case HYPOT: return sqrtl((long double)a * a + (long double)b * b);
    case ATAN2: return atan2l(a, b);
    case DIR_S: return a == 0.0f ? (long double)a : a / sqrtl((long double)a * a + (long double)b * b);
    case DIR_C:
        return a == 0.0f && b == 0.0f ? copysignl(1.0L, b)
                                      : b / sqrtl((long double)a * a + (long double)b * b);
    case ATANH: return atanhl(a);
    case COS: return cosl(a);
    case SIN_PI: return sinl((long double)0x1.921fb6p+1f * a);
    case TAN: return tanl(a);
    case COS2: return sqrtl((1.0L - (long double)a * a) * (1.0L - (long double)b * b));
    default: return remainderl(a, kTwoPi);
    }
}

static float library(int kind, float a, float b) {
    switch (kind) {
    case QUOTIENT:
    case DIVISOR: return a / b;
    case ROOT: return sqrtf(a);
    case HYPOT: return hypotf(a, b);
    case ATAN2: return (float)atan2((double)a, (double)b);
    case COS: return cosf(a);
    default: return atan2f(sinf(a), cosf(a));
    }
}

int main(void) {
    const size_t n = 1u << 21;
    std::vector<float> a(n), b(n), t(n), g(n);
    float *da, *db, *dt, *dg;
    CHECK(hipMalloc(&da, n * 4));
    CHECK(hipMalloc(&db, n * 4));
    CHECK(hipMalloc(&dt, n * 4));
    CHECK(hipMalloc(&dg, n * 4));
    const float inf = INFINITY;
    const float special[] = {0.0f, -0.0f, 1.0f, -1.0f, inf, -inf, NAN, 3.0e38f, -3.0e38f, 1.0e-40f, 5.0e4f, 1.0e9f};
    const int ns = (int)(sizeof special / sizeof special[0]);
    for (int kind = 0; kind < KINDS; ++kind) {
        // Tame arguments first, then (where the general form has limits)
        // every pair of special values.
        const bool limits = kind == QUOTIENT || kind == ROOT || kind == HYPOT || kind == ATAN2 ||
                            kind == COS || kind == WRAP;
        const size_t tail = limits ? (size_t)(ns * ns) : 0, tame_n = n - tail;
        for (size_t i = 0; i < tame_n; ++i) {
            a[i] = spread(-20, 13);
            b[i] = spread(-20, 13);
            if (kind == QUOTIENT || kind == DIVISOR) b[i] = fabsf(b[i]);
            if (kind == DIVISOR && i % 64 == 0) a[i] = spread(-126, 0) * 0x1p-20f;  // subnormal quotients
            if ((kind == QUOTIENT || kind == DIVISOR) && i % 16 == 1) hard_quotient(&a[i], &b[i]);
            if (kind == ROOT) a[i] = i % 64 ? fabsf(spread(-40, 26)) : 0.0f;
            if (kind == ROOT && i % 16 == 1) a[i] = hard_square();
            if (kind == ATANH) a[i] = sign() * (i % 2 ? 0.9999f * unit() : fminf(ldexpf(unit(), -(int)(next32() % 20)), 0.9999f));
            if (kind == ATANH && i % 1024 == 0) a[i] = sign() * 0.0f;
            if (kind == SIN_PI) a[i] = unit();
            if (kind == COS2) {
                a[i] = sign() * 0.35f * unit();
                b[i] = sign() * 0.44f * unit();
            }
            if (kind == TAN) a[i] = sign() * 0.75f * unit();
            if (kind == WRAP && i % 4 == 0) a[i] = sign() * 3.14159265f * (1.0f + ldexpf(sign() * unit(), -(int)(next32() % 24)));
            if ((kind == ATAN2 || kind == DIR_S || kind == DIR_C) && i % 8 == 0) {
                const float m = fabsf(spread(-20, 13));  // exact angles
                const int pick = (int)(next32() % 3);
                a[i] = sign() * (pick == 1 ? 0.0f : m);
                b[i] = sign() * (pick == 2 ? 0.0f : m);
            }
            if ((kind == HYPOT || kind == ATAN2 || kind == DIR_S || kind == DIR_C) && i % 32 == 5) {
                // zeros and the least floats
                a[i] = ldexpf((float)(hard32() % 4), -149) * (hard32() & 1 ? -1.0f : 1.0f);
                b[i] = ldexpf((float)(hard32() % 4), -149) * (hard32() & 1 ? -1.0f : 1.0f);
            }
        }
        for (size_t k = 0; k < tail; ++k) {
            a[tame_n + k] = special[k / ns];
            b[tame_n + k] = special[k % ns];
            if (kind == QUOTIENT && b[tame_n + k] == 0.0f) b[tame_n + k] = 2.0f;  // y is never 0
            if (kind == QUOTIENT) b[tame_n + k] = fabsf(b[tame_n + k]);
            if (kind == ROOT) a[tame_n + k] = fabsf(a[tame_n + k]);
        }
        CHECK(hipMemcpy(da, a.data(), n * 4, hipMemcpyHostToDevice));
        CHECK(hipMemcpy(db, b.data(), n * 4, hipMemcpyHostToDevice));
        run<<<1024, 256>>>(kind, da, db, dt, dg, n);
        CHECK(hipGetLastError());
        CHECK(hipMemcpy(t.data(), dt, n * 4, hipMemcpyDeviceToHost));
        CHECK(hipMemcpy(g.data(), dg, n * 4, hipMemcpyDeviceToHost));
        double worst = 0.0;
        size_t differ = 0, off = 0;
        for (size_t i = 0; i < tame_n; ++i) {
            differ += memcmp(&t[i], &g[i], 4) != 0;
            const long double want = truth(kind, a[i], b[i]);
            // An ulp of the result; the half turn's sine is added to 8, so an
            // ulp of 1, and a wrapped angle's remainder is within 2^-42.
            const float w = fabsf((float)want);
            const float floor_mag = kind == SIN_PI ? 1.0f : kind == WRAP ? 0x1p-20f : 0x1p-126f;
            const float mag = w > floor_mag ? w : floor_mag;
            const double ulp = (double)nextafterf(mag, inf) - (double)mag;
            const double e = (double)fabsl((long double)t[i] - want) / ulp;
            if (!(e <= worst)) worst = e;
            if (kind != SIN_PI && want == 0.0L && kind != HYPOT && kind != COS &&
                signbit(t[i]) != (want == 0.0L && signbit((float)want)))
                ++off;
        }
        for (size_t i = tame_n; i < n; ++i) {
            const float want = library(kind, a[i], b[i]);
            const bool nan = isnan(want) || isnan(g[i]);
            const bool same = nan ? isnan(want) == isnan(g[i])
                                  : fabsf(g[i] - want) <= 1.0e-6f * fabsf(want) + 1.0e-9f || g[i] == want;
            off += !same;
            if (!same) fprintf(stderr, "%s(%g, %g) = %g, library %g\n", kNames[kind], a[i], b[i], g[i], want);
        }
        printf("%s %zu %.9f %zu %zu\n", kNames[kind], n, worst, differ, off);
    }
    CHECK(hipFree(da));
    CHECK(hipFree(db));
    CHECK(hipFree(dt));
    CHECK(hipFree(dg));
    return 0;
}
