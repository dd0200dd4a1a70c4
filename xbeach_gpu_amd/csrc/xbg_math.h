// Deterministic elementary functions for the surf-beat step.
//
// The reference evaluates exp/log/pow/sinh/tanh/sin/cos with the host libm
// on its CPU path and with the CUDA device library on its GPU path; the two
// differ in the last bit now and then, and in the chaotic surf-zone flow a
// one-ulp difference grows to ~1e-3 relative after 1000 steps.  To make the
// HIP step reproduce its CPU oracle bit for bit, both use these functions.
//
// Every function is evaluated in double precision with only IEEE add,
// subtract, multiply, fused multiply-add, divide and exact scaling, in a fixed
// operation order; a multiply-add is fused where it is written so and nowhere
// else (both sides compile with -ffp-contract=off), so host and device produce
// identical bits.  The float entry points round the double result once; they
// agree with a correctly rounded libm except in double-rounding cases (about
// one input in 2^28).
//
// Methods.  The polynomials interpolate their functions at Chebyshev points
// (relative error of the result below 2e-17, fitted in extended precision).
//   exp   reduction by ln2 (two-part constant), 1 + r + r^2 Q(r), |r| <= ln2/2
//   sinh  the same reduction, r in [0, ln2), even and odd polynomials, no division
//   tanh  E / (E + 2), E = e^2a - 1 from exp's polynomial
//   log   reduction to [sqrt(1/2), sqrt(2)), s = f/(2+f), the odd series in s
//         and its reconstruction from f as in fdlibm e_log.c; 1/(2+f) from a
//         cubic and three Newton orders instead of a division
//   sin/cos  reduction by pi/2 (two-part constant, valid |x| < 2^19), kernel
//         polynomials of fdlibm k_sin.c / k_cos.c on |r| <= pi/4
//   expm1 fdlibm s_expm1.c rational form on |x| <= 1, exp(x)-1 outside
//   pow   exp(y * log|x|) with the integer-exponent sign rule; y = 2, 3, 4 and
//         8 as products in double
// A double division costs a wavefront of the GPU as much as some fifteen
// fused multiply-adds: exp with one took 2.5 times as long, tanh with three
// more than twice.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__) || defined(__HIP__)
#define XM_FN __host__ __device__ inline
#else
#define XM_FN inline
#endif

namespace xm {

XM_FN uint64_t bits(double x) { return __builtin_bit_cast(uint64_t, x); }
XM_FN double dbl(uint64_t b) { return __builtin_bit_cast(double, b); }
XM_FN bool isnan_(double x) { return x != x; }
XM_FN double inf_() { return dbl(0x7ff0000000000000ull); }
XM_FN double nan_() { return dbl(0x7ff8000000000000ull); }

XM_FN double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }

// x = k ln2 + hi - lo, hi exact; k = x / ln2 + shift rounded to an integer,
// from the low bits of a sum that rounds there (|x| < 2^20)
XM_FN double reduce_ln2(double x, double shift, int& k, double& lo) {
    const double ln2hi = 6.93147180369123816490e-01, ln2lo = 1.90821492927058770002e-10;
    const double invln2 = 1.44269504088896338700e+00, magic = 6755399441055744.0;  // 1.5 * 2^52
    const double t = shift == 0.0 ? fma_(x, invln2, magic) : fma_(x, invln2, shift) + magic, kd = t - magic;
    k = (int)(uint32_t)bits(t);
    lo = kd * ln2lo;
    return fma_(-kd, ln2hi, x);
}
// (e^r - 1 - r) / r^2 for |r| <= ln2/2
XM_FN double exp_q(double r) {
    double q = 2.0913209691564269e-09;
    q = fma_(q, r, 2.5105170644143384e-08);
    q = fma_(q, r, 2.755727803945201e-07);
    q = fma_(q, r, 2.7557255517955746e-06);
    q = fma_(q, r, 2.480158732088198e-05);
    q = fma_(q, r, 0.00019841269874720617);
    q = fma_(q, r, 0.0013888888888885856);
    q = fma_(q, r, 0.0083333333333261671);
    q = fma_(q, r, 0.041666666666666664);
    q = fma_(q, r, 0.16666666666666671);
    return fma_(q, r, 0.5);
}

XM_FN double exp(double x) {
    // at the ends the scaling gives inf and 0; NaN passes through
    const double xc = x > 710.0 ? 710.0 : (x < -746.0 ? -746.0 : x);
    int k;
    double lo;
    const double hi = reduce_ln2(xc, 0.0, k, lo), r = hi - lo;
    // with the part of hi - lo that r lost
    return __builtin_ldexp(1.0 + (r + fma_(r * r, exp_q(r), (hi - r) - lo)), k);
}

XM_FN double log(double x) {
    uint64_t b = bits(x);
    int k = 0;
    if (b - 0x0010000000000000ull >= 0x7fe0000000000000ull) {  // not a positive normal number
        if (isnan_(x) || x == inf_()) return x;
        if (x == 0.0) return -inf_();
        if (x < 0.0) return nan_();
        b = bits(x * dbl(0x4350000000000000ull));  // subnormal: 2^54
        k = -54;
    }
    // x = 2^k m, m in [sqrt(1/2), sqrt(2))
    uint32_t hi = (uint32_t)(b >> 32);
    const int e = (int)(hi - 0x3fe6a09eu) >> 20;
    k += e;
    hi -= (uint32_t)e << 20;
    const double f = dbl((uint64_t)hi << 32 | (uint32_t)b) - 1.0, d = 2.0 + f;
    double y = -0.057134684102826412;
    y = fma_(y, f, 0.12813395353460683);
    y = fma_(y, f, -0.25038631146362411);
    y = fma_(y, f, 0.49995694014279746);
    double g = fma_(-d, y, 1.0);
    y = fma_(y, fma_(g, g, g), y);
    g = fma_(-d, y, 1.0);
    y = fma_(y, g, y);
    const double s = f * y, w = s * s;
    double R = 0.14616719870254904;
    R = fma_(R, w, 0.15331699733323692);
    R = fma_(R, w, 0.18182889783543663);
    R = fma_(R, w, 0.22222211125751612);
    R = fma_(R, w, 0.28571428626030954);
    R = fma_(R, w, 0.39999999999899383);
    R = fma_(R, w, 0.66666666666666696);
    R = R * w;
    const double ln2hi = 6.93147180369123816490e-01, ln2lo = 1.90821492927058770002e-10;
    const double hfsq = 0.5 * f * f, dk = (double)k;
    return fma_(dk, ln2hi, -((hfsq - fma_(s, hfsq + R, dk * ln2lo)) - f));
}

XM_FN double log10(double x) { return log(x) * 0.43429448190325182765; }

XM_FN double expm1(double x) {
    if (isnan_(x)) return x;
    if (x > 1.0 || x < -1.0) return exp(x) - 1.0;
    // fdlibm s_expm1.c on |x| <= 1: reduction by one ln2 above 0.5 ln2,
    // rational approximation of the remainder, exact reconstruction
    const double ln2hi = 6.93147180369123816490e-01, ln2lo = 1.90821492927058770002e-10;
    const double Q1 = -3.33333333333331316428e-02, Q2 = 1.58730158725481460165e-03,
                 Q3 = -7.93650757867487942473e-05, Q4 = 4.00821782732936239552e-06,
                 Q5 = -2.01099218183624371326e-07;
    double ax = x < 0.0 ? -x : x;
    int k = 0;
    double c = 0.0;
    if (ax > 0.5 * 6.93147180559945286227e-01) {
        double hi, lo;
        if (x > 0.0) {
            hi = x - ln2hi;
            lo = ln2lo;
            k = 1;
        } else {
            hi = x + ln2hi;
            lo = -ln2lo;
            k = -1;
        }
        x = hi - lo;
        c = (hi - x) - lo;
    } else if (ax < 5.55111512312578270212e-17) {  // 2^-54
        return x;
    }
    double hfx = 0.5 * x;
    double hxs = x * hfx;
    double r1 = 1.0 + hxs * (Q1 + hxs * (Q2 + hxs * (Q3 + hxs * (Q4 + hxs * Q5))));
    double t = 3.0 - r1 * hfx;
    double e = hxs * ((r1 - t) / (6.0 - x * t));
    if (k == 0) return x - (x * e - hxs);
    e = (x * (e - c) - c);
    e = e - hxs;
    if (k == -1) return 0.5 * (x - e) - 0.5;
    if (x < -0.25) return -2.0 * (e - (x + 0.5));
    return 1.0 + 2.0 * (x - e);
}

// a = k ln2 + r, 0 <= r < ln2: e^+-a = 2^+-k (cosh r +- sinh r), and every
// term of sinh a is positive
XM_FN double sinh(double x) {
    const double a = x < 0.0 ? -x : x;
    double y;
    if (a > 700.0) {
        const double h = exp(0.5 * a);
        y = 0.5 * h * h;
    } else {
        int k;
        double lo;
        const double hi = reduce_ln2(a, -0.5, k, lo), r = hi - lo, z = r * r;
        double p = 1.1554240745674529e-11;
        p = fma_(p, z, 2.0876182888828003e-09);
        p = fma_(p, z, 2.755732119004969e-07);
        p = fma_(p, z, 2.4801587298108202e-05);
        p = fma_(p, z, 0.0013888888888891858);
        p = fma_(p, z, 0.041666666666666657);
        p = fma_(p, z, 0.5);
        double q = 7.69436449999226e-13;
        q = fma_(q, z, 1.6058738300383107e-10);
        q = fma_(q, z, 2.5052109335427469e-08);
        q = fma_(q, z, 2.7557319222561107e-06);
        q = fma_(q, z, 0.00019841269841270736);
        q = fma_(q, z, 0.0083333333333333332);
        q = fma_(q, z, 0.16666666666666666);
        const double e = (hi - r) - lo, s = r + fma_(q * z, r, e), c = 1.0 + fma_(p, z, e * r);
        const double u = dbl((uint64_t)(k + 1022) << 52), v = dbl((uint64_t)(1022 - k) << 52);  // 2^(k-1), 2^(-k-1)
        y = fma_(c, u - v, s * (u + v));
    }
    return __builtin_copysign(y, x);
}

// E / (E + 2), E = e^2a - 1 = 2^k (e^r - 1) + (2^k - 1)
XM_FN double tanh(double x) {
    double a = x < 0.0 ? -x : x;
    a = a > 22.0 ? 22.0 : a;  // 1 from there on
    int k;
    double lo;
    const double hi = reduce_ln2(2.0 * a, 0.0, k, lo), r = hi - lo;
    const double p = r + fma_(r * r, exp_q(r), (hi - r) - lo), u = dbl((uint64_t)(k + 1023) << 52);
    const double E = fma_(u, p, u - 1.0);
    const double y = E / (E + 2.0);
    return __builtin_copysign(y, x);
}

XM_FN double ksin(double r) {
    const double S1 = -1.66666666666666324348e-01, S2 = 8.33333333332248946124e-03,
                 S3 = -1.98412698298579493134e-04, S4 = 2.75573137070700676789e-06,
                 S5 = -2.50507602534068634195e-08, S6 = 1.58969099521155010221e-10;
    const double z = r * r, v = z * r;
    double q = fma_(S6, z, S5);
    q = fma_(q, z, S4);
    q = fma_(q, z, S3);
    q = fma_(q, z, S2);
    return fma_(v, fma_(q, z, S1), r);
}
XM_FN double kcos(double r) {
    const double C1 = 4.16666666666666019037e-02, C2 = -1.38888888888741095749e-03,
                 C3 = 2.48015872894767294178e-05, C4 = -2.75573143513906633035e-07,
                 C5 = 2.08757232129817482790e-09, C6 = -1.13596475577881948265e-11;
    const double z = r * r;
    double q = fma_(C6, z, C5);
    q = fma_(q, z, C4);
    q = fma_(q, z, C3);
    q = fma_(q, z, C2);
    q = fma_(q, z, C1) * z;
    const double hz = 0.5 * z, w = 1.0 - hz;
    return w + fma_(z, q, (1.0 - w) - hz);
}
// reduce by pi/2: r in [-pi/4, pi/4], quadrant q
XM_FN double rpio2(double x, int& q) {
    const double invpio2 = 6.36619772367581382433e-01, magic = 6755399441055744.0;
    const double pio2_1 = 1.57079632673412561417e+00, pio2_1t = 6.07710050650619224932e-11;
    const double t = fma_(x, invpio2, magic), k = t - magic;
    q = (int)(uint32_t)bits(t) & 3;
    return fma_(-k, pio2_1t, fma_(-k, pio2_1, x));
}
XM_FN double sin(double x) {
    int q;
    const double r = rpio2(x, q), v = q & 1 ? kcos(r) : ksin(r);
    return q & 2 ? -v : v;
}
XM_FN double cos(double x) {
    int q;
    const double r = rpio2(x, q), v = q & 1 ? ksin(r) : kcos(r);
    return (q + 1) & 2 ? -v : v;
}
// both, from one reduction (the same values)
XM_FN void sincos(double x, double& s, double& c) {
    int q;
    const double r = rpio2(x, q), ks = ksin(r), kc = kcos(r);
    s = q & 1 ? kc : ks;
    c = q & 1 ? ks : kc;
    s = q & 2 ? -s : s;
    c = (q + 1) & 2 ? -c : c;
}

XM_FN bool is_int(double y) {
    if (y != y || y == inf_() || y == -inf_()) return false;
    double a = y < 0 ? -y : y;
    if (a >= 4503599627370496.0) return true;  // 2^52
    double t = (double)(int64_t)a;
    return t == a;
}
XM_FN bool is_odd_int(double y) {
    if (!is_int(y)) return false;
    double a = y < 0 ? -y : y;
    if (a >= 9007199254740992.0) return false;  // 2^53: even
    return ((int64_t)a & 1) != 0;
}

XM_FN double pow(double x, double y) {
    if (y == 0.0) return 1.0;
    if (y == 2.0) return x * x;
    if (y == 3.0) return x * x * x;
    if (y == 4.0 || y == 8.0) {
        const double x2 = x * x, x4 = x2 * x2;
        return y == 4.0 ? x4 : x4 * x4;
    }
    if (x > 0.0 && x < inf_() && y - y == 0.0) return exp(y * log(x));
    if (x == 1.0) return 1.0;
    if (isnan_(x) || isnan_(y)) return nan_();
    if (x == 0.0) {
        if (y > 0.0) return is_odd_int(y) ? x : 0.0;
        return is_odd_int(y) && bits(x) >> 63 ? -inf_() : inf_();
    }
    double a = x;
    double sign = 1.0;
    if (x < 0.0) {
        if (!is_int(y)) return nan_();
        a = -x;
        if (is_odd_int(y)) sign = -1.0;
    }
    if (a == inf_()) return y > 0.0 ? sign * inf_() : sign * 0.0;
    return sign * exp(y * log(a));
}

// ---- correctly rounded float operations through double ----
// With a in double exactly, a few double operations that leave a relative
// error below 2^-51 give the IEEE float result, since no exact result that is
// not itself a float lies that near to a midpoint between floats: a square
// root of a float no nearer than 2^-51 (relative), a normal quotient of two
// floats no nearer than 2^-49.  A subnormal quotient can be an exact midpoint:
// subnormal results of div_by and div_near are to be formed by a division.

// sqrt(s) for a float s within a factor 1 +- 2^-20 of c*c, c a float in
// [1e-10, 1e10], hc = 0.5 / (double)c: with s = c^2 + d and t = d / (2c),
// sqrt(s) = c + t - t^2/(2c) + ..., the next term below 2^-62 of c; d is exact.
XM_FN float sqrt_near(float s, double c, double hc) {
    const double d = __builtin_fma(-c, c, (double)s), t = d * hc;
    return (float)__builtin_fma(t, __builtin_fma(-t, hc, 1.0), c);
}
// a / q for a float q within a factor 1 +- 2^-20 of c, rc = 1 / (double)c:
// 1/q = rc (1 + e + e^2 + ..), e = 1 - q rc.
XM_FN float div_near(float a, float q, double rc) {
    const double e = __builtin_fma(-(double)q, rc, 1.0);
    return (float)((double)a * __builtin_fma(rc, __builtin_fma(e, e, e), rc));
}
// a / b with rb = 1 / (double)b
XM_FN float div_by(float a, double rb) { return (float)((double)a * rb); }

// The wave dissipation's bins take these forms where no quotient of the cell
// can be subnormal.  The quotients are (a D) / E of the ee bins after a cap by
// idiv >= 1, and (gb b) / q of the rr bins, q within a factor 1 +- 2^-20 of c.
// small: nonzero_min over the ee bins before the cap and the rr bins; E >= 1e-7.
// Bins of at least 2^-90 after the cap and factors of at least 2^-31 leave
// quotients above 2^-122.
XM_FN uint32_t nonzero_min(uint32_t small, float v) {
    const uint32_t m = (__builtin_bit_cast(uint32_t, v) << 1) - 1u;  // zero wraps to the largest
    return m < small ? m : small;
}
XM_FN bool no_subnormal(float c, float D, float E, float gb, float idiv, uint32_t small) {
    return c > 1e-10f && c < 1e10f && !(D != 0.0f && D < 9.3e-10f * E) && (gb == 0.0f || gb >= 1e-5f * c) &&
           idiv < 1e6f && small >= (__builtin_bit_cast(uint32_t, 8.1e-28f * idiv) << 1);
}

// ---- float entry points: one rounding of the double result ----
XM_FN float expf(float x) { return (float)exp((double)x); }
XM_FN float logf(float x) { return (float)log((double)x); }
XM_FN float log10f(float x) { return (float)log10((double)x); }
XM_FN float powf(float x, float y) { return (float)pow((double)x, (double)y); }
XM_FN float sinhf(float x) { return (float)sinh((double)x); }
XM_FN float tanhf(float x) { return (float)tanh((double)x); }
XM_FN float sinf(float x) { return (float)sin((double)x); }
XM_FN float cosf(float x) { return (float)cos((double)x); }
XM_FN void sincosf(float x, float& s, float& c) {
    double ds, dc;
    sincos((double)x, ds, dc);
    s = (float)ds;
    c = (float)dc;
}

}  // namespace xm
