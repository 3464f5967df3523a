// at_math.h -- device-side Axilrod-Teller arithmetic for gfx950.
//
// Two formulations of the same potential:
//  * the reference's gradient expression (potential/AxilrodTeller.cpp:22-93),
//    evaluated operation for operation in IEEE FP64 (this translation unit is
//    compiled with -ffp-contract=off, so nothing is fused), used by the
//    bit-exact path;
//  * the squared-distance form used by the fast paths:
//      u = |xj-xi|^2, v = |xk-xi|^2, w = |xk-xj|^2, s = (u v w)^-1/2,
//      A = u+v-w, B = u-v+w, C = -u+v+w, K = 3 nu / 8,
//      E = s^3 (nu + K Q),  Q = A B C s^2,
//      dE/du = s^5 (R v w + K (S - 2 A B)), dE/dv = s^5 (R u w + K (S - 2 A C)),
//      dE/dw = s^5 (R u v + K (S - 2 B C)),
//      S = BC + AC + AB, R = -3 nu / 2 - 5 K Q / 2.
//    Fused multiply-adds are written explicitly with fma() so the rounding of
//    this form is fixed by the source, not by the compiler.
#pragma once

#include <hip/hip_runtime.h>

namespace tb3 {

// Utility::Particle::GetSqrDistPeriodic (utility/structs.hpp:106-115):
// per axis t = |b - a|, e = min(t, L - t) with std::min's (b < a) ? b : a,
// result ex*ex + ey*ey + ez*ez.  No wrapping of positions: for t > L the
// second operand is negative and squares to (t - L)^2, exactly as the reference.
__device__ __forceinline__ double sqr_dist_periodic(double ax, double ay, double az, double bx, double by,
                                                    double bz, double Lx, double Ly, double Lz)
{
    const double tx = __builtin_fabs(bx - ax);
    const double ty = __builtin_fabs(by - ay);
    const double tz = __builtin_fabs(bz - az);
    const double lx = Lx - tx, ly = Ly - ty, lz = Lz - tz;
    const double ex = (lx < tx) ? lx : tx;
    const double ey = (ly < ty) ? ly : ty;
    const double ez = (lz < tz) ? lz : tz;
    return ex * ex + ey * ey + ez * ez;
}

// The same value with one v_min_f64 per axis instead of a compare and two
// selects.  It is bit-identical to sqr_dist_periodic for every input: t is
// |b - a| >= +0 and L > 0, so t and L - t are never both zero (no +0/-0
// tie), t is NaN exactly when L - t is (both operands NaN), and t = +inf gives
// L - t = -inf, which both forms return.
__device__ __forceinline__ double sqr_dist_periodic_min(double ax, double ay, double az, double bx, double by,
                                                        double bz, double Lx, double Ly, double Lz)
{
    const double tx = __builtin_fabs(bx - ax);
    const double ty = __builtin_fabs(by - ay);
    const double tz = __builtin_fabs(bz - az);
    const double ex = __builtin_fmin(tx, Lx - tx);
    const double ey = __builtin_fmin(ty, Ly - ty);
    const double ez = __builtin_fmin(tz, Lz - tz);
    return ex * ex + ey * ey + ez * ez;
}

// Correctly rounded FP64 division and square root for operands in range.
//
// gfx950 has no FP64 divide or square-root instruction; the compiler expands
// a / b into a Newton-Raphson sequence (reciprocal estimate, two refinements
// r <- r + r (1 - b r), quotient q = a r, and the Markstein correction
// q + r (a - b q), each step one FMA) wrapped in three range steps:
// v_div_scale scales an operand by a power of two when the quotient or the
// reciprocal would leave the normal range or the numerator is near the
// bottom of it, v_div_fmas undoes that scaling in the last FMA, and
// v_div_fixup handles zeros, infinities, NaNs and overflow.  For finite
// operands far inside the normal range (every caller here keeps numerators,
// denominators and quotients within 2^-500 .. 2^500, or a zero numerator)
// the scale step leaves both operands as they are, the last FMA is a plain
// FMA, and the fixup returns the quotient unchanged.
//
// div_rn_from leaves out those range steps and also the estimate and the
// first refinement: the caller gives an approximation r of 1 / b that is
// within 2^-46.  The refinement squares that error, so what goes into the
// quotient is 1 / b to within half an ulp and 2^-92, and the rest is the
// same: the bits of a / b in 5 instructions where the estimate (which issues
// at a quarter of the FMA's rate) and two refinements take 8, four of them
// for the estimate's slots.
// Why the bits: what the last FMA rounds is off from a / b by
// |a / b - q| |1 - b r|.  Near a midpoint m of two doubles q is half an ulp
// away, so with b scaled to [1, 2) that is at most ulp(q) b 2^-55 (1 + 2^-38),
// while a quotient that is no midpoint is at least ulp(q) 2^-53 / b away from
// it: it falls on the right side for b^2 < 4 (1 - 2^-38).  Left are b within
// 2^-38 of 2, b = 2 - t 2^-52.  There 1 / b is t^2 2^-107 past a midpoint of
// two doubles for odd t, and the refinement, short of 1 / b by 2^-93, rounds
// to the other side of it for odd t < 128 (how far past a midpoint the caller's
// r has to be off: t / 2 ulp); a correctly rounded reciprocal gives the right
// quotient.  Over those t the quotient is wrong for the one numerator that
// comes next to a midpoint: a power of two for t = 1, some other mantissa for
// t = 5, 11, 13, 25, ... 123, never 3 or 5 (all r within 2^-46, in exact
// rational arithmetic).  Callers whose numerator may be anything but those
// two send the denominators whose low word says that they may lie within 128
// steps under a power of two (div_is_hard) to div_rn.
//
// div_rn is the compiler's division with that set right: its reciprocal comes
// from two refinements of the estimate and is misrounded over t = 5, 11 and
// 13, so over the same denominators the exact remainders of the quotient and of
// its neighbour decide between the two (no quotient is a midpoint).
//
// The square root likewise: sqrt(x) rescales x when it is tiny and passes
// +-0 and +inf through around a Newton iteration on the reciprocal
// square-root estimate; for x within 2^-500 .. 2^500 those steps are the
// identity and sqrt_rn_inrange is the iteration alone (10 instructions
// instead of 17).  Its by-product h, half the reciprocal root, gives
// 1 / sqrt(x) to within 2^-52 in two more, from whose powers the reciprocals
// of the brackets' denominators are formed.
// Both are checked bit for bit on the device (tb3_selftest_fp64_inrange).
__device__ __forceinline__ unsigned low_word(double b) { return (unsigned)__double_as_longlong(b); }
__device__ __forceinline__ bool div_is_hard(unsigned low) { return low >= 0xffffff80u; }

__device__ __forceinline__ double div_rn_from(double a, double b, double r)
{
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    const double q = a * r;
    const double rem = __builtin_fma(-b, q, a);
    return __builtin_fma(rem, r, q);
}

__device__ __forceinline__ double div_rn(double a, double b)
{
    const double q = a / b, rem = __builtin_fma(-b, q, a);
    const long long away = (rem < 0.0) == (a < 0.0) ? 1 : -1;  // from zero, where |a| > |b q|
    const double next = __longlong_as_double(__double_as_longlong(q) + away);
    // (a remainder below 2^-960 may not be exact)
    const bool nearer =
        (__builtin_fabs(rem) >= 0x1p-960) & (__builtin_fabs(__builtin_fma(-b, next, a)) < __builtin_fabs(rem));
    return div_is_hard(low_word(b)) & nearer ? next : q;
}

__device__ __forceinline__ double sqrt_rn_inrange(double x, double &inv)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = y * 0.5;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    const double r = h + h;
    inv = __builtin_fma(r, __builtin_fma(-g, r, 1.0), r);
    return g;
}

// A side's powers (AxilrodTeller.cpp:33-51) and, for the in-range sequences,
// approximations of the reciprocals of those that the denominators take.
struct RefSide {
    double d1, d2, d3, d4, d5, d6;
    double i1, i2;
};

template <bool INRANGE>
__device__ __forceinline__ RefSide ref_powers(double d1, double i1)
{
    RefSide p;
    p.d1 = d1;
    p.d2 = p.d1 * d1;
    p.d3 = p.d2 * d1;
    p.d4 = p.d3 * d1;
    p.d5 = p.d4 * d1;
    p.d6 = p.d5 * d1;
    if constexpr (INRANGE) {
        p.i1 = i1;
        p.i2 = i1 * i1;
    }
    return p;
}

// a / b: the division proper, or the in-range sequence from r, the product of the
// sides' reciprocal powers (rounded powers and products: within 40 ulp of
// 1 / b), when the caller has checked the operands' range.
template <bool INRANGE>
__device__ __forceinline__ double ref_div(double a, double b, double r)
{
    if constexpr (INRANGE) return div_rn_from(a, b, r);
    else return div_rn(a, b);
}

// One dVdR bracket (AxilrodTeller.cpp:68-81) for own side x and the two other
// sides y, z in the order the source names them: dVdRa = (a; b, c),
// dVdRb = (b; a, c), dVdRc = (c; b, a).  Left-to-right sums and products.
// `low` collects the largest low word of the denominators whose numerators
// are or may be other than 3 and 5 (powers of two, 6, 5 d and 3 nu), for
// div_is_hard.
template <bool INRANGE>
__device__ __forceinline__ double ref_bracket(double nu, const RefSide &x, const RefSide &y, const RefSide &z,
                                              unsigned &low)
{
    // r1 = 1 / (x^4 y^3 z^3); the other denominators differ from it by even
    // powers of the ratios of two sides
    double a = 0, b = 0, ai = 0, bi = 0, r1 = 0, r3 = 0, r4 = 0, r5 = 0, r6 = 0;
    if constexpr (INRANGE) {
        a = x.d2 * y.i2;
        b = x.d2 * z.i2;
        ai = y.d2 * x.i2;
        bi = z.d2 * x.i2;
        const double yz = (y.i1 * z.i1) * (y.i2 * z.i2), x4 = x.i2 * x.i2;
        r1 = x4 * yz;
        r5 = r1 * b;
        r6 = r1 * a;
        r3 = (r5 * x4) * y.d3;
        r4 = (r6 * x4) * z.d3;
    }
    const double b1 = x.d4 * y.d3 * z.d3, b2 = y.d5 * z.d5, b3 = x.d6 * z.d5, b4 = x.d6 * y.d5;
    const double b5 = x.d2 * y.d3 * z.d5, b6 = x.d2 * y.d5 * z.d3;
    const double b0 = 8. * x.d1;
    if constexpr (INRANGE) {
        low = max(max(low, low_word(b1)), low_word(b2));
        low = max(max(low, low_word(b3)), low_word(b4));
        low = max(max(low, low_word(b5)), low_word(b6));
        low = max(low, low_word(b0));
    }
    double t = ref_div<INRANGE>(-8., b1, r1);
    t = t - ref_div<INRANGE>(1., b2, r5 * a);
    t = t + ref_div<INRANGE>(5. * y.d1, b3, r3);
    t = t + ref_div<INRANGE>(5. * z.d1, b4, r4);
    t = t - ref_div<INRANGE>(1., b5, r5);
    t = t - ref_div<INRANGE>(1., b6, r6);
    t = t - ref_div<INRANGE>(3., x.d4 * y.d1 * z.d5, r5 * ai);
    t = t - ref_div<INRANGE>(3., x.d4 * y.d5 * z.d1, r6 * bi);
    t = t - ref_div<INRANGE>(5., x.d6 * y.d1 * z.d3, r1 * ai);
    t = t - ref_div<INRANGE>(5., x.d6 * y.d3 * z.d1, r1 * bi);
    t = t + ref_div<INRANGE>(6., b1, r1);
    return ref_div<INRANGE>(3. * nu, b0, 0.125 * x.i1) * t;
}

// The range the in-range sequences need, per triplet: every squared side in
// [2^-80, 2^80] puts the sides in [2^-40, 2^40], so every product of powers
// in the brackets (at most the 11th power of a side in total) lies within
// 2^-440 .. 2^440, every quotient within 2^-500 .. 2^500 and the square
// roots' arguments within 2^-80 .. 2^80; nu must be 0 or within 2^-200 ..
// 2^200 (nu_inrange, checked once per launch), which keeps 3 nu / (8 d1)
// within 2^-250 .. 2^250.
__host__ __device__ inline bool nu_inrange(double nu)
{
    const double m = nu < 0 ? -nu : nu;
    return nu == 0.0 || (m >= 0x1p-200 && m <= 0x1p200);
}

// What AxilrodTeller::CalculateForces (AxilrodTeller.cpp:22-93) subtracts
// from the force of one particle p of a triplet, whose others are e and o in
// the triplet's order.  Written out for p as i (e = j, o = k; ROLE 0), as j
// (e = i, o = k; ROLE 1) and as k (e = i, o = j; ROLE 2), the three
// contributions have one form:
//   (e - p) S + (o - p) T,
// S and T being the brackets of the sides s = |e - p| and t = |o - p|; the
// reference's negated differences and brackets come in pairs, and negation is
// exact.  Only the order of a bracket's other two sides depends on p's place:
// the third side m = |o - e| comes last in both for i, first in both for j,
// and first in S, last in T for k.  Each operation is the reference's, so the
// result is bit-identical; the third bracket, which p's force does not take,
// is not evaluated.
template <int ROLE, bool INRANGE>
__device__ __forceinline__ void ref_pair_brackets(const RefSide &s, const RefSide &t, const RefSide &m, double nu,
                                                  double &S, double &T, unsigned &low)
{
    if constexpr (ROLE == 0) S = ref_bracket<INRANGE>(nu, s, t, m, low);
    else S = ref_bracket<INRANGE>(nu, s, m, t, low);
    if constexpr (ROLE == 1) T = ref_bracket<INRANGE>(nu, t, m, s, low);
    else T = ref_bracket<INRANGE>(nu, t, s, m, low);
}

// A squared side: |b|^2 and |-b|^2 are the same bits.
__device__ __forceinline__ double ref_sqr(double dx, double dy, double dz) { return (dx * dx + dy * dy) + dz * dz; }

// A side's length and its reciprocal, for the in-range sequences; zeros where
// the square is out of their range.
__device__ __forceinline__ double2 ref_root(double sq)
{
    double2 r = make_double2(0.0, 0.0);
    if (sq >= 0x1p-80 && sq <= 0x1p80) r.x = sqrt_rn_inrange(sq, r.y);
    return r;
}

// The contribution, given the three sides' ref_root.  The in-range sequences
// run where the sides and nu allow them (nu_ok = nu_inrange(nu), hoisted by
// the caller) and no denominator is a hard one, div_rn and the compiler's root
// elsewhere: the same bits either way.
template <int ROLE>
__device__ __forceinline__ void ref_contrib(double xp, double yp, double zp, double xe, double ye, double ze,
                                            double xo, double yo, double zo, double2 ss, double2 st, double2 sm,
                                            double nu, bool nu_ok, double &cx, double &cy, double &cz)
{
    const double ex = xe - xp, ey = ye - yp, ez = ze - zp;
    const double ox = xo - xp, oy = yo - yp, oz = zo - zp;
    double S = 0.0, T = 0.0;
    bool done = false;
    if (nu_ok && ss.y != 0.0 && st.y != 0.0 && sm.y != 0.0) {
        unsigned low = 0;
        ref_pair_brackets<ROLE, true>(ref_powers<true>(ss.x, ss.y), ref_powers<true>(st.x, st.y),
                                      ref_powers<true>(sm.x, sm.y), nu, S, T, low);
        done = !div_is_hard(low);
    }
    if (!done) {
        unsigned low;
        auto side = [](double sq) { return ref_powers<false>(__builtin_sqrt(sq), 0.0); };
        ref_pair_brackets<ROLE, false>(side(ref_sqr(ex, ey, ez)), side(ref_sqr(ox, oy, oz)),
                                       side(ref_sqr(xo - xe, yo - ye, zo - ze)), nu, S, T, low);
    }
    cx = ex * S + ox * T;
    cy = ey * S + oy * T;
    cz = ez * S + oz * T;
}

// The same from the positions alone.
template <int ROLE>
__device__ __forceinline__ void ref_contrib(double xp, double yp, double zp, double xe, double ye, double ze,
                                            double xo, double yo, double zo, double nu, bool nu_ok, double &cx,
                                            double &cy, double &cz)
{
    ref_contrib<ROLE>(xp, yp, zp, xe, ye, ze, xo, yo, zo, ref_root(ref_sqr(xe - xp, ye - yp, ze - zp)),
                      ref_root(ref_sqr(xo - xp, yo - yp, zo - zp)), ref_root(ref_sqr(xo - xe, yo - ye, zo - ze)), nu,
                      nu_ok, cx, cy, cz);
}

// ---------------------------------------------------------------------------
// Fast formulation.

// 1/sqrt(x) in FP64 from the hardware estimate.
__device__ __forceinline__ double rsqrt_f64(double x)
{
    // v_rsq_f64 is good to ~2^-24 (checked on device); one third-order step
    // y (1 + r/2 + 3 r^2/8) with r = 1 - x y^2 leaves an error of order r^3,
    // below the rounding of the FP64 result, in five operations.
    const double y = __builtin_amdgcn_rsq(x);
    const double r = __builtin_fma(-(x * y), y, 1.0);
    const double t = __builtin_fma(0.375, r, 0.5);
    return __builtin_fma(y * r, t, y);
}

// 1/sqrt(x) in FP32: hardware estimate refined by one Newton step.
__device__ __forceinline__ float rsqrt_f32(float x)
{
    float y = __builtin_amdgcn_rsqf(x);
    const float r = __builtin_fmaf(-(x * y), y, 1.0f);
    return __builtin_fmaf(0.5f * y, r, y);
}

// Mixed-precision form: u, v, w arrive in FP64 and A = u+v-w, B = u-v+w,
// C = -u+v+w are formed in FP64 before rounding to FP32, because for
// elongated triangles (two long sides of nearly equal length) the difference
// cancels and FP32 inputs would leave only a few correct bits; everything
// after that is FP32, and the coefficients come back in FP64.
//
// A triplet with one short side (a close pair) gives its third particle two
// huge, nearly opposite terms, -(eu dij + ev dik) for particle i when w is
// the short side: the FP32 rounding of eu and ev alone would leave that
// gradient with ~1e-6 relative error.  Two exact identities avoid this:
// X + Y = 2uC, X + Z = 2vB and Y + Z = 2wA give S = X + Y + Z and the third
// particle's coefficient sum (eu + ev for w, ev + ew for u, eu + ew for v)
// without cancellation; the coefficient paired with the sum is then rebuilt
// as sum - partner in FP64 (exact for FP32 operands), so that the third
// particle sees sum * (its vector) plus partner * (the short side).
// `live` scales the reciprocal root: 1, or 0 for a triplet that does not
// count (its coefficients and energy are then zero).
__device__ __forceinline__ void at_coeffs_mixed(double u64, double v64, double w64, float nu, float K, double &cu,
                                                double &cv, double &cw, float &e, bool need_w, float live = 1.0f)
{
    const float u = (float)u64, v = (float)v64, w = (float)w64;
    const float A = (float)((u64 + v64) - w64);
    const float B = (float)((u64 - v64) + w64);
    const float C = (float)((v64 - u64) + w64);
    const float uv = u * v;
    const float s = rsqrt_f32(uv * w) * live;
    const float s2 = s * s;
    const float X = B * C, Y = A * C, Z = A * B;
    const float Q = (A * X) * s2;
    const float R = __builtin_fmaf(-2.5f * K, Q, -1.5f * nu);
    // the shortest side m, the sum o of the other two, the factor P of 2 m P
    // in S, and the product G that completes S = G + 2 m P
    const bool wmin = w64 <= u64 && w64 <= v64;
    const bool umin = !wmin && u64 <= v64;
    const float m = wmin ? w : (umin ? u : v);
    const float o = wmin ? u + v : (umin ? v + w : w + u);
    const float P = wmin ? A : (umin ? C : B);
    const float G = wmin ? X : (umin ? Z : Y);
    const float S = __builtin_fmaf(2.0f * m, P, G);
    const float KS = K * S;
    const float m2K = -2.0f * K;
    const float c2s5 = 2.0f * (s2 * s2 * s);
    const double du = (double)(c2s5 * __builtin_fmaf(R, v * w, __builtin_fmaf(m2K, Z, KS)));
    const double dv = (double)(c2s5 * __builtin_fmaf(R, u * w, __builtin_fmaf(m2K, Y, KS)));
    e = (s2 * s) * __builtin_fmaf(K, Q, nu);
    if (need_w) {
        const double dw = (double)(c2s5 * __builtin_fmaf(R, uv, __builtin_fmaf(m2K, X, KS)));
        const double sum = (double)(c2s5 * __builtin_fmaf(R, m * o, __builtin_fmaf(m2K, 2.0f * m * P, 2.0f * KS)));
        // w shortest, third particle i: -(cu dij + cv dik), rebuild cv;
        // u shortest, k: cv dik + cw djk, rebuild cw; v shortest, j:
        // cu dij - cw djk with djk ~ -dij, rebuild cw
        const double rebuilt = sum - (umin ? dv : du);
        cu = du;
        cv = wmin ? rebuilt : dv;
        cw = wmin ? dw : rebuilt;
    } else {
        cu = du;
        cv = dv;
        cw = 0.0;
    }
}

// Gradient coefficients of one triplet in the squared-distance form, in FP64
// with s = (u v w)^-1/2 given; s = 0 (u, v, w finite) gives zero coefficients
// and energy.  Returns eu = 2 dE/du, ev = 2 dE/dv, ew = 2 dE/dw and the energy
// e, so that
//   dE/dxi = -(eu dij + ev dik), dE/dxj = eu dij - ew djk, dE/dxk = ev dik + ew djk
// with dij = xj - xi, dik = xk - xi, djk = xk - xj.
template <bool WANT_E>
__device__ __forceinline__ void at_coeffs_roots(double u, double v, double w, double s, double nu, double K,
                                                double &eu, double &ev, double &ew, double &e)
{
    const double s2 = s * s;
    const double d = u - v;
    const double A = (u + v) - w;
    const double B = d + w;
    const double C = w - d;
    const double X = B * C, Y = A * C, Z = A * B;
    const double Q = (A * X) * s2;
    const double R = __builtin_fma(-5.0 * K, Q, -3.0 * nu);
    const double S = (X + Y) + Z;
    const double KS = (2.0 * K) * S;
    const double m4K = -4.0 * K;
    const double s3 = s2 * s;
    const double s5 = s2 * s3;
    eu = s5 * __builtin_fma(R, v * w, __builtin_fma(m4K, Z, KS));
    ev = s5 * __builtin_fma(R, u * w, __builtin_fma(m4K, Y, KS));
    ew = s5 * __builtin_fma(R, u * v, __builtin_fma(m4K, X, KS));
    e = WANT_E ? s3 * __builtin_fma(K, Q, nu) : 0.0;
}

// Dispatch on the per-triplet type: FP64 throughout, or the mixed form; the
// gradient coefficients come back in FP64 either way.
template <class T, bool NEED_W>
__device__ __forceinline__ void at_coeffs_from64(double u, double v, double w, T nu, T K, double &cu, double &cv,
                                                 double &cw, T &e)
{
    if constexpr (sizeof(T) == 8) at_coeffs_roots<true>(u, v, w, rsqrt_f64(u * v * w), nu, K, cu, cv, cw, e);
    else at_coeffs_mixed(u, v, w, nu, K, cu, cv, cw, e, NEED_W);
}

}  // namespace tb3
