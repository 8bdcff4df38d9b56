// pump_device.hpp -- device arithmetic for PUMP's 2pBVP and collision tests
// on gfx950.
//
// Results are bit-identical to the reference's host build (x86-64, no FP
// contraction, pow(float,int) promoted to double):
//   * contraction is disabled for every function in this header (and the
//     library is compiled with -ffp-contract=off);
//   * pow(x,2) of a float is formed as x*x in double (exact); pow(x,3) and
//     pow(x,4) as (x*x)*x and (x*x)*(x*x), the correctly rounded powers.
//     glibc's pow differs from the correctly rounded value by one double ulp
//     for about 0.2% of arguments; after the final rounding to float the
//     outputs agree except in rare last-place cases, which the parity tests
//     count and bound;
//   * per-pair quantities that do not depend on tau are formed once (same
//     operations, same order) and reused by every cost evaluation.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#pragma clang fp contract(off)

namespace pump {

constexpr int kDim = 6;
constexpr float kGravity = -9.81f;  // 2pBVP.cu:3

// ---------------------------------------------------------------------------
// cost(tau, x0, x1), 2pBVP.cu:97-107, split into the tau-independent part
// (terms 1-7 of the numerator, summed in source order) and per-term factors.
// ---------------------------------------------------------------------------
struct CostTerms {
    double s7;                                     // 12a0^2+12a2^2+12a1^2+12b0^2+12b2^2-24a1b1+12b1^2
    float f8, f9, f10, f11, f12, f13, f14, f15;    // float products multiplied by tau
    double d16, d17, d18, d20, d22, d24;           // 4*pow(v,2), times tau^2
    double f19, f21, f23;                          // 4*v0*v1 (a float, held widened), times tau^2
    double f25, f26;                               // 2*g*vz (a float, held widened), times tau^3
    float f29a, f29b, f29c, f30a, f30b, f30c;      // 12*p0*(-2*p1 + (v0+v1)*tau)
};

__host__ __device__ __forceinline__ double sq(float x) { return (double)x * (double)x; }

__host__ __device__ __forceinline__ void cost_terms(CostTerms &c, const float *a, const float *b)
{
    const float g = kGravity;
    double s = 12.0 * sq(a[0]);
    s = s + 12.0 * sq(a[2]);
    s = s + 12.0 * sq(a[1]);
    s = s + 12.0 * sq(b[0]);
    s = s + 12.0 * sq(b[2]);
    s = s - (double)(24.0f * a[1] * b[1]);
    s = s + 12.0 * sq(b[1]);
    c.s7 = s;
    c.f8 = 12.0f * a[4] * a[1];
    c.f9 = 12.0f * a[1] * b[4];
    c.f10 = 12.0f * a[3] * b[0];
    c.f11 = 12.0f * b[3] * b[0];
    c.f12 = 12.0f * a[5] * b[2];
    c.f13 = 12.0f * b[5] * b[2];
    c.f14 = 12.0f * a[4] * b[1];
    c.f15 = 12.0f * b[4] * b[1];
    c.d16 = 4.0 * sq(a[4]);
    c.d17 = 4.0 * sq(a[3]);
    c.d18 = 4.0 * sq(a[5]);
    c.f19 = (double)(4.0f * a[4] * b[4]);
    c.d20 = 4.0 * sq(b[4]);
    c.f21 = (double)(4.0f * a[3] * b[3]);
    c.d22 = 4.0 * sq(b[3]);
    c.f23 = (double)(4.0f * a[5] * b[5]);
    c.d24 = 4.0 * sq(b[5]);
    c.f25 = (double)(2.0f * g * a[5]);
    c.f26 = (double)(2.0f * g * b[5]);
    c.f29a = 12.0f * a[0];
    c.f29b = -2.0f * b[0];
    c.f29c = a[3] + b[3];
    c.f30a = 12.0f * a[2];
    c.f30b = -2.0f * b[2];
    c.f30c = a[5] + b[5];
}

__host__ __device__ __forceinline__ float cost_eval(const CostTerms &c, float tau)
{
    const double g2 = (double)kGravity * (double)kGravity;
    const double t = (double)tau;
    const double t2 = t * t;   // exact
    const double t3 = t2 * t;  // correctly rounded
    const double t4 = t2 * t2; // correctly rounded
    double s = c.s7;
    s = s + (double)(c.f8 * tau);
    s = s + (double)(c.f9 * tau);
    s = s - (double)(c.f10 * tau);
    s = s - (double)(c.f11 * tau);
    s = s - (double)(c.f12 * tau);
    s = s - (double)(c.f13 * tau);
    s = s - (double)(c.f14 * tau);
    s = s - (double)(c.f15 * tau);
    s = s + c.d16 * t2;
    s = s + c.d17 * t2;
    s = s + c.d18 * t2;
    s = s + c.f19 * t2;
    s = s + c.d20 * t2;
    s = s + c.f21 * t2;
    s = s + c.d22 * t2;
    s = s + c.f23 * t2;
    s = s + c.d24 * t2;
    s = s + c.f25 * t3;
    s = s - c.f26 * t3;
    s = s + t4;
    s = s + g2 * t4;
    s = s + (double)(c.f29a * (c.f29b + c.f29c * tau));
    s = s + (double)(c.f30a * (c.f30b + c.f30c * tau));
    return (float)(1.0 / t3 * s);
}

// |RN(d / 1e-6f)| > 0.0001 exactly when |d| >= kDcostBig, for every float d
// (the quotient is monotone in d; the one transition over all finite
// positive floats lies between 0x1.b7cdfcp-34 and 0x1.b7cdfep-34).  NaN
// fails both tests.  It lets the bisection test dcost's magnitude without
// forming the quotient: toptBisection's loop condition (2pBVP.cu:85) and
// the signs it branches on (2pBVP.cu:75,79,88) depend on dcost only
// through this test and the sign of d, which the division by a positive
// dtau keeps.
constexpr float kDcostBig = 0x1.b7cdfep-34f;

// dcost, 2pBVP.cu:109-115: float central difference, dtau = 1e-6f
__host__ __device__ __forceinline__ float dcost_eval(const CostTerms &c, float tau)
{
    const float h = 0.000001f;
    float up = cost_eval(c, tau + h / 2.0f);
    float dn = cost_eval(c, tau - h / 2.0f);
    return (up - dn) / h;
}

// toptBisection, 2pBVP.cu:71-95 (halving loop capped at 400: the reference
// would not terminate once tl underflows to zero).
__host__ __device__ __forceinline__ float topt_bisection(const CostTerms &c, float tmax)
{
    float tu = tmax;
    if (dcost_eval(c, tmax) < 0.0f)
        return tmax;
    float tl = 0.01f;
    for (int k = 0; k < 400 && dcost_eval(c, tl) > 0.0f; ++k)
        tl = tl / 2.0f;
    float topt = 0.0f;
    float dcval = 1.0f;
    int itr = 0;
    while ((double)fabsf(dcval) > 0.0001 && itr < 50) {
        ++itr;
        topt = (tu + tl) / 2.0f;
        dcval = dcost_eval(c, topt);
        if (dcval > 0.0f)
            tu = topt;
        else
            tl = topt;
    }
    return topt;
}

// ---------------------------------------------------------------------------
// The same bisection with few full cost evaluations.
//
// toptBisection only uses the sign of dc = cost(xa) - cost(xb), xa = x + h/2
// and xb = x - h/2 rounded to float, and whether |dc| >= kDcostBig.  Far from
// the root both follow from the derivative, so most steps need no cost
// evaluation (deriv_sign); near it the cost is evaluated by a shorter FP64
// expression whose rounding to float is proven, case by case, to be that of
// cost_eval (cost_certified), which runs itself where the proof fails.
//
// Notation: u = 2^-24, t the evaluation point, and with the float products of
// CostTerms kept as they are, the numerator of the cost before the last
// division is s(t) = s7 + sum_i fl(l_i t) + fl(a29 fl(b29 + fl(c29 t))) +
// fl(a30 fl(b30 + fl(c30 t))) + n2 t^2 + n3 t^3 + k4 t^4, each fl one float
// rounding.  Without those roundings it is p(t) = n0 + n1 t + n2 t^2 + n3 t^3
// + k4 t^4, and C(t) = p(t) / t^3 has C'(t) = q(t) / t^4 with
// q(t) = k4 t^4 - n2 t^2 - 2 n1 t - 3 n0.
// MP(t) = |n0| + |n1| t + |n2| t^2 + |n3| t^3 + k4 t^4.
// ---------------------------------------------------------------------------
struct PairTerms {
    float l[8];                   // f8..f15 with the sign of their term
    float a29, b29, c29, a30, b30, c30;
    double s7, n2, n3;
};

// deriv_sign's constants of a pair
struct DerivTerms {
    float n0x3, n1x2, n2; // 3 n0, 2 n1, n2
    float n0, n1, n3;     // signed, for p and MP
    float k0, k1;         // bound of the float roundings at both points: (k0 + k1 t) / t^3
};

constexpr float kK4 = 1.0f + kGravity * kGravity;
constexpr float kTMin = 0x1p-7f, kTMax = 0x1p7f; // where deriv_sure holds
constexpr float kFastMin = 0x1p-10f;             // cost_fast's bound holds from here to kTMax

__host__ __device__ __forceinline__ void pair_terms(PairTerms &T, DerivTerms &D, const float *a,
                                                    const float *b)
{
    CostTerms c;
    cost_terms(c, a, b);
    T.l[0] = c.f8;
    T.l[1] = c.f9;
    T.l[2] = -c.f10;
    T.l[3] = -c.f11;
    T.l[4] = -c.f12;
    T.l[5] = -c.f13;
    T.l[6] = -c.f14;
    T.l[7] = -c.f15;
    T.a29 = c.f29a;
    T.b29 = c.f29b;
    T.c29 = c.f29c;
    T.a30 = c.f30a;
    T.b30 = c.f30b;
    T.c30 = c.f30c;
    T.s7 = c.s7;
    T.n2 = ((c.d16 + c.d17) + (c.d18 + c.f19)) + ((c.d20 + c.f21) + (c.d22 + c.f23)) + c.d24;
    T.n3 = c.f25 - c.f26;
    const double ab29 = (double)T.a29 * T.b29, ab30 = (double)T.a30 * T.b30;
    const double ac29 = (double)T.a29 * T.c29, ac30 = (double)T.a30 * T.c30;
    double n1 = ac29 + ac30;
    float F = 0.0f;
    for (int i = 0; i < 8; ++i) {
        n1 = n1 + (double)T.l[i];
        F = F + fabsf(T.l[i]);
    }
    const double n0 = (T.s7 + ab29) + ab30;
    D.n0 = (float)n0;
    D.n0x3 = (float)(3.0 * n0);
    D.n1 = (float)n1;
    D.n1x2 = 2.0f * D.n1;
    D.n2 = (float)T.n2;
    D.n3 = (float)T.n3;
    // fl(l t) is off by u |l| t, and fl(a fl(b + fl(c t))) by
    // |a| (2u (|b| + |c| t) + u |c| t); twice that for the two points
    D.k0 = 0x1p-22f * ((float)fabs(ab29) + (float)fabs(ab30));
    D.k1 = 0x1p-23f * (F + 3.0f * ((float)fabs(ac29) + (float)fabs(ac30)));
}

__host__ __device__ __forceinline__ float pair_mp(const DerivTerms &D, float t)
{
    return fmaf(fmaf(fmaf(fmaf(kK4, t, fabsf(D.n3)), t, fabsf(D.n2)), t, fabsf(D.n1)), t,
                fabsf(D.n0));
}

// The sign of dc at x: kPos (dc >= kDcostBig for certain), kNeg
// (dc <= -kDcostBig for certain), kZero (dc = 0 for certain) or kUnsure.
// With d = xa - xb (exact: both lie within a factor of two of each other):
//   * d = 0 makes both points equal, dc = 0.
//   * C(xa) - C(xb) = d C'(y) for a y in [xb, xa], and |C'(y) - C'(x)| <=
//     d max |C''| <= d 12 MP(x) / x^5 (1 + 1e-3) (|C''| <= 4 (k4 t^4 + n2 t^2
//     + 2 |n1| t + 3 |n0|) / t^5, and d/x <= 2^-12.8 for x >= 2^-7).
//   * cost_eval's float roundings before the final one move s by at most
//     (k0 + k1 t) / 2 at either point; its FP64 roundings by 2^-47 A(t), A the
//     sum of all terms' magnitudes (s7 as one).  A <= |n0| + (k0 + k1 t) 2^23
//     + 4.1 n2 t^2 + 2 k4 t^4 <= 5 MP + (k0 + k1 t) 2^23: s7 is n0 less ab29
//     and ab30; the velocity terms of n2 are in magnitude at most three times
//     n2; and 2|g| (|vz0| + |vz1|) t^3 <= n2 t^2 + k4 t^4.
//   * The final roundings add at most u |C| each (2^-150 for a subnormal, far
//     inside the slack of the kDcostBig term), with |C| t^3 <=
//     |p| + 2^-10 MP for p as evaluated here (rounding, and t within d).
// So the sign is sure, and |dc| >= kDcostBig, when
//   d |q| > x (k0 + k1 x + 2^-23 (|p| + 2^-10 MP)) + x^4 kDcostBig
//           + d MP (q's own rounding, 18u, and 12 d / x).
// Both sides are multiplied by x below, with the constants rounded up; the
// FP32 evaluation of the right side (positive terms) is covered by 1.002.
// A NaN or an infinity fails the comparison.
enum : int { kUnsure = 0, kPos = 1, kNeg = 2, kZero = 3 };

// The test above at x (within [kTMin, kTMax]), and q(x)
__host__ __device__ __forceinline__ bool deriv_sure(const DerivTerms &D, float x, float &q)
{
    const float h = 0.000001f;
    const float d = (x + h / 2.0f) - (x - h / 2.0f);
    const float x2 = x * x;
    q = fmaf(fmaf(fmaf(kK4, x2, -D.n2), x, -D.n1x2), x, -D.n0x3);
    const float p = fmaf(fmaf(fmaf(fmaf(kK4, x, D.n3), x, D.n2), x, D.n1), x, D.n0);
    const float mp = pair_mp(D, x);
    const float e = fmaf(D.k1, x, D.k0) + 0x1p-23f * fmaf(0x1p-10f, mp, fabsf(p));
    const float bound = fmaf(x2, fmaf(x2 * x, 1.1e-10f, e),
                             d * mp * fmaf(32.0f * 0x1p-24f, x, 24.0f * d));
    return d * fabsf(q) * x > 1.002f * bound;
}

__host__ __device__ __forceinline__ int deriv_sign(const DerivTerms &D, float x)
{
    const float h = 0.000001f;
    if (x + h / 2.0f == x - h / 2.0f)
        return kZero;
    float q;
    const bool sure = deriv_sure(D, x, q);
    if (!(x >= kTMin && x <= kTMax && sure))
        return kUnsure;
    return q > 0.0f ? kPos : kNeg;
}

// Approximations of 1/a and 1/b within 2^-51 relative, for b within 2^-8.3
// of a (the cubes of two points h apart, x >= kFastMin).
__host__ __device__ __forceinline__ void recip_near(double a, double b, double &ra, double &rb)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double r0 = __builtin_amdgcn_rcp(a);
    const double r1 = fma(r0, fma(-a, r0, 1.0), r0);
    ra = fma(r1, fma(-a, r1, 1.0), r1);
#else
    ra = 1.0 / a;
#endif
    // e = 1 - b ra: ra (1 + e + e^2) is within e^3 < 2^-24.9 of 1/b,
    // relative, and one Newton step squares that
    const double e = fma(-b, ra, 1.0);
    const double r = fma(ra, fma(e, e, e), ra);
    rb = fma(r, fma(-b, r, 1.0), r);
}

// The cost at x before its rounding to float, within 2^-47 A(x) / x^3 of
// cost_eval's: the float products are cost_eval's own; the other terms are
// summed by their common power.  In units of 2^-53 A / x^3: cost_eval's
// roundings on s after s7 are at most 25 (23 sums; the products and powers
// together 2), this form's 23 (the sum n2 8, n3 and k4 2, the Horner steps 3,
// the other sums 10), and t^3, reciprocal and final product 3 there and 7
// here: 58, and the rest to 64 covers the bound's FP32 evaluation, its value at
// the midpoint for both points, and its division by one's cube (the cubes
// differ by 0.3% at most).  r3: recip_near's 1/x^3.
__host__ __device__ __forceinline__ double cost_fast(const PairTerms &T, float x, double r3)
{
    const double k4 = 1.0 + (double)kGravity * (double)kGravity;
    const double t = (double)x;
    const double s0 = (double)(T.l[0] * x) + (double)(T.l[1] * x);
    const double s1 = (double)(T.l[2] * x) + (double)(T.l[3] * x);
    const double s2 = (double)(T.l[4] * x) + (double)(T.l[5] * x);
    const double s3 = (double)(T.l[6] * x) + (double)(T.l[7] * x);
    const double s4 = (double)(T.a29 * (T.b29 + T.c29 * x)) +
                      (double)(T.a30 * (T.b30 + T.c30 * x));
    const double lin = ((s0 + s1) + (s2 + s3)) + (s4 + T.s7);
    const double s = fma(t * t, fma(t, fma(t, k4, T.n3), T.n2), lin);
    return s * r3;
}

// cost_eval's result from cost_fast's C and the bound w of its distance:
// every value within w of C rounds to the same float.  False where that is
// not so (once in 10^4 evaluations) and for NaNs.  The sign of a zero is not
// settled.
__host__ __device__ __forceinline__ bool cost_certified(double C, double w, float &out)
{
    const float lo = (float)(C - w);
    out = (float)(C + w);
    return out == lo;
}

// A pair's place in toptBisection.  x is the next point: tmax (ST_TMAX), tl
// (ST_LOW), the bracket's midpoint (ST_BIS), the result, whose cost is still
// to be evaluated (ST_FIN) or has been (ST_DONE).
enum : int { ST_TMAX = 0, ST_LOW = 1, ST_BIS = 2, ST_FIN = 3, ST_DONE = 4, ST_IDLE = 5 };

// w (1 + x^4) / x^3 bounds |cost_fast - cost_eval| (w is infinite where that
// is not known, so that every cost comes from cost_eval).
struct BisectState {
    float tl, tu, x, w;
    int state, itr; // itr: bisection steps (ST_BIS), halvings (ST_LOW)
};

// The leading steps of toptBisection(tmax) that deriv_sign decides; steps
// is incremented by their number.  With tl >= kTMin and tu <= kTMax the
// bracket reaches neighbouring floats in fewer than 40 halvings, so no
// 50-step limit binds here; the loop's own limit only ends it should every
// sign be sure down to there, and the remaining steps follow one by one.
__host__ __device__ __forceinline__ void bisect_start(const DerivTerms &D, float tmax,
                                                      BisectState &S, int &steps)
{
    S.tl = 0.01f;
    S.tu = tmax;
    S.x = tmax;
    S.itr = 0;
    S.state = ST_TMAX;
    const int up = deriv_sign(D, tmax);
    if (up != kUnsure) {
        ++steps;
        S.state = up == kNeg ? ST_FIN : ST_LOW;
        S.tl = up == kNeg ? tmax : 0.01f;
        S.x = S.tl;
    }
    if (S.state == ST_LOW) {
        const int low = deriv_sign(D, S.tl);
        if (low == kNeg || low == kZero) {
            ++steps;
            S.state = ST_BIS;
            S.x = (S.tu + S.tl) / 2.0f;
        }
    }
    bool go = S.state == ST_BIS && S.tu <= kTMax;
    for (int k = 0; k < 40 && go; ++k) {
        float q;
        go = deriv_sure(D, S.x, q);
        if (go) {
            S.tu = q > 0.0f ? S.x : S.tu;
            S.tl = q > 0.0f ? S.tl : S.x;
            S.x = (S.tu + S.tl) / 2.0f;
            ++S.itr;
        }
    }
    steps += S.itr;
    // 2^-47 A(t) <= w (1 + t^4), as t <= 0.57 (1 + t^4) and t^2 <= 0.5 (1 + t^4)
    const float mid = fmaf(0x1p23f * 0.57f, D.k1, 2.05f * D.n2);
    const float w = 0x1p-47f * (mid + fmaxf(fmaf(0x1p23f, D.k0, fabsf(D.n0)), 2.0f * kK4));
    S.w = (S.x >= kFastMin && S.tl >= kFastMin && S.tu <= kTMax) ? w : INFINITY;
}

// One further step from the costs ca, cb at the step's two points (ca alone
// in ST_FIN).  dcost = (ca - cb) / h (2pBVP.cu:109-115) enters only through
// its sign, which is that of dc = ca - cb, and through |dcost| > 0.0001,
// which is |dc| >= kDcostBig.
// A midpoint that leaves the bracket as it was is a fixed point: every later
// step would evaluate the same x and do the same, up to the 50th, so the
// bisection ends there with the same result; skipped is their number.
__host__ __device__ __forceinline__ void bisect_update(BisectState &S, float ca, float cb,
                                                       int &skipped)
{
    const float dc = ca - cb;
    const bool pos = dc > 0.0f;
    skipped = 0;
    if (S.state == ST_BIS) {
        const float tu = pos ? S.x : S.tu, tl = pos ? S.tl : S.x;
        ++S.itr;
        const bool go_on = fabsf(dc) >= kDcostBig && S.itr < 50;
        const bool fixed = tu == S.tu && tl == S.tl;
        skipped = go_on && fixed ? 50 - S.itr : 0;
        S.tu = tu;
        S.tl = tl;
        S.state = go_on && !fixed ? ST_BIS : ST_FIN;
        S.x = go_on && !fixed ? (tu + tl) / 2.0f : S.x;
    } else if (S.state == ST_FIN) {
        S.state = ST_DONE;
    } else if (S.state == ST_TMAX) {
        S.state = dc < 0.0f ? ST_FIN : ST_LOW;
        S.x = dc < 0.0f ? S.x : S.tl;
    } else if (pos && S.itr < 400) {
        S.tl = S.tl / 2.0f;
        S.x = S.tl;
        ++S.itr;
        if (!(S.tl >= kFastMin))
            S.w = INFINITY;
    } else {
        S.state = ST_BIS;
        S.itr = 0;
        S.x = (S.tu + S.tl) / 2.0f;
    }
}

// The step's two points and costs; false where a rounding is not settled
// (the costs are cost_eval's at xa and xb then).
__host__ __device__ __forceinline__ bool bisect_costs(const PairTerms &T, const BisectState &S,
                                                      float &xa, float &xb, float &ca, float &cb)
{
    const float h = S.state == ST_FIN ? 0.0f : 0.000001f / 2.0f;
    xa = S.x + h;
    xb = S.x - h;
    const double a = (double)xa, b = (double)xb;
    double ra, rb;
    recip_near(a * a * a, b * b * b, ra, rb);
    const float x2 = S.x * S.x;
    const double w = (double)fmaf(S.w, x2 * x2, S.w) * ra;
    const bool oka = cost_certified(cost_fast(T, xa, ra), w, ca);
    const bool okb = cost_certified(cost_fast(T, xb, rb), w, cb);
    return oka && okb;
}

// ---------------------------------------------------------------------------
// pathPoint(t, tau, x0, x1), 2pBVP.cu:117-131
// ---------------------------------------------------------------------------
// Unsigned 32-bit division by a fixed d >= 1 (Granlund and Montgomery,
// PLDI 1994, the round-up form with a 33-bit multiplier 2^32 + m):
// l = ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1, and for every
// n < 2^32, n / d = (t + ((n - t) >> s1)) >> s2 with t = mulhi(m, n),
// s1 = min(l, 1), s2 = max(l - 1, 0).  m >= 1, so m = 0 can mark "not in use".
struct DivMagic {
    uint32_t m;
    uint32_t s1, s2;
};

inline DivMagic div_magic(uint32_t d)
{
    uint32_t l = 0;
    while (l < 32 && (1ull << l) < d)
        ++l;
    const uint64_t m = ((1ull << 32) * ((1ull << l) - d)) / d + 1;
    return DivMagic{(uint32_t)m, l ? 1u : 0u, l ? l - 1 : 0u};
}

__host__ __device__ __forceinline__ uint32_t div_magic_apply(uint32_t n, const DivMagic &dm)
{
    const uint32_t t = (uint32_t)(((uint64_t)dm.m * n) >> 32);
    return (t + ((n - t) >> dm.s1)) >> dm.s2;
}

struct TauPowers {
    float tau;
    double t3;     // tau^3 (tau^2 is exact and formed where it is used)
    double r2, r3; // correctly rounded 1/tau^2, 1/tau^3
};

__host__ __device__ __forceinline__ TauPowers tau_powers(float tau)
{
    TauPowers p;
    const double t2 = (double)tau * (double)tau;
    p.tau = tau;
    p.t3 = t2 * (double)tau;
    p.r2 = 1.0 / t2;
    p.r3 = 1.0 / p.t3;
    return p;
}

// Correctly rounded a/b from r = RN(1/b) (Markstein, IBM J. Res. Dev. 34(1),
// 1990): q0 = RN(a r) is within 1.5 ulp of a/b; one residual step
// q1 = RN(q0 + (a - b q0) r), with a - b q0 exact by FMA, brings it within
// 1 ulp, and a second step from a quotient within 1 ulp and a reciprocal
// within 1/2 ulp rounds correctly.  Valid while a/b, a and b stay clear of
// overflow and subnormals (|a| < 1e300, 1e-300 < |b| < 1e300 here).
// The residuals are formed as b q - a and subtracted, which keeps the sign
// of a zero quotient (a = -0 gives -0).
__host__ __device__ __forceinline__ double div_rn(double a, double b, double r)
{
    const double q0 = a * r;
    const double e0 = fma(b, q0, -a);
    const double q1 = fma(-e0, r, q0);
    const double e1 = fma(b, q1, -a);
    return fma(-e1, r, q1);
}

// Correctly rounded a/b for a divisor b = tau^2, the exact square of a float,
// from r = RN(1/b), in one residual step.  Write b = M^2 2^(2k) with M < 2^24
// an integer, so b is a multiple of u = 2^(2k) >= 2^-48 b, and q = a/b.
//   * q0 = RN(a r) is within 1.5 ulp(q) of q.  a - b q0 is a multiple of
//     u ulp(q0) and at most 1.5 ulp(q) b < 2^49 u ulp(q) in magnitude, so the
//     FMA forms it exactly.
//   * q0 + (a - b q0) r = q + (q - q0)(b r - 1), |b r - 1| <= 2^-53: the
//     exact value rounded by the second FMA is within 1.5 * 2^-53 ulp(q) of q.
//   * A rounding midpoint m (odd multiple of ulp(q)/2) is not q: m b has at
//     least 54 significant bits, a has 53.  And |q - m| = |a - m b| / b with
//     a - m b a non-zero multiple of min(ulp(a), u ulp(q) / 2), so
//     |q - m| >= 2^-49 ulp(q).
// Hence the rounding lands on RN(q).  Same range conditions as div_rn.
__host__ __device__ __forceinline__ double div_sq(double a, double b, double r)
{
    const double q0 = a * r;
    const double e0 = fma(b, q0, -a);
    return fma(-e0, r, q0);
}

// Per-edge constants of pathPoint (2pBVP.cu:117-131): every subexpression
// that depends only on (x0, x1, tau), formed with the same operations in the
// same order as the full expression, so a waypoint evaluated from them is
// bit-identical to the expression evaluated from scratch.  Per waypoint only
// the terms in t remain (about 100 FP64 operations instead of 165).  The
// products z0 tau^3 and vz0 tau^3 are one multiplication each and are
// formed where they are used.
struct EdgePoly {
    float c3[2], c2[2], cv[2]; // x, y: cubic and quadratic position terms, velocity term
    float e[2];                // x, y: velocity term of -(2 t e)
    double kz, dz;             // z position: bracket of s^2 tau, bracket of s^3
    double bv, cz;             // z velocity: bracket of t tau, bracket of s^2
};

__host__ __device__ __forceinline__ EdgePoly edge_poly(const float *x0, const float *x1,
                                                       const TauPowers &P)
{
    EdgePoly E;
    const float tau = P.tau;
    for (int d = 0; d < 2; ++d) {
        const float p0 = x0[d], v0 = x0[d + 3], p1 = x1[d], v1 = x1[d + 3];
        const float c3 = 2.0f * p0 - 2.0f * p1 + (v0 + v1) * tau;
        const float c2 = 3.0f * p0 - 3.0f * p1 + (2.0f * v0 + v1) * tau;
        const float c = 2.0f * p0 - 2.0f * p1 + v1 * tau;
        E.c3[d] = c3;
        E.c2[d] = c2;
        E.cv[d] = c;
        E.e[d] = 3.0f * p0 - 3.0f * p1 + v1 * tau;
    }
    const double z0 = (double)x0[2], z1 = (double)x1[2];
    const double vz0 = (double)x0[5], vz1 = (double)x1[5], td = (double)tau;
    E.kz = -3.0 * z0 + 3.0 * z1 - 2.0 * vz0 * td - 1.0 * vz1 * td;
    E.dz = 2.0 * z0 - 2.0 * z1 + (double)((x0[5] + x1[5]) * tau);
    E.bv = -6.0 * z0 + 6.0 * z1 - 4.0 * vz0 * td - 2.0 * vz1 * td;
    E.cz = 6.0 * z0 - 6.0 * z1 + 3.0 * vz0 * td + 3.0 * vz1 * td;
    return E;
}

// pathPoint at time t from the edge's constants; x0 supplies p0, v0 of x, y
// and z0, vz0
__host__ __device__ __forceinline__ void path_point(float t, const TauPowers &P, const EdgePoly &E,
                                                    const float *x0, float *x)
{
    const float tau = P.tau;
    const double t2 = (double)tau * (double)tau; // exact
    const double s2 = (double)t * (double)t;
    const double s3 = s2 * (double)t;
    const double q = 3.0 * s2 - (double)(4.0f * t * tau) + t2;
    for (int d = 0; d < 2; ++d) {
        const float p0 = x0[d], v0 = x0[d + 3];
        const float lin = t * v0 + p0;
        x[d] = (float)((double)lin + div_rn(s3 * (double)E.c3[d], P.t3, P.r3) -
                       div_sq(s2 * (double)E.c2[d], t2, P.r2));
        const float f = -(2.0f * t * E.e[d]);
        x[d + 3] = (float)(div_sq((double)f, t2, P.r2) + div_rn(3.0 * s2 * (double)E.cv[d], P.t3, P.r3) +
                           div_sq((double)v0 * q, t2, P.r2));
    }
    {
        const double a = (double)(t * x0[5]) * P.t3;
        const double c = s2 * (double)tau * E.kz;
        const double d = s3 * E.dz;
        const double bz = (double)x0[2] * P.t3;
        x[2] = (float)div_rn(a + bz + c + d, P.t3, P.r3);
    }
    {
        const double b = (double)(t * tau) * E.bv;
        const double c = s2 * E.cz;
        const double av = (double)x0[5] * P.t3;
        x[5] = (float)div_rn(av + b + c, P.t3, P.r3);
    }
}

__host__ __device__ __forceinline__ void path_point(float t, const TauPowers &P, const float *x0,
                                                    const float *x1, float *x)
{
    path_point(t, P, edge_poly(x0, x1, P), x0, x);
}

// Waypoint k of an edge with W waypoints (findDiscretizedPath,
// 2pBVP.cu:53-69): endpoints are copies, interior points at (tau/(W-1))*k.
// dt = tau/(W-1) is passed in when the caller has formed it once per edge.
__host__ __device__ __forceinline__ void waypoint_dt(int k, int W, const TauPowers &P, float dt,
                                            const float *x0, const float *x1, float *x)
{
    if (k == 0) {
        for (int d = 0; d < kDim; ++d)
            x[d] = x0[d];
    } else if (k == W - 1) {
        for (int d = 0; d < kDim; ++d)
            x[d] = x1[d];
    } else {
        path_point(dt * (float)k, P, x0, x1, x);
    }
}

__host__ __device__ __forceinline__ void waypoint_dt(int k, int W, const TauPowers &P,
                                                     const EdgePoly &E, float dt, const float *x0,
                                                     const float *x1, float *x)
{
    if (k == 0) {
        for (int d = 0; d < kDim; ++d)
            x[d] = x0[d];
    } else if (k == W - 1) {
        for (int d = 0; d < kDim; ++d)
            x[d] = x1[d];
    } else {
        path_point(dt * (float)k, P, E, x0, x);
    }
}

__host__ __device__ __forceinline__ void waypoint(int k, int W, const TauPowers &P, const float *x0,
                                         const float *x1, float *x)
{
    waypoint_dt(k, W, P, P.tau / (float)(W - 1), x0, x1, x);
}

// Bounding box of the positions of every waypoint of an edge.  The position
// part of pathPoint (2pBVP.cu:117-131) is the cubic Hermite segment through
// (x0, v0) and (x1, v1) over [0, tau], which lies in the convex hull of its
// Bezier control points x0, x0 + v0 tau/3, x1 - v1 tau/3, x1.  The waypoints
// are that cubic with FP32-rounded coefficients, rounded to FP32: their
// distance from it is below 30 * 2^-24 * S, S = |p0| + |p1| + |v0 tau| +
// |v1 tau|.  The hull is formed here in FP32 (within 4 * 2^-24 * S of the
// exact one, and lo/hi round by at most 2^-24 of their magnitude), so the
// margin 1e-5 (1 + S) covers every deviation with room to spare.
__host__ __device__ __forceinline__ void edge_bbox(const float *x0, const float *x1, float tau, float *lo,
                                          float *hi)
{
    const float t3 = tau * (1.0f / 3.0f);
    for (int d = 0; d < 3; ++d) {
        const float p0 = x0[d], p3 = x1[d];
        const float w0 = x0[d + 3] * t3, w1 = x1[d + 3] * t3;
        const float p1 = p0 + w0, p2 = p3 - w1;
        const float mn = fminf(fminf(p0, p1), fminf(p2, p3));
        const float mx = fmaxf(fmaxf(p0, p1), fmaxf(p2, p3));
        const float m = 1e-5f * (1.0f + fabsf(p0) + fabsf(p3) + 3.0f * (fabsf(w0) + fabsf(w1)));
        const float l = mn - m, h = mx + m;
        const bool finite = fabsf(l) < INFINITY && fabsf(h) < INFINITY; // false for NaN too
        lo[d] = finite ? l : -INFINITY;
        hi[d] = finite ? h : INFINITY;
    }
}

// ---------------------------------------------------------------------------
// Segment vs axis-aligned box, collisionCheck.cu:65-143 (isMotionValid,
// broadphaseValidQ, motionValidQ, faceContainsProjection).
// Boxes are given by their position bounds lo[3], hi[3].
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ bool face_contains(const float *v, const float *w, float lambda, int j,
                                              const float *lo, const float *hi)
{
    for (int d = 0; d < 3; ++d) {
        float proj = v[d] + (w[d] - v[d]) * lambda;
        if (d != j && !(lo[d] <= proj && proj <= hi[d]))
            return false;
    }
    return true;
}

// true if the segment v->w collides with the box (broad phase overlap and a
// face projection inside the box)
__host__ __device__ __forceinline__ bool segment_hits_box(const float *v, const float *w,
                                                 const float *bmin, const float *bmax,
                                                 const float *lo, const float *hi)
{
    for (int d = 0; d < 3; ++d)
        if (bmax[d] <= lo[d] || hi[d] <= bmin[d])
            return false;
    for (int d = 0; d < 3; ++d) {
        float vw = w[d] - v[d];
        float lambda = (v[d] < lo[d]) ? (lo[d] - v[d]) / vw : (hi[d] - v[d]) / vw;
        if (face_contains(v, w, lambda, d, lo, hi))
            return true;
    }
    return false;
}

__host__ __device__ __forceinline__ void seg_bbox(const float *v, const float *w, float *bmin, float *bmax)
{
    for (int d = 0; d < 3; ++d) {
        if (v[d] > w[d]) {
            bmin[d] = w[d];
            bmax[d] = v[d];
        } else {
            bmin[d] = v[d];
            bmax[d] = w[d];
        }
    }
}

// ---------------------------------------------------------------------------
// Obstacle boxes staged in LDS (position bounds only, structure of arrays);
// boxes past the capacity are read from global memory by the callers.
// ---------------------------------------------------------------------------
constexpr int kMaxObsLds = 512;

template <int N> struct ObsLdsN {
    float lo[3][N];
    float hi[3][N];
};
using ObsLds = ObsLdsN<kMaxObsLds>;

template <int N>
__device__ __forceinline__ void stage_obstacles(ObsLdsN<N> &o, const float *__restrict__ obs, int n)
{
    const int m = n < N ? n : N;
    for (int q = threadIdx.x; q < m * 3; q += blockDim.x) {
        int b = q / 3, d = q - 3 * (q / 3);
        o.lo[d][b] = obs[b * 12 + d];
        o.hi[d][b] = obs[b * 12 + 6 + d];
    }
}

// The staged rows are read through LDS-typed pointers: with two generic
// pointers the compiler merges the branches into one flat load through a
// selected address.
template <int N>
__device__ __forceinline__ void box_bounds(const ObsLdsN<N> &o, const float *__restrict__ obs, int b,
                                           float *lo, float *hi)
{
    typedef __attribute__((address_space(3))) const float LdsFloat;
    if (b < N) {
        for (int d = 0; d < 3; ++d) {
            lo[d] = ((LdsFloat *)o.lo[d])[b];
            hi[d] = ((LdsFloat *)o.hi[d])[b];
        }
    } else {
        for (int d = 0; d < 3; ++d) {
            lo[d] = obs[b * 12 + d];
            hi[d] = obs[b * 12 + 6 + d];
        }
    }
}

// true if segment v->w hits any of the n_obs boxes
__device__ __forceinline__ bool segment_blocked(const float *v, const float *w, const ObsLds &o,
                                                const float *__restrict__ obs, int n_obs)
{
    float bmin[3], bmax[3];
    seg_bbox(v, w, bmin, bmax);
    for (int b = 0; b < n_obs; ++b) {
        float lo[3], hi[3];
        box_bounds(o, obs, b, lo, hi);
        if (segment_hits_box(v, w, bmin, bmax, lo, hi))
            return true;
    }
    return false;
}

// index of the edge (within a block's edge run) holding global waypoint g,
// off[0] <= g < off[ne]
__device__ __forceinline__ int find_edge(const int64_t *off, int ne, int64_t g)
{
    int lo = 0, hi = ne;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (off[mid] <= g)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// index k of the instance whose blocks [prefix[k], prefix[k+1]) hold block b
// (prefix[0] = 0 <= b < prefix[n_inst]) in a batched launch over instances
__device__ __forceinline__ int instance_of(const int64_t *__restrict__ prefix, int n_inst,
                                           int64_t b)
{
    int lo = 0, hi = n_inst;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= b)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// DPP lane move: lane i of the result reads src from the lane that kCtrl
// names (wave_shl:1 = 0x130: from lane i + 1; row_ror:n = 0x120 + n within
// each row of 16); lanes without a source keep 0.
template <int kCtrl> __device__ __forceinline__ float dpp_move(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xf, 0xf, false));
}

__device__ __forceinline__ float read_lane(float x, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// Min / max over the 64 lanes of a wave (all lanes active): rotations within
// each row of 16, then the four row results.  They work on integers in the
// floats' order (x -> ordered_int(x), its own inverse): an integer min takes
// the rotation as its DPP operand, one instruction per step, and combines
// the row results on the scalar unit, where a float min needs a separate
// move and a canonicalisation per step.  A NaN orders beyond the infinity of
// its sign: a positive one is the result of the max and passed over by the
// min, a negative one the other way round.  A lane whose bounds may be NaN and
// must not be passed over gives infinite ones instead (edge_bbox, the
// half-space cache); in the full Monte Carlo a NaN segment hits nothing.
__device__ __forceinline__ int ordered_int(int i) { return i ^ ((i >> 31) & 0x7fffffff); }

template <int kCtrl> __device__ __forceinline__ int dpp_rotate(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, kCtrl, 0xf, 0xf, true);
}

__device__ __forceinline__ int wave_min_i(int x)
{
    x = min(x, dpp_rotate<0x121>(x));
    x = min(x, dpp_rotate<0x122>(x));
    x = min(x, dpp_rotate<0x124>(x));
    x = min(x, dpp_rotate<0x128>(x));
    return min(min(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
               min(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

__device__ __forceinline__ int wave_max_i(int x)
{
    x = max(x, dpp_rotate<0x121>(x));
    x = max(x, dpp_rotate<0x122>(x));
    x = max(x, dpp_rotate<0x124>(x));
    x = max(x, dpp_rotate<0x128>(x));
    return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
               max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

__device__ __forceinline__ float wave_min(float x)
{
    return __int_as_float(ordered_int(wave_min_i(ordered_int(__float_as_int(x)))));
}

__device__ __forceinline__ float wave_max(float x)
{
    return __int_as_float(ordered_int(wave_max_i(ordered_int(__float_as_int(x)))));
}

} // namespace pump


