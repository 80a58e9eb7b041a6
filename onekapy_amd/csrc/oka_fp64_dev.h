// oka_fp64_dev.h -- FP64-exact tracing device code shared by the trace
// kernels (the workgroup tracer in oka_fp64.hip, the wave pool in
// oka_pool64.hip).
//
// Every floating-point expression is evaluated in the reference's operation
// order with contraction disabled, so that for identical inputs the results
// are bit-identical to the reference's numpy scalar arithmetic:
//   velocity           oneka/model.py:299-315, 343-350, 377-389, 423-427
//   feval              oneka/stochastic.py:253-260
//   Dormand-Prince     oneka/capturezone.py:198-253
//   segment raster     oneka/probabilityfield.py:292-310, 407-427
// Translation units that include it are compiled with -ffp-contract=off.
#pragma once

#include <math.h>

#include "oka_internal.h"
#include "oka_math.h"

#pragma clang fp contract(off)

namespace oka {
namespace fp64 {

// capturezone.py:202-209, each entry the correctly rounded quotient.
constexpr double A21 = 1.0 / 5.0;
constexpr double A31 = 3.0 / 40.0, A32 = 9.0 / 40.0;
constexpr double A41 = 44.0 / 45.0, A42 = -56.0 / 15.0, A43 = 32.0 / 9.0;
constexpr double A51 = 19372.0 / 6561.0, A52 = -25360.0 / 2187.0, A53 = 64448.0 / 6561.0,
                 A54 = -212.0 / 729.0;
constexpr double A61 = 9017.0 / 3168.0, A62 = -355.0 / 33.0, A63 = 46732.0 / 5247.0,
                 A64 = 49.0 / 176.0, A65 = -5103.0 / 18656.0;
constexpr double B1 = 35.0 / 384.0, B3 = 500.0 / 1113.0, B4 = 125.0 / 192.0,
                 B5 = -2187.0 / 6784.0, B6 = 11.0 / 84.0;
constexpr double E1 = 71.0 / 57600.0, E2 = -1.0 / 40.0, E3 = -71.0 / 16695.0,
                 E4 = 71.0 / 1920.0, E5 = -17253.0 / 339200.0, E6 = 22.0 / 525.0;

constexpr double kC2Pi = 0.15915494309189535;  // model.py:312-313
constexpr double kC4Pi = 0.07957747154594767;  // model.py:264
constexpr double kEps = 2.220446049250313e-16; // capturezone.py:199

// One well of a realization's field: position and -q (16-byte aligned, so
// that x and y load as one 128-bit LDS read and one address serves the well).
struct __align__(16) Well64 {
    double x, y, nq, pad;
};

// One realization's velocity field, but for its wells.
struct Field64 {
    int nw;
    int plain;           // kPlain*: when the short division sequences apply
    double xo, yo;
    double A, B, C, D, E, F;
    double A2, B2;       // 2.0*A, 2.0*B (exact)
    double K, bt, bn;    // conductivity, thickness, thickness*porosity
    double rbn;          // recip_plain(bn)
    double por, half_kb2;
};

// The field with its wells in LDS, a record each (the pool, whose lanes may be
// on different sites).
struct FieldLds : Field64 {
    const Well64 *w;
    static constexpr int kBlock = 2;   // wells per loop iteration (confined)
    __device__ __forceinline__ Well64 well(int i) const { return w[i]; }
};

// The field of a workgroup that is on one site: the wells' places come by
// scalar loads from the site's array (wave-uniform, in the scalar cache for
// every realization), and only the strengths are in LDS.  A broadcast LDS read
// of 16 bytes takes 16 cycles of the CU's LDS, so with whole records the four
// SIMDs' 24 bytes a well kept the LDS nearly as busy as their 24 issue slots
// kept them; a lone trace waits for one round trip per 4 wells instead of per
// 2.  Against records: 100 x 100 particles of a 4-well site 3 % less time,
// 10^4 x 1000 of a 25-well site 1-2 %.
typedef const __attribute__((address_space(4))) double *ConstF64;   // constant: scalar loads
struct FieldSite : Field64 {
    ConstF64 xy;         // nw x 2
    const double *nq;    // LDS
    static constexpr int kBlock = 4;
    __device__ __forceinline__ Well64 well(int i) const
    {
        return {xy[2 * i], xy[2 * i + 1], nq[i], 0.0};
    }
};

// a1 / b and a2 / b as the compiler divides: correctly rounded (IEEE division,
// as numpy's) but for some numerators of the divisors with mantissa 2 - k 2^-52,
// k = 5, 11 and 13 (see quot_plain; recip_plain's step here too would mend
// those and costs the tiled tracers 2 %).  gfx950 has no division instruction; the compiler expands every FP64 `/`
// into one fixed sequence:
//   d = div_scale(b; b, a)  r = rcp(d)  r += r (1 - d r)  r += r (1 - d r)
//   n, s = div_scale(a; b, a)  m = n r  q = div_fmas(fma(-d, m, n), r, m; s)
//   q = div_fixup(q, b, a)
// Only d and r depend on the numerator, through d's scaling of extreme
// exponents.  When both numerators leave d the same (always, in the normal
// range), this runs that sequence once for d and r and twice for the rest,
// so each result has the bits `a / b` would have; otherwise it divides twice.
__device__ __forceinline__ void div_pair(double a1, double a2, double b, double &q1, double &q2)
{
    bool s1, s2;
    const double d = __builtin_amdgcn_div_scale(a1, b, false, &s1);
    const double d2 = __builtin_amdgcn_div_scale(a2, b, false, &s2);
    if (__double_as_longlong(d) != __double_as_longlong(d2)) {
        q1 = a1 / b;
        q2 = a2 / b;
        return;
    }
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    const double n1 = __builtin_amdgcn_div_scale(a1, b, true, &s1);
    const double n2 = __builtin_amdgcn_div_scale(a2, b, true, &s2);
    const double m1 = n1 * r, m2 = n2 * r;
    q1 = __builtin_amdgcn_div_fixup(
        __builtin_amdgcn_div_fmas(fma(-d, m1, n1), r, m1, s1), b, a1);
    q2 = __builtin_amdgcn_div_fixup(
        __builtin_amdgcn_div_fmas(fma(-d, m2, n2), r, m2, s2), b, a2);
}

// 1 / b for a divisor that needs no scaling (see plain_coord): the hardware
// estimate r0 (relative error e0 below 2^-23, measured 2^-24.3 at most over
// 4e9 divisors) and one third-order step, r0 (1 + e0 + e0^2), whose error
// before its rounding is e0^3 < 2^-69.  One instruction less than two Newton
// steps.  With quot_plain a well term takes 21 VALU instructions instead of 24
// (the tracer is bound by their issue): 10^4 x 1000 particles of a 25-well
// site 149.8 -> 132.7 ms, with the regional quotient's shared reciprocal.
__device__ __forceinline__ double recip_plain(double b)
{
    const double r0 = __builtin_amdgcn_rcp(b);
    const double e = fma(-b, r0, 1.0);
    return fma(r0, fma(e, e, e), r0);
}

// a / b correctly rounded from r = recip_plain(b), for operands that need no
// scaling.  With |r b - 1| <= (1 + 2^-16) 2^-54 m (m in [1, 2) the mantissa of
// b), q0 = RN(a r) is one of the two doubles around any rounding boundary
// next to a / b, the residual a - b q0 is exact, and q0 + residual r lies
// within 2^-107 m (1 + 2^-16) (times the exponent of the quotient) of a / b.
// A quotient differs from a rounding boundary by at least 2^-105 / m, so the
// final rounding is that of a / b for every m < 2 - 2^-16.  Above it the proof
// needs r to be the double nearest to 1 / b.  There b is 2 - k 2^-52 (times a
// power of two) and 1 / b, for odd k, lies a relative k^2 2^-106 above the
// middle of two doubles, which the e0^3 that recip_plain leaves out could reach for k below
// 2^16.6.  But the hardware's estimate is then above 1 / b (it is one value for
// k = 2 to 2^20), so leaving out e0^3 < 0 errs upwards, and r is the upper of
// the two, the nearer one: checked on the GPU for every k up to 2^20 and six
// exponents.  (Two Newton steps give the lower one for k = 3, 5 .. 13, and the
// other double for some numerators of k = 5, 11 and 13.)  With the nearer r the
// quotients of the 32,080 numerators closest to a boundary, for the odd k up to
// 4,000 and four larger ones, are those of exact arithmetic.  The residual is
// formed negated, b q0 - a, so that a zero numerator keeps its sign through the
// sum (-(+0) r + (-0) = -0) and no div_fixup is needed.  0 / 0 gives NaN: r0 is
// infinite and e0 NaN.
__device__ __forceinline__ double quot_plain(double a, double b, double r)
{
    const double q0 = a * r;
    return fma(-fma(b, q0, -a), r, q0);
}

// The well terms' divisions (-q dx) / r2 and (-q dy) / r2 need no scaling
// when every coordinate involved (evaluation point and wells) is 0 or has a
// magnitude in [2^-200, 2^60), and every |q| is 0 or in [2^-100, 2^100]:
// a nonzero difference of two such coordinates is a multiple of 2^-252 below
// 2^61, so a nonzero r2 lies in [2^-504, 2^123), a nonzero numerator in
// [2^-353, 2^161], their exponents differ by less than 768 and no quotient
// is subnormal -- none of div_scale's conditions (tiny or huge denominator,
// exponent gap >= 768, subnormal quotient, numerator exponent <= 53) holds.
// r2 = 0 implies zero numerators: 0 / 0 gives NaN in both sequences.
// A point coordinate below 2^-200 is as good as 0 where every well's (and the
// origin's) coordinate is at least 2^-200 in magnitude: their difference is
// then the well's coordinate to within rounding.
__device__ __forceinline__ bool plain_coord(double v)
{
    const double a = fabs(v);
    return a == 0.0 || (a >= 0x1p-200 && a < 0x1p60);
}

__device__ __forceinline__ bool plain_strength(double nq)
{
    const double a = fabs(nq);
    return a == 0.0 || (a >= 0x1p-100 && a <= 0x1p100);
}

// Field64::plain: the short sequences never; where the point passes
// plain_coord; or, when no well coordinate is 0, where it is below 2^60.
enum { kPlainNever = 0, kPlainCoord = 1, kPlainBelow = 2 };

// What well w allows: combine over the wells with min().
__device__ __forceinline__ int plain_well(const Well64 &w)
{
    if (!(plain_coord(w.x) && plain_coord(w.y) && plain_strength(w.nq)))
        return kPlainNever;
    return w.x != 0.0 && w.y != 0.0 ? kPlainBelow : kPlainCoord;
}

// The same of one coordinate of the origin.
__device__ __forceinline__ int plain_origin(double v)
{
    return !plain_coord(v) ? kPlainNever : (v != 0.0 ? kPlainBelow : kPlainCoord);
}

// Whether the regional part allows the short quotient Q / bn: with these
// bounds Q is 0 or a multiple of 2^-540, bn and its reciprocal are far from
// the range's ends, and the residual of quot_plain is exact.
__device__ __forceinline__ bool plain_term(double c)
{
    const double a = fabs(c);
    return a == 0.0 || (a >= 0x1p-200 && a <= 0x1p100);
}

__device__ __forceinline__ bool plain_field(const Field64 &f)
{
    return plain_term(f.A2) && plain_term(f.B2) && plain_term(f.C) && plain_term(f.D) &&
           plain_term(f.E) && f.bn >= 0x1p-100 && f.bn <= 0x1p100;
}

// Whether the point (x, y) allows the short sequences, given that the field
// does (f.plain != kPlainNever).  NaN coordinates may pass: every sequence
// gives NaN for them.
__device__ __forceinline__ bool plain_point(const Field64 &f, double x, double y)
{
    return f.plain == kPlainBelow ? fmax(fabs(x), fabs(y)) < 0x1p60
                                  : plain_coord(x) && plain_coord(y);
}

__device__ __forceinline__ FieldSite make_field(const TraceArgs &a, int r, const double *nq,
                                                int plain)
{
    FieldSite f;
    f.xy = (ConstF64)a.wells_xy;
    f.nq = nq;
    f.nw = a.nwells;
    f.xo = a.xo;
    f.yo = a.yo;
    const double *c = a.coef + 6 * (int64_t)r;
    f.A = c[0];
    f.B = c[1];
    f.C = c[2];
    f.D = c[3];
    f.E = c[4];
    f.F = c[5];
    f.A2 = 2.0 * f.A;
    f.B2 = 2.0 * f.B;
    f.K = a.K[r];
    f.bt = a.b[r];
    f.por = a.n[r];
    f.bn = f.bt * f.por;
    f.rbn = recip_plain(f.bn);
    f.half_kb2 = (0.5 * f.K) * (f.bt * f.bt);
    f.plain = plain_field(f) ? plain : kPlainNever;
    return f;
}

// The wells' part of the discharge at (x, y) (model.py:307-313) and, for the
// unconfined field, of the potential (model.py:258-264).
template <bool kConfined, bool kPlain, class F>
__device__ __forceinline__ void well_sums(const F &f, double x, double y, double &Qx, double &Qy,
                                          double &pw)
{
    auto term = [&](const Well64 &wl) {
        const double ddx = x - wl.x;
        const double ddy = y - wl.y;
        const double r2 = ddx * ddx + ddy * ddy;
        double sx, sy;
        if (kPlain) {
            const double r = recip_plain(r2);
            sx = quot_plain(wl.nq * ddx, r2, r);
            sy = quot_plain(wl.nq * ddy, r2, r);
        } else {
            div_pair(wl.nq * ddx, wl.nq * ddy, r2, sx, sy);
        }
        Qx = Qx + sx * kC2Pi;
        Qy = Qy + sy * kC2Pi;
        if (!kConfined)
            pw = pw + ((-wl.nq) * log_rn(r2)) * kC4Pi;
    };
    // several wells per iteration in the confined field, their loads issued
    // together (the unconfined loop, with its logarithms, is slower unrolled)
    constexpr int kBlock = kConfined && kPlain ? F::kBlock : 1;
    int w = 0;
    for (; w + kBlock <= f.nw; w += kBlock) {
        Well64 wl[kBlock];
#pragma unroll
        for (int k = 0; k < kBlock; ++k)
            wl[k] = f.well(w + k);
#pragma unroll
        for (int k = 0; k < kBlock; ++k)
            term(wl[k]);
    }
    if (kBlock > 1)
        for (; w < f.nw; ++w)
            term(f.well(w));
}

// feval(xy) = -V(xy) (stochastic.py:253-260).  Returns false where the
// reference raises AquiferError (unconfined only).  kPlain uses the short
// division sequences and clears `ok` when (x, y) does not allow them: the
// result is then discarded and computed again without kPlain.
template <bool kConfined, bool kPlain, class F>
__device__ __forceinline__ bool feval(const F &f, double x, double y, double &kx, double &ky,
                                      bool &ok)
{
    const double dx = x - f.xo;
    const double dy = y - f.yo;
    double Qx = -((f.A2 * dx + f.C * dy) + f.D);
    double Qy = -((f.B2 * dy + f.C * dx) + f.E);
    double pw = 0.0;
    if (kPlain)
        ok = ok && plain_point(f, x, y);
    well_sums<kConfined, kPlain>(f, x, y, Qx, Qy, pw);
    double vx, vy;
    if (kConfined) {
        if (kPlain) {
            vx = quot_plain(Qx, f.bn, f.rbn);
            vy = quot_plain(Qy, f.bn, f.rbn);
        } else {
            div_pair(Qx, Qy, f.bn, vx, vy);
        }
        kx = -vx;
        ky = -vy;
        return true;
    }
    double pot = f.A * (dx * dx) + f.B * (dy * dy);
    pot = pot + (f.C * dx) * dy;
    pot = pot + f.D * dx;
    pot = pot + f.E * dy;
    pot = pot + f.F;
    pot = pot + pw;
    if (pot <= 0.0)
        return false;
    const double head = pot < f.half_kb2 ? sqrt((2.0 * pot) / f.K) : (pot + f.half_kb2) / (f.K * f.bt);
    if (head <= 0.0)
        return false;
    const double den = head > f.bt ? f.bn : head * f.por;
    div_pair(Qx, Qy, den, vx, vy);
    kx = -vx;
    ky = -vy;
    return true;
}

// One field evaluation of every active lane: with the short sequences, and
// again without them when the field or any lane's point does not allow them.
// Both give the same bits where they apply (but for div_pair's exception), so
// one such lane may take its wave along, and the long sequence stays off the
// usual path.
template <bool kConfined, class F>
__device__ __forceinline__ bool eval64(const F &f, double x, double y, double &kx, double &ky)
{
    bool ok = f.plain != kPlainNever, wet = false;
    if (ok)
        wet = feval<kConfined, true>(f, x, y, kx, ky, ok);
    if (__ballot(!ok) != 0ull)
        wet = feval<kConfined, false>(f, x, y, kx, ky, ok);
    return wet;
}

struct Integ {
    double dur, absdur, tol, maxstep, sg;
    int64_t cap;
};

struct Trace64 {
    double x, y, t, dt, k1x, k1y;
    double bx0, bx1, by0, by1;
    int64_t att, acc;
    int status;
};

// pow_fifth(x), by a shorter way that gives the same bits: w ~ u^(-1/5) from
// the hardware's base-2 logarithm and exponential (relative error below 2^-18)
// and one third-order step (then below 2^-52), y = u w^4, and pow_fifth's own
// double-double Newton step, with w^4 in place of its division.  x^(0.2 - 1/5)
// = 1 + t takes a logarithm good to 2^-20.  The sum hi + lo is within 2^-75 of
// the power, so it decides the rounding unless the two ends of hi + lo
// (1 +- 2^-70) round apart (once in some 10^5 calls), or x is not an ordinary
// number: pow_fifth then decides.  A third of its instructions, and no
// division.  With step_factor, 10^4 x 1000 particles of the 25-well site 131.2
// -> 126.2 ms, 100 x 100 of the 4-well site (whose lone traces wait for the
// chain) 9 % less.
__device__ __forceinline__ double pow_fifth_fast(double x)
{
    if (x >= 0x1p-900 && x <= 0x1p900) {
        int e;
        const double m = split_exponent(x, &e);
        const int q = (e + 1000) / 5 - 200;
        const int r = e - 5 * q;                              // 0..4
        const double u = m * (double)(1 << r);                // exact, in [1, 32)
        const float lm = __builtin_amdgcn_logf((float)m);     // base 2
        double w = (double)__builtin_amdgcn_exp2f(-0.2f * (lm + (float)r));
        double w2 = w * w;
        double w4 = w2 * w2;
        const double d = fma_(-u, w4 * w, 1.0);
        w = fma_(w, d * fma_(0.12, d, 0.2), w);
        w2 = w * w;
        w4 = w2 * w2;
        const double y = u * w4;
        const dd y2 = two_prod(y, y);
        const dd y4 = dd_mul(y2, y2);
        const dd y5 = dd_mul_d(y4, y);
        dd rho = two_sum(u, -y5.hi);
        rho.lo = rho.lo - y5.lo;
        const double dy = (rho.hi + rho.lo) * (0.2 * w4);
        const dd root = fast_two_sum(y, dy);
        const double t = 0x1.999999999999ap-57 * (((double)e + (double)lm) * OKA_LN2_HI);
        const double lo = root.lo + root.hi * t;
        const double err = root.hi * 0x1p-70;
        const double a = root.hi + (lo - err), b = root.hi + (lo + err);
        if (a == b)
            return a * pow2i(q);
    }
    return pow_fifth(x);
}

// The step factor min(pow(tol / (est + EPS), 0.2), maxstep / (ds + EPS), 10)
// of capturezone.py:243-247, as its comparisons give it.  Where the power is
// certainly above the lesser of the other two, tol > (est + EPS) c^5 (1 +
// 2^-30) with c^5 in double, it is not evaluated: away from wells the length
// of the step decides.
__device__ __forceinline__ double step_factor(double tol, double maxstep, double est, double ds)
{
    const double c2 = maxstep / (ds + kEps);
    double c = c2 < 10.0 ? c2 : 10.0;
    const double p2 = c * c, p5 = (p2 * p2) * c;
    const bool above = tol >= 0x1p-500 && ((est + kEps) * p5) * (1.0 + 0x1p-30) < tol;
    if (!above) {
        c = pow_fifth_fast(tol / (est + kEps));
        if (c2 < c)
            c = c2;
        if (10.0 < c)
            c = 10.0;
    }
    return c;
}

// Opens a trace at (xs, ys) (capturezone.py:211-217).  Its k1 = f(start) is
// the next advance64's evaluation.
__device__ __forceinline__ void open64(Trace64 &s, const Integ &I, double xs, double ys)
{
    s.x = xs;
    s.y = ys;
    s.t = 0.0;
    s.dt = 0.1 * I.sg;
    s.k1x = s.k1y = 0.0;
    s.att = 0;
    s.acc = 0;
    s.bx0 = s.bx1 = xs;
    s.by0 = s.by1 = ys;
    s.status = OKA_TRACE_OK;
}

// The stages of an attempted step.
struct Stages64 {
    double k3x, k3y, k4x, k4y, k5x, k5y, k6x, k6y, k7x, k7y, xn, yn;
};

// Stages 3 to 7 of an attempted step of size dt given k2
// (capturezone.py:228-240); false where an evaluation raises.
template <bool kConfined, bool kPlain, class F>
__device__ __forceinline__ bool dp5_stages(const F &f, const Trace64 &s, double dt,
                                           double k2x, double k2y, Stages64 &k, bool &ok)
{
    const double x = s.x, y = s.y, k1x = s.k1x, k1y = s.k1y;
    if (!feval<kConfined, kPlain>(f, x + dt * (A31 * k1x + A32 * k2x),
                                  y + dt * (A31 * k1y + A32 * k2y), k.k3x, k.k3y, ok))
        return false;
    if (!feval<kConfined, kPlain>(f, x + dt * ((A41 * k1x + A42 * k2x) + A43 * k.k3x),
                                  y + dt * ((A41 * k1y + A42 * k2y) + A43 * k.k3y), k.k4x, k.k4y,
                                  ok))
        return false;
    if (!feval<kConfined, kPlain>(
            f, x + dt * (((A51 * k1x + A52 * k2x) + A53 * k.k3x) + A54 * k.k4x),
            y + dt * (((A51 * k1y + A52 * k2y) + A53 * k.k3y) + A54 * k.k4y), k.k5x, k.k5y, ok))
        return false;
    if (!feval<kConfined, kPlain>(
            f, x + dt * ((((A61 * k1x + A62 * k2x) + A63 * k.k3x) + A64 * k.k4x) + A65 * k.k5x),
            y + dt * ((((A61 * k1y + A62 * k2y) + A63 * k.k3y) + A64 * k.k4y) + A65 * k.k5y),
            k.k6x, k.k6y, ok))
        return false;
    k.xn = x + dt * ((((B1 * k1x + B3 * k.k3x) + B4 * k.k4x) + B5 * k.k5x) + B6 * k.k6x);
    k.yn = y + dt * ((((B1 * k1y + B3 * k.k3y) + B4 * k.k4y) + B5 * k.k5y) + B6 * k.k6y);
    return feval<kConfined, kPlain>(f, k.xn, k.yn, k.k7x, k.k7y, ok);
}

// One iteration of a trace: k1 of a fresh trace (capturezone.py:218-219), else
// an attempted step (capturezone.py:221-247).  Returns bit 0 = accepted
// (segment (ox, oy) -> (s.x, s.y)), bit 1 = the trace has ended.  A fresh
// trace's k1 is its lane's share of the evaluation that the wave's other
// lanes spend on their step's second stage, so starting a trace costs the
// wave no evaluation of its own.
template <bool kConfined, class F>
__device__ __forceinline__ int advance64(const F &f, const Integ &I, Trace64 &s, bool &fresh,
                                         double &ox, double &oy)
{
    double dt = s.dt;
    if (fabs(s.t + dt) > I.absdur)
        dt = I.dur - s.t;
    const double x = s.x, y = s.y, k1x = s.k1x, k1y = s.k1y;
    double k2x, k2y;
    bool wet = eval64<kConfined>(f, fresh ? x : x + dt * (A21 * k1x),
                                 fresh ? y : y + dt * (A21 * k1y), k2x, k2y);
    if (fresh) {
        fresh = false;
        s.k1x = k2x;
        s.k1y = k2y;
        if (!wet)
            s.status = OKA_TRACE_TRUNCATED;
        return wet && 0.0 < I.absdur ? 0 : 2;
    }
    s.att += 1;
    Stages64 k;
    bool ok = f.plain != kPlainNever;
    if (wet) {
        if (ok)
            wet = dp5_stages<kConfined, true>(f, s, dt, k2x, k2y, k, ok);
        if (__ballot(!ok) != 0ull)
            wet = dp5_stages<kConfined, false>(f, s, dt, k2x, k2y, k, ok);
    }
    if (!wet) {
        s.status = OKA_TRACE_TRUNCATED;
        return 2;
    }
    const double ex =
        dt * (((((E1 * k1x + E2 * k.k7x) + E3 * k.k3x) + E4 * k.k4x) + E5 * k.k5x) + E6 * k.k6x);
    const double ey =
        dt * (((((E1 * k1y + E2 * k.k7y) + E3 * k.k3y) + E4 * k.k4y) + E5 * k.k5y) + E6 * k.k6y);
    const double ax = fabs(ex), ay = fabs(ey);
    const double est = (isnan(ax) || isnan(ay)) ? (double)NAN : (ay > ax ? ay : ax);
    const double d0 = k.xn - x, d1 = k.yn - y;
    const double ds = sqrt(fma_(d1, d1, d0 * d0));  // numpy norm: sqrt of a contracted ddot
    int res = 0;
    if (est < I.tol && ds < I.maxstep) {
        s.t = s.t + dt;
        s.k1x = k.k7x;
        s.k1y = k.k7y;
        ox = x;
        oy = y;
        s.x = k.xn;
        s.y = k.yn;
        s.acc += 1;
        s.bx0 = k.xn < s.bx0 ? k.xn : s.bx0;
        s.bx1 = k.xn > s.bx1 ? k.xn : s.bx1;
        s.by0 = k.yn < s.by0 ? k.yn : s.by0;
        s.by1 = k.yn > s.by1 ? k.yn : s.by1;
        res = 1;
    }
    const double c = step_factor(I.tol, I.maxstep, est, ds);
    dt = (0.9 * c) * dt;
    s.dt = dt;
    if (fabs(s.t) < I.absdur) {
        if (isnan(dt) || dt == 0.0) {
            s.status = OKA_TRACE_STALLED;
            res |= 2;
        } else if (I.cap > 0 && s.att >= I.cap) {
            s.status = OKA_TRACE_STEP_CAP;
            res |= 2;
        }
    } else {
        res |= 2;
    }
    return res;
}

struct EpochReg {
    double xmin, ymin;
    int nrows, ncols, roff, coff;
};

__device__ __forceinline__ EpochReg find_epoch(const TraceArgs &a, int64_t k)
{
    int lo = 0, hi = a.nepochs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.epochs[mid].first_trace <= k)
            lo = mid;
        else
            hi = mid - 1;
    }
    const oka_epoch &e = a.epochs[lo];
    return {e.xmin, e.ymin, e.nrows, e.ncols, e.row_off, e.col_off};
}

// The rasterizer's constants: the lattice spacing with its reciprocals and
// the umbra; the rest serve the outer chords of raster_segment, in float.
struct Raster64 {
    double dx, dy, rdx, rdy, umbra, u2;
    float idx, fdy, slack, outer, outer2;   // 1 / dx, dy; 2^-10 umbra; umbra + slack; its square
    int fast;                               // the chords and the short quotients apply
};

// gmax: the largest magnitude of the lattice's coordinates.
__device__ __forceinline__ Raster64 make_raster(double dx, double dy, double umbra, double gmax)
{
    Raster64 g;
    g.dx = dx;
    g.dy = dy;
    g.rdx = recip_plain(dx);
    g.rdy = recip_plain(dy);
    g.umbra = umbra;
    g.u2 = umbra * umbra;
    g.idx = (float)g.rdx;
    g.fdy = (float)dy;
    g.slack = (float)umbra * 0x1p-10f;
    g.outer = (float)umbra + g.slack;
    g.outer2 = g.outer * g.outer;
    // float range; the window at most 1,000 umbras per spacing; the rounding
    // of the coordinates far below the slack
    g.fast = umbra >= 1e-12 && umbra <= 1e12 && dx <= 1e3 * umbra && dy <= 1e3 * umbra &&
             dx >= 1e-6 * umbra && dy >= 1e-6 * umbra && gmax <= 0x1p36 * umbra;
    return g;
}

__device__ __forceinline__ double grid_extent(const TraceArgs &a)
{
    return fmax(fmax(fabs(a.gxmin), fabs(a.gxmax)), fmax(fabs(a.gymin), fabs(a.gymax)));
}

// probabilityfield.py:296-310, 407-427 for one node (row, col of the final
// grid; j, i of the epoch's): marks it if it is strictly within umbra.
template <typename Bits>
__device__ __forceinline__ void raster_node(Bits &bits, const EpochReg &e, const Raster64 &g,
                                            double ax, double ay, double bax, double bay, double l2,
                                            int i, int j)
{
    const double cx = e.xmin + (double)j * g.dx;
    const double cax = cx - ax;
    const double cy = e.ymin + (double)i * g.dy;
    const double cay = cy - ay;
    const double perp = bax * cay - bay * cax;
    const double dot = bax * cax + bay * cay;
    double al, be;
    div_pair(perp * perp, dot * dot, l2, al, be);
    double d2;
    if (dot < 0.0)
        d2 = al + be;
    else if (be > l2)
        d2 = ((al + be) - 2.0 * dot) + l2;
    else
        d2 = al;
    if (d2 < g.u2)
        bits.set(i + e.roff, j + e.coff);
}

// probabilityfield.py:292-310 for one segment, marking nodes of the final grid
// in `bits` (FlatBits, TileBits or PoolBits).  Already-marked nodes are
// skipped, as the reference does.  Returns the size of the reference's
// candidate window.
//
// Most of a window's nodes lie outside the umbra or are marked already, so
// each row first takes, in float, the chord of the capsule around the segment
// at a radius 2^-10 larger than umbra (raster32's, with its clip widened by as
// much), which contains every node the exact test could mark.  The widening is
// sized for segments of up to 1,000 umbras: a float coordinate of 1,000 umbras
// is rounded by 2^-14 umbras, the row's offset c carries up to three such
// errors, and with those of the slopes and of the columns the band's sides are
// off by at most three quarters of the 2^-10.  The end lines may be off by a
// little more than all of it, but the discs around the ends, off by less than a
// quarter, hold the nodes that this could cost.  (A replay of the arithmetic on
// 4e7 nodes inside the umbra, segments up to 998 umbras: c off by 2^-13, no
// node lost.)  Only the chord's unmarked nodes, read a word at a time, take the
// exact test.  Against the exact test at every unmarked node of the window: 10^4 x 1000 particles of
// the 25-well site 126.2 -> 119.9 ms, 100 x 100 of the 4-well site 14 % less.
template <typename Bits>
__device__ __forceinline__ int raster_segment(Bits &bits, const EpochReg &e, const Raster64 &g,
                                               double ax, double ay, double bx, double by)
{
    const double lox = bx < ax ? bx : ax, hix = bx > ax ? bx : ax;
    const double loy = by < ay ? by : ay, hiy = by > ay ? by : ay;
    const double nxl = (lox - g.umbra) - e.xmin, nxr = (hix + g.umbra) - e.xmin;
    const double nyl = (loy - g.umbra) - e.ymin, nyr = (hiy + g.umbra) - e.ymin;
    double qxl, qxr, qyl, qyr;
    const bool plain = g.fast && fmin(fmin(fabs(nxl), fabs(nxr)), fmin(fabs(nyl), fabs(nyr))) >= 0x1p-300 &&
                       fmax(fmax(fabs(nxl), fabs(nxr)), fmax(fabs(nyl), fabs(nyr))) <= 0x1p300;
    if (__ballot(!plain) == 0ull) {
        qxl = quot_plain(nxl, g.dx, g.rdx);
        qxr = quot_plain(nxr, g.dx, g.rdx);
        qyl = quot_plain(nyl, g.dy, g.rdy);
        qyr = quot_plain(nyr, g.dy, g.rdy);
    } else {
        div_pair(nxl, nxr, g.dx, qxl, qxr);
        div_pair(nyl, nyr, g.dy, qyl, qyr);
    }
    double jl = floor(qxl);
    double jr = floor(qxr) + 1.0;
    double il = floor(qyl);
    double ir = floor(qyr) + 1.0;
    if (jl < 0.0) jl = 0.0;
    if (il < 0.0) il = 0.0;
    if (jr > (double)e.ncols) jr = (double)e.ncols;
    if (ir > (double)e.nrows) ir = (double)e.nrows;
    if (!(jl < jr) || !(il < ir))
        return 0;
    const int j0 = (int)jl, j1 = (int)jr, i0 = (int)il, i1 = (int)ir;
    const double bax = bx - ax, bay = by - ay;
    const double l2 = bax * bax + bay * bay;
    const int ncand = (j1 - j0) * (i1 - i0);
    // the row's chord: x - ax in (lo, hi) with c = y_row - ay; in columns from j0
    const float fbx = (float)bax, fby = (float)bay, fl2 = (float)l2;
    // the length's limit and g.slack depend on each other
    const bool chord = g.fast && fabsf(fbx) > 1e-20f && fabsf(fby) > 1e-20f &&
                       fl2 < 1e6f * g.outer2 && j1 - j0 < 4096 && i1 - i0 < 4096;
    const float ibx = __builtin_amdgcn_rcpf(fbx), iby = __builtin_amdgcn_rcpf(fby);
    const float len = __builtin_amdgcn_sqrtf(fl2);
    const float kb = -fby * ibx, ka = fbx * iby;
    const float clip = g.slack * len * fabsf(ibx), l2b = fl2 * ibx;
    const float blo = fminf(l2b, 0.0f) - clip, bhi = fmaxf(l2b, 0.0f) + clip;
    const float wr = g.outer * len * fabsf(iby);
    const float xa = (float)((ax - (e.xmin + jl * g.dx)) * g.rdx);   // A's column from j0
    const float c0 = (float)((e.ymin + il * g.dy) - ay);
    const float last = (float)(j1 - j0 - 1);
    for (int i = i0; i < i1; ++i) {
        int ja = j0, jb = j1 - 1;
        if (chord) {
            const float c = fmaf((float)(i - i0), g.fdy, c0);
            float lo = fmaxf(fmaf(kb, c, blo), fmaf(ka, c, -wr));
            float hi = fminf(fmaf(kb, c, bhi), fmaf(ka, c, wr));
            if (!(lo < hi)) {
                lo = INFINITY;
                hi = -INFINITY;
            }
            const float ha = fmaf(-c, c, g.outer2);
            if (ha > 0.0f) {
                const float r = __builtin_amdgcn_sqrtf(ha);
                lo = fminf(lo, -r);
                hi = fmaxf(hi, r);
            }
            const float cb = c - fby;
            const float hb = fmaf(-cb, cb, g.outer2);
            if (hb > 0.0f) {
                const float r = __builtin_amdgcn_sqrtf(hb);
                lo = fminf(lo, fbx - r);
                hi = fmaxf(hi, fbx + r);
            }
            const float fa = fmaxf(ceilf(fmaf(lo, g.idx, xa - 0x1p-8f)), 0.0f);
            const float fb = fminf(floorf(fmaf(hi, g.idx, xa + 0x1p-8f)), last);
            if (!(fa <= fb))
                continue;
            ja = j0 + (int)fa;
            jb = j0 + (int)fb;
        }
        for (; ja <= jb; ja += 32) {
            const int n = min(jb - ja + 1, 32);
            uint32_t todo = ~bits.window(i + e.roff, ja + e.coff, n) & span_mask(n, 0);
            while (todo) {
                const int k = __ffs(todo) - 1;
                todo &= todo - 1u;
                raster_node(bits, e, g, ax, ay, bax, bay, l2, i, ja + k);
            }
        }
    }
    return ncand;
}

__device__ __forceinline__ Integ make_integ(const TraceArgs &a)
{
    Integ I;
    I.dur = a.duration;
    I.absdur = fabs(a.duration);
    I.tol = a.tol;
    I.maxstep = a.maxstep;
    I.sg = a.duration > 0.0 ? 1.0 : (a.duration < 0.0 ? -1.0 : (a.duration == 0.0 ? 0.0 : (double)NAN));
    I.cap = a.max_steps;
    return I;
}

}  // namespace fp64
}  // namespace oka
