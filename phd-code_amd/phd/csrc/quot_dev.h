// quot_dev.h -- how a face's quotients and square roots are evaluated.
//
// The face functions (riemann_dev.h, states_dev.h) take an arithmetic policy:
//
//   Ieee    the language's / and sqrt.  Always right.
//   Shared  the same quotients and roots, bit for bit, for operands whose
//           ranges have been checked, at a fraction of the instructions.
//
// hipcc lowers a / b to two div_scale, rcp, two Newton steps on the
// reciprocal, q = a r, e = a - b q, div_fmas and div_fixup (11 instructions,
// 57 cycles a wavefront on MI355X with the quarter-rate rcp), and sqrt to an
// rsq, a Goldschmidt iteration with two residual corrections, and the scaling
// of tiny arguments (85 cycles).  Far from the overflow and underflow limits
// the scaling steps are identities; leaving them out, and computing a
// divisor's reciprocal once for all its numerators, gives the same correctly
// rounded results (Markstein 1990: q + e r with q = a r, e = a - b q exact, is
// the correctly rounded quotient) in 8 instructions per divisor and 3 per
// numerator, 10 for a root.  A 2D HLLC face has about 20 quotients and 8 roots,
// half of its kernel's instructions; a 2D gradient entry divides 8 numerators by
// one divisor, a 3D entry 15.  (The 3D face kernel waits on its gathers instead and
// keeps the operators.)
//
// Shared keeps one flag: `ok` falls when an operand leaves the ranges for
// which the comment at the place shows the sequence to be exact, and the
// caller then evaluates the face again with Ieee.  Every check is written so
// that a NaN fails it.
//
// The residual's form carries the sign of a zero numerator: div() is for
// divisors > 0, divn() for divisors < 0; the two agree for other numerators.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#ifndef PHD_HD
#define PHD_HD __host__ __device__
#endif

namespace phd {

struct Ieee {
    using Rcp = double;                       // the divisor itself
    static constexpr bool fast = false;
    bool ok = true;
    PHD_HD __forceinline__ Rcp rcp(double b) const { return b; }
    PHD_HD __forceinline__ Rcp twice(Rcp c) const { return 2. * c; }
    PHD_HD __forceinline__ Rcp pick(bool first, Rcp a, Rcp b) const { return first ? a : b; }
    PHD_HD __forceinline__ double div(double a, Rcp c) const { return a / c; }
    PHD_HD __forceinline__ double divn(double a, Rcp c) const { return a / c; }
    PHD_HD __forceinline__ double root(double x) const { return sqrt(x); }
    PHD_HD __forceinline__ void need(bool) {}
};

// divisor and the reciprocal two Newton steps give
struct SharedRcp {
    double b, r;
};

struct Shared {
    using Rcp = SharedRcp;
    static constexpr bool fast = true;
    bool ok = true;

    // |b| in [2^-360, 2^610]
    PHD_HD __forceinline__ Rcp rcp(double b) const
    {
#ifdef __HIP_DEVICE_COMPILE__
        double r = __builtin_amdgcn_rcp(b);
        double e = fma(-b, r, 1.0);
        r = fma(r, e, r);
        e = fma(-b, r, 1.0);
        return {b, fma(r, e, r)};
#else
        return {b, 1.0 / b};
#endif
    }
    PHD_HD __forceinline__ Rcp twice(Rcp c) const { return {2. * c.b, .5 * c.r}; }
    PHD_HD __forceinline__ Rcp pick(bool first, Rcp a, Rcp b) const
    {
        return {first ? a.b : b.b, first ? a.r : b.r};
    }
    // a zero or |a| in [2^-900, 2^700], |a / b| in [2^-1000, 2^1000] or zero:
    // the residual is then exact (a multiple of 2^-1006).  A smaller nonzero
    // a is fine where only 1 + a/b is used.
    PHD_HD __forceinline__ double div(double a, Rcp c) const
    {
        const double q = a * c.r;
        const double e = fma(c.b, q, -a);
        return fma(-e, c.r, q);
    }
    PHD_HD __forceinline__ double divn(double a, Rcp c) const
    {
        const double q = a * c.r;
        const double e = fma(-c.b, q, a);
        return fma(e, c.r, q);
    }
    // x in [2^-700, 2^1000]
    PHD_HD __forceinline__ double root(double x) const
    {
#ifdef __HIP_DEVICE_COMPILE__
        const double y = __builtin_amdgcn_rsq(x);
        double g = x * y, h = y * 0.5;
        const double r = fma(-h, g, 0.5);
        g = fma(g, r, g);
        h = fma(h, r, h);
        double d = fma(-g, g, x);
        g = fma(d, h, g);
        d = fma(-g, g, x);
        return fma(d, h, g);
#else
        return sqrt(x);
#endif
    }
    PHD_HD __forceinline__ void need(bool c) { ok &= c; }
};

// range checks; all false for NaN
PHD_HD __forceinline__ bool within(double x, double lo, double hi) { return (x >= lo) & (x <= hi); }
PHD_HD __forceinline__ bool zero_or_above(double x, double lo)
{
    const double a = fabs(x);
    return (a >= lo) | (x == 0.0);
}
PHD_HD __forceinline__ bool zero_or_within(double x, double lo, double hi)
{
    return zero_or_above(x, lo) & (fabs(x) <= hi);
}

// Operands of the gradient sums area * (d_dif cfx - d_sum dr / 2) / (r vol).
// Coordinates (positions and face centroids) zero or >= 2^-100 are multiples of
// 2^-152, so their differences and cfx are zero or >= 2^-153, and primitives zero or
// >= 2^-240 give d_dif and d_sum / 2 zero or >= 2^-293.  Each product is zero or >=
// 2^-445 and a multiple of 2^-498, so their difference is zero or >= 2^-498, and the
// numerator, with an area zero or >= 2^-200, zero or >= 2^-698.  Above, it stays
// below 2^(151 + 151 + 1 + 150) = 2^453.  The distance r = sqrt(sum dr^2) lies in
// [2^-153, 2^152] unless zero, and r vol in [2^-353, 2^302]; so the quotients lie in
// [2^-1000, 2^806].  (The limits leave room for cells of 2^-66 to 2^50 length units,
// densities and pressures in any units, and velocities decaying ahead of a front.
// One upper limit for all: a pair of registers for each further one made the 2D
// kernel spill, 12.15 -> 12.24 ms a pass of the 256-problem ensemble.)
constexpr double SUM_MAX = 0x1p150;
PHD_HD __forceinline__ bool coord_ok(double x) { return zero_or_within(x, 0x1p-100, SUM_MAX); }
PHD_HD __forceinline__ bool prim_ok(double x) { return zero_or_within(x, 0x1p-240, SUM_MAX); }
PHD_HD __forceinline__ bool area_ok(double x) { return zero_or_within(x, 0x1p-200, SUM_MAX); }
PHD_HD __forceinline__ bool vol_ok(double x) { return within(x, 0x1p-200, SUM_MAX); }

// densities and pressures, and the ratios of specific heats, that Shared takes
PHD_HD __forceinline__ bool state_ok(double x) { return within(x, 0x1p-132, 0x1p132); }
inline bool shared_gamma(double gamma) { return gamma >= 1. + 0x1p-10 && gamma <= 64.; }

} // namespace phd
