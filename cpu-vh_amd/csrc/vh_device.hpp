// Device-side physics of the viscous-hydro step (gfx950, FP64).
//
// Arithmetic is written to round exactly like cpu-vh's compiled C++: every
// expression keeps the reference's operand order, the file is compiled with
// -ffp-contract=off (no fused multiply-add unless written as fma()), and the
// reference's single-precision islands (sqrtf/fabsf/powf on double operands)
// are reproduced bit for bit:
//   * sqrtf(x)   == (float)sqrt((double)x): the double square root of a float
//                   rounded back to float is the correctly rounded float root;
//   * powf(x,.25f) (glibc) == the correctly rounded fourth root, except on a
//                   list of inputs where glibc's result differs; that list is
//                   computed at start-up from the host's own glibc and looked
//                   up here (eos_fourth_root).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace vh {

constexpr double HBARC = 0.197326938;   // rhic/src/FullyDiscreteKurganovTadmorScheme.cpp:886
constexpr double EOS_FACTOR = 13.8997;  // rhic/include/EquationOfState.h:19
constexpr double THETA = 1.1;           // rhic/include/FluxLimiter.h:13
constexpr int EOS_LEN = 100000;         // rhic/src/EquationOfState.cpp:295
constexpr int MAX_ITERS_NR = 10000;     // rhic/src/EnergyMomentumTensor.cpp:18-20
constexpr int MAX_ITERS_BI = 1000000;
constexpr double ACC = 1.0e-3;
constexpr double delta_pipi = 1.33333;  // rhic/src/SourceTerms.cpp:50-53
constexpr double tau_pipi = 1.42857;
constexpr double delta_PiPi = 0.666667;
constexpr double lambda_piPi = 1.2;

enum : int { NAN_NONE = 0, NAN_ENERGY = 1, NAN_ROOT = 2, NAN_REG_SHEAR = 3, NAN_REG_BULK = 4 };

// Division by a divisor used several times: one correctly rounded reciprocal
// r = RN(1/b) and, per numerator, q0 = RN(a*r), rem = a - b*q0 (exact with
// FMA), q = RN(q0 + rem*r).  By Markstein's theorem (IBM J. Res. Dev. 34,
// 1990; Muller et al., Handbook of Floating-Point Arithmetic, ch. 5) q is the
// correctly rounded a/b, i.e. the division operator's value, when nothing
// underflows or overflows.  Sufficient here: |b| in [2^-100, 2^100] (so r is
// normal) and |q0| in [2^-860, 2^1000] (then rem is a multiple of 2^-1064,
// exactly representable, and q is normal); a == +-0 gives a*r, the
// correctly signed zero.
//
// DivFast uses the reciprocal form and, for the lanes whose quotient leaves
// that range (tiny or huge values, NaN), the division operator; DivExact
// always uses the division operator.  Either way every result equals the
// division operator's.
struct Recip {
    double b, r;
    bool ok;
};
__host__ __device__ __forceinline__ Recip make_recip(double b) {
    Recip R;
    R.b = b;
    R.r = 1.0 / b;
    const double ab = __builtin_fabs(b);
    R.ok = ab >= 0x1p-100 && ab <= 0x1p100;
    return R;
}
// Divisors 3 and 5.  b q0 of a small integer b is exact wherever q0 is, and so is
// the residual, subnormal numerators and quotients included; no quotient lies
// half way between two numbers, and the residual's part of a unit in the last
// place is a third or a fifth of a unit, far from the half a rounding error
// could cross.  div_mid therefore gives the operator's bits for every finite
// numerator, and no check is needed.
struct IntRecip {
    double b, r;
};
struct DivFast {
    __host__ __device__ __forceinline__ Recip recip(double b) { return make_recip(b); }
    __host__ __device__ __forceinline__ void see(double) {}
    __host__ __device__ __forceinline__ void in(bool) {}
    __host__ __device__ __forceinline__ double operator()(double a, const Recip &R) {
        const double q0 = a * R.r;
        const double rem = __builtin_fma(-R.b, q0, a);
        double q = __builtin_fma(rem, R.r, q0);
        const double aq = __builtin_fabs(q0);
        const bool zero = a == 0.0;
        if (zero) q = q0;
        if (__builtin_expect(!(R.ok && ((aq >= 0x1p-860 && aq <= 0x1p1000) || zero)), 0)) q = a / R.b;
        return q;
    }
    __host__ __device__ __forceinline__ double operator()(double a, const IntRecip &R) {
        return (*this)(a, Recip{R.b, R.r, true});
    }
};
struct DivExact {
    __device__ __forceinline__ double operator()(double a, const Recip &R) { return a / R.b; }
};

// Quotients of operands known to be far from overflow and underflow: the
// hardware reciprocal refined by two Newton steps, the quotient and one
// residual correction.  These are the operations the division operator
// expands to on this target, less its scaling and fix-up instructions, which
// leave such operands and results alone: the same bits in 8 instructions
// instead of 11, and without the mask register every scaled division passes
// its flag through, so independent divisions overlap.  Sufficient: |a| and
// |b| in [2^-300, 2^300], or a zero.  The residual is taken as b q0 - a so
// that a zero a keeps its sign for b > 0.  near_rcp(b) serves several
// numerators of one divisor.
__host__ __device__ __forceinline__ double near_rcp(double b) {
#ifdef __HIP_DEVICE_COMPILE__
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
#else
    return 1.0 / b;  // host checks of the division policies
#endif
}
__host__ __device__ __forceinline__ double div_mid(double a, double b, double r) {
    const double q0 = a * r;
    const double rem = __builtin_fma(b, q0, -a);
    return __builtin_fma(-rem, r, q0);
}
__host__ __device__ __forceinline__ double div_mid(double a, double b) { return div_mid(a, b, near_rcp(b)); }

__host__ __device__ __forceinline__ uint32_t high_word(double x) {
    return (uint32_t)(__builtin_bit_cast(uint64_t, x) >> 32);
}
// The high word of |x| less that of 2^LO as an unsigned number lies below this
// span exactly when 2^LO <= |x| < 2^HI; NaN, infinities, zeros and, for the
// signed form, negative x fall outside.
template <int LO, int HI>
__host__ __device__ __forceinline__ bool in_range(double x) {
    return high_word(x) - (uint32_t)((1023 + LO) << 20) < (uint32_t)((HI - LO) << 20);
}
template <int LO, int HI>
__host__ __device__ __forceinline__ bool abs_in_range(double x) {
    return (high_word(x) << 1) - ((uint32_t)(1023 + LO) << 21) < ((uint32_t)(HI - LO) << 21);
}
// x's exponent, |x| in [2^(k-1), 2^k), subnormal x included; 0 for zeros,
// infinities and NaN.
__host__ __device__ __forceinline__ int exponent(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_frexp_exp(x);
#else
    int k = 0;
    if (__builtin_isfinite(x)) __builtin_frexp(x, &k);
    return k;
#endif
}

// sqrtf of a float x that is zero or >= 2^-96 (NaN and infinity keep their
// value), correctly rounded: the hardware root is within one unit in the last
// place, so the result is it or a neighbour, and s s' >= x (or < x) tells on
// which side of the midpoint of two neighbours s, s' the root lies (x and s s'
// are multiples of the same power of two below which the midpoint's square
// differs from s s').
__device__ __forceinline__ float sqrt_mid(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float lo = __uint_as_float(__float_as_uint(s) - 1u), hi = __uint_as_float(__float_as_uint(s) + 1u);
    float r = __builtin_fmaf(-lo, s, x) <= 0.0f ? lo : s;
    r = __builtin_fmaf(-hi, s, x) > 0.0f ? hi : r;
    return r;
}

// Division policy of the FP64 stage: every quotient by the reciprocal form,
// unchecked, with what the check needs accumulated beside it.  The caller
// asks fails() once at the end and, if some lane's operands left the range,
// evaluates the whole expression again with DivFast (quotients that meet small
// numerators often have a check of their own, checked()).  What has to hold: every
// divisor b in [2^-100, 2^50), every numerator a zero or |a| >= 2^-969, nothing
// overflowed.  Then q0 is normal (at least 2^-1020) and the residual b q0 - a is
// a multiple of 2^-1074, so it is exactly representable and the corrected
// quotient is the division operator's; a == +-0 gives the correctly signed
// zero.  The check is on a, not on q0: a subnormal quotient's high word can be
// zero, as a zero's is, and a's exponent does not wait for the product.
// Divisors reach down to 2^-100 because t, t^2, t^3 and dt are among them (with
// a floor of 2^-16 every cell below t = 0.025 or dt = 1.5e-5 took the checked
// evaluation: 40 steps of 61x57x31 at t = 0.001 and dt = 1e-5 took 11.3 ms
// instead of 5.7).  A quotient that overflows or is NaN makes the results NaN
// or infinite, which see() notes.  DivFast compares, selects and branches
// at each of about 300 divisions a cell and stage (three 64-bit compares, a
// select and a branch each); here a division costs its four instructions and
// two 32-bit ones.  With nr_step_try the 3+1D kernel issued 2.36e8 VALU
// instructions per launch at 131x131x61 (2.23e8 with checked() and IntRecip
// since) where it issued 3.35e8; with their
// copies, 60 steps of that event took 112.8 instead of 122.8 ms, 100 steps of
// a 147x129 event 6.48 instead of 8.32 ms, 200 conformal steps at 201x201 9.87
// instead of 12.2 ms, 40 steps of 16 batched events 16.6 instead of 18.9 ms.
struct DivTry {
    static constexpr int MIN_EXPONENT = -968;  // of a numerator that is not zero
    int lo = 0;
    uint32_t hi = 0;
    bool ok = true;
    __host__ __device__ __forceinline__ Recip recip(double b) {
        double r = near_rcp(b);
        r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);  // 1/b correctly rounded
        ok = ok && in_range<-100, 50>(b);
        return Recip{b, r, true};
    }
    __host__ __device__ __forceinline__ double operator()(double a, const Recip &R) {
        const int k = exponent(a);
        lo = k < lo ? k : lo;
        return div_mid(a, R.b, R.r);
    }
    __host__ __device__ __forceinline__ double operator()(double a, const IntRecip &R) { return div_mid(a, R.b, R.r); }
    __host__ __device__ __forceinline__ void see(double x) {
        const uint32_t u = high_word(x) << 1;
        hi = u > hi ? u : hi;
    }
    __host__ __device__ __forceinline__ void in(bool inside) { ok = ok && inside; }
    __host__ __device__ __forceinline__ bool small() const { return lo < MIN_EXPONENT; }
    __host__ __device__ __forceinline__ bool fails() const { return !ok || small() || hi >= 0x7ffu << 21; }
};
// A few of DivTry's quotients, f, with a check of their own: where a numerator
// is small, f again by the division operator, in place.  For the fluxes and
// speeds of the three directions, four fifths of all quotients: ahead of a hot
// region in a uniform medium velocity and shear fall by powers, and products of
// them pass through the small numbers over tens of cells.  150 steps of 261x261
// around such a region (34 and 38 % of the source's and the directions' waves
// had a small numerator): 18.1 ms with one check per role, 12.4 with this and
// IntRecip, 15.3 with a check per division everywhere; conformal 15.1, 10.8, 11.9;
// 40 steps of 101x101x61 39.1, 29.4, 34.5; a Glauber event of 131x131x61, 60 steps,
// 96.8, 90.0, 130; an event without such cells the same within 1 %.
struct DivOperator {
    __device__ __forceinline__ double operator()(double a, const Recip &R) { return a / R.b; }
};
template <class DV, class F>
__device__ __forceinline__ auto checked(DV &div, F &&f) {
    if constexpr (std::is_same_v<DV, DivTry>) {
        DivTry d;
        auto x = f(d);
        if (__builtin_expect(d.small(), 0)) {
            DivOperator o;
            x = f(o);
        }
        return x;
    } else {
        return f(div);
    }
}
// The table lookups of DivTry's callers: their quotients need no check (a
// quotient too small for the residual to be exact changes neither the index
// nor the interpolated value, a NaN or infinite energy density gives the
// same 1e-15 floor).
struct DivTable {
    __device__ __forceinline__ double operator()(double a, const Recip &R) { return div_mid(a, R.b, R.r); }
};
template <class DV>
using TableDiv = std::conditional_t<std::is_same_v<DV, DivTry>, DivTable, DV>;

// Quotient policies of the root solve and the primitive recovery.  QuotExact
// is the division operator (the FP64 path).  QuotFast (mixed form only) is a
// hardware reciprocal refined by two Newton steps and one residual
// correction: within an ulp of the quotient, not correctly rounded.  With
// DivRecip the table lookups multiply by the precomputed reciprocal spacing.
struct QuotExact {
    static __device__ __forceinline__ double q(double a, double b) { return a / b; }
    // the reference's sqrtf of a double (a float island): correctly rounded
    static __device__ __forceinline__ float sqrt_island(float x) { return (float)__builtin_sqrt((double)x); }
};
struct QuotFast {
    // hardware reciprocal and one Newton step: relative error about 2^-46
    static __device__ __forceinline__ double rcp1(double b) {
        const double r = __builtin_amdgcn_rcp(b);
        return __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    }
    static __device__ __forceinline__ double rcp(double b) {
        double r = __builtin_amdgcn_rcp(b);
        r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
        return __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    }
    static __device__ __forceinline__ double q(double a, double b) {
        double r = __builtin_amdgcn_rcp(b);
        r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
        r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
        const double q0 = a * r;
        return __builtin_fma(__builtin_fma(-b, q0, a), r, q0);
    }
    // the hardware's single-precision square root (within an ulp)
    static __device__ __forceinline__ float sqrt_island(float x) { return __builtin_amdgcn_sqrtf(x); }
};
struct DivRecip {
    __device__ __forceinline__ double operator()(double a, const Recip &R) { return a * R.r; }
};

struct EosDev {
    int kind;        // 0 conformal, 1 table
    int cs2_const;   // table: host verified that the reference's c_s^2 is 1/3 for every e
    int cs2_mode;    // table: 0 the reference's delta_e/delta_p, 1 the sound speed delta_p/delta_e
    double e_min, e_spacing, e_max;
    double r_spacing;  // RN(1/e_spacing)
    const double *p_tb;
    const double *T_tb;
    // FP32 segments of the pressure table for the mixed form's face solves:
    // entry k = {p_k, d_k, d_k / de, (d_{k+1} - d_k) / de}, d_k = p_{k+1} - p_k
    // formed in FP64 (the last segment's slope continues past the table)
    const float4 *p4;
    // glibc powf(x, 0.25f) exceptions: sorted (x bits, result bits) pairs,
    // bucketed by (xbits - exc_lo) >> exc_shift.
    const uint2 *exc;
    const uint32_t *exc_bucket;
    uint32_t exc_lo, exc_hi;
    int exc_shift;
};

__device__ __forceinline__ float f32_sqrt(float x) { return (float)__builtin_sqrt((double)x); }
__device__ __forceinline__ float f32_fabs(float x) { return __builtin_fabsf(x); }

// glibc powf(x, 0.25f) for the conformal temperature (EquationOfState.cpp:196).
__device__ __forceinline__ float eos_fourth_root(const EosDev &E, float x) {
    float r = (float)__builtin_sqrt(__builtin_sqrt((double)x));
    uint32_t xb = __float_as_uint(x);
    if (xb >= E.exc_lo && xb < E.exc_hi) {
        uint32_t b = (xb - E.exc_lo) >> E.exc_shift;
        uint32_t lo = E.exc_bucket[b], hi = E.exc_bucket[b + 1];
        while (lo < hi) {
            uint32_t mid = (lo + hi) >> 1;
            uint32_t k = E.exc[mid].x;
            if (k < xb) lo = mid + 1;
            else hi = mid;
        }
        if (lo < E.exc_bucket[b + 1] && E.exc[lo].x == xb) r = __uint_as_float(E.exc[lo].y);
    }
    return r;
}

// rhic/src/EquationOfState.cpp:329-360
template <class DV>
__device__ __forceinline__ double eos_interp(const EosDev &E, double e, const double *__restrict__ tb, DV &div) {
    const double e0 = E.e_min, de = E.e_spacing;
    const Recip Rde{de, E.r_spacing, true};
    TableDiv<DV> dt;
    int idx = (int)dt(e - e0, Rde);
    idx = idx < EOS_LEN - 2 ? idx : EOS_LEN - 2;
    idx = idx > 0 ? idx : 0;
    const double frac = dt(e - (idx * de + e0), Rde);
    double t1 = tb[idx], t2 = tb[idx + 1];
    return t1 * (1. - frac) + t2 * frac;
}

template <bool TABLE, class DV>
__device__ __forceinline__ double eos_pressure(const EosDev &E, double e, DV &div) {
    if constexpr (TABLE) {
        double f = eos_interp(E, e, E.p_tb, div);
        return 1.e-15 < f ? f : 1.e-15;  // std::max(1.e-15, f)
    } else {
        TableDiv<DV> dt;
        return dt(e, Recip{3., 1. / 3., true});
    }
}

// Mixed form: the same linear interpolation from one scaled coordinate
// x = (e - e_min) / de (idx = trunc(x), frac = x - idx), within a few ulps of
// the reference's two divisions.
__device__ __forceinline__ double eos_pressure_fast(const EosDev &E, double e) {
    const double x = (e - E.e_min) * E.r_spacing;
    int idx = (int)x;
    idx = idx < EOS_LEN - 2 ? idx : EOS_LEN - 2;
    idx = idx > 0 ? idx : 0;
    const double frac = x - (double)idx;
    const double t1 = E.p_tb[idx], t2 = E.p_tb[idx + 1];
    const double f = __builtin_fma(frac, t2 - t1, t1);
    return 1.e-15 < f ? f : 1.e-15;
}

template <bool TABLE, class DV>
__device__ __forceinline__ double eos_cs2(const EosDev &E, double e, DV &div) {
    if constexpr (TABLE) {
        if (E.cs2_const) return 1. / 3.;
        double v_min = 0.01, v_max = 1. / 3.;
        double delta_e = E.e_spacing;
        double p = eos_pressure<true>(E, e, div);
        double p_r = eos_pressure<true>(E, e + delta_e, div);
        double delta_p = p_r - p;
        double v;
        if (E.cs2_mode) {
            if constexpr (std::is_same_v<DV, DivTry>) v = div_mid(delta_p, delta_e, E.r_spacing);
            else v = delta_p / delta_e;
        } else {
            v = delta_e / delta_p;
        }
        v = v_max < v ? v_max : v;  // std::min(v_max, v)
        v = v_min < v ? v : v_min;  // std::max(v_min, .)
        return v;
    } else {
        return 1. / 3.;
    }
}

template <bool TABLE, class DV>
__device__ __forceinline__ double eos_temperature(const EosDev &E, double e, DV &div) {
    if constexpr (TABLE) {
        double f = eos_interp(E, e, E.T_tb, div);
        return 1.e-15 < f ? f : 1.e-15;
    } else {
        return (double)eos_fourth_root(E, (float)(e / EOS_FACTOR));
    }
}

// approximateDerivative (rhic/src/FluxLimiter.cpp:14-32): minmod(l, minmod(c, r))
// with minmod(a, b) = (sign(a) + sign(b)) min(|a|, |b|) / 2 and sign(0) = +1.
// Its value is the smallest of the three where all are >= 0, the largest where
// all are < 0, and +0 otherwise: max(lo, min(hi, 0)) of the smallest lo and
// the largest hi, with + 0.0 turning a -0 into the reference's +0.  Bit for bit
// the sign form's value for finite arguments (scaling by 2 and 1/2 is exact);
// it differs only where the line already holds NaN or infinite values.  Seven
// min, max and add instructions in place of the sign form's eighteen compares,
// selects, conversions and products; each stage evaluates it 72 times a cell
// and direction: 60 steps of a 131x131x61 event with their copies 130.2 ->
// 122.8 ms, 100 steps of a 147x129 event 8.86 -> 8.29 ms.
__device__ __forceinline__ double approx_deriv(double x, double y, double z) {
    const double l = THETA * (y - x);
    const double c = (z - x) / 2.0;
    const double r = THETA * (z - y);
    const double lo = __builtin_fmin(l, __builtin_fmin(c, r));
    const double hi = __builtin_fmax(l, __builtin_fmax(c, r));
    return __builtin_fmax(lo, __builtin_fmin(hi, 0.0)) + 0.0;
}

struct Prim {
    double e, p, ut, ux, uy, un;
};

// getInferredVariables, rhic/src/EnergyMomentumTensor.cpp:117-233, in two
// parts: the energy density from the conserved variables (the closed form
// below ePrev = 0.1, else the root solve), then pressure, floors and
// velocity.  ttt..pitn are q[0..7]; Pi = q[14] when bulk is evolved.
struct Moments {
    double M0, M1, M2, M3, M;
};

__device__ __forceinline__ Moments moments(double t, double ttt, double ttx, double tty, double ttn, double pitt,
                                           double pitx, double pity, double pitn) {
    Moments m;
    m.M0 = ttt - pitt;
    m.M1 = ttx - pitx;
    m.M2 = tty - pity;
    m.M3 = ttn - pitn;
    m.M = m.M1 * m.M1 + m.M2 * m.M2 + t * t * m.M3 * m.M3;
    return m;
}

// Newton-Raphson + bisection root solve of the table EoS,
// rhic/src/EnergyMomentumTensor.cpp:26-111, with the division operator
// throughout.  Callers instantiate it inside loops so each kernel carries
// few copies.
struct RootResult {
    double e;
    int nan;
};
// One Newton step of energyDensityFromConservedVariables
// (rhic/src/EnergyMomentumTensor.cpp:26-47) from e0; bad is set when the
// step is NaN (the reference's "f/fp is nan").
template <class QD, class DV>
__device__ __forceinline__ double nr_step(const EosDev &E, double e0, double M0, double M, double Pi, DV &dx,
                                          bool &bad) {
    if constexpr (std::is_same_v<QD, QuotFast>) {
        // mixed form: the same iteration with two reciprocals in place of
        // five quotients.  R = 1/(e0 p) gives 1/e0 and 1/p; with
        // X = c (B + D H - c cst2 D M0 / e0) and cst2 e0 H = p H the step
        // f / fp = f (1 - X / (p H))^-1 is f p H / (p H - X).
        const double p = eos_pressure_fast(E, e0);
        const double cs2 = eos_cs2<true>(E, e0, dx);
        const double R = QuotFast::rcp1(e0 * p);
        const double ie0 = p * R, ip = e0 * R;
        const double cst2 = p * ie0;
        const double A = __builtin_fma(-M0, cst2, M0) + Pi;
        const double B = M0 * (M0 + Pi) - M;
        const double H = (double)QuotFast::sqrt_island(f32_fabs((float)__builtin_fma(A, A, 4 * cst2 * B)));
        const double D = (A - H) * (0.5 * e0 * ip);
        const double f = e0 + D;
        const double c = cs2 - cst2;
        const double X = c * (B + D * H - c * cst2 * D * M0 * ie0);
        const double pH = p * H;
        const double step = f * pH * QuotFast::rcp1(pH - X);
        bad = __builtin_isnan(step);
        return e0 - step;
    }
    double p = eos_pressure<true>(E, e0, dx);
    double cs2 = eos_cs2<true>(E, e0, dx);
    double cst2 = QD::q(p, e0);
    double A = M0 * (1.0 - cst2) + Pi;
    double B = M0 * (M0 + Pi) - M;
    double H = (double)QD::sqrt_island(f32_fabs((float)(A * A + 4 * cst2 * B)));
    double D = QD::q(A - H, 2 * cst2);
    double f = e0 + D;
    double fp = 1.0 - QD::q((cs2 - cst2) * (B + D * H - QD::q((cs2 - cst2) * cst2 * D * M0, e0)), cst2 * e0 * H);
    const double step = QD::q(f, fp);
    bad = __builtin_isnan(step);
    return e0 - step;
}

// nr_step's QuotExact form with the same bits from div_mid and sqrt_mid, and
// ok cleared where an operand leaves their range: e0 in [2^-100, 2^100], H in
// [2^-47, 2^60] and |f'| in [2^-60, 2^100] bound the others (p is 1e-15 or
// more, |A| < 2^90 where H is bounded, A - H is zero or at least 2^-124; an
// intermediate that overflows makes f' NaN, and one that underflows is too
// small to change f').  e0's reciprocal serves both quotients by e0.  The
// iteration is about half the instructions of the operator's, which spends
// eleven on each of ten divisions and some twenty on the double square root.
// CS: how c_s^2 is found (eos_cs2): 0 it is 1/3, 1 delta_p/delta_e, 2 the reference's delta_e/delta_p.
template <int CS>
__device__ __forceinline__ double nr_step_try(const EosDev &E, double e0, double M0, double B, double Pi, bool &ok) {
    DivTry dx;
    const double p = eos_pressure<true>(E, e0, dx);
    double cs2 = 1. / 3.;
    if constexpr (CS != 0) {
        const double delta_p = eos_pressure<true>(E, e0 + E.e_spacing, dx) - p;
        double v = CS == 1 ? div_mid(delta_p, E.e_spacing, E.r_spacing) : E.e_spacing / delta_p;
        v = cs2 < v ? cs2 : v;
        cs2 = 0.01 < v ? v : 0.01;
    }
    const double r0 = near_rcp(e0);
    const double cst2 = div_mid(p, e0, r0);
    const double A = M0 * (1.0 - cst2) + Pi;
    const double H = (double)sqrt_mid(f32_fabs((float)(A * A + 4 * cst2 * B)));
    const double D = div_mid(A - H, 2 * cst2);
    const double f = e0 + D;
    const double fp = 1.0 - div_mid((cs2 - cst2) * (B + D * H - div_mid((cs2 - cst2) * cst2 * D * M0, e0, r0)),
                                    cst2 * e0 * H);
    ok = in_range<-100, 100>(e0) && in_range<-47, 60>(H) && abs_in_range<-60, 100>(fp);
    return e0 - div_mid(f, fp);
}

// the reference's stop test, evaluated in float (:44); the mixed form
// evaluates it in double
template <class QD>
__device__ __forceinline__ bool nr_converged(double e, double e0) {
    if constexpr (std::is_same_v<QD, QuotFast>) return __builtin_fabs(e - e0) <= ACC * __builtin_fabs(e);
    return (double)f32_fabs((float)(e - e0)) <= ACC * (double)f32_fabs((float)e);
}

// bisection fallback after MAX_ITERS_NR Newton steps (:48-111)
template <class QD, class DV>
__device__ __forceinline__ double table_bisect(const EosDev &E, double ePrev, double M0, double M, double Pi) {
    DV dx;
    double e_lo = 0.0, e_mid = ePrev, e_hi = 2.0 * (ePrev + 1.0);
    for (int j = 0; j < MAX_ITERS_BI; ++j) {
        double p_lo = eos_pressure<true>(E, e_lo, dx), p_mid = eos_pressure<true>(E, e_mid, dx),
               p_hi = eos_pressure<true>(E, e_hi, dx);
        double cst2_lo = QD::q(p_lo, e_lo), cst2_mid = QD::q(p_mid, e_mid), cst2_hi = QD::q(p_hi, e_hi);
        double A_lo = M0 * (1.0 - cst2_lo) + Pi;
        double A_mid = M0 * (1.0 - cst2_mid) + Pi;
        double A_hi = M0 * (1.0 - cst2_hi) + Pi;
        double B = M0 * (M0 + Pi) - M;
        double H_lo = (double)QD::sqrt_island(f32_fabs((float)(A_lo * A_lo + 4 * cst2_lo * B)));
        double H_mid = (double)QD::sqrt_island(f32_fabs((float)(A_mid * A_mid + 4 * cst2_mid * B)));
        double H_hi = (double)QD::sqrt_island(f32_fabs((float)(A_hi * A_hi + 4 * cst2_hi * B)));
        double D_lo = QD::q(A_lo - H_lo, 2 * cst2_lo);
        double D_mid = QD::q(A_mid - H_mid, 2 * cst2_mid);
        double D_hi = QD::q(A_hi - H_hi, 2 * cst2_hi);
        double f_lo = e_lo + D_lo, f_mid = e_mid + D_mid, f_hi = e_hi + D_hi;
        if ((e_hi - e_lo) < (ACC * e_hi) / 2.0) return e_mid;
        if (f_lo * f_mid < 0.0) {
            e_hi = e_mid;
            e_mid = (e_lo + e_hi) / 2.0;
        } else if (f_mid * f_hi < 0.0) {
            e_lo = e_mid;
            e_mid = (e_lo + e_hi) / 2.0;
        } else {
            // no sign change (or NaN): the bracket never moves again, so the
            // reference's remaining iterations all repeat this one and its
            // loop ends with ePrev -- return that now
            return ePrev;
        }
    }
    return ePrev;
}

// Table-EoS root solve (rhic/src/EnergyMomentumTensor.cpp:22-111): Newton
// from ePrev, then bisection.
template <class QD = QuotExact, class DV = DivExact>
__device__ __forceinline__ RootResult table_root(const EosDev &E, double ePrev, double M0, double M, double Pi) {
    DV dx;
    double e0 = ePrev;
    for (int j = 0; j < MAX_ITERS_NR; ++j) {
        bool bad;
        const double e = nr_step<QD, DV>(E, e0, M0, M, Pi, dx, bad);
        if (bad) return RootResult{ePrev, NAN_ROOT};
        if (nr_converged<QD>(e, e0)) return RootResult{e, NAN_NONE};
        e0 = e;
    }
    return RootResult{table_bisect<QD, DV>(E, ePrev, M0, M, Pi), NAN_NONE};
}

// Table-EoS root solves from one start value, stepped together: table_root of
// each state with nr_step_try.  Each takes exactly the steps table_root takes
// (a state that has converged keeps its value while the others go on); a step
// of all N evaluates them side by side, so their table gathers and chains
// overlap where one state's step after another's waited for each gather: 60
// steps of 131x131x61 with their copies 117.5 -> 110.6 ms, 100 steps of
// 147x129 6.49 -> 6.24 ms, 16 batched events 16.9 -> 16.1 ms (one box).  A
// state that leaves nr_step_try's range (a NaN among the causes), or has not
// converged after TRY_ITERS steps, ends the attempt (ok false): the caller
// solves again with table_root, which alone goes on to MAX_ITERS_NR and the
// bisection.
constexpr int TRY_ITERS = 64;
template <int CS, int N>
__device__ __forceinline__ void roots_try(const EosDev &E, double ePrev, const Moments (&m)[N], const double (&Pi)[N],
                                          double (&e)[N], bool &ok) {
    double B[N];
    bool done[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        B[k] = m[k].M0 * (m[k].M0 + Pi[k]) - m[k].M;
        e[k] = ePrev;
        done[k] = false;
    }
    bool any = true;
    for (int j = 0; j < TRY_ITERS && any; ++j) {
        any = false;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            bool in;
            const double en = nr_step_try<CS>(E, e[k], m[k].M0, B[k], Pi[k], in);
            const bool conv = nr_converged<QuotExact>(en, e[k]);
            ok = ok && (in || done[k]);
            e[k] = done[k] ? e[k] : en;
            done[k] = done[k] || conv || !in;
            any = any || !done[k];
        }
    }
    ok = ok && !any;
}
// Four states go two at a time (four at once keep too much live: the
// 131x131x61 step takes 1.3 % longer).
template <int CS, int N>
__device__ __forceinline__ void roots_by_two(const EosDev &E, double ePrev, const Moments (&m)[N], const double (&Pi)[N],
                                             double (&e)[N], bool &ok) {
    if constexpr (N == 4) {
#pragma unroll
        for (int h = 0; h < 4; h += 2) {
            const Moments mh[2] = {m[h], m[h + 1]};
            const double Ph[2] = {Pi[h], Pi[h + 1]};
            double eh[2];
            roots_try<CS, 2>(E, ePrev, mh, Ph, eh, ok);
            e[h] = eh[0];
            e[h + 1] = eh[1];
        }
    } else {
        roots_try<CS, N>(E, ePrev, m, Pi, e, ok);
    }
}
template <int N>
__device__ __forceinline__ void table_roots_try(const EosDev &E, double ePrev, const Moments (&m)[N],
                                                const double (&Pi)[N], double (&e)[N], bool &ok) {
    if (E.cs2_const) roots_by_two<0, N>(E, ePrev, m, Pi, e, ok);
    else if (E.cs2_mode) roots_by_two<1, N>(E, ePrev, m, Pi, e, ok);
    else roots_by_two<2, N>(E, ePrev, m, Pi, e, ok);
}

// The segment of E.p4 holding e (clamped to the table's ends, where its
// line extends) and e's fraction within it.
__device__ __forceinline__ float4 eos_segment_f32(const EosDev &E, float e, float emin, float rsp, float &frac) {
    const float x = (e - emin) * rsp;
    int idx = (int)x;
    idx = idx < EOS_LEN - 2 ? idx : EOS_LEN - 2;
    idx = idx > 0 ? idx : 0;
    frac = x - (float)idx;
    return E.p4[idx];
}

// The mixed form's Newton iteration in FP32: the reference's iteration
// (EnergyMomentumTensor.cpp:26-47, the formulas of nr_step's QuotFast form)
// in single precision from the FP64 moments, with B = M0 (M0 + Pi) - M
// formed in FP64 (it cancels for fast flow), hardware reciprocals and square
// root, and the reference's stop test |e - e0| <= 1e-3 |e| evaluated in FP32,
// as the reference evaluates it (fabsf).  One FP32 segment per step gives p
// and, unless CONST_CS2 (the table's c_s^2 is 1/3 for every e), c_s^2(e0) as
// eos_cs2's one-segment quotient: the pressure one table spacing up at the
// same fraction, clamped alike.  The bisection fallback is the FP64 one.
template <bool CONST_CS2>
__device__ __forceinline__ RootResult table_root_f32(const EosDev &E, double ePrev, double M0d, double Md, double Pid) {
    const float M0 = (float)M0d, Pi = (float)Pid;
    const float B = (float)(M0d * (M0d + Pid) - Md);
    const float emin = (float)E.e_min, rsp = (float)E.r_spacing;
    float e0 = (float)ePrev;
    int how = 0;  // 1: converged, 2: NaN step, 0: iterations spent
    for (int j = 0; j < MAX_ITERS_NR; ++j) {
        float frac;
        const float4 T = eos_segment_f32(E, e0, emin, rsp, frac);
        float p = __builtin_fmaf(frac, T.y, T.x);
        p = 1.e-15f < p ? p : 1.e-15f;
        float cs2 = 1.0f / 3.0f;
        if constexpr (!CONST_CS2) {
            const float dpde = __builtin_fmaf(frac, T.w, T.z);
            float v = E.cs2_mode ? dpde : __builtin_amdgcn_rcpf(dpde);
            v = (1.0f / 3.0f) < v ? (1.0f / 3.0f) : v;
            v = 0.01f < v ? v : 0.01f;
            cs2 = v;
        }
        const float R = __builtin_amdgcn_rcpf(e0 * p);
        const float ie0 = p * R, ip = e0 * R;
        const float cst2 = p * ie0;
        const float A = __builtin_fmaf(-M0, cst2, M0) + Pi;
        const float H = __builtin_amdgcn_sqrtf(__builtin_fabsf(__builtin_fmaf(A, A, 4 * cst2 * B)));
        const float D = (A - H) * (0.5f * e0 * ip);
        const float f = e0 + D;
        const float c = cs2 - cst2;
        const float X = c * (B + D * H - c * cst2 * D * M0 * ie0);
        const float pH = p * H;
        const float step = f * pH * __builtin_amdgcn_rcpf(pH - X);
        if (__builtin_isnan(step)) {
            how = 2;
            break;
        }
        const float e = e0 - step;
        const bool done = __builtin_fabsf(e - e0) <= 1.0e-3f * __builtin_fabsf(e);
        e0 = e;
        if (done) {
            how = 1;
            break;
        }
    }
    if (how == 1) return RootResult{(double)e0, NAN_NONE};
    if (how == 2) return RootResult{ePrev, NAN_ROOT};
    return RootResult{table_bisect<QuotFast, DivRecip>(E, ePrev, M0d, Md, Pid), NAN_NONE};
}

// energyDensityFromConservedVariables, rhic/src/EnergyMomentumTensor.cpp:22-115
template <bool TABLE, class QD = QuotExact, class DV = DivExact>
__device__ __forceinline__ double energy_from_conserved(const EosDev &E, double ePrev, double M0, double M, double Pi,
                                                        int &nan) {
    if constexpr (!TABLE) {
        (void)E; (void)ePrev; (void)Pi; (void)nan;
        return (double)f32_fabs((float)((double)QD::sqrt_island(f32_fabs((float)(4 * M0 * M0 - 3 * M))) - M0));
    } else {
        const RootResult r = table_root<QD, DV>(E, ePrev, M0, M, Pi);
        if (r.nan) nan = r.nan;
        return r.e;
    }
}

template <bool TABLE, class DV, class QD>
__device__ __forceinline__ Prim recover_finish(const EosDev &E, const Moments &m, double e, double Pi, int &nan,
                                               DV &div) {
    Prim r;
    r.e = e;
    if (__builtin_isnan(r.e)) nan = NAN_ENERGY;
    constexpr bool FAST = std::is_same_v<QD, QuotFast>, TRY = std::is_same_v<DV, DivTry>;
    if constexpr (FAST && TABLE) r.p = eos_pressure_fast(E, r.e);
    else r.p = eos_pressure<TABLE>(E, r.e, div);
    if (r.e < 1.e-7) {
        r.e = 1.e-7;
        r.p = 1.e-7;
    }
    double P = r.p + Pi;
    double Ei, E2;
    if constexpr (TRY) {
        const double w = r.e + P;
        Ei = div_mid(1.0, w);
        r.ut = (double)sqrt_mid(f32_fabs((float)((m.M0 + P) * Ei)));
        E2 = div_mid(Ei, r.ut);
        div.ok = div.ok && in_range<-100, 100>(w) && in_range<-16, 100>(r.ut);
    } else {
        if constexpr (FAST) Ei = QuotFast::rcp1(r.e + P);
        else Ei = QD::q(1.0, r.e + P);
        r.ut = (double)QD::sqrt_island(f32_fabs((float)((m.M0 + P) * Ei)));
        if constexpr (FAST) E2 = Ei * QuotFast::rcp1(r.ut);
        else E2 = QD::q(Ei, r.ut);
    }
    r.ux = m.M1 * E2;
    r.uy = m.M2 * E2;
    r.un = m.M3 * E2;
    if (r.ut > 1.0e3) {
        r.ut = 1.0;
        r.ux = 0.0;
        r.uy = 0.0;
        r.un = 0.0;
    }
    return r;
}

// getInferredVariables of N states sharing ePrev with DivTry: the values of
// recover_moments where nothing fails (div.fails() else, and nan is left to
// the evaluation that follows).
template <bool TABLE, int N>
__device__ __forceinline__ void recover_try(const EosDev &E, const Moments (&m)[N], const double (&Pi)[N],
                                            double ePrev, int &nan, DivTry &div, Prim (&out)[N]) {
    double e[N];
    if (ePrev <= 0.1) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            e[k] = m[k].M0 - div_mid(m[k].M, m[k].M0);
            div.ok = div.ok && in_range<-100, 100>(m[k].M0);
        }
    } else if constexpr (TABLE) {
        table_roots_try<N>(E, ePrev, m, Pi, e, div.ok);
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            int dummy = NAN_NONE;
            e[k] = energy_from_conserved<false>(E, ePrev, m[k].M0, m[k].M, Pi[k], dummy);
        }
    }
#pragma unroll
    for (int k = 0; k < N; ++k) out[k] = recover_finish<TABLE, DivTry, QuotExact>(E, m[k], e[k], Pi[k], nan, div);
}

// getInferredVariables from the moments of the conserved variables.
template <bool TABLE, class DV, class QD = QuotExact>
__device__ __forceinline__ Prim recover_moments(const EosDev &E, const Moments &m, double Pi, double ePrev, int &nan,
                                                DV &div) {
    if constexpr (std::is_same_v<DV, DivTry>) {
        Prim w[1];
        recover_try<TABLE, 1>(E, {m}, {Pi}, ePrev, nan, div, w);
        return w[0];
    }
    double e;
    if (ePrev <= 0.1) {
        if constexpr (std::is_same_v<QD, QuotFast>) e = m.M0 - m.M * QuotFast::rcp1(m.M0);
        else e = m.M0 - QD::q(m.M, m.M0);
    } else  // the FP64 path keeps the division operator inside the root solve's table lookups
        e = energy_from_conserved<TABLE, QD, std::conditional_t<std::is_same_v<QD, QuotFast>, DivRecip, DivExact>>(
            E, ePrev, m.M0, m.M, Pi, nan);
    return recover_finish<TABLE, DV, QD>(E, m, e, Pi, nan, div);
}

template <bool TABLE, class DV, class QD = QuotExact>
__device__ __forceinline__ Prim recover(const EosDev &E, double t, double ttt, double ttx, double tty, double ttn,
                                        double pitt, double pitx, double pity, double pitn, double Pi, double ePrev,
                                        int &nan, DV &div) {
    const Moments m = moments(t, ttt, ttx, tty, ttn, pitt, pitx, pity, pitn);
    return recover_moments<TABLE, DV, QD>(E, m, Pi, ePrev, nan, div);
}

// recover_moments with the division operator, for the cells whose DivTry
// recovery fails; out of line (see role_terms_slow).
struct RecoverSlow {
    Prim w;
    int nan;
};
template <bool TABLE>
__device__ __attribute__((noinline)) RecoverSlow recover_slow(const void *eos, Moments m, double Pi, double ePrev) {
    RecoverSlow r;
    r.nan = NAN_NONE;
    DivFast div;
    r.w = recover_moments<TABLE>(*(const EosDev *)eos, m, Pi, ePrev, r.nan, div);
    return r;
}

// Four root solves from one start value, stepped together: the table-EoS
// Newton iteration and bisection of table_root for each state, unchanged,
// with the four iterations interleaved so that their table lookups and
// divisions overlap (independent chains).  Each state takes exactly the
// steps table_root takes for it; rn[k] is its NaN site.
template <class DV>
__device__ __forceinline__ void table_root4(const EosDev &E, double ePrev, const Moments (&m)[4], const double (&Pi)[4],
                                            double (&e)[4], int (&rn)[4]) {
    DV dx;
    double e0[4];
    bool done[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        e0[k] = ePrev;
        done[k] = false;
        rn[k] = NAN_NONE;
        e[k] = ePrev;
    }
    for (int j = 0; j < MAX_ITERS_NR; ++j) {
        bool any = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (!done[k]) {
                bool bad;
                const double en = nr_step<QuotExact, DV>(E, e0[k], m[k].M0, m[k].M, Pi[k], dx, bad);
                if (bad) {
                    e[k] = ePrev;
                    rn[k] = NAN_ROOT;
                    done[k] = true;
                } else if (nr_converged<QuotExact>(en, e0[k])) {
                    e[k] = en;
                    done[k] = true;
                } else {
                    e0[k] = en;
                }
            }
            any = any || !done[k];
        }
        if (!any) break;
    }
#pragma unroll 1
    for (int k = 0; k < 4; ++k)
        if (!done[k]) e[k] = table_bisect<QuotExact, DV>(E, ePrev, m[k].M0, m[k].M, Pi[k]);
}

// getInferredVariables for four states sharing ePrev (the four half-site
// states of one cell's two faces along one direction): recover() of each,
// with the four root solves interleaved.  NaN sites are recorded in the
// order the four recover() calls would record them.
template <bool TABLE, class DV>
__device__ __forceinline__ void recover4(const EosDev &E, double t, const double (&x)[4][9], double ePrev, int &nan,
                                         DV &div, Prim (&out)[4]) {
    Moments m[4];
    double Pi[4], e[4];
    int rn[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        m[k] = moments(t, x[k][0], x[k][1], x[k][2], x[k][3], x[k][4], x[k][5], x[k][6], x[k][7]);
        Pi[k] = x[k][8];
        rn[k] = NAN_NONE;
    }
    if constexpr (std::is_same_v<DV, DivTry>) {
        recover_try<TABLE, 4>(E, m, Pi, ePrev, nan, div, out);
        return;
    }
    if (ePrev <= 0.1) {
#pragma unroll
        for (int k = 0; k < 4; ++k) e[k] = m[k].M0 - QuotExact::q(m[k].M, m[k].M0);
    } else if constexpr (TABLE) {
        table_root4<DivExact>(E, ePrev, m, Pi, e, rn);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int dummy = NAN_NONE;
            e[k] = energy_from_conserved<false>(E, ePrev, m[k].M0, m[k].M, Pi[k], dummy);
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (rn[k]) nan = rn[k];
        out[k] = recover_finish<TABLE, DV, QuotExact>(E, m[k], e[k], Pi[k], nan, div);
    }
}

}  // namespace vh
