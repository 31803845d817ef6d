// Per-value formulas of the FDTD step, shared by every sweep kernel.
//
// Each function maps already-loaded values to a result, so the naive and the
// tiled kernels run literally the same arithmetic.  Flavours (EXACT):
//
//  * 1 (FP64 parity mode): the expression order of the reference
//    (phonomena/simulation/base_solver.py:323-517), true division by the
//    spacings, no contraction (the library is built with -ffp-contract=off).
//    On the same inputs this reproduces the NumPy solver bit for bit.
//  * 2 (FP64 parity mode, every spacing a power of two): the same
//    expressions with each division by a spacing h taken as the product
//    with 1/h, which the spacing tables then hold.  1/h is exact for h = 2^k,
//    and x * 2^-k and x / 2^k are both the correctly rounded value of the
//    same real number (subnormal and overflowing results included), so this
//    is bit-identical to flavour 1, for the price of a multiply instead of a
//    correctly rounded division (about ten instructions in FP64).
//  * 3 (FP64 parity mode, where values allow it): the correctly rounded
//    quotient a / h from the spacing's reciprocal, see quotient() below; the
//    same bits as flavour 1 again (a zero may differ in sign, which no value
//    of the scheme depends on).
//  * 0 (FP32 modes): divisions replaced by products with inverse spacings,
//    explicit fused multiply-adds.
//
// Material rows hold 16 values: C00 C01 C02 C10 C11 C12 C20 C21 C22 C33 C44
// C55 coef pad pad pad, with coef = dt^2 / rho (pre-folded on the host the way
// the reference computes `self.m.dt**2/self.m.P`).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define PF_DEV __device__ __forceinline__

namespace pf {

enum : int { M_C00 = 0, M_C01, M_C02, M_C10, M_C11, M_C12, M_C20, M_C21, M_C22,
             M_C33, M_C44, M_C55, M_COEF, MAT_STRIDE = 16 };

// MODE_FP64P: MODE_FP64 on a mesh whose spacings are all powers of two
// (flavour 2 above); the host picks it, with reciprocal spacing tables.
// MODE_FP64Q: MODE_FP64 with flavour 3 where a block's values allow it and
// flavour 1 elsewhere; the host picks it when the spacings and stiffnesses do.
enum : int { MODE_FP64 = 0, MODE_FP32 = 1, MODE_FP32C = 2, MODE_FP64P = 3, MODE_FP64Q = 4 };

// The formula flavour of a mode.
constexpr int exact_of(int mode) {
    return mode == MODE_FP64 ? 1 : (mode == MODE_FP64P ? 2 : (mode == MODE_FP64Q ? 3 : 0));
}

PF_DEV float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
PF_DEV double mad(double a, double b, double c) { return __builtin_fma(a, b, c); }

// A spacing with its reciprocal y = RN(1 / h) (MODE_FP64Q).
template <class R> struct Div { R h, y; };
// What a mode's kernels hold for a spacing.
template <class R, int MODE> struct SpacingOf { typedef R type; };
template <> struct SpacingOf<double, MODE_FP64Q> { typedef Div<double> type; };
template <class R, int MODE> using Spacing = typename SpacingOf<R, MODE>::type;
template <class H, class R> PF_DEV H spacing(R h, R y) {
    if constexpr (sizeof(H) == sizeof(R)) return h;
    else return H{h, y};
}

// RN(a / h) in three operations (Markstein: a quotient from y = RN(1 / h),
// corrected by its remainder).  q = RN(a y) is within 1.5 ulp of a / h, so the
// corrected sum differs from a / h by less than 2^-51 ulp before it is
// rounded, and RN of it is RN(a / h) unless a / h is that near a rounding
// boundary.  For a given h only a few dividends come so near; the host tries
// the three operations on all of them (pf_quotient.hpp) and leaves
// a mesh with a spacing that fails to the divisions (none was found among
// 2 x 10^6 random spacings).  This holds while nothing on the way underflows
// or overflows, which follows from the displacements alone (in_range): with
// every spacing at most 2^H and every stiffness entry 0 or at least 2^-C,
// displacements that are 0 or at least 2^-L are multiples of 2^-(L+52),
// and so are their differences; quotients of those (times a stiffness) are 0
// or at least 2^-(L+52+C+H) and their sums multiples of 2^-(L+104+C+H), a
// shear stress, a stiffness times such a sum, of 2^-(L+156+C+H); so the stress
// differences that the update divides are 0 or at least that, their quotients
// are normal and their remainders, multiples of 2^-106 times the dividend,
// exact up to L = 812 - C - 2 H: QUOT_L = 752 for H = C = 20.  Upwards,
// displacements below 2^400, entries below 2^100 and spacings above 2^-60 keep
// everything below 2^630.  (A bound per mesh, as a kernel argument, measured 6 %
// slower than this constant.)
// The compiler's division takes about 14 issue slots (it scales, takes a
// quarter-rate reciprocal and fixes special cases up).  A step of the tiled
// sweep with quotients, with divisions: 205 x 193 x 101 nodes 101 us, 118; with
// an absorbing layer 121, 129; 257 x 257 x 129 with one 235, 250; 129 x 129 x
// 65 with one 46, 54.  Noting the range costs 8 of the 101; a second
// correction, which needs no check of the spacings, 10.  Where every tile is
// out of range the same mesh takes 146 us: the divisions of that branch cost
// more than in a kernel that only divides.  Displacements below 2^-752 are the
// tail ahead of a first wave.  With c dt / h = 0.5 it is short, and the first
// 150 to 1200 steps from rest run as the rest do (100 us, 119); with 0.17 it
// fills part of the mesh for some hundred steps, and they take 106, 123, 127
// and 113 us a step over the first 150, 300, 600 and 1200, against 119.  A byte
// per tile that keeps a tile dividing, a look at the dividends themselves and
// a copy of the whole step for each flavour cost the near case more (124, 103
// and spilled registers).
PF_DEV double quotient(double a, Div<double> d) {
    const double q = a * d.y;
    return __builtin_fma(__builtin_fma(-d.h, q, a), d.y, q);
}
// Whether a displacement is 0 or within 2^-QUOT_L .. 2^400.
constexpr int QUOT_L = 752;
PF_DEV bool in_range(double v) {
    constexpr unsigned lo = (1023u - QUOT_L) << 20, hi = (1023u + 400u) << 20;
    const unsigned e = (unsigned)(__double_as_longlong(v) >> 32) & 0x7fffffffu;
    return e - lo < hi - lo || v == 0.0;
}
PF_DEV bool in_range(float) { return true; }

// a / h in flavours 1 and 3; a * h (h holding 1/h) in flavour 2.
template <int EXACT, class R>
PF_DEV R over(R a, R h) {
    if constexpr (EXACT == 2) return a * h;
    else return a / h;
}
template <int EXACT>
PF_DEV double over(double a, Div<double> d) {
    if constexpr (EXACT == 3) return quotient(a, d);
    else return a / d.h;
}

// ---- normal stresses T1..T3 -------------------------------------------------
// Interior (base_solver.py:329-351): row a of C times the three normal
// differences, each divided by its staggered spacing.
template <int EXACT, class R, class H>
PF_DEV void normal3(const R* c, R dux, R duy, R duz, H hx, H hy, H hz, R& t1, R& t2, R& t3) {
    if constexpr (EXACT) {
        t1 = over<EXACT>(c[M_C00] * dux, hx) + over<EXACT>(c[M_C01] * duy, hy) + over<EXACT>(c[M_C02] * duz, hz);
        t2 = over<EXACT>(c[M_C10] * dux, hx) + over<EXACT>(c[M_C11] * duy, hy) + over<EXACT>(c[M_C12] * duz, hz);
        t3 = over<EXACT>(c[M_C20] * dux, hx) + over<EXACT>(c[M_C21] * duy, hy) + over<EXACT>(c[M_C22] * duz, hz);
    } else {
        // hx, hy, hz are inverse spacings here
        R ex = dux * hx, ey = duy * hy, ez = duz * hz;
        t1 = mad(c[M_C00], ex, mad(c[M_C01], ey, c[M_C02] * ez));
        t2 = mad(c[M_C10], ex, mad(c[M_C11], ey, c[M_C12] * ez));
        t3 = mad(c[M_C20], ex, mad(c[M_C21], ey, c[M_C22] * ez));
    }
}

// Free surface k = 0 (base_solver.py:408-418): same rows with the first
// spacing of each axis; the one-sided uz difference is uz[..,0] - 0; T3 = 0.
template <int EXACT, class R>
PF_DEV void normal3_surface(const R* c, R dux, R duy, R uz0, R hx0, R hy0, R hz0, R& t1, R& t2, R& t3) {
    R duz = uz0 - R(0);
    if constexpr (EXACT) {
        t1 = over<EXACT>(c[M_C00] * dux, hx0) + over<EXACT>(c[M_C01] * duy, hy0) + over<EXACT>(c[M_C02] * duz, hz0);
        t2 = over<EXACT>(c[M_C10] * dux, hx0) + over<EXACT>(c[M_C11] * duy, hy0) + over<EXACT>(c[M_C12] * duz, hz0);
    } else {
        R ex = dux * hx0, ey = duy * hy0, ez = duz * hz0;
        t1 = mad(c[M_C00], ex, mad(c[M_C01], ey, c[M_C02] * ez));
        t2 = mad(c[M_C10], ex, mad(c[M_C11], ey, c[M_C12] * ez));
    }
    t3 = R(0);
}

// ---- shear stresses T4..T6 --------------------------------------------------
// c * (a / h1 + b / h2); the caller passes the spacings in the order the
// reference divides by them (interior: base_solver.py:353-372, surface with
// its swapped spacings: :420-433).
template <int EXACT, class R, class H>
PF_DEV R shear(R c, R a, H h1, R b, H h2) {
    if constexpr (EXACT) {
        return c * (over<EXACT>(a, h1) + over<EXACT>(b, h2));
    } else {
        return c * mad(a, h1, b * h2);
    }
}

// ---- displacement divergence ------------------------------------------------
// (d1 / g1 + d2 / g2) + d3 / g3  (base_solver.py:444-446 and analogues)
template <int EXACT, class R, class H>
PF_DEV R div3(R d1, H g1, R d2, H g2, R d3, H g3) {
    if constexpr (EXACT) {
        return over<EXACT>(d1, g1) + over<EXACT>(d2, g2) + over<EXACT>(d3, g3);
    } else {
        return mad(d1, g1, mad(d2, g2, d3 * g3));
    }
}

// Free-surface u_z bracket with the reference's precedence
// (base_solver.py:514-516): (d1/g1 + d2/g2) + T3[..,1] - T3[..,0]/fdz0.
template <int EXACT, class R>
PF_DEV R div3_uz_surface(R d1, R g1, R d2, R g2, R t3k1, R t3k0, R fz0) {
    if constexpr (EXACT) {
        return over<EXACT>(d1, g1) + over<EXACT>(d2, g2) + t3k1 - over<EXACT>(t3k0, fz0);
    } else {
        return mad(d1, g1, mad(d2, g2, t3k1)) - t3k0 * fz0;
    }
}

// ---- leapfrog ---------------------------------------------------------------
// u_new = 2 u - u_old + coef * div (base_solver.py:441-443).  In FP32 the
// difference takes one fused operation (2 u is exact, and where it would
// overflow a difference that does not is kept); in FP64 two, since 2 u
// overflows there in the reference (fused it measured no faster).  With a
// damping term s > 0 (sponge extension): ((2u - (1-s) u_old) + coef*div) / (1+s);
// in FP32 the division is a product with the hardware reciprocal of 1+s
// (v_rcp_f32, within 1 ulp; one per node, shared by its three components:
// the same expression in every call, so the compiler forms it once), where
// a correctly rounded quotient costs about ten instructions and made the
// two-step pass 0.7 % slower.  At s = 0 both forms give the bits of the
// undamped update (the reciprocal of 1 is 1; 1 * x and x / 1 are exact).
template <int EXACT, bool SPONGE, class R>
PF_DEV R leap(R u, R uo, R coef, R dv, R s) {
    if constexpr (EXACT) {
        if constexpr (SPONGE) {
            // off the absorbing layer s = 0: (1 - 0) u_old = u_old and
            // x / (1 + 0) = x exactly, so the division is skipped there
            R r = 2 * u - (1 - s) * uo + coef * dv;
            if (s != R(0)) r = r / (1 + s);
            return r;
        }
        else return 2 * u - uo + coef * dv;
    } else {
        if constexpr (SPONGE) return mad(coef, dv, mad(R(2), u, -((1 - s) * uo))) * __builtin_amdgcn_rcpf(1 + s);
        else return mad(coef, dv, mad(R(2), u, -uo));
    }
}

// ---- compensated (hi + lo) arithmetic for PF_FP32C --------------------------
// Storage of the lo part: after every normalising TwoSum |lo| <= ulp(hi)/2,
// so lo is kept as a signed 16-bit multiple of 2^-16 ulp(hi) (ulp(hi) =
// 2^(e-24) for hi = m 2^e, 0.5 <= |m| < 1): hi + lo carries 24 + 16
// significant bits in 6 bytes instead of 8.  Both functions are exact
// scalings (ldexp) around one round-to-nearest; hi = 0 has lo = 0.  The sum
// with 1.5 x 2^23 rounds to an integer, ties to even, and leaves it in its low
// bits (one operation for the rounding and the conversion).  This, the sums
// with 2 u and the short last sum of the damped update took 385 x 371 x 193 nodes
// FP32C from 451 to 431 us a step (62 % of the issue slots are VALU work there).
typedef int16_t lo_t;

PF_DEV lo_t lo_encode(float hi, float lo) {
    const int e = __builtin_amdgcn_frexp_expf(hi);
    const float q = __builtin_amdgcn_fmed3f(__builtin_amdgcn_ldexpf(lo, 40 - e), -32767.0f, 32767.0f);
    return (lo_t)__float_as_int(q + 12582912.0f);
}
PF_DEV float lo_decode(float hi, lo_t q) {
    return __builtin_amdgcn_ldexpf((float)q, __builtin_amdgcn_frexp_expf(hi) - 40);
}
// FP64 fields carry no lo part.
PF_DEV lo_t lo_encode(double, double) { return 0; }
PF_DEV double lo_decode(double, lo_t) { return 0.0; }

// Error-free transformations (Knuth TwoSum, FMA TwoProd); a value is the
// unevaluated sum hi + lo with |lo| <= ulp(hi)/2 after normalisation.
PF_DEV void two_sum(float a, float b, float& s, float& e) {
    s = a + b;
    float bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}
// two_sum(2 a, b): 2 a is exact, so it needs no operation of its own.
PF_DEV void two_sum_2a(float a, float b, float& s, float& e) {
    s = mad(2.0f, a, b);
    float bb = mad(-2.0f, a, s);
    e = mad(2.0f, a, -(s - bb)) + (b - bb);
}
// two_sum for |a| >= |b| or a = b = 0 (Dekker): the same s and e.
PF_DEV void fast_two_sum(float a, float b, float& s, float& e) {
    s = a + b;
    e = b - (s - a);
}

// U_new = 2 U - U_old + f (+ damping), with U = hi + lo.  The increment f is
// an ordinary FP32 value; what is compensated is the accumulation of the
// displacement itself, so the small per-step increments are never lost
// against the large running value.
template <bool SPONGE>
PF_DEV void leap_comp(float hi, float lo, float ohi, float olo, float f, float s, float& nhi, float& nlo) {
    if constexpr (!SPONGE) {
        float a, e;
        two_sum_2a(hi, -ohi, a, e);
        float low = (mad(2.0f, lo, -olo) + e) + f;
        two_sum(a, low, nhi, nlo);
    } else {
        float q = 1.0f - s;
        float p = q * ohi;
        float pe = mad(q, ohi, -p);
        float plow = mad(q, olo, pe);
        float a, e;
        two_sum_2a(hi, -p, a, e);
        float low = (mad(2.0f, lo, -plow) + e) + f;
        float nh, nl;
        two_sum(a, low, nh, nl);
        float r = __builtin_amdgcn_rcpf(1.0f + s);  // as in leap()
        float h2 = nh * r;
        float l2 = mad(nh, r, -h2) + nl * r;
        // |nl r| <= ulp(nh) r / 2 <= ulp(h2): |l2| < 2 ulp(h2) <= |h2|
        fast_two_sum(h2, l2, nhi, nlo);
    }
}

// a + c * (b - d) for the Mur faces in compensated form; c = ch + cl.
PF_DEV void mur_comp(float ah, float al, float ch, float cl, float bh, float bl, float dh, float dl,
                     float& rh, float& rl) {
    float sh, se;
    two_sum(bh, -dh, sh, se);
    se += bl - dl;
    float ph = ch * sh;
    float pe = mad(ch, sh, -ph);
    pe = mad(ch, se, mad(cl, sh, pe));
    float th, te;
    two_sum(ah, ph, th, te);
    te += al + pe;
    two_sum(th, te, rh, rl);
}

}  // namespace pf
