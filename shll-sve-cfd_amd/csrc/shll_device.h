// shll_device.h -- device arithmetic of the SHLL step for gfx950.
//
// The precisions share one set of templates:
//   PREC_F64   : every value double, the reference association (FP64 oracle form)
//   PREC_REF32 : float values with the reference's double promotions, so results are
//                bitwise those of the reference C on x86-64
//   PREC_C32   : float arithmetic, (hi, lo) float state, conservative face update
//                with TwoSum (the FP32-compensated form)
//   PREC_C32K  : PREC_C32 with one Kahan step per cell for the update
//   PREC_F64F  : FP64 values in the compensated forms' arrangement (fused multiply-adds,
//                1/rho and 1/a from faithful Newton sequences, face-term update); 1D
//
// The library is compiled with -ffp-contract=off: every + - * below is one IEEE-754
// operation in source order (fused multiply-adds only where written), and division
// and square root are correctly rounded, so the F64 and REF32 kernels reproduce the CPU
// results bit for bit (F64F alone uses faithful sequences).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "shll_types.h"

namespace shll {

// ---------------------------------------------------------------------------
// cross-lane moves inside one wavefront (DPP wave_shr:1 / wave_shl:1)
// from_left(x)  : the value x of lane-1 (lane 0 keeps its own)
// from_right(x) : the value x of lane+1 (lane 63 keeps its own)
// Every lane of the wave executes these with the same control flow.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int dpp_from_left(int x) {
    return __builtin_amdgcn_update_dpp(x, x, 0x138, 0xf, 0xf, false);
}
__device__ __forceinline__ int dpp_from_right(int x) {
    return __builtin_amdgcn_update_dpp(x, x, 0x130, 0xf, 0xf, false);
}
__device__ __forceinline__ float from_left(float x) {
    return __int_as_float(dpp_from_left(__float_as_int(x)));
}
__device__ __forceinline__ float from_right(float x) {
    return __int_as_float(dpp_from_right(__float_as_int(x)));
}
__device__ __forceinline__ double from_left(double x) {
    int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(dpp_from_left(hi), dpp_from_left(lo));
}
__device__ __forceinline__ double from_right(double x) {
    int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(dpp_from_right(hi), dpp_from_right(lo));
}

// from_left_z(x) / from_right_z(x): as from_left / from_right, except that lane 0 (lane 63)
// reads 0 -- for values whose edge lanes are don't-cares; without an "old" operand the
// shift can be folded into the instruction that uses it
__device__ __forceinline__ float from_left_z(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_right_z(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double from_left_z(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_right_z(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// from_left_or(x, e) / from_right_or(x, e): as from_left / from_right, except that lane 0
// (lane 63) takes e, a value the lane brings from outside the wavefront
__device__ __forceinline__ float from_left_or(float x, float e) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(e), __float_as_int(x), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float from_right_or(float x, float e) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(e), __float_as_int(x), 0x130, 0xf, 0xf, false));
}
__device__ __forceinline__ double from_left_or(double x, double e) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(e), __double2loint(x), 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(e), __double2hiint(x), 0x138, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double from_right_or(double x, double e) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(e), __double2loint(x), 0x130, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(e), __double2hiint(x), 0x130, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// wave-uniform value (moves it to a scalar register)
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// ---------------------------------------------------------------------------
// Correctly rounded division and square root.  The fast paths are the instruction sequences the
// compiler emits for IEEE '/', sqrtf and sqrt (-fhip-fp32-correctly-rounded-divide-sqrt; FP64 is
// always IEEE) minus their range handling -- the exponent pre-scaling of v_div_scale /
// v_div_fmas, the special-value pass of v_div_fixup, the square roots' pre-scaling of tiny
// radicands and their pass-through of 0 and inf.  With operands and results of moderate size (no
// intermediate leaves the normal range) they give the same bits as the operators.
// The reference forms (F64, REF32) call them through RefArith::prim1_fast / prim2_fast, which
// say whether every intermediate stayed in that range (below), and hand the other cells -- a
// vacuum, a tiny velocity, a non-finite state -- to the operators themselves (prim1_exact /
// prim2_exact), so they are always bitwise '/' and sqrt.  The compensated scheme calls the fast
// paths directly: its divisors (density, sound speed) and radicand (gamma*R*T) are of order one,
// and its one possibly tiny quotient, the Mach number M, only enters as M/2 +- 1/2 and 1 - M^2,
// which absorb any last-place difference of a tiny M.
// ---------------------------------------------------------------------------
// rcp_fast(b): 1/b correctly rounded -- v_rcp_f32 (within 1 ulp) and one Newton step with
// fused multiply-adds.  Checked against IEEE 1.0f/b on the MI355X for every normal float b
// whose reciprocal is normal (2^23 mantissas x 252 exponents, no difference).
__device__ __forceinline__ float rcp_fast(float b) {
    const float r = __builtin_amdgcn_rcpf(b);
    const float e = __builtin_fmaf(-b, r, 1.0f);
    return __builtin_fmaf(e, r, r);
}
// a/b from its correctly rounded reciprocal y: q = a*y is within one ulp of a/b, the residual
// a - b*q is exact in one fma, and q + residual*y is the correctly rounded quotient (Markstein's
// theorem; also checked against IEEE a/b on 2^31 random float and 2^28 random double pairs)
template <class RT>
__device__ __forceinline__ RT quot(RT a, RT b, RT y) {
    const RT q = a * y;
    const RT d = __builtin_elementwise_fma(-b, q, a);
    return __builtin_elementwise_fma(d, y, q);
}
__device__ __forceinline__ float div_fast(float a, float b) { return quot(a, b, rcp_fast(b)); }
__device__ __forceinline__ float sqrt_fast(float x) {
    float s = __builtin_amdgcn_sqrtf(x);   // within 1 ulp
    const float sdn = __int_as_float(__float_as_int(s) - 1);
    const float sup = __int_as_float(__float_as_int(s) + 1);
    const float rdn = __builtin_fmaf(-sdn, s, x);
    const float rup = __builtin_fmaf(-sup, s, x);
    s = rdn <= 0.0f ? sdn : s;
    return rup > 0.0f ? sup : s;
}
// 1/b: the hardware's seed (v_rcp_f64, relative error about 2^-24, measured) and two Newton steps;
// equal to the correctly rounded 1/b on each of 8e8 random arguments with exponents -1000..1000
// (MI355X).  Zero gives NaN (not inf).
__device__ __forceinline__ double rcp_nr2(double b) {
    double r = __builtin_amdgcn_rcp(b);
    double e = __builtin_fma(-b, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-b, r, 1.0);
    return __builtin_fma(r, e, r);
}
// s = sqrt(x) correctly rounded, and y = 1/s: the square root's iteration already holds
// h = 1/(2 sqrt(x)) to about 2^-46, so one Newton step on 2h replaces a reciprocal seed and two
// (checked with quot against IEEE sqrt and v/sqrt(x) on 2^28 random arguments)
__device__ __forceinline__ void sqrt_rcp(double x, double& s, double& y) {
    const double q = __builtin_amdgcn_rsq(x);
    double g = x * q, h = q * 0.5;  // sqrt(x) and 1/(2 sqrt(x)) estimates
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    s = __builtin_fma(d, h, g);
    const double w = h + h;
    const double e = __builtin_fma(-s, w, 1.0);
    y = __builtin_fma(w, e, w);
}
__device__ __forceinline__ void sqrt_rcp(float x, float& s, float& y) {
    s = sqrt_fast(x);
    y = rcp_fast(s);
}

// Faithful FP64 reciprocal square root and square root (the F64F form, with rcp_nr2): the hardware
// seed (v_rsq_f64, relative error about 2^-24, measured) and one third-order step
// y <- y (1 + e/2 + 3 e^2/8), e = 1 - x y^2 (its remainder is 5/16 e^3, about 2^-73; two Newton steps
// took one operation more and rounded twice), and the same correction of x y for the root.  y is
// within 2 ulp of 1.0/sqrt(x), s within 1 of sqrt(x) on random arguments with exponents -1000..1000
// (MI355X); neither is correctly rounded, and the seeds are the hardware's, so the F64F results are
// reproduced on a CPU to within round-off, not bit for bit.  Zero, negative and NaN arguments
// give NaN.
__device__ __forceinline__ void rsq_sqrt(double x, double& y, double& s) {
    const double q = __builtin_amdgcn_rsq(x);
    const double g = x * q;
    const double e = __builtin_fma(-g, q, 1.0);
    const double c = __builtin_fma(0.375, e, 0.5) * e;
    y = __builtin_fma(q, c, q);
    s = __builtin_fma(g, c, g);
}
__device__ __forceinline__ double rsq_nr2(double x) {
    double y, s;
    rsq_sqrt(x, y, s);
    return y;
}

// ---------------------------------------------------------------------------
// Reference association (F64 and REF32).  RT is the storage/arithmetic type;
// (double) conversions sit where the reference's double literals and its double
// sqrt() put them (base_shll.c:135-139, :172-175; base_shll_2d.c:313-317).
// For RT = double every conversion is the identity.
//
// prim*_fast give the bits of prim*_exact in about half the instructions, and say where they
// may not:
//   - quotients with one divisor share its reciprocal (u1/u0, u2/u0, u3/u0; vx/a, vy/a); 1/cv
//     is a constant (Consts::d_rcv, f_rcv, correctly rounded by the host);
//   - e - kin is one fused multiply-add: kin/2's product is exact (a power of two times a
//     rounded square, or in REF32 1D first order a 48-bit square in double);
//   - (float)sqrt((double)x) of a float x is the float square root (rounding twice is
//     harmless from 53 to 24 bits), so REF32 takes it in float;
//   - a quotient of +-0 comes out as +0, a zero whose sign no sum here keeps.
// A quotient is right to the last bit while it and the reciprocal are normal and its remainder is
// exact, the dividend 48 (FP64: 106) binary orders above the smallest denormal.  What covers that:
//   - RefSpan: the radicand x = gamma R T and the density within [LO, HI) (else the cell takes
//     prim*_exact).  T > 0 then bounds e = cv T + kin below, the energy with it, and a away from
//     the ends of the range; non-finite states fail here;
//   - then only a velocity of |M| < 2^-35 (FP64: 2^-500), of a momentum |u| < ULO, can be off: M/2 +-
//     1/2 is +-1/2 and 1 - M^2 is 1 all the same, and next to the sound speed nothing of it is left
//     in the fluxes, except in the transverse momentum's (rho u v).  So 2D divides again with the
//     operator where a momentum is below ULO and not zero (*tiny).  Transverse velocities ahead of a
//     front square from cell to cell (1e-9, 1e-18, 1e-36, 0), so a wavefront that holds a front
//     often has such a lane: REF32 at 128^2, four steps per launch, 10.7 us with the whole cell
//     redone there, 8.4 us with the divisions only, 7.6 us once the fronts are gone.
// Before, each of the five (2D: seven) operations carried its own compare and branch, and a
// gas at rest (u = 0) took the slow path of two of them: 1D first order FP64, 1024 cells,
// 5.43 us per 8-step launch, 4.2 us now; second order, 4 cells per lane: 894 VALU instructions per
// step, 581 now; the whole 2D second-order REF32 run at 1024^2 1.12x.
// ---------------------------------------------------------------------------
template <class RT> struct RefRange;
template <> struct RefRange<double> {
    static constexpr double ULO = 0x1p-800;
    static constexpr int LO = (1023 - 200) << 20, HI = (1023 + 200) << 20;  // 2^-200, 2^200
    __device__ static __forceinline__ int bits(double x) { return __double2hiint(x); }
};
template <> struct RefRange<float> {
    static constexpr float ULO = 0x1p-80f;
    static constexpr int LO = (127 - 30) << 23, HI = (127 + 40) << 23;  // 2^-30, 2^40
    __device__ static __forceinline__ int bits(float x) { return __float_as_int(x); }
};
// Radicands and densities of any number of cells within [LO, HI): their (high) words as integers,
// which order like the values; a negative value is below, a NaN below or above.  Two full-rate
// instructions per cell.
template <class RT>
struct RefSpan {
    using R = RefRange<RT>;
    int top = R::LO, low = R::LO;
    __device__ __forceinline__ void take(RT x, RT rho) {
        top = max(top, max(R::bits(x), R::bits(rho)));
        low = min(low, min(R::bits(x), R::bits(rho)));
    }
    __device__ __forceinline__ bool ok() const { return low >= R::LO && top < R::HI; }
};
// The same by the smallest magnitude, as floats, which order alike and pass over a NaN, and the
// largest unsigned integer, where a negative value or a NaN is above any other: thin() is true only of
// a magnitude below LO, not of a cell without a temperature.
template <class RT>
struct ThinSpan {
    using R = RefRange<RT>;
    unsigned top = 0;
    float low = __builtin_inff();
    __device__ __forceinline__ void take(RT x, RT rho) {
        top = max(top, max((unsigned)R::bits(x), (unsigned)R::bits(rho)));
        asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(low) : "v"(R::bits(x)), "v"(R::bits(rho)));
    }
    __device__ __forceinline__ bool thin() const { return __float_as_int(low) < R::LO; }
    __device__ __forceinline__ bool ok() const { return !thin() && top < (unsigned)R::HI; }
};

template <class RT>
struct RefArith {
    static constexpr bool F32 = sizeof(RT) == 4;
    // Compute_P_from_U, 1D.  KE = 0: (0.5*u)*u (base_shll.c:174); KE = 1: 0.5*(u*u)
    // (the 2D files' association, used by the derived 1D second-order scheme).
    // M = vx/a (base_shll.c:136).
    __device__ static __forceinline__ void prim1_exact(RT u0, RT u1, RT u2, int ke, RT cv, RT gR, RT& vx, RT& T,
                                                       RT& a, RT& M) {
        vx = u1 / u0;
        double kin = ke == 0 ? (0.5 * (double)vx) * (double)vx : 0.5 * (double)(vx * vx);
        T = (RT)(((double)(u2 / u0) - kin) / (double)cv);
        a = (RT)sqrt((double)(gR * T));
        M = vx / a;
    }
    template <class Span>
    __device__ static __forceinline__ void prim1_fast(RT u0, RT u1, RT u2, int ke, RT cv, double rcv, RT gR, RT& vx,
                                                      RT& T, RT& a, RT& M, Span& span) {
        RT y;
        if constexpr (F32) y = rcp_fast(u0);
        else y = rcp_nr2(u0);
        vx = quot(u1, u0, y);
        const double e = (double)quot(u2, u0, y);
        const double vv = ke == 0 && F32 ? (double)vx * (double)vx : (double)(vx * vx);
        T = (RT)quot(__builtin_fma(-0.5, vv, e), (double)cv, rcv);
        const RT x = gR * T;
        sqrt_rcp(x, a, y);
        M = quot(vx, a, y);
        span.take(x, u0);
    }
    // the range test on a momentum
    __device__ static __forceinline__ bool small(RT um) {
        return !(fabs(um) >= RefRange<RT>::ULO || um == (RT)0);
    }
    // Compute_P_from_U, 2D (base_shll_2d.c:313-317), and the two Mach numbers
    __device__ static __forceinline__ void prim2_exact(RT u0, RT u1, RT u2, RT u3, RT cv, RT gR, RT& vx, RT& vy,
                                                       RT& T, RT& a, RT& Mx, RT& My) {
        vx = u1 / u0;
        vy = u2 / u0;
        T = (RT)(((double)(u3 / u0) - 0.5 * (double)(vx * vx + vy * vy)) / (double)cv);
        a = (RT)sqrt((double)(gR * T));
        Mx = vx / a;
        My = vy / a;
    }
    __device__ static __forceinline__ void prim2_fast(RT u0, RT u1, RT u2, RT u3, RT cv, double rcv, RT gR, RT& vx,
                                                      RT& vy, RT& T, RT& a, RT& Mx, RT& My, RefSpan<RT>& span,
                                                      bool& tiny) {
        RT y;
        if constexpr (F32) y = rcp_fast(u0);
        else y = rcp_nr2(u0);
        vx = quot(u1, u0, y);
        vy = quot(u2, u0, y);
        const double e = (double)quot(u3, u0, y);
        T = (RT)quot(__builtin_fma(-0.5, (double)(vx * vx + vy * vy), e), (double)cv, rcv);
        const RT x = gR * T;
        sqrt_rcp(x, a, y);
        Mx = quot(vx, a, y);
        My = quot(vy, a, y);
        span.take(x, u0);
        tiny |= small(u1) || small(u2);
    }
    // Z invariants (base_shll.c:137-139): 0.5*(M +- 1) in double, stored to RT, is M/2 +- 1/2
    // rounded once: M/2 is exact, and for a float M the double sum is exact or nowhere near the
    // middle of two floats
    __device__ static __forceinline__ void zinv(RT M, RT a, RT& z1, RT& z2, RT& z3) {
        z1 = __builtin_elementwise_fma((RT)0.5, M, (RT)0.5);
        z2 = (RT)((0.5 * (double)a) * (1.0 - (double)(M * M)));
        z3 = __builtin_elementwise_fma((RT)0.5, M, (RT)-0.5);
    }
    // minmod (2nd_order_base_shll.c:191-201): product sign test, ties -> right
    __device__ static __forceinline__ RT mm(RT l, RT r) {
        RT pick = fabs(l) < fabs(r) ? l : r;
        return l * r < (RT)0 ? (RT)0 : pick;
    }
    // 0.5*(difference) with the double literal of base-omp/2nd_order_base_shll.c:317,
    // rounded to RT as minmod's argument (halving is exact, or rounds once, in either type)
    __device__ static __forceinline__ RT half(RT x) { return (RT)0.5 * x; }
};

// FP32-compensated arithmetic: float, with explicit fused multiply-adds where a
// product feeds a sum (one rounding instead of two, and one instruction).
struct C32Arith {
    __device__ static __forceinline__ void prim1(float u0, float u1, float u2, float rcv, float gR, float& vx,
                                                 float& T, float& a) {
        float inv = rcp_fast(u0);
        vx = u1 * inv;
        float e = u2 * inv;
        T = __builtin_fmaf(-0.5f * vx, vx, e) * rcv;  // (e - vx^2/2) / cv
        a = sqrt_fast(gR * T);
    }
    __device__ static __forceinline__ void prim2(float u0, float u1, float u2, float u3, float rcv, float gR,
                                                 float& vx, float& vy, float& T, float& a) {
        float inv = rcp_fast(u0);
        vx = u1 * inv;
        vy = u2 * inv;
        float e = u3 * inv;
        T = __builtin_fmaf(-0.5f, __builtin_fmaf(vx, vx, vy * vy), e) * rcv;
        a = sqrt_fast(gR * T);
    }
    // z1 = (M+1)/2, z2 = (a/2)(1-M^2), z3 = (M-1)/2.  z1 and z3 are RN(M/2 +- 1/2): M/2 is
    // exact (or, below 2^-125, off by less than 2^-150, which the sum rounds away), so one
    // fused multiply-add gives the bits of the product-then-sum
    __device__ static __forceinline__ void zinv(float M, float a, float& z1, float& z2, float& z3) {
        z1 = __builtin_fmaf(0.5f, M, 0.5f);
        z2 = (0.5f * a) * __builtin_fmaf(-M, M, 1.0f);
        z3 = __builtin_fmaf(0.5f, M, -0.5f);
    }
    // minmod as the median of (l, r, 0): the smaller magnitude when the signs agree,
    // zero otherwise -- one v_med3_f32.  Unlike the reference's product test it also
    // clips slopes of opposite sign whose float product underflows, and the sign of a
    // zero result is unspecified (a zero slope only ever meets a nonzero or +0 face
    // flux, where the sign of the zero cannot change the sum).
    __device__ static __forceinline__ float mm(float l, float r) { return __builtin_amdgcn_fmed3f(l, r, 0.0f); }
    __device__ static __forceinline__ float half(float x) { return 0.5f * x; }
};

// FP64 in the compensated scheme's arrangement (PREC_F64F): the limiter of the C32 forms in
// double (the split fluxes are flux1_f64f in shll_flux.h), on fluxes scaled by SC.
// minmod is the median of (l, r, 0): the smaller magnitude when the signs agree, zero otherwise
// (sign of a zero result unspecified, as in C32Arith::mm).
//   UNIT   SC = 2^-512, so that every |l|, |r| < 1: max(min(l, r), 0) and max(min(-l, -r), 0) are
//          one v_min_f64 each, whose result the output clamp limits to [0, 1] for free; one of
//          the two is zero.  Three instructions instead of four, the same values.
//   else   SC = 1, any magnitude.
template <bool UNIT>
struct F64FArith {
    static constexpr double SC = UNIT ? 0x1p-512 : 1.0;
    // min(l, r) and min(-l, -r), each limited to [0, 1] (the compiler turns the second into a
    // negated maximum, which takes the clamp as an instruction of its own)
    __device__ static __forceinline__ double min01(double l, double r) {
        double d;
        asm("v_min_f64 %0, %1, %2 clamp" : "=v"(d) : "v"(l), "v"(r));
        return d;
    }
    __device__ static __forceinline__ double nmin01(double l, double r) {
        double d;
        asm("v_min_f64 %0, -%1, -%2 clamp" : "=v"(d) : "v"(l), "v"(r));
        return d;
    }
    __device__ static __forceinline__ double mm(double l, double r) {
        if constexpr (UNIT) return min01(l, r) - nmin01(l, r);
        else return __builtin_fmax(__builtin_fmin(l, r), __builtin_fmin(__builtin_fmax(l, r), 0.0));
    }
    __device__ static __forceinline__ double half(double x) { return 0.5 * x; }
};

// the same split in FP64: U*Z2 once, two fused multiply-adds
__device__ __forceinline__ void split_f64f(double f, double u, double z1, double z2, double z3, double& fp,
                                           double& fm) {
    const double uz = u * z2;
    fp = __builtin_fma(f, z1, uz);
    fm = __builtin_fma(-f, z3, -uz);
}

// Limited slope of a split flux from its values at c-1, c, c+1 (interior cells):
//   LIM_MINMOD  mm(qc - ql, qr - qc)                                 2nd_order_base_shll.c:268-276
//   LIM_MC      mm((qr - ql)/2, theta * mm(qc - ql, qr - qc))        base-omp/2nd_order_base_shll.c:317-325
template <class A, int LIM, class RT>
__device__ __forceinline__ RT limited_slope(RT ql, RT qc, RT qr, RT theta) {
    const RT s = A::mm(qc - ql, qr - qc);
    if constexpr (LIM == LIM_MINMOD) return s;
    else return A::mm(A::half(qr - ql), theta * s);
}

// TwoSum (Knuth, TAOCP vol. 2, 4.2.2): s + e == a + b exactly
__device__ __forceinline__ void two_sum(float a, float b, float& s, float& e) {
    s = a + b;
    float bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}

// Fast2Sum (Dekker 1971): s + e == a + b exactly when |a| >= |b| (the renormalisation
// of a (hi, lo) pair, whose lo is below an ulp of hi)
__device__ __forceinline__ void fast_two_sum(float a, float b, float& s, float& e) {
    s = a + b;
    e = b - (s - a);
}

// SHLL split of one flux component: F+ = F*Z1 + U*Z2, F- = -F*Z3 - U*Z2 (base_shll.c:149-157)
template <class RT>
__device__ __forceinline__ void split(RT f, RT u, RT z1, RT z2, RT z3, RT& fp, RT& fm) {
    fp = f * z1 + u * z2;
    fm = -f * z3 - u * z2;
}

// the same split in the compensated scheme's float arithmetic: U*Z2 once, two FMAs
__device__ __forceinline__ void split_c32(float f, float u, float z1, float z2, float z3, float& fp, float& fm) {
    const float uz = u * z2;
    fp = __builtin_fmaf(f, z1, uz);
    fm = __builtin_fmaf(-f, z3, -uz);
}

}  // namespace shll
