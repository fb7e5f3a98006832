// shll_flux.h -- the split fluxes of one cell (Compute_P_from_U followed by
// Compute_F_from_P for that cell), shared by the step kernels and the stage kernel so
// that both evaluate exactly the same operations.
#pragma once

#include "shll_device.h"

namespace shll {

// storage / arithmetic type of a precision
template <int PREC> struct Real { using T = double; };
template <> struct Real<PREC_REF32> { using T = float; };
template <> struct Real<PREC_C32> { using T = float; };
template <> struct Real<PREC_C32K> { using T = float; };

// constants of the reference forms, by type
template <class RT>
__device__ __forceinline__ void ref_consts(const Inst& in, RT& cv, double& rcv, RT& gR) {
    if constexpr (sizeof(RT) == 8) {
        cv = in.k.d_cv;
        rcv = in.k.d_rcv;
        gR = in.k.d_gR;
    } else {
        cv = in.k.f_cv;
        rcv = in.k.f_rcv;
        gR = in.k.f_gR;
    }
}
// Compute_P_from_U of one cell: the fast form (for cells that pass span), the exact form
template <class RT, class Span>
__device__ __forceinline__ void ref_prim1(RT u0, RT u1, RT u2, const Inst& in, RT& vx, RT& T, RT& a, RT& M,
                                          Span& span) {
    RT cv, gR;
    double rcv;
    ref_consts<RT>(in, cv, rcv, gR);
    RefArith<RT>::prim1_fast(u0, u1, u2, in.ke, cv, rcv, gR, vx, T, a, M, span);
}
template <class RT>
__device__ __forceinline__ void ref_prim1_exact(RT u0, RT u1, RT u2, const Inst& in, RT& vx, RT& T, RT& a, RT& M) {
    RT cv, gR;
    double rcv;
    ref_consts<RT>(in, cv, rcv, gR);
    RefArith<RT>::prim1_exact(u0, u1, u2, in.ke, cv, gR, vx, T, a, M);
}
// Compute_F_from_P of one cell (base_shll.c:134-157)
template <class RT>
__device__ __forceinline__ void ref_flux1(RT u0, RT u1, RT u2, RT vx, RT T, RT a, RT M, RT (&fp)[3], RT (&fm)[3]) {
    RT z1, z2, z3;
    RefArith<RT>::zinv(M, a, z1, z2, z3);
    const RT P = u0 * T;  // (rho*R)*T with R = 1 (base_shll.c:17, :141)
    const RT f0 = u1, f1 = u1 * vx + P, f2 = vx * (u2 + P);
    split<RT>(f0, u0, z1, z2, z3, fp[0], fm[0]);
    split<RT>(f1, u1, z1, z2, z3, fp[1], fm[1]);
    split<RT>(f2, u2, z1, z2, z3, fp[2], fm[2]);
}

// 1D, F64F: F+ and F- of the three variables scaled by SC (a power of two), and the sound speed
// a (base_shll.c:134-157 in the compensated forms' arrangement).  With R = 1 and
// c = gamma R/CV:
//   q = E - (rho u) u / 2,  p = q/CV                 (no E/rho; p itself is never formed)
//   a^2 = c q/rho,  from x = q/rho: y = 1/sqrt(x), s = sqrt(x)   (rsq_sqrt)
//   Mh = SC M/2 = (u y) SC/(2 sqrt c),  Z1 = Mh + SC/2,  Z3 = Mh - SC/2
//   Z2 = SC (a/2)(1 - M^2) = s SC sqrt(c)/2 - Mh u
// 32 FP64 operations and two seeds (36 with p, a^2 and 1 - M^2 formed).  With the limiter's
// three-instruction form the step of 8 cells issues 626 VALU instructions instead of 715 (and 12
// that bound the scaled fluxes, Extremes), and a batch of 400 tubes ran in 85.8 instead of 92.6 ms.
// Rounding error of a step against 80-bit arithmetic (rho, m, E relative): 9.6e-18, 1.22e-16,
// 1.00e-17 with 36 operations, 9.4e-18, 1.22e-16, 9.8e-18 so; after 20 steps 3.42e-17, 4.73e-16,
// 2.64e-17 and 3.29e-17, 4.42e-16, 2.58e-17.  sqrt c and its reciprocal are the nearest doubles (host).
template <bool UNIT>
__device__ __forceinline__ void flux1_f64f(double u0, double u1, double u2, const Inst& in, double (&fp)[3],
                                           double (&fm)[3], double& a) {
    constexpr double H = 0.5 * F64FArith<UNIT>::SC;
    const double km = UNIT ? in.k.u_hrc : 0.5 * in.k.d_rsc;  // SC/(2 sqrt c)
    const double ka = UNIT ? in.k.u_hsc : 0.5 * in.k.d_sc;   // SC sqrt(c)/2
    const double inv = rcp_nr2(u0);
    const double vx = u1 * inv;
    const double k = u1 * vx;
    const double q = __builtin_fma(-0.5, k, u2);
    double y, s;
    rsq_sqrt(q * inv, y, s);
    const double Mh = km * (vx * y);
    const double z1 = Mh + H, z3 = Mh - H;
    const double z2 = __builtin_fma(-Mh, vx, ka * s);
    a = in.k.d_sc * s;
    const double f1 = __builtin_fma(in.k.d_rcv, q, k), f2 = vx * __builtin_fma(in.k.d_rcv, q, u2);
    split_f64f(u1, u0, z1, z2, z3, fp[0], fm[0]);
    split_f64f(f1, u1, z1, z2, z3, fp[1], fm[1]);
    split_f64f(f2, u2, z1, z2, z3, fp[2], fm[2]);
}

// 1D: F+ and F- of the three variables and the sound speed a (base_shll.c:134-177;
// the second-order scheme's kinetic-energy association through in.ke).  U: the state
// (F64/REF32) or its hi word (C32/C32K).
template <int PREC, class RT>
__device__ __forceinline__ void flux1(RT u0, RT u1, RT u2, const Inst& in, RT (&fp)[3], RT (&fm)[3], RT& a) {
    RT vx, T, z1, z2, z3;
    if constexpr (PREC == PREC_F64F) {
        flux1_f64f<false>(u0, u1, u2, in, fp, fm, a);
    } else if constexpr (PREC == PREC_C32 || PREC == PREC_C32K) {
        C32Arith::prim1(u0, u1, u2, in.k.c_rcv, in.k.c_gR, vx, T, a);
        C32Arith::zinv(div_fast(vx, a), a, z1, z2, z3);
        const RT P = u0 * T;  // R = 1
        const RT f0 = u1, f1 = __builtin_fmaf(u1, vx, P), f2 = vx * (u2 + P);
        split_c32(f0, u0, z1, z2, z3, fp[0], fm[0]);
        split_c32(f1, u1, z1, z2, z3, fp[1], fm[1]);
        split_c32(f2, u2, z1, z2, z3, fp[2], fm[2]);
    } else {
        RT M;
        RefSpan<RT> span;
        ref_prim1<RT>(u0, u1, u2, in, vx, T, a, M, span);
        if (!span.ok()) ref_prim1_exact<RT>(u0, u1, u2, in, vx, T, a, M);
        ref_flux1<RT>(u0, u1, u2, vx, T, a, M, fp, fm);
    }
}

// 2D reference forms: Compute_P_from_U of one cell and the Mach numbers (as ref_prim1; tiny: divide
// for the velocities again)
template <class RT>
struct Prim2 {
    RT vx, vy, T, a, Mx, My;
};
template <class RT>
__device__ __forceinline__ void ref_prim2(const RT (&U)[4], const Inst& in, Prim2<RT>& q, RefSpan<RT>& span, bool& tiny) {
    RT cv, gR;
    double rcv;
    ref_consts<RT>(in, cv, rcv, gR);
    RefArith<RT>::prim2_fast(U[0], U[1], U[2], U[3], cv, rcv, gR, q.vx, q.vy, q.T, q.a, q.Mx, q.My, span, tiny);
}
template <class RT>
__device__ __forceinline__ void ref_prim2_exact(const RT (&U)[4], const Inst& in, Prim2<RT>& q) {
    RT cv, gR;
    double rcv;
    ref_consts<RT>(in, cv, rcv, gR);
    RefArith<RT>::prim2_exact(U[0], U[1], U[2], U[3], cv, gR, q.vx, q.vy, q.T, q.a, q.Mx, q.My);
}
// redo what the fast form could not (ok: span's)
template <class RT>
__device__ __forceinline__ void ref_prim2_redo(const RT (&U)[4], const Inst& in, bool ok, Prim2<RT>& q) {
    if (!ok) {
        ref_prim2_exact<RT>(U, in, q);
    } else {
        q.vx = U[1] / U[0];
        q.vy = U[2] / U[0];
    }
}
// Compute_F_from_P of one cell, x and y (base_shll_2d.c:239-298)
template <class RT>
__device__ __forceinline__ void ref_flux2(const RT (&U)[4], const Prim2<RT>& q, RT (&xp)[4], RT (&xm)[4], RT (&yp)[4],
                                          RT (&ym)[4]) {
    RT z1, z2, z3;
    const RT P = U[0] * q.T;  // (rho*R)*T with R = 1 (base_shll_2d.c:24, :246)
    RefArith<RT>::zinv(q.Mx, q.a, z1, z2, z3);
    split<RT>(U[1], U[0], z1, z2, z3, xp[0], xm[0]);
    split<RT>(U[1] * q.vx + P, U[1], z1, z2, z3, xp[1], xm[1]);
    split<RT>(U[1] * q.vy, U[2], z1, z2, z3, xp[2], xm[2]);
    split<RT>(q.vx * (U[3] + P), U[3], z1, z2, z3, xp[3], xm[3]);
    RefArith<RT>::zinv(q.My, q.a, z1, z2, z3);
    split<RT>(U[2], U[0], z1, z2, z3, yp[0], ym[0]);
    split<RT>(U[2] * q.vx, U[1], z1, z2, z3, yp[1], ym[1]);
    split<RT>(U[2] * q.vy + P, U[2], z1, z2, z3, yp[2], ym[2]);
    split<RT>(q.vy * (U[3] + P), U[3], z1, z2, z3, yp[3], ym[3]);
}

// The reference's update terms: u - lam*x, and the second-order u - 0.5*lam*x formed in double and
// stored to RT.
//   EIGHTH: lam = CFL/(R + 1) = 1/8 (DT/DX always, base_shll.c:18,84; DT/DY on square cells).  A
//     float x's second-order product is exact in double, and rounding the difference to double first
//     is harmless, so one fused multiply-add gives the same bits.
//   FUSED: so does it in one type while the product is exact, which a product with bits below the
//     denormal range is not.  The caller has seen that no cell is thin (ThinSpan).  Then a flux has no
//     bits below 2^-510 (float: 2^-126): it is a sum of two products, of which one at least has
//     factors of the order of density, energy or pressure and of the sound speed or M +- 1; and x
//     is a sum of such fluxes, or of their limited slopes.  (In 2D the transverse momentum's flux
//     has none of them, and the wavefronts of a tile meet each other's rows: two operations.)
template <bool FUSED, class RT>
__device__ __forceinline__ RT ref_first(RT u, RT lam, RT x) {
    if constexpr (FUSED) return __builtin_elementwise_fma((RT)-0.125, x, u);
    else return u - lam * x;
}
template <bool EIGHTH, bool FUSED = false, class RT>
__device__ __forceinline__ RT ref_second(RT u, RT lam, RT x) {
    if constexpr (FUSED || (EIGHTH && sizeof(RT) == 4)) return __builtin_elementwise_fma((RT)-0.0625, x, u);
    else return (RT)((double)u - 0.5 * (double)lam * (double)x);
}

// x and y split fluxes of one cell (Compute_P_from_U + Compute_F_from_P, base_shll_2d.c:239-319)
// and its sound speed a.  U: conserved (F64/REF32: the state; C32: hi).
template <int PREC, class RT>
__device__ __forceinline__ void fluxes2(const RT (&U)[4], const Inst& in, RT (&xp)[4], RT (&xm)[4], RT (&yp)[4],
                                        RT (&ym)[4], RT& a) {
    if constexpr (PREC == PREC_C32 || PREC == PREC_C32K) {
        // the compensated scheme's float form: fused multiply-adds (split_c32)
        RT vx, vy, T, z1, z2, z3;
        C32Arith::prim2(U[0], U[1], U[2], U[3], in.k.c_rcv, in.k.c_gR, vx, vy, T, a);
        const RT P = U[0] * T;
        C32Arith::zinv(div_fast(vx, a), a, z1, z2, z3);
        split_c32(U[1], U[0], z1, z2, z3, xp[0], xm[0]);
        split_c32(__builtin_fmaf(U[1], vx, P), U[1], z1, z2, z3, xp[1], xm[1]);
        split_c32(U[1] * vy, U[2], z1, z2, z3, xp[2], xm[2]);
        split_c32(vx * (U[3] + P), U[3], z1, z2, z3, xp[3], xm[3]);
        C32Arith::zinv(div_fast(vy, a), a, z1, z2, z3);
        split_c32(U[2], U[0], z1, z2, z3, yp[0], ym[0]);
        split_c32(U[2] * vx, U[1], z1, z2, z3, yp[1], ym[1]);
        split_c32(__builtin_fmaf(U[2], vy, P), U[2], z1, z2, z3, yp[2], ym[2]);
        split_c32(vy * (U[3] + P), U[3], z1, z2, z3, yp[3], ym[3]);
    } else {
        Prim2<RT> q;
        bool tiny = false;
        RefSpan<RT> span;
        ref_prim2<RT>(U, in, q, span, tiny);
        const bool ok = span.ok();
        if (__builtin_expect(!ok || tiny, 0)) ref_prim2_redo<RT>(U, in, ok, q);
        ref_flux2<RT>(U, q, xp, xm, yp, ym);
        a = q.a;
    }
}

template <int PREC, class RT>
__device__ __forceinline__ void fluxes2(const RT (&U)[4], const Inst& in, RT (&xp)[4], RT (&xm)[4], RT (&yp)[4],
                                        RT (&ym)[4]) {
    RT a;
    fluxes2<PREC, RT>(U, in, xp, xm, yp, ym, a);
}

}  // namespace shll
