// shll_k2d.hip -- fused 2D SHLL step kernels along the rows for gfx950: second order, and first
// order in FP64 on large domains (the other first-order launches: shll_k2t.hip).
//
// Layout: SoA planes, cell (i, j) at i*ny + j, y contiguous (base_shll_2d.c:146-221).
// One wavefront takes a strip of 64 consecutive columns j (lane = j - j0) and streams
// down the rows i.  For each row it loads the state once (64 consecutive cells per
// variable: one coalesced access), recovers the primitives, forms the x and y split
// fluxes, and keeps the few rows its x stencil needs in registers; the y neighbours come
// from the adjacent lanes (DPP wave shifts).  The outer lanes of a strip are recomputed
// halo.  No LDS, no barriers.
//
// The update keeps the reference's unsplit order: x term, (second-order x term),
// y term, (second-order y term), all from the same state (base_shll_2d.c:225-236,
// 2nd_order_base_shll.c:436-458).  Walls: reflective with per-component signs
// (base_shll_2d.c:150-216) or outflow (2nd_order_base_shll.c:214-323).  Second-order
// slopes: minmod or the MC limiter of base-omp/2nd_order_base_shll.c:317-325,385-392.
#include "shll_flux.h"

#ifndef PF_DEPTH
#define PF_DEPTH 2
#endif

namespace shll {

// reflective wall signs: x walls (-,+,-,-), y walls (-,-,+,-)
__device__ __forceinline__ int sgn_x(int v) { return v == 1 ? 1 : -1; }
__device__ __forceinline__ int sgn_y(int v) { return v == 2 ? 1 : -1; }

// A lane's y walls, as per-lane flags (lane-varying, so the wall choices are selects
// rather than branches): lo / hi = the lane is column 0 / ny-1, *_refl = and reflective;
// edge = on or beyond such a column (no slope)
struct LaneWalls {
    bool lo, hi, lo_refl, hi_refl, refl, edge;
};

// ---------------------------------------------------------------------------
// Second order, one step per launch: a wavefront streams a strip of 64 columns down the rows.
//
// Row t's state is loaded two rows ahead; its fluxes, its y terms and the limited x slopes of
// row t-1 complete when it arrives, and row c = t-2 is advanced.  Between rows a wavefront
// keeps rows c and c+1 (state, x fluxes, y terms), the slopes of row c and, of row c-1, what
// row c's lower face needs; every slope is limited once.  Inner rows run one straight-line
// body (walls only enter where an item starts, and in the two drain rows past the last one).
// Bound: VALU issue, and on small domains the latency of an item's rows (default_rows2d in
// shll_api.cpp).  Before, each row re-limited half of its x slopes and walked through some
// thirty branch blocks and 100 register moves (REF32 MC: about 700 VALU instructions per row,
// now about 500).  Measured, us per step before and now at the best item heights of each: REF32
// MC 1024^2 28 and 19.6, 4096^2 273 and 191; FP64 minmod 777x613 25.3 and 15.1, 2048^2 118 and
// 70 (268 MB read and written: 48% of the copy rate); C32K 1024^2 24.3 and 15.5.
// ---------------------------------------------------------------------------
template <int PREC>
struct Row2 {
    using RT = typename Real<PREC>::T;
    RT u[4], l[4];          // state (C32: hi, lo)
    RT xp[4], xm[4];        // x split fluxes
    RT y1[4], y2[4];        // y terms (y_terms2)
};

// y terms of a row: reference forms y1 = hp - hm + T - B and y2 = the same of the slopes; C32
// the lower and upper face terms, C32K their difference in y1
template <int PREC, int LIM, bool YW, class A, class RT>
__device__ __forceinline__ void y_terms2(const RT (&yp)[4], const RT (&ym)[4], const LaneWalls& w, RT lamy, RT th,
                                         RT (&y1)[4], RT (&y2)[4]) {
    constexpr bool CMP = PREC == PREC_C32 || PREC == PREC_C32K;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const RT sy = (RT)sgn_y(v);
        const RT hp = yp[v], hm = ym[v];
        RT B = from_left_z(hp), T = from_right_z(hm);
        RT dhp = limited_slope<A, LIM>(B, hp, from_right_z(hp), th);
        RT dhm = limited_slope<A, LIM>(from_left_z(hm), hm, T, th);
        if constexpr (YW) {
            dhp = w.edge ? (RT)0 : dhp;
            dhm = w.edge ? (RT)0 : dhm;
        }
        if constexpr (YW) B = w.lo ? (w.lo_refl ? sy * hm : hp) : B;
        if constexpr (!CMP) {
            if constexpr (YW) T = w.hi ? (w.hi_refl ? sy * hp : hm) : T;
            y1[v] = hp - hm + T - B;
            RT Bd = from_left_z(dhp), Td = from_right_z(dhm);
            if constexpr (YW) {
                Bd = w.lo ? (RT)0 : Bd;
                Td = w.hi ? (RT)0 : Td;
            }
            y2[v] = dhp + dhm - Td - Bd;
        } else {
            RT d = from_left_z(dhp) - dhm;
            if constexpr (YW) d = w.lo ? (RT)0 : d;
            const RT tb = __builtin_fmaf((RT)0.5 * lamy, d, lamy * (B + hm));
            RT tt = from_right_z(tb);
            if constexpr (YW) tt = w.hi ? lamy * (hp + (w.hi_refl ? sy * hp : hm)) : tt;
            if constexpr (PREC == PREC_C32K) {
                y1[v] = tb - tt;
                y2[v] = 0;
            } else {
                y1[v] = tb;
                y2[v] = tt;
            }
        }
    }
}

template <int PREC, int LIM, bool YW, bool SQ>
__device__ __forceinline__ void rows2(const StepArgs& a, const Item2& it, const Inst& in, int lane) {
    using RT = typename Real<PREC>::T;
    constexpr bool CMP = PREC == PREC_C32 || PREC == PREC_C32K;
    using A = typename std::conditional<CMP, C32Arith, RefArith<RT>>::type;
    const int nx = in.nx, ny = in.ny;
    const int64_t P = a.plane;
    const int j = it.j0 + lane;
    const int jc = j < 0 ? 0 : (j < ny ? j : ny - 1);  // lanes off the domain hold a copy of its edge
    const bool jown = j >= it.jx0 && j < it.jx0 + it.jw;
    const bool refl = in.bc == BC_REFLECT;
    const LaneWalls w{j == 0, j == ny - 1, j == 0 && refl, j == ny - 1 && refl, refl, j <= 0 || j >= ny - 1};
    const RT lamx = PREC == PREC_F64 ? (RT)in.k.d_lamx : (PREC == PREC_REF32 ? (RT)in.k.f_lamx : (RT)in.k.c_lamx);
    const RT lamy = PREC == PREC_F64 ? (RT)in.k.d_lamy : (PREC == PREC_REF32 ? (RT)in.k.f_lamy : (RT)in.k.c_lamy);
    const RT th = PREC == PREC_F64 ? (RT)in.k.d_theta : (PREC == PREC_REF32 ? (RT)in.k.f_theta : (RT)in.k.c_theta);
    const RT hlx = (RT)0.5 * lamx;
    const RT* __restrict__ p0 = (const RT*)a.in0 + in.off + jc;
    const RT* __restrict__ p1 = CMP ? (const RT*)a.in1 + in.off + jc : nullptr;
    RT* __restrict__ q0 = (RT*)a.out0 + in.off + jc;
    RT* __restrict__ q1 = CMP ? (RT*)a.out1 + in.off + jc : nullptr;

    auto load = [&](int t, Row2<PREC>& r) {
        const int64_t o = (int64_t)(t < nx ? t : nx - 1) * ny;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            r.u[v] = p0[v * P + o];
            if constexpr (CMP) r.l[v] = p1[v * P + o];
        }
    };
    const int end = it.ix0 + it.iw;
    // fluxes of row t, and the y terms of an owned row
    auto take = [&](int t, Row2<PREC>& r) {
        RT yp[4], ym[4];
        fluxes2<PREC, RT>(r.u, in, r.xp, r.xm, yp, ym);
        RT y1[4] = {0, 0, 0, 0}, y2[4] = {0, 0, 0, 0};
        if (t >= it.ix0 && t < end) y_terms2<PREC, LIM, YW, A, RT>(yp, ym, w, lamy, th, y1, y2);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            r.y1[v] = y1[v];
            r.y2[v] = y2[v];
        }
    };

    // of row c-1 the upper-face parts (reference forms: F+ and its slope; C32: the face term);
    // the slopes of row c
    RT L[4], sPl[4], sP[4], sM[4];
    // iteration t advances row c = t - 2 from rows c, c+1 and t (ra, rb, rn), whose arrival
    // completes the slopes of row t-1; INNER false: t = nx, nx + 1, the last rows at the wall
    auto advance = [&](int t, const Row2<PREC>& ra, const Row2<PREC>& rb, const Row2<PREC>& rn, auto inner) {
        constexpr bool INNER = decltype(inner)::value;
        const int c = t - 2;
        RT nP[4], nM[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            nP[v] = INNER ? limited_slope<A, LIM>(ra.xp[v], rb.xp[v], rn.xp[v], th) : (RT)0;
            nM[v] = INNER ? limited_slope<A, LIM>(ra.xm[v], rb.xm[v], rn.xm[v], th) : (RT)0;
        }
        const int64_t o = (int64_t)c * ny;
        RT tr[4];
        if constexpr (CMP) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                RT R = rb.xm[v];
                if constexpr (!INNER) R = c == nx - 1 ? (refl ? (RT)sgn_x(v) * ra.xp[v] : ra.xm[v]) : R;
                tr[v] = __builtin_fmaf(hlx, sP[v] - nM[v], lamx * (ra.xp[v] + R));
            }
        }
        if (c >= it.ix0) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if constexpr (!CMP) {
                    RT R = rb.xm[v];
                    if constexpr (!INNER) R = c == nx - 1 ? (refl ? (RT)sgn_x(v) * ra.xp[v] : ra.xm[v]) : R;
                    RT uu = ra.u[v] - lamx * (ra.xp[v] - ra.xm[v] + R - L[v]);
                    uu = ref_second<true>(uu, lamx, sP[v] + sM[v] - nM[v] - sPl[v]);
                    uu = uu - lamy * ra.y1[v];
                    uu = ref_second<SQ>(uu, lamy, ra.y2[v]);
                    if (jown) q0[v * P + o] = uu;
                } else {
                    RT hi = ra.u[v], lo = ra.l[v], e;
                    if constexpr (PREC == PREC_C32K) {
                        const RT y = ((L[v] - tr[v]) + ra.y1[v]) + lo;
                        const RT s = hi + y;
                        e = y - (s - hi);
                        hi = s;
                    } else {
                        two_sum(hi, L[v], hi, e);
                        lo = lo + e;
                        two_sum(hi, -tr[v], hi, e);
                        lo = lo + e;
                        two_sum(hi, ra.y1[v], hi, e);
                        lo = lo + e;
                        two_sum(hi, -ra.y2[v], hi, e);
                        lo = lo + e;
                        fast_two_sum(hi, lo, hi, e);
                    }
                    if (jown) {
                        q0[v * P + o] = hi;
                        q1[v * P + o] = e;
                    }
                }
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if constexpr (CMP) {
                L[v] = tr[v];
            } else {
                L[v] = ra.xp[v];
                sPl[v] = sP[v];
            }
            sP[v] = nP[v];
            sM[v] = nM[v];
        }
    };
    auto drain = [&](int t, const Row2<PREC>& ra, const Row2<PREC>& rb) {
        if (t < end + 2) advance(t, ra, rb, rb, std::false_type{});
        if (t + 1 < end + 2) advance(t + 1, rb, rb, rb, std::false_type{});
    };
    // four rows in rotation (so none is ever moved): c, c+1, t, and t+1 on its way from memory
    Row2<PREC> r0, r1, r2, r3;
    const int first = it.ix0 - 2 < 0 ? 0 : it.ix0 - 2;
    load(first, r0);
    load(first + 1, r1);
    load(first + 2, r2);
    take(first, r0);
    take(first + 1, r1);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        // the first row's lower face: the wall (at a cut: spoils rows that are not stored)
        const RT f = refl ? (RT)sgn_x(v) * r0.xm[v] : r0.xp[v];
        L[v] = CMP ? lamx * (f + r0.xm[v]) : f;
        sPl[v] = sP[v] = sM[v] = (RT)0;
    }
    int t = first + 2;
    const int tin = end + 2 < nx ? end + 2 : nx;  // iterations below this take a row
    // unrolled by four only where that keeps the wavefronts per SIMD: REF32 needs 152 registers
    // unrolled (3 per SIMD) and 128 rolled, and ran 4% slower unrolled at 4096^2; FP64 ran 7%
    // faster.  (Leaving the unrolled loop from its middle cost 100 registers.)
    for (; PREC != PREC_REF32 && t + 4 <= tin; t += 4) {
        load(t + 1, r3);
        take(t, r2);
        advance(t, r0, r1, r2, std::true_type{});
        load(t + 2, r0);
        take(t + 1, r3);
        advance(t + 1, r1, r2, r3, std::true_type{});
        load(t + 3, r1);
        take(t + 2, r0);
        advance(t + 2, r2, r3, r0, std::true_type{});
        load(t + 4, r2);
        take(t + 3, r1);
        advance(t + 3, r3, r0, r1, std::true_type{});
    }
    for (; t < tin; ++t) {
        load(t + 1, r3);
        take(t, r2);
        advance(t, r0, r1, r2, std::true_type{});
        r0 = r1;
        r1 = r2;
        r2 = r3;
    }
    drain(t, r0, r1);
}

template <int PREC, int WPB, int LIM>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(PREC == PREC_F64 ? 2 : 1)))
void k_row2d(StepArgs a) {
    const LaunchView lv = launch_view(a);
    const int blk = xcd_work((int)blockIdx.x, (lv.n_items + WPB - 1) / WPB);
    const int wave = blk * WPB + uniform((int)threadIdx.x >> 6);
    if (blk < 0 || wave >= lv.n_items) return;
    const int lane = (int)threadIdx.x & 63;
    const Item2 it = ((const Item2*)a.items)[wave];
    const Inst in = a.inst[it.inst];
    if (in.nsteps - lv.step_base <= 0) return;
    // strips away from both y walls take the copy without wall choices, REF32 on square cells the
    // one with DT/DY = 1/8 (ref_second)
    const bool yw = it.j0 <= 0 || it.j0 + 64 >= in.ny;
    if constexpr (PREC == PREC_REF32) {
        const bool sq = in.k.f_lamy == 0.125f;
        if (yw) {
            if (sq) rows2<PREC, LIM, true, true>(a, it, in, lane);
            else rows2<PREC, LIM, true, false>(a, it, in, lane);
        } else {
            if (sq) rows2<PREC, LIM, false, true>(a, it, in, lane);
            else rows2<PREC, LIM, false, false>(a, it, in, lane);
        }
    } else {
        if (yw) rows2<PREC, LIM, true, false>(a, it, in, lane);
        else rows2<PREC, LIM, false, false>(a, it, in, lane);
    }
}

// ---------------------------------------------------------------------------
// First order in FP64 on domains whose state exceeds the last-level cache, K = 1 or 2 steps per
// launch: a pipeline of K stages along the rows.  Every other first-order launch takes the
// register tiles of shll_k2t.hip; there these large FP64 domains leave too few wavefronts per
// SIMD to keep HBM busy (4096^2, us per step: pipeline 237 and 172 at 1 and 2 steps per launch,
// tiles 257 and 192; 2048^2, in the cache: 58 and 51).
//
// Stage s takes the rows of its input level one at a time (stage 0 from HBM, stage s
// from stage s-1) and holds the last row it took.  When row t arrives, the x face
// between rows t-1 and t is known, so the held row t-1 is advanced one step and
// passed on; row t is held in its place.  After the last row a stage drains its held
// row with the wall face.  Each stage keeps only one row (state, x split fluxes and
// the row's face and y terms), so K steps cost K times the arithmetic of one step but
// one read and one write of the state.  The row next to a cut (an item edge that is
// not a wall) gets a made-up face and a strip's edge lanes get their own values from
// the DPP shifts, so each stage spoils one more row and column next to every cut: the
// items' halos are K rows and K columns wide and only owned cells are stored.  Stages
// at or past the instance's remaining step count pass rows through.
// ---------------------------------------------------------------------------
struct Held2 {
    double u[4];   // state
    double fp[4];  // x split flux F+ (the next row's lower face)
    double d[4];   // F+ - F- of the row
    double tl[4];  // L: F+ of the row below
    double yb[4];  // (hp - hm) + T - B
};

enum { ST_TAKE_FIRST = 0, ST_TAKE = 1, ST_DRAIN = 2 };

// One stage, one row.  io: the incoming row (ST_TAKE_FIRST / ST_TAKE); on return the
// outgoing row (ST_TAKE / ST_DRAIN).  act: the stage advances (else it only delays).
template <bool YW>
__device__ __forceinline__ void stage2(Held2& h, double (&io)[4], int mode, bool act, const Inst& in,
                                       const LaneWalls& w, double lamx, double lamy) {
    const bool refl = w.refl;
    if (!act) {
        // pass-through with the stage's one-row delay
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double u = h.u[v];
            if (mode != ST_DRAIN) h.u[v] = io[v];
            io[v] = u;
        }
        return;
    }
    double xp[4], xm[4], yp[4], ym[4], nu[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) nu[v] = io[v];  // the incoming row (io is overwritten by the outgoing one)
    // the x fluxes of the row that meets the held row's upper face: the incoming row, or
    // at a drain the held row itself (its F- for the outflow wall)
    fluxes2<PREC_F64, double>(mode == ST_DRAIN ? h.u : nu, in, xp, xm, yp, ym);
    if (mode != ST_TAKE_FIRST) {
        // advance the held row
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double Rv = mode == ST_DRAIN && refl ? sgn_x(v) * h.fp[v] : xm[v];
            const double uu = h.u[v] - lamx * (h.d[v] + Rv - h.tl[v]);
            io[v] = uu - lamy * h.yb[v];
        }
    }
    if (mode == ST_DRAIN) return;
    // hold the incoming row: its lower x face (the wall rule on a stage's first row), y terms
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const double sx = sgn_x(v), sy = sgn_y(v);
        const double fpc = xp[v], fmc = xm[v], hpc = yp[v], hmc = ym[v];
        const double hpl = from_left_z(hpc), hmr = from_right_z(hmc);
        h.tl[v] = mode == ST_TAKE_FIRST ? (refl ? sx * fmc : fpc) : h.fp[v];
        const double Bv = YW ? (w.lo_refl ? sy * hmc : (w.lo ? hpc : hpl)) : hpl;
        const double Tv = YW ? (w.hi_refl ? sy * hpc : (w.hi ? hmc : hmr)) : hmr;
        h.yb[v] = hpc - hmc + Tv - Bv;
        h.d[v] = fpc - fmc;
        h.u[v] = nu[v];
        h.fp[v] = fpc;
    }
}

template <int K, bool YW>
__device__ __forceinline__ void pipeline2(const StepArgs& a, const Item2& it, const Inst& in, int lane, int ns) {
    const int nx = in.nx, ny = in.ny;
    const int64_t P = a.plane;
    const int j = it.j0 + lane;
    const bool jok = j >= 0 && j < ny;
    const bool jown = j >= it.jx0 && j < it.jx0 + it.jw;
    const int jc = jok ? j : (j < 0 ? 0 : ny - 1);
    const double* __restrict__ ip = (const double*)a.in0 + in.off;
    double* __restrict__ op = (double*)a.out0 + in.off;
    const double lamx = in.k.d_lamx, lamy = in.k.d_lamy;
    const bool refl = in.bc == BC_REFLECT;
    const LaneWalls w{j == 0, j == ny - 1, j == 0 && refl, j == ny - 1 && refl, refl, j <= 0 || j >= ny - 1};

    // rows taken by every stage: [r0, r1), then a drain
    const int r0 = it.ix0 - K < 0 ? 0 : it.ix0 - K;
    const int r1 = it.ix0 + it.iw + K > nx ? nx : it.ix0 + it.iw + K;
    Held2 h[K];
#pragma unroll
    for (int s = 0; s < K; ++s)
#pragma unroll
        for (int v = 0; v < 4; ++v) h[s].u[v] = h[s].fp[v] = h[s].d[v] = h[s].tl[v] = h[s].yb[v] = 0.0;

    constexpr int D = PF_DEPTH;
    double nu[D][4];
    // jc is clamped into the domain: every lane loads, lanes off the domain keep a benign state
    auto load_row = [&](int t, double (&U)[4]) {
        if (t < r1) {
            const int64_t o = (int64_t)t * ny + jc;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double x = ip[v * P + o];
                U[v] = jok ? x : (v == 0 ? 1.0 : (v == 3 ? 2.5 : 0.0));
            }
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load_row(r0 + d, nu[d]);
    // Stage s is at row t - s in iteration t: it takes rows [r0, r1) (from stage s-1,
    // which gives up its held row when it takes the next one or drains) and drains at r1.
    // Stage K-1 gives row t - K.
    const int tend = r1 + K;
    auto iter = [&](int t, bool steady) {
        double U[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) U[v] = nu[0][v];
#pragma unroll
        for (int d = 0; d + 1 < D; ++d)
#pragma unroll
            for (int v = 0; v < 4; ++v) nu[d][v] = nu[d + 1][v];
        load_row(t + D, nu[D - 1]);
        // live: U holds a row at the current stage's input level
        bool live = true;
        if (steady) {
            // every stage takes an inner row and advances: one straight-line body
#pragma unroll
            for (int s = 0; s < K; ++s) stage2<YW>(h[s], U, ST_TAKE, true, in, w, lamx, lamy);
        } else {
#pragma unroll
            for (int s = 0; s < K; ++s) {
                const int ts = t - s;
                if (ts < r0 || ts > r1) {
                    live = false;
                } else if (ts == r1) {
                    stage2<YW>(h[s], U, ST_DRAIN, s < ns, in, w, lamx, lamy);
                    live = true;
                } else if (live) {
                    const int mode = ts == r0 ? ST_TAKE_FIRST : ST_TAKE;
                    stage2<YW>(h[s], U, mode, s < ns, in, w, lamx, lamy);
                    live = mode == ST_TAKE;
                }
            }
        }
        const int c = t - K;
        if (live && jown && c >= it.ix0 && c < it.ix0 + it.iw) {
            const int64_t o = (int64_t)c * ny + jc;
#pragma unroll
            for (int v = 0; v < 4; ++v) op[v * P + o] = U[v];
        }
    };
    // iterations t in [r0 + K, r1) are steady when every stage advances (ns == K): they run
    // in a loop of their own, K at a time, apart from the ramp-up and drain iterations
    int t = r0;
    if (ns == K && r1 - (r0 + K) >= K) {
        for (; t < r0 + K; ++t) iter(t, false);
        for (; t + K <= r1; t += K)
#pragma unroll
            for (int q = 0; q < K; ++q) iter(t + q, true);
    }
    for (; t < tend; ++t) iter(t, ns == K && t - (K - 1) > r0 && t < r1);
}

template <int K, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_step2d_tb(StepArgs a) {
    const LaunchView lv = launch_view(a);
    const int blk = xcd_work((int)blockIdx.x, (lv.n_items + WPB - 1) / WPB);
    const int wave = blk * WPB + uniform((int)threadIdx.x >> 6);
    if (blk < 0 || wave >= lv.n_items) return;
    const int lane = (int)threadIdx.x & 63;
    const Item2 it = ((const Item2*)a.items)[wave];
    const Inst in = a.inst[it.inst];
    const int64_t left = in.nsteps - lv.step_base;
    if (left <= 0) return;
    const int kk = a.ksteps < K ? a.ksteps : K;
    const int ns = left < (int64_t)kk ? (int)left : kk;  // stages that advance
    // strips away from both y walls take the copy without wall choices
    const bool yw = it.j0 <= 0 || it.j0 + 64 >= in.ny;
    if (yw) pipeline2<K, true>(a, it, in, lane, ns);
    else pipeline2<K, false>(a, it, in, lane, ns);
}

// ---------------------------------------------------------------------------
// Second order (FP32-compensated forms), K steps per launch: the same row pipeline with a
// delay of two rows per stage.  The face between rows c and c+1 needs the limited slopes
// of rows c and c+1, and the slope of row c+1 needs row c+2, so a stage advances row t-2
// when row t arrives.  It keeps two pending rows (state, x split fluxes, y terms), the F+
// slope of the first one and that row's lower face term.  Slopes of the domain's first
// and last rows are zero (2nd_order_base_shll.c:227-276); at a cut the first row's slope
// and the last row's F- slope are taken as zero, which spoils two rows per stage, like
// the radius-2 y stencil spoils two lanes at a strip edge: items carry 2K halo rows and
// columns.  Bitwise equal to K launches of k_row2d.
// ---------------------------------------------------------------------------
template <int PREC>
struct Held2o2 {
    using RT = typename Real<PREC>::T;
    RT u0[4], l0[4], u1[4], l1[4];  // pending rows: the older (0) and the newer (1)
    RT xp0[4], xm0[4], xp1[4], xm1[4];
    RT dfp0[4];                     // limited F+ slope of row 0
    RT tl0[4];                      // lower face term of row 0
    RT yb0[4], yt0[4], yb1[4], yt1[4];  // y face terms (C32K: yb = tb - tt)
};

enum { S2_FIRST = 0, S2_SECOND = 1, S2_TAKE = 2, S2_DRAIN1 = 3, S2_DRAIN2 = 4 };

template <int PREC, bool YW, int LIM>
__device__ __forceinline__ void stage2o2(Held2o2<PREC>& h, float (&iou)[4], float (&iol)[4], int mode, bool act,
                                         int ts, const Inst& in, const LaneWalls& w, bool yedge, float lamx,
                                         float lamy, float th) {
    using A = C32Arith;
    const int nx = in.nx;
    const bool refl = w.refl;
    const float hl = 0.5f * lamx, hly = 0.5f * lamy;
    float nu[4], nl[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        nu[v] = iou[v];
        nl[v] = iol[v];
    }
    if (!act) {
        // pass-through with the stage's two-row delay
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float u = h.u0[v], l = h.l0[v];
            if (mode == S2_FIRST) {
                h.u0[v] = nu[v]; h.l0[v] = nl[v];
            } else if (mode == S2_SECOND) {
                h.u1[v] = nu[v]; h.l1[v] = nl[v];
            } else if (mode == S2_TAKE) {
                h.u0[v] = h.u1[v]; h.l0[v] = h.l1[v]; h.u1[v] = nu[v]; h.l1[v] = nl[v];
            } else if (mode == S2_DRAIN1) {
                h.u0[v] = h.u1[v]; h.l0[v] = h.l1[v];
            }
            iou[v] = u;
            iol[v] = l;
        }
        return;
    }
    float xp[4], xm[4], yp[4], ym[4], yb[4], yt[4];
    const bool take = mode == S2_FIRST || mode == S2_SECOND || mode == S2_TAKE;
    if (take) {
        fluxes2<PREC, float>(nu, in, xp, xm, yp, ym);
        // y face terms of the incoming row: lower face tb, upper face tt (lane above)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float sy = (float)sgn_y(v);
            const float hpc = yp[v], hmc = ym[v];
            const float hpl = from_left_z(hpc), hpr = from_right_z(hpc);
            const float hml = from_left_z(hmc), hmr = from_right_z(hmc);
            float dhp = limited_slope<A, LIM>(hpl, hpc, hpr, th);
            float dhm = limited_slope<A, LIM>(hml, hmc, hmr, th);
            if constexpr (YW) {
                dhp = yedge ? 0.0f : dhp;
                dhm = yedge ? 0.0f : dhm;
            }
            const float dhpl = from_left_z(dhp);
            float Gb = hpl + hmc, db = dhpl - dhm;
            if constexpr (YW) {
                Gb = w.lo ? (w.lo_refl ? hmc + sy * hmc : hpc + hmc) : Gb;
                db = w.lo ? 0.0f : db;
            }
            const float tb = __builtin_fmaf(hly, db, lamy * Gb);
            float tt = from_right_z(tb);
            if constexpr (YW)
                tt = w.hi ? __builtin_fmaf(hly, 0.0f, lamy * (w.hi_refl ? hpc + sy * hpc : hpc + hmc)) : tt;
            if constexpr (PREC == PREC_C32K) {
                yb[v] = tb - tt;
                yt[v] = 0.0f;
            } else {
                yb[v] = tb;
                yt[v] = tt;
            }
        }
    }
    if (mode == S2_FIRST) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float sx = (float)sgn_x(v);
            h.u0[v] = nu[v]; h.l0[v] = nl[v];
            h.xp0[v] = xp[v]; h.xm0[v] = xm[v];
            h.yb0[v] = yb[v]; h.yt0[v] = yt[v];
            // the wall face below the first row (made up at a cut)
            h.tl0[v] = __builtin_fmaf(hl, 0.0f, lamx * (refl ? xm[v] + sx * xm[v] : xp[v] + xm[v]));
        }
        return;
    }
    if (mode == S2_SECOND) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            h.u1[v] = nu[v]; h.l1[v] = nl[v];
            h.xp1[v] = xp[v]; h.xm1[v] = xm[v];
            h.yb1[v] = yb[v]; h.yt1[v] = yt[v];
            h.dfp0[v] = 0.0f;  // the first row: a wall row, or a cut
        }
        return;
    }
    // advance row 0 with its upper face
    const int r = ts - 1;  // the row whose slopes complete now (TAKE)
    const bool bnd = r <= 0 || r >= nx - 1;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float sx = (float)sgn_x(v);
        float face, dfp1 = 0.0f;
        if (mode == S2_TAKE) {
            const float dfm1 = bnd ? 0.0f : limited_slope<A, LIM>(h.xm0[v], h.xm1[v], xm[v], th);
            dfp1 = bnd ? 0.0f : limited_slope<A, LIM>(h.xp0[v], h.xp1[v], xp[v], th);
            face = __builtin_fmaf(hl, h.dfp0[v] - dfm1, lamx * (h.xp0[v] + h.xm1[v]));
        } else if (mode == S2_DRAIN1) {
            face = __builtin_fmaf(hl, h.dfp0[v] - 0.0f, lamx * (h.xp0[v] + h.xm1[v]));
        } else {
            const float fpc = h.xp0[v], fmc = h.xm0[v];
            face = __builtin_fmaf(hl, 0.0f, lamx * (refl ? fpc + sx * fpc : fpc + fmc));
        }
        const float tl = h.tl0[v];
        float aa = h.u0[v], bb = h.l0[v], e;
        if constexpr (PREC == PREC_C32K) {
            const float y = ((tl - face) + h.yb0[v]) + bb;
            const float s2 = aa + y;
            e = y - (s2 - aa);
            aa = s2;
        } else {
            two_sum(aa, tl, aa, e);
            bb = bb + e;
            two_sum(aa, -face, aa, e);
            bb = bb + e;
            two_sum(aa, h.yb0[v], aa, e);
            bb = bb + e;
            two_sum(aa, -h.yt0[v], aa, e);
            bb = bb + e;
            fast_two_sum(aa, bb, aa, e);
        }
        iou[v] = aa;
        iol[v] = e;
        if (mode != S2_DRAIN2) {
            // row 1 becomes row 0
            h.u0[v] = h.u1[v]; h.l0[v] = h.l1[v];
            h.xp0[v] = h.xp1[v]; h.xm0[v] = h.xm1[v];
            h.yb0[v] = h.yb1[v]; h.yt0[v] = h.yt1[v];
            h.tl0[v] = face;
            h.dfp0[v] = dfp1;
        }
        if (mode == S2_TAKE) {
            h.u1[v] = nu[v]; h.l1[v] = nl[v];
            h.xp1[v] = xp[v]; h.xm1[v] = xm[v];
            h.yb1[v] = yb[v]; h.yt1[v] = yt[v];
        }
    }
}

template <int PREC, int K, bool YW, int LIM>
__device__ __forceinline__ void pipeline2o2(const StepArgs& a, const Item2& it, const Inst& in, int lane, int ns) {
    const int nx = in.nx, ny = in.ny;
    const int64_t P = a.plane;
    const int j = it.j0 + lane;
    const bool jok = j >= 0 && j < ny;
    const bool jown = j >= it.jx0 && j < it.jx0 + it.jw;
    const int jc = jok ? j : (j < 0 ? 0 : ny - 1);
    const float* __restrict__ i0p = (const float*)a.in0 + in.off;
    const float* __restrict__ i1p = (const float*)a.in1 + in.off;
    float* __restrict__ o0p = (float*)a.out0 + in.off;
    float* __restrict__ o1p = (float*)a.out1 + in.off;
    const float lamx = in.k.c_lamx, lamy = in.k.c_lamy, th = in.k.c_theta;
    const bool refl = in.bc == BC_REFLECT;
    const LaneWalls w{j == 0, j == ny - 1, j == 0 && refl, j == ny - 1 && refl, refl, j <= 0 || j >= ny - 1};
    const bool yedge = j <= 0 || j >= ny - 1;  // zero y slopes (2nd_order_base_shll.c:293-344)

    constexpr int H = 2 * K;
    const int r0 = it.ix0 - H < 0 ? 0 : it.ix0 - H;
    const int r1 = it.ix0 + it.iw + H > nx ? nx : it.ix0 + it.iw + H;
    Held2o2<PREC> h[K];
#pragma unroll
    for (int s = 0; s < K; ++s)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            h[s].u0[v] = h[s].l0[v] = h[s].u1[v] = h[s].l1[v] = 0.0f;
            h[s].xp0[v] = h[s].xm0[v] = h[s].xp1[v] = h[s].xm1[v] = h[s].dfp0[v] = h[s].tl0[v] = 0.0f;
            h[s].yb0[v] = h[s].yt0[v] = h[s].yb1[v] = h[s].yt1[v] = 0.0f;
        }
    constexpr int D = PF_DEPTH;
    float nu[D][4], nl[D][4];  // rows t+1 .. t+D, loaded ahead
    auto load_row = [&](int t, float (&U)[4], float (&Ul)[4]) {
        if (t < r1) {
            const int64_t o = (int64_t)t * ny + jc;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float x = i0p[v * P + o], y = i1p[v * P + o];
                U[v] = jok ? x : (v == 0 ? 1.0f : (v == 3 ? 2.5f : 0.0f));
                Ul[v] = jok ? y : 0.0f;
            }
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load_row(r0 + d, nu[d], nl[d]);
    // Stage s is at row t - 2s in iteration t: it takes rows [r0, r1) and drains at r1 and
    // r1 + 1, giving row t - 2s - 2 from its third row on.  Stage K-1 gives row t - 2K.
    const int tend = r1 + 2 * K;
    auto iter = [&](int t, bool steady) {
        float U[4], Ul[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            U[v] = nu[0][v];
            Ul[v] = nl[0][v];
        }
#pragma unroll
        for (int d = 0; d + 1 < D; ++d)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                nu[d][v] = nu[d + 1][v];
                nl[d][v] = nl[d + 1][v];
            }
        load_row(t + D, nu[D - 1], nl[D - 1]);
        bool live = true;  // U holds a row at the current stage's input level
        if (steady) {
#pragma unroll
            for (int s = 0; s < K; ++s)
                stage2o2<PREC, YW, LIM>(h[s], U, Ul, S2_TAKE, true, t - 2 * s, in, w, yedge, lamx, lamy, th);
        } else {
#pragma unroll
            for (int s = 0; s < K; ++s) {
                const int ts = t - 2 * s;
                if (ts < r0 || ts > r1 + 1) {
                    live = false;
                } else if (ts >= r1) {
                    stage2o2<PREC, YW, LIM>(h[s], U, Ul, ts == r1 ? S2_DRAIN1 : S2_DRAIN2, s < ns, ts, in, w, yedge,
                                            lamx, lamy, th);
                    live = true;
                } else if (live) {
                    const int mode = ts == r0 ? S2_FIRST : (ts == r0 + 1 ? S2_SECOND : S2_TAKE);
                    stage2o2<PREC, YW, LIM>(h[s], U, Ul, mode, s < ns, ts, in, w, yedge, lamx, lamy, th);
                    live = mode == S2_TAKE;
                }
            }
        }
        const int c = t - 2 * K;
        if (live && jown && c >= it.ix0 && c < it.ix0 + it.iw) {
            const int64_t o = (int64_t)c * ny + jc;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                o0p[v * P + o] = U[v];
                o1p[v * P + o] = Ul[v];
            }
        }
    };
    // iterations t in [r0 + 2K, r1) are steady when every stage advances (ns == K): they run
    // in a loop of their own, apart from the ramp-up and drain iterations
    int t = r0;
    if (ns == K && r1 - (r0 + 2 * K) >= 2 * K) {
        for (; t < r0 + 2 * K; ++t) iter(t, false);
        for (; t + 2 * K <= r1; t += 2 * K)
#pragma unroll
            for (int q = 0; q < 2 * K; ++q) iter(t + q, true);
    }
    for (; t < tend; ++t) iter(t, ns == K && t - 2 * (K - 1) >= r0 + 2 && t < r1);
}

template <int PREC, int K, int WPB, int LIM>
__global__ __launch_bounds__(64 * WPB) void k_step2d_tb2(StepArgs a) {
    const LaunchView lv = launch_view(a);
    const int blk = xcd_work((int)blockIdx.x, (lv.n_items + WPB - 1) / WPB);
    const int wave = blk * WPB + uniform((int)threadIdx.x >> 6);
    if (blk < 0 || wave >= lv.n_items) return;
    const int lane = (int)threadIdx.x & 63;
    const Item2 it = ((const Item2*)a.items)[wave];
    const Inst in = a.inst[it.inst];
    const int64_t left = in.nsteps - lv.step_base;
    if (left <= 0) return;
    const int kk = a.ksteps < K ? a.ksteps : K;
    const int ns = left < (int64_t)kk ? (int)left : kk;
    const bool yw = it.j0 <= 0 || it.j0 + 64 >= in.ny;
    if (yw) pipeline2o2<PREC, K, true, LIM>(a, it, in, lane, ns);
    else pipeline2o2<PREC, K, false, LIM>(a, it, in, lane, ns);
}

template <int PREC, int WPB, int LIM>
static hipError_t launch2_tb2_w(int k, int nblocks, hipStream_t s, const StepArgs& a) {
    const dim3 grid(nblocks), block(64 * WPB);
    switch (k) {
    case 2: hipLaunchKernelGGL((k_step2d_tb2<PREC, 2, WPB, LIM>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int PREC>
static hipError_t launch2_tb2(int k, int lim, int wpb, int nblocks, hipStream_t s, const StepArgs& a) {
    if (lim == LIM_MC)
        return wpb == 1 ? launch2_tb2_w<PREC, 1, LIM_MC>(k, nblocks, s, a) : launch2_tb2_w<PREC, 4, LIM_MC>(k, nblocks, s, a);
    return wpb == 1 ? launch2_tb2_w<PREC, 1, LIM_MINMOD>(k, nblocks, s, a)
                    : launch2_tb2_w<PREC, 4, LIM_MINMOD>(k, nblocks, s, a);
}

template <int WPB>
static hipError_t launch2_tb(int k, int nblocks, hipStream_t s, const StepArgs& a) {
    const dim3 grid(nblocks), block(64 * WPB);
    if (k == 1) hipLaunchKernelGGL((k_step2d_tb<1, WPB>), grid, block, 0, s, a);
    else if (k == 2) hipLaunchKernelGGL((k_step2d_tb<2, WPB>), grid, block, 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template <int PREC, int WPB>
static hipError_t launch2_row_w(int lim, int nblocks, hipStream_t s, const StepArgs& a) {
    const dim3 grid(nblocks), block(64 * WPB);
    if (lim == LIM_MINMOD) hipLaunchKernelGGL((k_row2d<PREC, WPB, LIM_MINMOD>), grid, block, 0, s, a);
    else if (lim == LIM_MC) hipLaunchKernelGGL((k_row2d<PREC, WPB, LIM_MC>), grid, block, 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template <int PREC>
static hipError_t launch2_row(int lim, int wpb, int nblocks, hipStream_t s, const StepArgs& a) {
    return wpb == 1 ? launch2_row_w<PREC, 1>(lim, nblocks, s, a) : launch2_row_w<PREC, 4>(lim, nblocks, s, a);
}

bool step2d_supported(int prec, int order, int k) {
    if (k == 1) return true;
    if (order == 1) return k == 2 || k == 3 || k == 4 || k == 8;
    return (prec == PREC_C32 || prec == PREC_C32K) && k == 2;
}

// the row kernels: second order, and first order in FP64 (k = 1, 2)
hipError_t launch_step2d(int prec, int order, int lim, int k, int wpb, int n_items, hipStream_t s,
                         const StepArgs& a) {
    const int nblocks = xcd_grid((n_items + wpb - 1) / wpb);
    if (nblocks <= 0) return hipSuccess;
    if (order == 1) {
        if (prec != PREC_F64 || lim != LIM_MINMOD) return hipErrorInvalidValue;
        return wpb == 1 ? launch2_tb<1>(k, nblocks, s, a) : launch2_tb<4>(k, nblocks, s, a);
    }
    if (order != 2) return hipErrorInvalidValue;
    if (k != 1) {
        if (prec == PREC_C32) return launch2_tb2<PREC_C32>(k, lim, wpb, nblocks, s, a);
        if (prec == PREC_C32K) return launch2_tb2<PREC_C32K>(k, lim, wpb, nblocks, s, a);
        return hipErrorInvalidValue;
    }
    switch (prec) {
    case PREC_F64: return launch2_row<PREC_F64>(lim, wpb, nblocks, s, a);
    case PREC_REF32: return launch2_row<PREC_REF32>(lim, wpb, nblocks, s, a);
    case PREC_C32: return launch2_row<PREC_C32>(lim, wpb, nblocks, s, a);
    case PREC_C32K: return launch2_row<PREC_C32K>(lim, wpb, nblocks, s, a);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace shll
