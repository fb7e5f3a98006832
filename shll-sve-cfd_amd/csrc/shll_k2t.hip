// shll_k2t.hip -- 2D SHLL step kernel on register tiles (first and second order) for gfx950.
//
// A block of W wavefronts holds a tile of W*RW rows by 64 columns in registers: wavefront w
// has RW consecutive rows, lane = column.  A step is
//   primitive recovery and the x and y split fluxes of the wavefront's RW rows,
//   the y terms of each row, from the adjacent lanes (DPP wave shifts),
//   one exchange of the edge rows' x fluxes with the wavefronts above and below (LDS, one
//   barrier, double-buffered by step parity),
//   limited x slopes (second order) and the conservative update, all in registers,
// so a launch of k steps reads the state once and writes it once; the outer order*k rows and
// columns of a tile are recomputed halo.  The RW rows of a wavefront are independent chains,
// where a wavefront that walks down its rows one after another (the row pipelines of
// shll_k2d.hip) has only one.
//
// Layout, update order, walls and limiters as in shll_k2d.hip (base_shll_2d.c:139-319,
// 2nd_order_base_shll.c:203-541, base-omp/2nd_order_base_shll.c:317-325,385-392).
#include "shll_flux.h"

namespace shll {

// x walls change the sign of all but the x momentum's flux, y walls of all but the y momentum's
template <class RT>
__device__ __forceinline__ RT wall_x(int v, RT f) { return v == 1 ? f : -f; }
template <class RT>
__device__ __forceinline__ RT wall_y(int v, RT f) { return v == 2 ? f : -f; }

// Edge rows' x fluxes in LDS, per buffer, wavefront and slot: 4 variables x 64 lanes.
// Slots for the wavefront below: F- of the first row (second order: and of the second, and F+
// of the first); for the one above: F+ of the last row (and of the last but one, and F- of the
// last).  First order double-buffers them by step parity, one barrier per step; second order,
// with three times the slots, keeps one buffer and takes a second barrier before it is
// written again.
template <int ORDER>
struct TileSlots {
    static constexpr int SIDE = ORDER == 1 ? 1 : 3, N = 2 * SIDE, NBUF = ORDER == 1 ? 2 : 1;
};

template <int PREC, int ORDER, int LIM, int RW, int W, bool EDGE, bool SQ>
struct Tile2 {
    using RT = typename Real<PREC>::T;
    static constexpr bool CMP = PREC == PREC_C32 || PREC == PREC_C32K;  // (hi, lo) state
    static constexpr bool KAHAN = PREC == PREC_C32K;
    using A = typename std::conditional<CMP, C32Arith, RefArith<RT>>::type;
    using Up = RefUpdate<RT>;
    static constexpr int SIDE = TileSlots<ORDER>::SIDE, SLOTS = TileSlots<ORDER>::N;

    const Inst& in;
    RT* lds;        // [NBUF][W][SLOTS][4][64]
    int wib, lane;  // wavefront in block
    int g0, j;      // the wavefront's first row, the lane's column
    bool jlo, jhi, refl;
    RT lamy, hlamx, hlamy, lamx, th;

    RT u[RW][4], l[CMP ? RW : 1][4];
    RT xp[RW][4], xm[RW][4];
    // y terms: reference forms Y1 = hp - hm + T - B and Y2 = the same of the slopes; C32 the
    // lower and upper face terms, C32K their difference in Y1
    RT Y1[RW][4], Y2[ORDER == 2 || PREC == PREC_C32 ? RW : 1][4];

    __device__ __forceinline__ RT* slot(int parity, int w, int s, int v) const {
        const int b = TileSlots<ORDER>::NBUF == 2 ? parity : 0;
        return lds + (((b * W + w) * SLOTS + s) * 4 + v) * 64 + lane;
    }

    // F and the y terms of row r
    __device__ __forceinline__ void y_terms(int r, const RT (&yp)[4], const RT (&ym)[4]) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const RT hp = yp[v], hm = ym[v];
            RT B = from_left_z(hp), dhp = 0, dhm = 0;
            if constexpr (ORDER == 2) {
                dhp = limited_slope<A, LIM>(B, hp, from_right_z(hp), th);
                dhm = limited_slope<A, LIM>(from_left_z(hm), hm, from_right_z(hm), th);
                if constexpr (EDGE) {
                    dhp = jlo || jhi ? (RT)0 : dhp;
                    dhm = jlo || jhi ? (RT)0 : dhm;
                }
            }
            if constexpr (EDGE) B = jlo ? (refl ? wall_y(v, hm) : hp) : B;
            if constexpr (!CMP) {
                RT T = from_right_z(hm);
                if constexpr (EDGE) T = jhi ? (refl ? wall_y(v, hp) : hm) : T;
                Y1[r][v] = hp - hm + T - B;
                if constexpr (ORDER == 2) {
                    RT Bd = from_left_z(dhp), Td = from_right_z(dhm);
                    if constexpr (EDGE) {
                        Bd = jlo ? (RT)0 : Bd;
                        Td = jhi ? (RT)0 : Td;
                    }
                    Y2[r][v] = dhp + dhm - Td - Bd;
                }
            } else {
                RT tb = lamy * (B + hm);
                if constexpr (ORDER == 2) {
                    RT d = from_left_z(dhp) - dhm;
                    if constexpr (EDGE) d = jlo ? (RT)0 : d;
                    tb = __builtin_fmaf(hlamy, d, tb);
                }
                RT tt = from_right_z(tb);
                if constexpr (EDGE) tt = jhi ? lamy * (hp + (refl ? wall_y(v, hp) : hm)) : tt;
                if constexpr (KAHAN) {
                    Y1[r][v] = tb - tt;
                } else {
                    Y1[r][v] = tb;
                    Y2[r][v] = tt;
                }
            }
        }
    }

    __device__ __forceinline__ void fluxes() {
        if constexpr (CMP) {
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                RT yp[4], ym[4];
                fluxes2<PREC, RT>(u[r], in, xp[r], xm[r], yp, ym);
                y_terms(r, yp, ym);
            }
        } else {
            // primitives of all rows, then one branch for the lanes with a cell outside the
            // fast form's range
            Prim2<RT> q[RW];
            bool ok = true;
#pragma unroll
            for (int r = 0; r < RW; ++r) ok &= ref_prim2<RT>(u[r], in, q[r]);
            if (__builtin_expect(!ok, 0)) {
#pragma unroll
                for (int r = 0; r < RW; ++r) ref_prim2_exact<RT>(u[r], in, q[r]);
            }
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                RT yp[4], ym[4];
                ref_flux2<RT>(u[r], q[r], xp[r], xm[r], yp, ym);
                y_terms(r, yp, ym);
            }
        }
    }

    // limited slope of row g from its three values; zero on the domain's first and last rows
    __device__ __forceinline__ RT xslope(RT a, RT b, RT c, int g) const {
        RT s = limited_slope<A, LIM>(a, b, c, th);
        if constexpr (EDGE) s = g <= 0 || g >= in.nx - 1 ? (RT)0 : s;
        return s;
    }

    // the conservative update of all rows, variable by variable
    __device__ __forceinline__ void update(int parity, bool again) {
        if constexpr (TileSlots<ORDER>::NBUF == 1) {
            if (again) __syncthreads();  // every wavefront has read the last step's rows
        }
        // publish the edge rows, wait, read the neighbours'; the block's end wavefronts read
        // their own rows for the missing ones (halo)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            *slot(parity, wib, 0, v) = xm[0][v];
            *slot(parity, wib, SIDE, v) = xp[RW - 1][v];
            if constexpr (ORDER == 2) {
                *slot(parity, wib, 1, v) = xm[1][v];
                *slot(parity, wib, 2, v) = xp[0][v];
                *slot(parity, wib, SIDE + 1, v) = xp[RW - 2][v];
                *slot(parity, wib, SIDE + 2, v) = xm[RW - 1][v];
            }
        }
        __syncthreads();
        const int wb = wib > 0 ? wib - 1 : 0, wa = wib + 1 < W ? wib + 1 : W - 1;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            // window rows -1 .. RW (second order: F+ also at -2, F- at RW+1), index r + 2
            RT P[RW + 4], M[RW + 4];
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                P[r + 2] = xp[r][v];
                M[r + 2] = xm[r][v];
            }
            P[0] = P[RW + 2] = P[RW + 3] = M[0] = M[1] = M[RW + 3] = (RT)0;
            P[1] = *slot(parity, wb, SIDE, v);
            M[RW + 2] = *slot(parity, wa, 0, v);
            RT sP[RW + 1], sM[RW + 1];  // sP[f] = F+ slope of row f-1, sM[f] = F- slope of row f
            if constexpr (ORDER == 2) {
                P[0] = *slot(parity, wb, SIDE + 1, v);
                M[1] = *slot(parity, wb, SIDE + 2, v);
                M[RW + 3] = *slot(parity, wa, 1, v);
                P[RW + 2] = *slot(parity, wa, 2, v);
#pragma unroll
                for (int f = 0; f <= RW; ++f) {
                    sP[f] = xslope(P[f], P[f + 1], P[f + 2], g0 + f - 1);
                    sM[f] = xslope(M[f + 1], M[f + 2], M[f + 3], g0 + f);
                }
            }
            if constexpr (CMP) {
                RT t[RW + 1];  // face terms between rows f-1 and f
#pragma unroll
                for (int f = 0; f <= RW; ++f) {
                    RT L = P[f + 1], R = M[f + 2];
                    if constexpr (EDGE) {
                        const int g = g0 + f;
                        L = g == 0 ? (refl ? wall_x(v, R) : P[f + 2]) : L;
                        R = g == in.nx ? (refl ? wall_x(v, L) : M[f + 1]) : R;
                    }
                    t[f] = lamx * (L + R);
                    if constexpr (ORDER == 2) {
                        t[f] = __builtin_fmaf(hlamx, sP[f] - sM[f], t[f]);
                    }
                }
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    RT hi = u[r][v], lo = l[r][v];
                    if constexpr (KAHAN) {
                        const RT y = ((t[r] - t[r + 1]) + Y1[r][v]) + lo;
                        const RT s = hi + y;
                        l[r][v] = y - (s - hi);
                        u[r][v] = s;
                    } else {
                        RT e;
                        two_sum(hi, t[r], hi, e);
                        lo = lo + e;
                        two_sum(hi, -t[r + 1], hi, e);
                        lo = lo + e;
                        two_sum(hi, Y1[r][v], hi, e);
                        lo = lo + e;
                        two_sum(hi, -Y2[r][v], hi, e);
                        lo = lo + e;
                        fast_two_sum(hi, lo, u[r][v], l[r][v]);
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    RT L = P[r + 1], R = M[r + 3];
                    if constexpr (EDGE) {
                        L = g0 + r == 0 ? (refl ? wall_x(v, xm[r][v]) : xp[r][v]) : L;
                        R = g0 + r == in.nx - 1 ? (refl ? wall_x(v, xp[r][v]) : xm[r][v]) : R;
                    }
                    RT uu = Up::template first<true>(v == 2, u[r][v], lamx, xp[r][v] - xm[r][v] + R - L);
                    if constexpr (ORDER == 2)
                        uu = Up::template second<true>(v == 2, uu, lamx, sP[r + 1] + sM[r] - sM[r + 1] - sP[r]);
                    uu = Up::template first<SQ>(v == 1, uu, lamy, Y1[r][v]);
                    if constexpr (ORDER == 2) uu = Up::template second<SQ>(v == 1, uu, lamy, Y2[r][v]);
                    u[r][v] = uu;
                }
            }
        }
    }
};

// One item: its owned rows in tiles of at most W*RW rows
template <int PREC, int ORDER, int LIM, int RW, int W, bool EDGE, bool SQ>
__device__ __forceinline__ void tile_steps(const StepArgs& a, const Item2& it, const Inst& in, int i0, int ns, int x0,
                                           int x1, typename Real<PREC>::T* lds, int& parity) {  // parity: steps this block has taken
    using T = Tile2<PREC, ORDER, LIM, RW, W, EDGE, SQ>;
    using RT = typename T::RT;
    constexpr bool CMP = T::CMP;
    const int wib = uniform((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int j = it.j0 + lane, nx = in.nx, ny = in.ny;
    const int jc = j < 0 ? 0 : (j < ny ? j : ny - 1);
    const int64_t P = a.plane;
    const int g0 = i0 + wib * RW;
    T t{in, lds, wib, lane, g0, j, j <= 0, j >= ny - 1, in.bc == BC_REFLECT};
    if constexpr (CMP) {
        t.lamx = in.k.c_lamx; t.lamy = in.k.c_lamy; t.th = in.k.c_theta;
    } else if constexpr (PREC == PREC_F64) {
        t.lamx = in.k.d_lamx; t.lamy = in.k.d_lamy; t.th = in.k.d_theta;
    } else {
        t.lamx = in.k.f_lamx; t.lamy = in.k.f_lamy; t.th = in.k.f_theta;
    }
    t.hlamx = (RT)0.5 * t.lamx;
    t.hlamy = (RT)0.5 * t.lamy;
    // rows and columns off the domain hold copies of its edge
    const RT* __restrict__ p0 = (const RT*)a.in0 + in.off;
    const RT* __restrict__ p1 = CMP ? (const RT*)a.in1 + in.off : nullptr;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int g = g0 + r < 0 ? 0 : (g0 + r < nx ? g0 + r : nx - 1);
        const int64_t o = (int64_t)g * ny + jc;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            t.u[r][v] = p0[v * P + o];
            if constexpr (CMP) t.l[r][v] = p1[v * P + o];
        }
    }
    for (int s = 0; s < ns; ++s) {
        t.fluxes();
        t.update(parity & 1, parity > 0);
        ++parity;
    }
    RT* __restrict__ o0 = (RT*)a.out0 + in.off;
    RT* __restrict__ o1 = CMP ? (RT*)a.out1 + in.off : nullptr;
    const bool jown = j >= it.jx0 && j < it.jx0 + it.jw;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int g = g0 + r;
        if (g >= x0 && g < x1 && jown) {
            const int64_t o = (int64_t)g * ny + j;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                o0[v * P + o] = t.u[r][v];
                if constexpr (CMP) o1[v * P + o] = t.l[r][v];
            }
        }
    }
}

#ifndef T_EU32
#define T_EU32 1
#define T_EU64 1
#endif
template <int PREC, int ORDER, int LIM, int RW, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(PREC == PREC_F64 ? T_EU64 : T_EU32)))
void k_tile2d(StepArgs a) {
    using RT = typename Real<PREC>::T;
    __shared__ RT lds[TileSlots<ORDER>::NBUF * W * TileSlots<ORDER>::N * 4 * 64];
    const LaunchView lv = launch_view(a);
    const int item = xcd_work((int)blockIdx.x, lv.n_items);
    if (item < 0) return;
    const Item2 it = ((const Item2*)a.items)[item];
    const Inst in = a.inst[it.inst];
    const int64_t left = in.nsteps - lv.step_base;
    const int ns = left < (int64_t)a.ksteps ? (int)left : a.ksteps;
    if (ns <= 0) return;
    // tiles of the item: halo rows on the sides that are not walls
    const int H = ORDER * a.ksteps, end = it.ix0 + it.iw;
    int parity = 0;
    for (int x0 = it.ix0; x0 < end;) {
        const int i0 = x0 - H < 0 ? 0 : x0 - H;
        int x1 = i0 + W * RW >= in.nx ? in.nx : i0 + W * RW - H;
        x1 = x1 < end ? x1 : end;
        const bool edge = i0 <= 0 || i0 + W * RW >= in.nx || it.j0 <= 0 || it.j0 + 64 >= in.ny;
        if constexpr (PREC == PREC_F64 || PREC == PREC_REF32) {
            const bool sq = PREC == PREC_F64 ? in.k.d_lamy == 0.125 : in.k.f_lamy == 0.125f;
            if (edge) {
                if (sq) tile_steps<PREC, ORDER, LIM, RW, W, true, true>(a, it, in, i0, ns, x0, x1, lds, parity);
                else tile_steps<PREC, ORDER, LIM, RW, W, true, false>(a, it, in, i0, ns, x0, x1, lds, parity);
            } else {
                if (sq) tile_steps<PREC, ORDER, LIM, RW, W, false, true>(a, it, in, i0, ns, x0, x1, lds, parity);
                else tile_steps<PREC, ORDER, LIM, RW, W, false, false>(a, it, in, i0, ns, x0, x1, lds, parity);
            }
        } else {
            if (edge) tile_steps<PREC, ORDER, LIM, RW, W, true, false>(a, it, in, i0, ns, x0, x1, lds, parity);
            else tile_steps<PREC, ORDER, LIM, RW, W, false, false>(a, it, in, i0, ns, x0, x1, lds, parity);
        }
        x0 = x1;
    }
}

// rows per wavefront and wavefronts per block, by precision and order
#ifndef T_RW32
#define T_RW32 4
#define T_W32 4
#define T_RW64 4
#define T_W64 4
#endif
template <int PREC, int ORDER>
struct TileShape {
    static constexpr int RW = PREC == PREC_F64 ? T_RW64 : T_RW32, W = PREC == PREC_F64 ? T_W64 : T_W32;
};

int tile2d_rows(int prec, int order) {
    (void)order;
    return prec == PREC_F64 ? TileShape<PREC_F64, 1>::RW * TileShape<PREC_F64, 1>::W
                            : TileShape<PREC_REF32, 1>::RW * TileShape<PREC_REF32, 1>::W;
}

template <int PREC, int ORDER, int LIM>
static hipError_t launch_tile(int nblocks, hipStream_t s, const StepArgs& a) {
    constexpr int RW = TileShape<PREC, ORDER>::RW, W = TileShape<PREC, ORDER>::W;
    hipLaunchKernelGGL((k_tile2d<PREC, ORDER, LIM, RW, W>), dim3(nblocks), dim3(64 * W), 0, s, a);
    return hipGetLastError();
}

template <int PREC>
static hipError_t launch_tile_p(int order, int lim, int nblocks, hipStream_t s, const StepArgs& a) {
    if (order == 1) return launch_tile<PREC, 1, LIM_MINMOD>(nblocks, s, a);
    return lim == LIM_MC ? launch_tile<PREC, 2, LIM_MC>(nblocks, s, a) : launch_tile<PREC, 2, LIM_MINMOD>(nblocks, s, a);
}

// one block per item
hipError_t launch_tile2d(int prec, int order, int lim, int n_items, hipStream_t s, const StepArgs& a) {
    const int nblocks = xcd_grid(n_items);
    if (nblocks <= 0) return hipSuccess;
    switch (prec) {
    case PREC_F64: return launch_tile_p<PREC_F64>(order, lim, nblocks, s, a);
    case PREC_REF32: return launch_tile_p<PREC_REF32>(order, lim, nblocks, s, a);
    case PREC_C32: return launch_tile_p<PREC_C32>(order, lim, nblocks, s, a);
    case PREC_C32K: return launch_tile_p<PREC_C32K>(order, lim, nblocks, s, a);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace shll
