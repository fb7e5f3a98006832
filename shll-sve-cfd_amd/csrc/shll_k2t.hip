// shll_k2t.hip -- 2D first-order SHLL step kernel on register tiles for gfx950.
//
// A block of W wavefronts holds a tile of W*RW rows by 64 columns in registers: wavefront w
// has RW consecutive rows, lane = column.  A step is
//   primitive recovery and the x and y split fluxes of the wavefront's RW rows,
//   the y terms of each row, from the adjacent lanes (DPP wave shifts),
//   one exchange of the edge rows' x fluxes with the wavefronts above and below (LDS, one
//   barrier, double-buffered by step parity),
//   the conservative update, all in registers,
// so a launch of k steps reads the state once and writes it once; the outer k rows and columns
// of a tile are recomputed halo.  Bound: VALU issue and latency on small domains, HBM traffic
// (halo included) together with the blocks a CU holds on large ones.
//
// Why tiles: a wavefront that walks down its rows (the pipelines of shll_k2d.hip) has one serial
// chain of k stages per row and few wavefronts on a small domain; the RW rows of a tile's
// wavefront are independent chains, and a domain gives a wavefront per RW rows and strip.
// Measured, us per step before (row pipelines, their default items) and now: REF32 128^2 27 and
// 1.5, 2048^2 45 and 24; FP64 700^2 32 and 6.9, 1531x2049 45 and 30; C32K 600^2 28 and 4.6,
// 1500^2 29 and 13, 4096^2 104 and 74; C32 4096^2 151 and 112.  A pipeline of k wavefronts that
// hand rows on through LDS (one stage each, a barrier per row) was slower: C32K 4096^2 107,
// FP64 1531x2049 48.
//
// Layout, update order and walls as in shll_k2d.hip (base_shll_2d.c:139-319).
#include "shll_flux.h"

namespace shll {

// x walls change the sign of all but the x momentum's flux, y walls of all but the y momentum's
template <class RT>
__device__ __forceinline__ RT wall_x(int v, RT f) { return v == 1 ? f : -f; }
template <class RT>
__device__ __forceinline__ RT wall_y(int v, RT f) { return v == 2 ? f : -f; }

// One wavefront's rows.  EDGE: the tile touches a wall.
template <int PREC, int RW, int W, bool EDGE>
struct Tile2 {
    using RT = typename Real<PREC>::T;
    static constexpr bool CMP = PREC == PREC_C32 || PREC == PREC_C32K;  // (hi, lo) state
    static constexpr bool KAHAN = PREC == PREC_C32K;

    const Inst& in;
    RT* lds;        // [2 parity][W][2: F- of the first row, F+ of the last][4][64]
    int wib, lane;  // wavefront in block
    int g0;         // the wavefront's first row
    bool jlo, jhi, refl;
    RT lamx, lamy;

    RT u[RW][4], l[CMP ? RW : 1][4];
    RT xp[RW][4], xm[RW][4];
    // y terms: reference forms Y1 = hp - hm + T - B; C32 the lower and upper face terms, C32K
    // their difference in Y1
    RT Y1[RW][4], Y2[PREC == PREC_C32 ? RW : 1][4];

    __device__ __forceinline__ RT* slot(int parity, int w, int s, int v) const {
        return lds + (((parity * W + w) * 2 + s) * 4 + v) * 64 + lane;
    }

    __device__ __forceinline__ void y_terms(int r, const RT (&yp)[4], const RT (&ym)[4]) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const RT hp = yp[v], hm = ym[v];
            RT B = from_left_z(hp);
            if constexpr (EDGE) B = jlo ? (refl ? wall_y(v, hm) : hp) : B;
            if constexpr (!CMP) {
                RT T = from_right_z(hm);
                if constexpr (EDGE) T = jhi ? (refl ? wall_y(v, hp) : hm) : T;
                Y1[r][v] = hp - hm + T - B;
            } else {
                const RT tb = lamy * (B + hm);
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
            // fast form's range, so the rows' dependent chains overlap
            Prim2<RT> q[RW];
            RefSpan<RT> span;
            bool tiny = false;
#pragma unroll
            for (int r = 0; r < RW; ++r) ref_prim2<RT>(u[r], in, q[r], span, tiny);
            const bool ok = span.ok();
            if (__builtin_expect(!ok || tiny, 0)) {
#pragma unroll
                for (int r = 0; r < RW; ++r) ref_prim2_redo<RT>(u[r], in, ok, q[r]);
            }
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                RT yp[4], ym[4];
                ref_flux2<RT>(u[r], q[r], xp[r], xm[r], yp, ym);
                y_terms(r, yp, ym);
            }
        }
    }

    // publish the edge rows, wait, read the neighbours', update all rows; the block's end
    // wavefronts read their own rows for the missing ones (halo)
    __device__ __forceinline__ void update(int parity) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            *slot(parity, wib, 0, v) = xm[0][v];
            *slot(parity, wib, 1, v) = xp[RW - 1][v];
        }
        __syncthreads();
        const int wb = wib > 0 ? wib - 1 : 0, wa = wib + 1 < W ? wib + 1 : W - 1;
        // reference forms: all reads ahead of the updates; read one variable at a time they cost
        // 143 registers instead of 126 (FP64), and so the second block of 16 rows on a CU
        RT near[CMP ? 1 : 4][2];
        if constexpr (!CMP) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                near[v][0] = *slot(parity, wb, 1, v);
                near[v][1] = *slot(parity, wa, 0, v);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const RT below = CMP ? *slot(parity, wb, 1, v) : near[CMP ? 0 : v][0];
            const RT above = CMP ? *slot(parity, wa, 0, v) : near[CMP ? 0 : v][1];
            if constexpr (CMP) {
                RT t[RW + 1];  // face terms between rows f-1 and f
#pragma unroll
                for (int f = 0; f <= RW; ++f) {
                    RT L = f > 0 ? xp[f > 0 ? f - 1 : 0][v] : below;
                    RT R = f < RW ? xm[f < RW ? f : 0][v] : above;
                    if constexpr (EDGE) {
                        if (f < RW) L = g0 + f == 0 ? (refl ? wall_x(v, R) : xp[f < RW ? f : 0][v]) : L;
                        if (f > 0) R = g0 + f == in.nx ? (refl ? wall_x(v, L) : xm[f > 0 ? f - 1 : 0][v]) : R;
                    }
                    t[f] = lamx * (L + R);
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
                    RT L = r > 0 ? xp[r > 0 ? r - 1 : 0][v] : below;
                    RT R = r + 1 < RW ? xm[r + 1 < RW ? r + 1 : 0][v] : above;
                    if constexpr (EDGE) {
                        L = g0 + r == 0 ? (refl ? wall_x(v, xm[r][v]) : xp[r][v]) : L;
                        R = g0 + r == in.nx - 1 ? (refl ? wall_x(v, xp[r][v]) : xm[r][v]) : R;
                    }
                    const RT uu = u[r][v] - lamx * (xp[r][v] - xm[r][v] + R - L);
                    u[r][v] = uu - lamy * Y1[r][v];
                }
            }
        }
    }
};

// ns steps of rows [i0, i0 + W*RW), of which the item's are stored
template <int PREC, int RW, int W, bool EDGE>
__device__ __forceinline__ void tile_steps(const StepArgs& a, const Item2& it, const Inst& in, int i0, int ns,
                                           typename Real<PREC>::T* lds) {
    using T = Tile2<PREC, RW, W, EDGE>;
    using RT = typename T::RT;
    constexpr bool CMP = T::CMP;
    const int wib = uniform((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const int j = it.j0 + lane, nx = in.nx, ny = in.ny;
    const int jc = j < 0 ? 0 : (j < ny ? j : ny - 1);
    const int64_t P = a.plane;
    const int g0 = i0 + wib * RW;
    T t{in, lds, wib, lane, g0, j <= 0, j >= ny - 1, in.bc == BC_REFLECT};
    t.lamx = PREC == PREC_F64 ? (RT)in.k.d_lamx : (PREC == PREC_REF32 ? (RT)in.k.f_lamx : (RT)in.k.c_lamx);
    t.lamy = PREC == PREC_F64 ? (RT)in.k.d_lamy : (PREC == PREC_REF32 ? (RT)in.k.f_lamy : (RT)in.k.c_lamy);
    // rows and columns off the domain hold copies of its edge
    const RT* __restrict__ p0 = (const RT*)a.in0 + in.off;
    const RT* __restrict__ p1 = CMP ? (const RT*)a.in1 + in.off : nullptr;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int g = g0 + r < nx ? g0 + r : nx - 1;
        const int64_t o = (int64_t)g * ny + jc;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            t.u[r][v] = p0[v * P + o];
            if constexpr (CMP) t.l[r][v] = p1[v * P + o];
        }
    }
    for (int s = 0; s < ns; ++s) {
        t.fluxes();
        t.update(s & 1);
    }
    RT* __restrict__ o0 = (RT*)a.out0 + in.off;
    RT* __restrict__ o1 = CMP ? (RT*)a.out1 + in.off : nullptr;
    const bool jown = j >= it.jx0 && j < it.jx0 + it.jw;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int g = g0 + r;
        if (g >= it.ix0 && g < it.ix0 + it.iw && jown) {
            const int64_t o = (int64_t)g * ny + j;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                o0[v * P + o] = t.u[r][v];
                if constexpr (CMP) o1[v * P + o] = t.l[r][v];
            }
        }
    }
}

template <int PREC, int RW, int W>
__global__ __launch_bounds__(64 * W) void k_tile2d(StepArgs a) {
    using RT = typename Real<PREC>::T;
    __shared__ RT lds[2 * W * 2 * 4 * 64];
    const LaunchView lv = launch_view(a);
    const int item = xcd_work((int)blockIdx.x, lv.n_items);
    if (item < 0) return;
    const Item2 it = ((const Item2*)a.items)[item];
    const Inst in = a.inst[it.inst];
    const int64_t left = in.nsteps - lv.step_base;
    const int ns = left < (int64_t)a.ksteps ? (int)left : a.ksteps;
    if (ns <= 0) return;
    // the tile's rows: the item's owned rows [ix0, ix0 + iw) and, on the sides that are not
    // walls, the halo (the host makes no item of more than W*RW - 2k rows)
    const int i0 = it.ix0 - a.ksteps < 0 ? 0 : it.ix0 - a.ksteps;
    const bool edge = i0 <= 0 || i0 + W * RW >= in.nx || it.j0 <= 0 || it.j0 + 64 >= in.ny;
    if (edge) tile_steps<PREC, RW, W, true>(a, it, in, i0, ns, lds);
    else tile_steps<PREC, RW, W, false>(a, it, in, i0, ns, lds);
}

// ---------------------------------------------------------------------------
// Tile heights (rows = RW * W), by precision: the first of the list that the number of its tiles
// allows, else the last that leaves owned rows beside the 2k of the halo.  Measured, us per step.
//
// 12 rows, one per wavefront, while its tiles find a compute unit each: a block's step is bound
// by the issue of its own SIMDs, so fewer rows to a block are a shorter step (k = 4, 16 and 12
// rows: 128^2 REF32 1.74 and 1.51, FP64 2.48 and 1.98, C32K 1.72 and 1.50, C32 2.31 and 1.82;
// 180^2 REF32 1.75 and 1.56; 256^2, more tiles than units, 1.77 and 2.19).  16 rows of one per
// wavefront are no better than of two (1.75).
//
// Then a taller tile recomputes less halo and a shorter one gives more blocks.  C32K, k = 4:
// 300^2 16 rows 2.0, 32 rows 2.9; 500^2 3.6 and 3.1; 1024^2 32 rows 8.2, 40 rows 8.5; 1500^2
// 13.9 and 13.0; 4096^2 82 and 74.  REF32: 24 rows gain nothing up to 4096^2 (97 and 96); C32
// spills at 40 rows (4096^2 32 rows 112, 40 rows 142).  FP64 tiles of 16 rows hold two blocks on
// a CU (126 registers), of 24 rows one, so 24 rows win where their tiles fill the CUs once or
// twice (k = 3, 16 and 24 rows: 300^2 2.9 and 3.6, 500^2 4.4 and 3.8, 700^2 7.3 and 6.9) and
// lose beyond (1024^2 13.0 and 13.6, 2048^2 42 and 44; k = 2: 12.1 and 13.6, 38 and 45), but for
// the halo of 4 steps, which leaves 8 of 16 rows (4096^2 189 and 183).  FP64 tiles of 32 rows,
// one block of 16 wavefronts, k = 2 and 3: 1024^2 13.7 and 12.7, 2048^2 42 and 40, behind the
// two blocks of 16 rows at k = 2.
// ---------------------------------------------------------------------------
struct TileRows {
    int rows, least;   // taken from `least` tiles on
    int most, most4;   // up to this many tiles per compute unit, below 4 steps and from 4 on (0: any)
};
static const TileRows* tile_rows(int prec) {
    static const TileRows f64[] = {{12, 0, 1, 1}, {24, 200, 2, 0}, {16, 0, 0, 0}, {0, 0, 0, 0}};
    static const TileRows ref32[] = {{12, 0, 1, 1}, {24, 1 << 30, 0, 0}, {16, 0, 0, 0}, {0, 0, 0, 0}};
    static const TileRows c32[] = {{12, 0, 1, 1}, {32, 150, 0, 0}, {16, 0, 0, 0}, {0, 0, 0, 0}};
    static const TileRows c32k[] = {{12, 0, 1, 1}, {40, 1000, 0, 0}, {32, 150, 0, 0}, {16, 0, 0, 0}, {0, 0, 0, 0}};
    return prec == PREC_F64 ? f64 : prec == PREC_REF32 ? ref32 : prec == PREC_C32 ? c32 : c32k;
}

// rows of the tiles for k steps per launch on cus compute units, 0 if none fits; tiles(owned):
// the number of tiles that own that many rows
int tile2d_rows(int prec, int k, int cus, int64_t (*tiles)(const void*, int), const void* arg) {
    int rows = 0;
    for (const TileRows* t = tile_rows(prec); t->rows > 0; ++t) {
        if (t->rows <= 2 * k) continue;
        rows = t->rows;
        const int64_t n = tiles(arg, rows - 2 * k);
        const int most = k < 4 ? t->most : t->most4;
        if (n >= t->least && (most == 0 || n <= (int64_t)most * cus)) break;
    }
    return rows;
}

template <int PREC, int RW, int W>
static hipError_t launch_tile(int nblocks, hipStream_t s, const StepArgs& a) {
    hipLaunchKernelGGL((k_tile2d<PREC, RW, W>), dim3(nblocks), dim3(64 * W), 0, s, a);
    return hipGetLastError();
}

// one block per item; rows as tile2d_rows gives them
hipError_t launch_tile2d(int prec, int rows, int n_items, hipStream_t s, const StepArgs& a) {
    const int nblocks = xcd_grid(n_items);
    if (nblocks <= 0) return hipSuccess;
    switch (prec * 64 + rows) {
    case PREC_F64 * 64 + 12: return launch_tile<PREC_F64, 1, 12>(nblocks, s, a);
    case PREC_F64 * 64 + 16: return launch_tile<PREC_F64, 2, 8>(nblocks, s, a);
    case PREC_F64 * 64 + 24: return launch_tile<PREC_F64, 2, 12>(nblocks, s, a);
    case PREC_REF32 * 64 + 12: return launch_tile<PREC_REF32, 1, 12>(nblocks, s, a);
    case PREC_REF32 * 64 + 16: return launch_tile<PREC_REF32, 2, 8>(nblocks, s, a);
    case PREC_REF32 * 64 + 24: return launch_tile<PREC_REF32, 2, 12>(nblocks, s, a);
    case PREC_C32 * 64 + 12: return launch_tile<PREC_C32, 1, 12>(nblocks, s, a);
    case PREC_C32 * 64 + 16: return launch_tile<PREC_C32, 2, 8>(nblocks, s, a);
    case PREC_C32 * 64 + 32: return launch_tile<PREC_C32, 4, 8>(nblocks, s, a);
    case PREC_C32K * 64 + 12: return launch_tile<PREC_C32K, 1, 12>(nblocks, s, a);
    case PREC_C32K * 64 + 16: return launch_tile<PREC_C32K, 2, 8>(nblocks, s, a);
    case PREC_C32K * 64 + 32: return launch_tile<PREC_C32K, 4, 8>(nblocks, s, a);
    case PREC_C32K * 64 + 40: return launch_tile<PREC_C32K, 5, 8>(nblocks, s, a);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace shll
