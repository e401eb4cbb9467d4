// tdw_resident.hip -- the constant-mass PECE step of lattices whose whole
// state (both components) fits in the LDS of one CU: one workgroup per state.
//
// With the state resident, everything between two density sums is one pass:
//   rs_pred   predictor and partial corrector (tdwslda_ode_integrator.h:26-135)
//             with the norm of y_p as a per-state factor: 8 S (AB5AM5);
//   dens, potentials of the prediction (weights f s^2): 1 S;
//   rs_h<1>   s y_p into LDS, its Laplacian in place (all axes), H psi and
//             <H> (pca_kernels.cu:233-391, 806-832), the corrector
//             (tdwslda_ode_integrator.h:138-220), its norm, the normalised y:
//             3 S;
//   dens, potentials of the corrected state: 1 S;
//   rs_h<0>   H psi - <H> psi of it into the newest history slot: 2 S.
// 15 S per state-step in nine launches.  The kernel-by-kernel step moves 31 S
// (2D plane kernels) to 35 S in some twenty launches, the six-pass step of
// tdw_fused.hip 20 S in sixteen.  Per step, before and after: 1D 64 points x
// 128 states 87 -> 59 us, 36 x 18 x 300 190 -> 98 us, 64 x 64 x 1024 924 ->
// 684 us, 12^3 x 1781 487 -> 400 us.
//
// Bounds: at 64 x 64 one 133 KB state fills a CU's LDS and its load, transform
// and store phases follow one another (rs_h<1> 169 us for 3 S of 134 MB,
// rs_h<0> 141 us for 2 S, against 292 and 169 us of the kernels they replace);
// small lattices wait for launches, cold instruction fetches and the chain of
// barriers of one state (15 us for up to 256 states of 36 x 18).
#include "tdw_device.hpp"
#include "tdw_fused.hpp"
#include "tdw_internal.hpp"
#include "tdw_physics.hpp"
#include "tdw_resident.hpp"
#include "tdw_planemm.hpp"
#include "tdw_rsfft.hpp"

#include <algorithm>
#include <math.h>
#include <vector>

namespace tdw {

struct RsPlan {
    int dim, inner, npc, ll;      // points per x plane (padded), padded points per component, last axis length
    unsigned mll;                 // division by the last axis length
    RsAxis ax[3];
    MmScale mm;                   // of the matrix-core planes
};

// Laplacian of both components in LDS, in place: the factor
// -(k_x^2 + k_y^2 + k_z^2) / N on the spectrum, kx its x part per position of
// the x axis, kin the rest per point of an x plane
__device__ __forceinline__ void rs_laplace(double2 *A, const double2 *tw, const RsPlan &pl,
                                           const double *__restrict__ kx, const double *__restrict__ kin)
{
    for (int d = pl.dim - 1; d > 0; d--) rs_forward(A, tw, pl.ax[d]);
    rs_filter(A, tw, pl.ax[0], [&](unsigned i, unsigned q, double2 &v) { v = v * (kx[i] + kin[q]); });
    for (int d = 1; d < pl.dim; d++) rs_inverse(A, tw, pl.ax[d]);
}

// Predictor: y <- y_p (unnormalised), c <- the partial corrector, s = 1 /
// sqrt(norm), s2 = s^2 per state; with nrm_out, the norm itself.  A state per
// workgroup, so the norm needs no second launch.
template <int SCH>
__global__ void __launch_bounds__(RS_NT)
rs_pred(const double2 *yin, double2 *y, double2 *c, const double2 *f1, const double2 *f2, const double2 *f3,
        const double2 *f4, const double2 *f5, int n, int N, double dt, double dv, double *__restrict__ s_out,
        double *__restrict__ s2_out, double *__restrict__ nrm_out)
{
    __shared__ double red[RS_NT / 64];
    const int a = blockIdx.x;
    double nrm = 0.0;
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
        // both components' loads before the stores, which may alias them
        const long idx[2] = {(long)a * N + i, ((long)n + a) * N + i};
        double2 yk[2], F[2][5];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            yk[q] = yin[idx[q]];
            F[q][0] = f1[idx[q]];
            F[q][1] = f2[idx[q]];
            F[q][2] = f3[idx[q]];
            F[q][3] = SCH >= 45 ? f4[idx[q]] : make_double2(0.0, 0.0);
            F[q][4] = SCH >= 55 ? f5[idx[q]] : make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
            double2 sp, sc;
            abm_sums<SCH>(F[q][0], F[q][1], F[q][2], F[q][3], F[q][4], sp, sc);
            const double2 yp = yk[q] + imul(sp, -dt);
            y[idx[q]] = yp;
            c[idx[q]] = yk[q] + imul(sc, -dt);
            nrm += cnorm(yp);
        }
    }
    nrm = block_sum(nrm, red) * dv;
    if (threadIdx.x) return;
    const double sc = 1.0 / sqrt(nrm);
    s_out[a] = sc;
    s2_out[a] = sc * sc;
    if (nrm_out) nrm_out[a] = nrm;
}

struct RsH {
    double mu_a, mu_b, dv, dta0;
    int bdg;
};

// CORR 0: out = H psi - <H> psi, psi = in; with lap, lap = its Laplacian.
// CORR 1: psi = s_a in (the normalised prediction), out = the normalised
// corrected state of -i dt a0 (H psi - <H> psi) + c (out may be in: a state
// is read whole before it is written).
// CORR 2: out = H psi, psi = in (out is not in); with c, e_out = dv Re <in|c>.
// <H> per state into e_out (and e_out2), or read from use_e; the corrected
// state's norm into nrm_out where given.  H as in k_apply_h, with the transverse momenta of 1D
// and 2D (kt, and kt2 in 1D) in the kinetic term.
template <int CORR>
__global__ void __launch_bounds__(RS_NT)
rs_h(const double2 *in, double2 *out, const double2 *__restrict__ c, const double *__restrict__ pots,
     const double *__restrict__ sc, const double *__restrict__ kt, const double *__restrict__ kt2, int n, int N,
     RsPlan pl, RsH hp, const double2 *__restrict__ twg, int ntw, const double *__restrict__ kx,
     const double *__restrict__ kin, const double *use_e, double *e_out, double *e_out2,
     double *__restrict__ nrm_out, double2 *lap)
{
    extern __shared__ double2 rs_sm[];
    __shared__ double red[RS_NT / 64];
    double2 *A = rs_sm, *tw = rs_sm + 2 * pl.npc;
    const int a = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const long gu = (long)a * N, gv = ((long)n + a) * N;
    const double s = CORR == 1 ? sc[a] : 1.0;
    for (int k = tid; k < ntw; k += nt) tw[k] = twg[k];
    // point i of a component sits at i + i / ll: rows of the last axis, ll + 1 apart
    const int pad = pl.dim > 1;
    for (int i = tid; i < N; i += nt) {
        const int pe = pad ? i + rs_div(i, pl.ll, pl.mll) : i;
        A[pe] = in[gu + i] * s;
        A[pl.npc + pe] = in[gv + i] * s;
    }
    __syncthreads();
    rs_laplace(A, tw, pl, kx, kin);
    double k2t = 0.0;
    if (kt) k2t = kt[a] * kt[a];
    if (kt2) k2t += kt2[a] * kt2[a];
    // H psi over the Laplacian, <psi|H psi>
    double e = 0.0;
    for (int i = tid; i < N; i += nt) {
        const int pe = pad ? i + rs_div(i, pl.ll, pl.mll) : i;
        const double aa = hp.bdg ? -0.5 : pots[4 * N + i] * -0.5, ab = hp.bdg ? -0.5 : pots[5 * N + i] * -0.5;
        const double Va = pots[i] - hp.mu_a - aa * k2t, Vb = pots[N + i] - hp.mu_b - ab * k2t;
        const double2 D = make_double2(pots[2 * N + 2 * i], pots[2 * N + 2 * i + 1]);
        const double2 tu = in[gu + i] * s, tv = in[gv + i] * s;
        if (CORR == 0 && lap) {
            lap[gu + i] = A[pe];
            lap[gv + i] = A[pl.npc + pe];
        }
        const double2 u = tu * Va + cmul(tv, D) + A[pe] * aa;
        const double2 v = tv * (-Vb) + cmulc(D, tu) - A[pl.npc + pe] * ab;
        if constexpr (CORR == 2) {
            out[gu + i] = u;
            out[gv + i] = v;
            if (c) e += cmulc(tu, c[gu + i]).x + cmulc(tv, c[gv + i]).x;
            continue;
        }
        A[pe] = u;
        A[pl.npc + pe] = v;
        e += cmulc(tu, u).x + cmulc(tv, v).x;
    }
    if constexpr (CORR == 2) {
        if (!c) return;
        e = block_sum(e, red) * hp.dv;
        if (tid == 0) e_out[a] = e;
        return;
    }
    if (use_e) {
        e = use_e[a];
    } else {
        e = block_sum(e, red) * hp.dv;
        if (tid == 0) {
            e_out[a] = e;
            if (e_out2) e_out2[a] = e;
        }
    }
    double nrm = 0.0;
    for (int i = tid; i < N; i += nt) {
        const int pe = pad ? i + rs_div(i, pl.ll, pl.mll) : i;
        const double2 u = A[pe] - in[gu + i] * s * e, v = A[pl.npc + pe] - in[gv + i] * s * e;
        if constexpr (CORR == 1) {
            const double2 yu = imul(u, -hp.dta0) + c[gu + i], yv = imul(v, -hp.dta0) + c[gv + i];
            A[pe] = yu;
            A[pl.npc + pe] = yv;
            nrm += cnorm(yu) + cnorm(yv);
        } else {
            out[gu + i] = u;
            out[gv + i] = v;
        }
    }
    if constexpr (CORR == 1) {
        nrm = block_sum(nrm, red) * hp.dv;
        const double r = 1.0 / sqrt(nrm);
        if (tid == 0 && nrm_out) nrm_out[a] = nrm;
        for (int i = tid; i < N; i += nt) {
            const int pe = pad ? i + rs_div(i, pl.ll, pl.mll) : i;
            out[gu + i] = A[pe] * r;
            out[gv + i] = A[pl.npc + pe] * r;
        }
    }
}

// ---------------------------------------------------------------------------
// The same for 2D planes of 32 or 64 points a side, on the matrix cores.
//
// The transforms of rs_h read and write the state seven times in LDS, behind
// as many barriers, and one 64 x 64 state occupies a CU alone.  Here the second
// derivatives are the products of tdw_planemm.hpp: a wave owns the points
// (ix, iy) of one component with ix in a 16-row tile or that plus LX/2, iy in a
// tile or that plus LY/2, and all that follows (H psi, <H>, corrector, norm)
// stays in its registers.
// More multiplications (64 per point and component at 64 x 64) but no index
// arithmetic and one barrier before H: at 64 x 64 the corrector form of 1024
// states 169 -> 128 us, the plain one 141 -> 99, of 192 states 39 -> 28 and
// 35 -> 25; 32 x 32 and 32 x 64 gain as much.  One 512-thread workgroup per CU
// at 64 x 64 (133 KB of LDS, 254 registers), bound by its load and store
// phases, which nothing overlaps.
// ---------------------------------------------------------------------------
template <int LX, int LY, int CORR>
__global__ void __launch_bounds__(64 * 2 * (LX / 32) * (LY / 32), 2)
rs_mm(const double2 *in, double2 *out, const double2 *__restrict__ c, const double *__restrict__ pots,
      const double *__restrict__ sc, const double *__restrict__ kt, int n, RsH hp, const double *__restrict__ mx,
      const double *__restrict__ my, double rx, double ry, const double *use_e, double *e_out, double *e_out2, double *__restrict__ nrm_out)
{
    constexpr int HX = LX / 2, HY = LY / 2, TX = HX / 16, TY = HY / 16, W = 2 * TX * TY, NT = 64 * W;
    constexpr int N = LX * LY, RS = LY + 1, NPC = LX * RS;
    extern __shared__ double2 rs_sm[];
    __shared__ double red[W];
    const int a = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int cmp = w / (TX * TY), tx = (w / TY) % TX, ty = w % TY;
    const long gu = (long)a * N, gv = ((long)n + a) * N;
    const double s = CORR == 1 ? sc[a] : 1.0;
#pragma unroll 4
    for (int i = tid; i < N; i += NT) {
        const int pe = i + i / LY;
        rs_sm[pe] = in[gu + i] * s;
        rs_sm[NPC + pe] = in[gv + i] * s;
    }
    const double2 *X = rs_sm + cmp * NPC, *Y = rs_sm + (1 - cmp) * NPC;   // own component, the other
    const int lr = lane >> 4, lc = lane & 15;
    // lap[h][g]: points (ix + h HX, iy + g HY), four rows each; re and im
    dbl4 lre[2][2], lim[2][2];
    __syncthreads();
    MmAcc acc;
    mm_product<true, HX, RS, HY>(X + lr * RS + 16 * ty + lc, mx + (long)tx * (HX / 4) * 128 + lane, acc);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            lre[h][g] = mm_outer_at(acc, h, g, 0) * rx;
            lim[h][g] = mm_outer_at(acc, h, g, 1) * rx;
        }
    __builtin_amdgcn_sched_barrier(0);
    mm_product<false, HY, RS, HX>(X + (16 * tx + lc) * RS + lr, my + (long)ty * (HY / 4) * 128 + lane, acc);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            lre[h][g] += mm_inner_at(acc, h, g, 0) * ry;
            lim[h][g] += mm_inner_at(acc, h, g, 1) * ry;
        }
    const double k2t = kt ? kt[a] * kt[a] : 0.0;
    const long own = cmp ? gv : gu;
    const double *V = pots + cmp * N, *al = pots + (4 + cmp) * N;
    const double sg = cmp ? -1.0 : 1.0, mu = cmp ? hp.mu_b : hp.mu_a;
    // The wave's points, one 16 x 16 tile (four rows r) at a time: tile (h, g)
    // starts h HX rows and g HY columns on, rows are 4 apart.  The offsets are
    // formed per tile and kept opaque, else all sixteen points' addresses are
    // (registers).
    const int i0 = (16 * tx + lr) * LY + 16 * ty + lc, j0 = (16 * tx + lr) * RS + 16 * ty + lc;
#define MM_TILES(h, g, i, j)                                                                     \
    _Pragma("unroll") for (int h = 0; h < 2; h++)                                                \
        _Pragma("unroll") for (int g = 0; g < 2; g++)                                            \
            if (int i = i0 + h * HX * LY + g * HY, j = j0 + h * HX * RS + g * HY; mm_tile(i, j))
    // H psi over the Laplacian, <psi|H psi>
    const double2 *co = CORR && c ? c + own : nullptr;
    double2 *oo = out + own;
    double e = 0.0;
    MM_TILES(h, g, i, j) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ir = i + 4 * r * LY, jr = j + 4 * r * RS;
            const double2 x = X[jr], y = Y[jr];
            const double av = al[ir];
            const double aa = hp.bdg ? -0.5 : av * -0.5;
            const double Vv = sg * (V[ir] - mu - aa * k2t);
            const double2 Dv = ((const double2 *)(pots + 2 * N))[ir];
            const double2 t = x * Vv + cmul(y, make_double2(Dv.x, sg * Dv.y)) +
                              make_double2(lre[h][g][r], lim[h][g][r]) * (sg * aa);
            if constexpr (CORR == 2) {
                oo[ir] = t;
                if (co) e += cmulc(x, co[ir]).x;
            } else {
                lre[h][g][r] = t.x;
                lim[h][g][r] = t.y;
                e += cmulc(x, t).x;
            }
        }
    }
    if constexpr (CORR == 2) {
        if (!co) return;
        e = block_sum(e, red) * hp.dv;
        if (tid == 0) e_out[a] = e;
        return;
    }
    if (use_e) {
        e = use_e[a];
    } else {
        e = block_sum(e, red) * hp.dv;
        if (tid == 0) {
            e_out[a] = e;
            if (e_out2) e_out2[a] = e;
        }
    }
    double nrm = 0.0;
    MM_TILES(h, g, i, j) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int ir = i + 4 * r * LY;
            double2 t = make_double2(lre[h][g][r], lim[h][g][r]) - X[j + 4 * r * RS] * e;
            if constexpr (CORR == 1) {
                t = imul(t, -hp.dta0) + co[ir];
                lre[h][g][r] = t.x;
                lim[h][g][r] = t.y;
                nrm += cnorm(t);
            } else {
                oo[ir] = t;
            }
        }
    }
    if constexpr (CORR == 1) {
        nrm = block_sum(nrm, red) * hp.dv;
        const double q = 1.0 / sqrt(nrm);
        if (tid == 0 && nrm_out) nrm_out[a] = nrm;
        MM_TILES(h, g, i, j) {
#pragma unroll
            for (int r = 0; r < 4; r++) oo[i + 4 * r * LY] = make_double2(lre[h][g][r], lim[h][g][r]) * q;
        }
    }
#undef MM_TILES
}

// ---------------------------------------------------------------------------
// First derivatives along both axes and the Laplacian of the same planes (a
// measurement's derivatives): a plane per workgroup, read and each result
// written once, where the axis passes read it twice and the Laplacian three
// times: 1024 states of 64 x 64 119 us for 592, near what the copies take.
// tab: second-, then first-derivative tables of x, then of y.
// ---------------------------------------------------------------------------
template <int LX, int LY>
__global__ void __launch_bounds__(64 * (LX / 32) * (LY / 32), 2)
rs_deriv(const double2 *in, double2 *ddx, double2 *ddy, double2 *lap, const double *__restrict__ tab, MmScale sc)
{
    constexpr int HX = LX / 2, HY = LY / 2, TX = HX / 16, TY = HY / 16, NT = 64 * TX * TY;
    constexpr int N = LX * LY, RS = LY + 1, MX = TX * (LX / 8) * 128, MY = TY * (LY / 8) * 128;
    extern __shared__ double2 rs_sm[];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, tx = w / TY, ty = w % TY;
    const long g0 = (long)blockIdx.x * N;
#pragma unroll 8
    for (int i = tid; i < N; i += NT) rs_sm[i + i / LY] = in[g0 + i];
    const int lr = lane >> 4, lc = lane & 15;
    const double *mx = tab + (long)tx * (HX / 4) * 128 + lane, *my = tab + 2 * MX + (long)ty * (HY / 4) * 128 + lane;
    const double2 *xo = rs_sm + lr * RS + 16 * ty + lc, *xi = rs_sm + (16 * tx + lc) * RS + lr;
    const long o = g0 + (16 * tx + lr) * LY + 16 * ty + lc;
    MmAcc acc;
    dbl4 lre[2][2], lim[2][2];
    __syncthreads();
    mm_product<true, HX, RS, HY>(xo, mx + MX, acc);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const dbl4 re = mm_outer_at(acc, h, g, 0) * sc.s[0][1], im = mm_outer_at(acc, h, g, 1) * sc.s[0][1];
#pragma unroll
            for (int r = 0; r < 4; r++) ddx[o + (h * HX + 4 * r) * LY + g * HY] = make_double2(re[r], im[r]);
        }
    __builtin_amdgcn_sched_barrier(0);
    mm_product<false, HY, RS, HX>(xi, my + MY, acc);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const dbl4 re = mm_inner_at(acc, h, g, 0) * sc.s[1][1], im = mm_inner_at(acc, h, g, 1) * sc.s[1][1];
#pragma unroll
            for (int r = 0; r < 4; r++) ddy[o + (h * HX + 4 * r) * LY + g * HY] = make_double2(re[r], im[r]);
        }
    __builtin_amdgcn_sched_barrier(0);
    mm_product<true, HX, RS, HY>(xo, mx, acc);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            lre[h][g] = mm_outer_at(acc, h, g, 0) * sc.s[0][0];
            lim[h][g] = mm_outer_at(acc, h, g, 1) * sc.s[0][0];
        }
    __builtin_amdgcn_sched_barrier(0);
    mm_product<false, HY, RS, HX>(xi, my, acc);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int g = 0; g < 2; g++) {
            const dbl4 re = lre[h][g] + mm_inner_at(acc, h, g, 0) * sc.s[1][0],
                       im = lim[h][g] + mm_inner_at(acc, h, g, 1) * sc.s[1][0];
#pragma unroll
            for (int r = 0; r < 4; r++) lap[o + (h * HX + 4 * r) * LY + g * HY] = make_double2(re[r], im[r]);
        }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static size_t rs_lds(const RsPlan &pl, int ntw) { return sizeof(double2) * (2 * (size_t)pl.npc + ntw); }

// 2D planes of the matrix-core form: tiles of 16 in both halves of an axis
static bool mm_plane(const tdw_ctx *c)
{
    return c->dim == 2 && (c->nx == 32 || c->nx == 64) && (c->ny == 32 || c->ny == 64);
}

int resident_setup(tdw_ctx *c)
{
    const int len[3] = {c->nx, c->ny, c->nz};
    const int dim = c->dim, ll = len[dim - 1], row = dim > 1 ? ll + 1 : 1;
    RsPlan pl;
    pl.dim = dim;
    pl.ll = ll;
    pl.mll = rs_magic(ll);
    const size_t npc = dim == 1 ? (size_t)c->nx : c->N / ll * row;
    const int ntw = len[0] + (dim > 1 ? len[1] : 0) + (dim > 2 ? len[2] : 0);
    // the state, the twiddles and the static reduction slots within a CU's LDS
    if (sizeof(double2) * (2 * npc + ntw) + 1024 > (size_t)c->max_lds) return 0;
    pl.npc = (int)npc;
    pl.inner = (int)(npc / c->nx);
    std::vector<double2> tw;
    std::vector<double> kk[3];
    int t0 = 0;
    for (int d = 0; d < dim; d++) {
        RsAxis &ax = pl.ax[d];
        const int L = len[d];
        bool ok;
        if (d == 0) ok = rs_axis(ax, L, pl.inner, 2 * pl.inner, pl.inner, pl.npc, t0);
        else if (d == dim - 1) ok = rs_axis(ax, L, 1, 2 * (pl.npc / row), 0, row, t0);
        else ok = rs_axis(ax, L, row, 2 * c->nx * row, row, c->ny * row, t0);
        if (!ok || (d == 0 && ax.nst < 1)) return 0;
        t0 += L;
        // -k^2 / N at each position of the spectrum
        for (int f : rs_order(ax)) {
            const double k = rs_k(f, L, c->Lphys[d]);
            kk[d].push_back(-(k * k) / (double)c->N);
        }
        for (int t = 0; t < L; t++) {
            const double an = 2.0 * M_PI * (double)t / (double)L;
            tw.push_back(make_double2(cos(an), -sin(an)));
        }
    }
    // tables: twiddles of all axes, then k_x^2, then the rest per point of an
    // x plane (pads included)
    std::vector<double> kt(kk[0]);
    for (int i = 0; i < pl.inner; i++) {
        const int z = i % row, y = i / row;
        double v = 0.0;
        if (dim == 2 && z < ll) v = kk[1][z];
        if (dim == 3 && z < ll) v = kk[1][y] + kk[2][z];
        kt.push_back(v);
    }
    // the halves of the second-derivative circulants in rs_mm's operand order
    if (mm_plane(c))
        for (int d = 0; d < 2; d++)
            for (int order = 2; order > 0; order--) pl.mm.s[d][2 - order] = mm_tables(len[d], c->Lphys[d], order, kt);
    const size_t btw = sizeof(double2) * tw.size(), bk = sizeof(double) * kt.size();
    TDW_HIP(hipMalloc(&c->d_rtab, btw + bk));
    TDW_HIP(hipMemcpy(c->d_rtab, tw.data(), btw, hipMemcpyHostToDevice));
    TDW_HIP(hipMemcpy((char *)c->d_rtab + btw, kt.data(), bk, hipMemcpyHostToDevice));
    c->rplan = new RsPlan(pl);
    return 0;
}

void resident_release(tdw_ctx *c)
{
    if (c->d_rtab) hipFree(c->d_rtab);
    c->d_rtab = nullptr;
    delete c->rplan;
    c->rplan = nullptr;
}

bool resident_supported(const tdw_ctx *c)
{
    return c->rplan && !varying_mass(c) && c->p.precision == TDW_FP64;
}

// The six passes move 19-20 S for the resident step's 15 S, in twice the
// launches, but stream them from a full chip.  A state that shares its CU's LDS
// with a second one is faster resident, as is one of a plane whose points are
// not whole waves (the passes' norm partials are then one per pencil instead of
// one per wave).  us per step of 4, 600, 4000 states, six passes and resident:
// 12^3 80, 182, 1009 and 75, 181, 884; 32 x 12 x 12 100, 439, 2601 and 111, 435,
// 2474; but 12 x 16 x 16 76, 270, 1654 and 97, 314, 1824; 8 x 24 x 24 80, 366, 2340
// and 116, 444, 2556; 16^3 82, 341, 2188 and 117, 426, 2484.
bool resident_pays3d(const tdw_ctx *c)
{
    if (!resident_supported(c)) return false;
    const size_t lds = rs_lds(*c->rplan, c->nx + c->ny + c->nz) + 1024;
    return 2 * lds <= (size_t)c->max_lds || c->S % 64 != 0;
}

// Threads of a workgroup: 16 waves per CU (four per SIMD, what 103 VGPRs of
// rs_h leave) over the workgroups that share it, as many as the LDS holds or
// as the states give; a whole number of waves, no more than one point per
// thread.  With 20 waves a second workgroup did not fit beside the first: 300
// states of 36 x 18 took 26 us against 15 for 128.
static int rs_threads(size_t lds, int n, int N)
{
    const int fit = lds ? (int)std::max<size_t>(1, (160 * 1024) / (lds + 256)) : 8;
    const int wg = std::min(std::min(fit, 16), std::max(1, (n + 255) / 256));
    const int nt = 64 * std::max(1, 16 / wg);
    return std::min(nt, (N + 63) / 64 * 64);
}

template <int CORR>
static int launch_h(tdw_ctx *c, int n, const double2 *in, double2 *out, const double2 *cc, const double *pots,
                    const double *sc, const double *use_e, double *e_out, double *e_out2, double *nrm_out,
                    double2 *lap = nullptr)
{
    const RsPlan &pl = *c->rplan;
    const int N = (int)c->N, ntw = pl.ax[0].L + (pl.dim > 1 ? pl.ax[1].L : 0) + (pl.dim > 2 ? pl.ax[2].L : 0);
    const double2 *tw = (const double2 *)c->d_rtab;
    const double *kx = (const double *)(tw + ntw);
    const double a0 = (c->p.scheme == TDW_AB3AM4) ? 9. / 24. : 251. / 720.;
    const RsH hp{c->p.mu_a, c->p.mu_b, dvol_norm(c), c->p.dt * a0, c->p.functional == TDW_BDG};
    const size_t lds = rs_lds(pl, ntw);
    const double *kt = c->dim < 3 ? c->d_kt : nullptr, *kt2 = c->dim == 1 ? c->d_kt + n : nullptr;
    TDW_TIMED(c, CORR ? "rs_hcorr" : "rs_h");
    if (mm_plane(c)) {
        const double *mx = kx + pl.ax[0].L + pl.inner;
        const double *my = mx + 2 * mm_doubles(c->nx);
        const dim3 g(n), b(128 * (c->nx / 32) * (c->ny / 32));
        const size_t sm = sizeof(double2) * 2 * (size_t)pl.npc;
#define RS_MM(LX, LY)                                                                                               \
    hipLaunchKernelGGL((rs_mm<LX, LY, CORR>), g, b, sm, c->stream, in, out, cc, pots, sc, kt, n, hp, mx, my, \
                       pl.mm.s[0][0], pl.mm.s[1][0], use_e, e_out, e_out2, nrm_out)
        if (c->nx == 32) {
            if (c->ny == 32) RS_MM(32, 32);
            else RS_MM(32, 64);
        } else {
            if (c->ny == 32) RS_MM(64, 32);
            else RS_MM(64, 64);
        }
#undef RS_MM
        return (int)hipGetLastError();
    }
    hipLaunchKernelGGL(rs_h<CORR>, dim3(n), dim3(rs_threads(lds, n, N)), lds, c->stream, in, out, cc, pots, sc, kt, kt2,
                       n, N, pl, hp, tw, ntw, kx, kx + pl.ax[0].L, use_e, e_out, e_out2, nrm_out, lap);
    return (int)hipGetLastError();
}

int plane_derivatives(tdw_ctx *c, int m, const double2 *in, double2 *ddx, double2 *ddy, double2 *lap, int *done)
{
    *done = c->rplan && mm_plane(c);
    if (!*done) return 0;
    const RsPlan &pl = *c->rplan;
    const double *tab = (const double *)((const double2 *)c->d_rtab + pl.ax[0].L + pl.ax[1].L) + pl.ax[0].L + pl.inner;
    const auto fn = c->nx == 32 ? (c->ny == 32 ? rs_deriv<32, 32> : rs_deriv<32, 64>)
                                : (c->ny == 32 ? rs_deriv<64, 32> : rs_deriv<64, 64>);
    TDW_TIMED(c, "rs_deriv");
    hipLaunchKernelGGL(fn, dim3((unsigned)m), dim3(64 * (c->nx / 32) * (c->ny / 32)), sizeof(double2) * (size_t)pl.npc,
                       c->stream, in, ddx, ddy, lap, tab, pl.mm);
    return (int)hipGetLastError();
}

int resident_h(tdw_ctx *c, int n, const double2 *in, double2 *out, const double *pots, double *qpe,
               const double *use_e)
{
    return launch_h<0>(c, n, in, out, nullptr, pots, nullptr, use_e, qpe, nullptr, nullptr);
}

int resident_h_only(tdw_ctx *c, int n, const double2 *in, double2 *out, const double *pots, const double2 *dotw,
                    double *d_dot)
{
    return launch_h<2>(c, n, in, out, dotw, pots, nullptr, nullptr, d_dot, nullptr, nullptr);
}

int resident_step(tdw_ctx *c, tdw_state *s, int it, int grad_last, tdw_tape_step *tape, tdw_complex *y_out,
                  double2 *cbuf, tdw_complex *f_next)
{
    // a gradient step's derivative arrays: refused before anything is written
    if (grad_last && (!s->lap || !s->ddx || (c->dim >= 2 && !s->ddy) || (c->dim >= 3 && !s->ddz))) return TDW_EINVAL;
    const int n = s->n, N = (int)c->N;
    const int h = c->p.scheme == TDW_AB3AM4 ? 3 : c->p.scheme == TDW_AB4AM5 ? 4 : 5;
    TDW_TRY(fused_state_vecs(c));
    double *qpe = s->qpe ? s->qpe : c->d_qpe;
    const double2 *y0 = (const double2 *)s->wf, *f[5];
    for (int j = 0; j < 5; j++) f[j] = (const double2 *)s->f[j];
    double2 *y = y_out ? (double2 *)y_out : (double2 *)s->wf;
    double2 *cc = cbuf ? cbuf : (double2 *)s->f[h - 1];
    const double dv = dvol_norm(c);
    {
        TDW_TIMED(c, "rs_pred");
        const int nt = rs_threads(0, n, N);
        double *nrm = tape ? tape->scal : nullptr;
#define RS_PRED(S)                                                                                                       hipLaunchKernelGGL(rs_pred<S>, dim3(n), dim3(nt), 0, c->stream, y0, y, cc, f[0], f[1], f[2], f[3], f[4], n, N,                        c->p.dt, dv, c->d_sp, c->d_s2, nrm)
        if (h == 3) RS_PRED(34);
        else if (h == 4) RS_PRED(45);
        else RS_PRED(55);
#undef RS_PRED
        TDW_HIP(hipGetLastError());
    }
    if (y_out) s->wf = y_out;
    TDW_TRY(densities(c, n, y, nullptr, nullptr, nullptr, nullptr, c->d_fbeta, c->d_s2, c->d_kt, c->d_cnt, s->dens, 0));
    TDW_TRY(step_potentials(c, it + 1, s->dens, s->pots));
    TDW_TRY(hkf_fields(c, s->pots, true));
    if (tape) TDW_TRY(tape_fields(c, s->dens, tape->dens_p, s->pots, tape->pots_p));
    const double *hp = h_view(c, it + 1, s->pots);
    if (!hp) return TDW_EINVAL;
    TDW_TRY(launch_h<1>(c, n, y, y, cc, hp, c->d_sp, nullptr, qpe, tape ? tape->scal + n : nullptr,
                        tape ? tape->scal + 2 * n : nullptr));
    // the corrected state: densities (a measurement step's with gradients,
    // tau and j), potentials, the new history entry
    if (grad_last && dens_grad_fused_supported(c)) {
        // 3D lattices with the in-pass gradient densities (as the six-pass
        // step does it: no derivative array is stored)
        TDW_TRY(dens_grad_fused(c, n, y, c->d_fbeta, nullptr, s->dens));
    } else {
        if (grad_last)
            TDW_TRY(derivatives(c, 2 * n, y, (double2 *)s->ddx, (double2 *)s->ddy, (double2 *)s->ddz,
                                (double2 *)s->lap));
        TDW_TRY(densities(c, n, y, (double2 *)s->ddx, (double2 *)s->ddy, (double2 *)s->ddz, (double2 *)s->lap,
                          c->d_fbeta, nullptr, c->d_kt, c->d_cnt, s->dens, grad_last));
    }
    if (grad_last) TDW_TRY(density_tau(c, s->dens));
    TDW_TRY(step_potentials(c, it + 1, s->dens, s->pots));
    TDW_TRY(hkf_fields(c, s->pots, true));
    if (tape) TDW_TRY(tape_fields(c, s->dens, tape->dens_c, s->pots, tape->pots_c));
    hp = h_view(c, it + 1, s->pots);
    if (!hp) return TDW_EINVAL;
    tdw_complex *tmp = f_next ? f_next : s->f[h - 1];
    for (int j = h - 1; j > 0; j--) s->f[j] = s->f[j - 1];
    s->f[0] = tmp;
    // 1D and 2D steps leave the Laplacian of y in lap (a gradient step's
    // derivatives have): rs_h stores it on its way (1 S, 1-2 % of a step).
    // rs_mm does not (64 x 64 x 1024: 552 -> 640 us a step with the store, and
    // the plane-wise step before it left H y_p there), so lap is scratch on
    // 32 x 32 and 64 x 64; planes of 32 x 64 points take a pass of their own.
    double2 *lap = c->dim < 3 && !grad_last ? (double2 *)s->lap : nullptr;
    if (lap && mm_plane(c)) {
        if (c->nx != c->ny) TDW_TRY(laplace(c, 2 * n, y, lap));
        lap = nullptr;
    }
    return launch_h<0>(c, n, y, (double2 *)s->f[0], nullptr, hp, nullptr, nullptr, qpe,
                       tape ? tape->scal + 3 * n : nullptr, nullptr, lap);
}

}  // namespace tdw
