// tdw_planemm.hpp -- spectral derivatives along the axes of a plane in LDS as
// products on v_mfma_f64_16x16x4.
//
// A spectral derivative along an axis of L points is a real circulant L x L
// matrix (even for the second, odd for the first with its Nyquist mode zero).
// With H = L / 2, p = x_j + x_{j + H} and m = x_j - x_{j + H} it falls into two
// H x H products: y_i = P p + M m, y_{i + H} = P p - M m.  A wave forms the
// outputs of a 16 x 16 tile of one quarter of the plane and of its three
// images, for either axis: along the outer axis the matrix is the A operand
// and the plane B, along the inner one the plane is A and the matrix B, and
// both leave the results in the same registers, D element r in row
// lane / 16 + 4 r, column lane % 16 of the tile.  So a plane is written to LDS
// once, is never overwritten, and what is formed from several derivatives at a
// point needs no exchange.
#pragma once
#include "tdw_device.hpp"
#include <cmath>
#include <vector>

namespace tdw {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// units of the tables of two axes (mm_tables): second derivative, then first
struct MmScale {
    double s[2][2];
};

// P and M products of a wave, [image along the other axis][re, im]
struct MmAcc {
    dbl4 P[2][2], Q[2][2];
};

__device__ __forceinline__ void mm_clear(MmAcc &a)
{
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int q = 0; q < 2; q++) a.P[g][q] = a.Q[g][q] = dbl4{0.0, 0.0, 0.0, 0.0};
}

// Products along the outer axis (rows, H = half its length, RS apart): x at
// row lane / 16 and the lane's column of the tile, whose image is G columns
// on; along the inner axis: x at row lane % 16 of the tile and column
// lane / 16, the tile's image G rows on.  One step of four columns of the
// matrix (mp, mm: its P and M elements).
template <bool OUTER, int H, int RS, int G>
__device__ __forceinline__ void mm_step(const double2 *x, int ks, double mp, double mm, MmAcc &a)
{
#pragma unroll
    for (int g = 0; g < 2; g++) {
        const double2 u = OUTER ? x[4 * ks * RS + g * G] : x[g * G * RS + 4 * ks];
        const double2 v = OUTER ? x[(4 * ks + H) * RS + g * G] : x[g * G * RS + 4 * ks + H];
        if constexpr (OUTER) {
            a.P[g][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(mp, u.x + v.x, a.P[g][0], 0, 0, 0);
            a.P[g][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(mp, u.y + v.y, a.P[g][1], 0, 0, 0);
            a.Q[g][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(mm, u.x - v.x, a.Q[g][0], 0, 0, 0);
            a.Q[g][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(mm, u.y - v.y, a.Q[g][1], 0, 0, 0);
        } else {
            a.P[g][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x + v.x, mp, a.P[g][0], 0, 0, 0);
            a.P[g][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y + v.y, mp, a.P[g][1], 0, 0, 0);
            a.Q[g][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x - v.x, mm, a.Q[g][0], 0, 0, 0);
            a.Q[g][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y - v.y, mm, a.Q[g][1], 0, 0, 0);
        }
    }
}

// M: the tile's tables (mm_tables) plus the lane
template <bool OUTER, int H, int RS, int G>
__device__ __forceinline__ void mm_product(const double2 *x, const double *M, MmAcc &a)
{
    mm_clear(a);
#pragma unroll 2
    for (int ks = 0; ks < H / 4; ks++) mm_step<OUTER, H, RS, G>(x, ks, M[ks * 128], M[ks * 128 + 64], a);
}

// the same with the tables in registers (mm_load)
template <int H> struct MmTab {
    double p[H / 4], m[H / 4];
};
template <int H>
__device__ __forceinline__ void mm_load(const double *M, MmTab<H> &t)
{
#pragma unroll
    for (int ks = 0; ks < H / 4; ks++) {
        t.p[ks] = M[ks * 128];
        t.m[ks] = M[ks * 128 + 64];
    }
}
template <bool OUTER, int H, int RS, int G>
__device__ __forceinline__ void mm_product(const double2 *x, const MmTab<H> &t, MmAcc &a)
{
    mm_clear(a);
#pragma unroll
    for (int ks = 0; ks < H / 4; ks++) mm_step<OUTER, H, RS, G>(x, ks, t.p[ks], t.m[ks], a);
}

// results at row image h, column image g: re (q 0) or im (q 1), four rows
__device__ __forceinline__ dbl4 mm_outer_at(const MmAcc &a, int h, int g, int q)
{
    return h ? a.P[g][q] - a.Q[g][q] : a.P[g][q] + a.Q[g][q];
}
__device__ __forceinline__ dbl4 mm_inner_at(const MmAcc &a, int h, int g, int q)
{
    return g ? a.P[h][q] - a.Q[h][q] : a.P[h][q] + a.Q[h][q];
}

// a tile's offsets, opaque to the compiler; the previous tile is done with
__device__ __forceinline__ bool mm_tile(int &i, int &j)
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+v"(i), "+v"(j));
    return true;
}

// v is formed here: a sum whose only use is a store that padding lanes skip is
// otherwise moved down to it, and its operands held until then
__device__ __forceinline__ void mm_keep(dbl4 &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void mm_keep(double &v) { asm volatile("" : "+v"(v)); }

static inline int mm_tiles(int L) { return (L / 2 + 15) / 16; }
// doubles of an axis' table
static inline size_t mm_doubles(int L) { return (size_t)mm_tiles(L) * (L / 8) * 128; }

// Scale of the entries of an axis' tables, below.  Rounding of the entries is
// an error of the operator, the same at every point and step, where an FFT's
// rounding averages out: with the entries rounded as they come, <psi|D psi> of
// smooth states of 64 points was off by 1.7e-16 where the FFT's was 6e-18, and
// the adjoint's gradient over 64 x 64 points by 1.7e-14 (relative, rms) where
// the FFT's was 1.1e-14.  Two or three of the entries are nearly all of it, so
// a scale is chosen with which those are nearly exact: of 4e9 values in [1, 2)
// (6e9 for 64 points) the one with the least rms rounding over all entries,
// 7 to 140 times below that of scale 1.
static inline double mm_unit(int L, int order)
{
    switch (L) {
    case 24: return order == 2 ? 0x1.e56c429bb0f6p+0 : 0x1.75dcd1ca8d826p+0;
    case 32: return order == 2 ? 0x1.c83dc8037e289p+0 : 0x1.552546a3a8664p+0;
    case 64: return order == 2 ? 0x1.e08d722a80c9p+0 : 0x1.37fab3f8c34dap+0;
    default: return 1.0;
    }
}

// The tables of an axis of L points (a multiple of 8) for the derivative of
// the given order, in units of (2 pi / len)^order mm_unit, which is returned
// for the products to be multiplied with: tile t, step ks, P then M, lane l:
// the element of row 16 t + l % 16 (0 past the half's rows) and column 4 ks +
// l / 16.  Summed in extended precision (in double the sums' own rounding gave
// the gradient an error of 1e-13).  Not scaled: the unit is 1.
static inline double mm_tables(int L, double len, int order, std::vector<double> &out, bool scaled = true)
{
    const int H = L / 2;
    const long double pi = 3.141592653589793238462643383L, k1 = 2.0L * pi / len;
    const long double dim = order == 2 ? k1 * k1 : k1, unit = scaled ? mm_unit(L, order) : 1.0L / dim;
    std::vector<long double> cs(L), sn(L), cc(L, 0.0L);
    for (int t = 0; t < L; t++) {
        cs[t] = cosl(2.0L * pi * t / L);
        sn[t] = sinl(2.0L * pi * t / L);
    }
    for (int x = 0; x < L; x++)
        for (int f = 0; f < L; f++) {
            const int m = f < H ? f : f - L;
            if (order == 2) cc[x] -= (long double)(m * m) / L * cs[(f * x) % L];
            else if (m != -H) cc[x] -= (long double)m / L * sn[(f * x) % L];
        }
    for (int t = 0; t < mm_tiles(L); t++)
        for (int ks = 0; ks < H / 4; ks++)
            for (int pm = 0; pm < 2; pm++)
                for (int l = 0; l < 64; l++) {
                    const int row = 16 * t + l % 16, x = row - (4 * ks + l / 16) + L;
                    const long double v = cc[x % L], h = cc[(x + H) % L];
                    out.push_back(row < H ? (double)(0.5L * (pm ? v - h : v + h) / unit) : 0.0);
                }
    return (double)(unit * dim);
}

}  // namespace tdw
