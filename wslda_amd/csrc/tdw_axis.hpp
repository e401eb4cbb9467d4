// tdw_axis.hpp -- transforms and derivatives along one axis of pencils held
// in LDS, of compile-time length L = R1 * R2.
#pragma once
#include "tdw_device.hpp"
#include "tdw_regfft.hpp"

namespace tdw {

// In-place transforms along one axis of P pencils held in LDS, for
// L = R1*R2: with n = n1*R2 + n2 and f = k1 + R1*k2,
//   X[f] = sum_n2 W_R2^{n2 k2} W_L^{n2 k1} sum_n1 x[n1 R2 + n2] W_R1^{n1 k1},
// stage 1 (per n2): R1-point DFT over n1, twiddle W_L^{n2 k1}, stored at k1*R2 + n2;
// stage 2 (per k1): R2-point DFT over n2 -> X[k1 + R1 k2], times mul(m(f), q)
//   for pencil q, inverse R2-point DFT and the conjugate twiddle, stored at
//   k1*R2 + n2;
// stage 3 (per n2): inverse R1-point DFT over k1, stored at n1*R2 + n2.
// MODE 0 runs all three (with mul = -ks m^2 the second derivative); MODE 1
// stops after the forward R2-point DFT and leaves X[k1 + R1 k2] at position
// k1*R2 + k2; MODE 2 starts from that layout and runs the inverse half.
// Every stage reads and writes the same positions, so one buffer suffices.
// Consecutive lanes take consecutive pencils: with pencils one element or one
// padded row apart, a wave's LDS accesses fall in distinct banks.

// frequency index m(f) in (-L/2, L/2] of the DFT output at position p (MODE 1 layout)
template <int L> __host__ __device__ constexpr int axis_freq(int p)
{
    constexpr int R1 = rf::fac2<L>::R1, R2 = rf::fac2<L>::R2;
    const int f = R2 > 1 ? p / R2 + R1 * (p % R2) : p;
    return f < L / 2 ? f : f - L;
}

struct KsMul {
    double ks;
    __device__ double operator()(int m, int) const { return -ks * (double)(m * m); }
};

template <int L, int P, int QD, int QH, int QL, int IS, int NT, int MODE, typename C, typename MUL>
__device__ __forceinline__ void dft_axis(C *A, const C *tw, int tid, MUL mul)
{
    typedef decltype(C().x) Rl;
    constexpr int R1 = rf::fac2<L>::R1, R2 = rf::fac2<L>::R2;
    // stage 1
    if constexpr (R2 > 1 && MODE != 2) {
        for (int b = tid; b < P * R2; b += NT) {
            const int n2 = b / P, q = b - n2 * P;
            C *pa = A + (q / QD) * QH + (q % QD) * QL;
            C v[R1];
#pragma unroll
            for (int n1 = 0; n1 < R1; n1++) v[n1] = pa[(n1 * R2 + n2) * IS];
            rf::dft_inplace<R1, -1, C>(v);
#pragma unroll
            for (int k1 = 1; k1 < R1; k1++) v[k1] = cmul(v[k1], tw[(n2 * k1) % L]);
#pragma unroll
            for (int k1 = 0; k1 < R1; k1++) pa[(k1 * R2 + n2) * IS] = v[k1];
        }
        __syncthreads();
    }
    // stage 2 (for R2 == 1 the whole transform)
    for (int b = tid; b < P * R1; b += NT) {
        const int k1 = b / P, q = b - k1 * P;
        C *pa = A + (q / QD) * QH + (q % QD) * QL;
        if constexpr (R2 > 1) {
            C v[R2];
#pragma unroll
            for (int n2 = 0; n2 < R2; n2++) v[n2] = pa[(k1 * R2 + n2) * IS];
            if constexpr (MODE != 2) {
                rf::dft_inplace<R2, -1, C>(v);
                if constexpr (MODE == 1) {
#pragma unroll
                    for (int k2 = 0; k2 < R2; k2++) pa[(k1 * R2 + k2) * IS] = v[k2];
                    continue;
                }
#pragma unroll
                for (int k2 = 0; k2 < R2; k2++) {
                    const int f = k1 + R1 * k2;
                    const int m = (f < L / 2) ? f : f - L;
                    v[k2] = v[k2] * (Rl)mul(m, q);
                }
            }
            rf::dft_inplace<R2, +1, C>(v);
#pragma unroll
            for (int n2 = 0; n2 < R2; n2++) {
                C w = tw[(n2 * k1) % L];
                w.y = -w.y;
                pa[(k1 * R2 + n2) * IS] = n2 == 0 ? v[n2] : cmul(v[n2], w);
            }
        } else if (k1 == 0) {
            // R2 == 1: one group per pencil holds the whole pencil
            C v[R1];
#pragma unroll
            for (int n = 0; n < R1; n++) v[n] = pa[n * IS];
            if constexpr (MODE != 2) {
                rf::dft_inplace<R1, -1, C>(v);
                if constexpr (MODE == 0) {
#pragma unroll
                    for (int f = 0; f < R1; f++) {
                        const int m = (f < L / 2) ? f : f - L;
                        v[f] = v[f] * (Rl)mul(m, q);
                    }
                }
            }
            if constexpr (MODE != 1) rf::dft_inplace<R1, +1, C>(v);
#pragma unroll
            for (int n = 0; n < R1; n++) pa[n * IS] = v[n];
        }
    }
    __syncthreads();
    // stage 3
    if constexpr (R2 > 1 && MODE != 1) {
        for (int b = tid; b < P * R2; b += NT) {
            const int n2 = b / P, q = b - n2 * P;
            C *pa = A + (q / QD) * QH + (q % QD) * QL;
            C v[R1];
#pragma unroll
            for (int k1 = 0; k1 < R1; k1++) v[k1] = pa[(k1 * R2 + n2) * IS];
            rf::dft_inplace<R1, +1, C>(v);
#pragma unroll
            for (int n1 = 0; n1 < R1; n1++) pa[(n1 * R2 + n2) * IS] = v[n1];
        }
        __syncthreads();
    }
}

// second derivative along one axis, in place (ks = (2 pi / L_phys)^2 / L)
template <int L, int P, int QD, int QH, int QL, int IS, int NT, typename C>
__device__ __forceinline__ void lap_axis(C *A, const C *tw, int tid, double ks)
{
    dft_axis<L, P, QD, QH, QL, IS, NT, 0>(A, tw, tid, KsMul{ks});
}

// multiplier of the y pass of a 2D transform: -(k_y^2 + k_z^2) / (LY LZ),
// with the z part per position of the z-transformed row in zt
struct YZMul {
    double ky;
    const double *zt;
    int lz;
    __device__ double operator()(int m, int q) const { return -(ky * (double)(m * m) + zt[q % lz]); }
};

// ---------------------------------------------------------------------------
// In-place derivatives along one axis of P pencils held in LDS (L = R1*R2,
// n = n1*R2 + n2, frequency f = k1 + R1*k2 at position k1*R2 + n2 between
// the stages; consecutive lanes take consecutive pencils, so layouts whose
// pencils start one element apart, or a padded row apart, are read without
// LDS bank conflicts).  A receives the second derivative (factor -k2s m^2, the
// inverse transform's 1/L folded into k2s); with GRAD, B (same layout)
// receives the first derivative (factor i k1s m, Nyquist mode zero).  Pencil q starts at
// (q / QD) * QH + (q % QD) * QL, element stride IS.
// ---------------------------------------------------------------------------
template <int L, int P, int QD, int QH, int QL, int IS, int NT, bool GRAD, typename C = double2>
__device__ __forceinline__ void axis_d12(C *A, C *B, const C *tw, int tid, double k1s, double k2s)
{
    typedef decltype(C().x) R;
    constexpr int R1 = rf::fac2<L>::R1, R2 = rf::fac2<L>::R2;
    static_assert(R2 > 1, "axis_d12 needs L = R1 * R2 with R2 > 1");
    // stage 1: R1-point DFTs over n1, twiddle W_L^{n2 k1}
    for (int b = tid; b < P * R2; b += NT) {
        const int n2 = b / P, q = b - n2 * P;
        C *pa = A + (q / QD) * QH + (q % QD) * QL;
        C v[R1];
#pragma unroll
        for (int n1 = 0; n1 < R1; n1++) v[n1] = pa[(n1 * R2 + n2) * IS];
        rf::dft_inplace<R1, -1, C>(v);
#pragma unroll
        for (int k1 = 1; k1 < R1; k1++) v[k1] = cmul(v[k1], tw[(n2 * k1) % L]);
#pragma unroll
        for (int k1 = 0; k1 < R1; k1++) pa[(k1 * R2 + n2) * IS] = v[k1];
    }
    __syncthreads();
    // stage 2: R2-point DFTs over n2, the derivative factors, inverse R2 DFTs
    for (int b = tid; b < P * R1; b += NT) {
        const int k1 = b / P, q = b - k1 * P;
        const int off = (q / QD) * QH + (q % QD) * QL;
        C *pa = A + off;
        C v[R2], g[R2];
#pragma unroll
        for (int n2 = 0; n2 < R2; n2++) v[n2] = pa[(k1 * R2 + n2) * IS];
        rf::dft_inplace<R2, -1, C>(v);
#pragma unroll
        for (int k2 = 0; k2 < R2; k2++) {
            const int f = k1 + R1 * k2;
            const int m = (f < L / 2) ? f : f - L;
            if constexpr (GRAD) g[k2] = (f == L / 2) ? cvt<C>(make_double2(0.0, 0.0)) : imul(v[k2], (R)(k1s * (double)m));
            v[k2] = v[k2] * (R)(-k2s * (double)(m * m));
        }
        rf::dft_inplace<R2, +1, C>(v);
        if constexpr (GRAD) rf::dft_inplace<R2, +1, C>(g);
#pragma unroll
        for (int n2 = 0; n2 < R2; n2++) {
            C wc = tw[(n2 * k1) % L];
            wc.y = -wc.y;
            pa[(k1 * R2 + n2) * IS] = n2 == 0 ? v[n2] : cmul(v[n2], wc);
            if constexpr (GRAD) B[off + (k1 * R2 + n2) * IS] = n2 == 0 ? g[n2] : cmul(g[n2], wc);
        }
    }
    __syncthreads();
    // stage 3: inverse R1-point DFTs over k1
    for (int b = tid; b < P * R2; b += NT) {
        const int n2 = b / P, q = b - n2 * P;
        const int off = (q / QD) * QH + (q % QD) * QL;
        C v[R1];
        C *pa = A + off;
#pragma unroll
        for (int k1 = 0; k1 < R1; k1++) v[k1] = pa[(k1 * R2 + n2) * IS];
        rf::dft_inplace<R1, +1, C>(v);
#pragma unroll
        for (int n1 = 0; n1 < R1; n1++) pa[(n1 * R2 + n2) * IS] = v[n1];
        if constexpr (GRAD) {
            C *pb = B + off;
#pragma unroll
            for (int k1 = 0; k1 < R1; k1++) v[k1] = pb[(k1 * R2 + n2) * IS];
            rf::dft_inplace<R1, +1, C>(v);
#pragma unroll
            for (int n1 = 0; n1 < R1; n1++) pb[(n1 * R2 + n2) * IS] = v[n1];
        }
    }
    __syncthreads();
}

}  // namespace tdw
