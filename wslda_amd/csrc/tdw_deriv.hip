// tdw_deriv.hip -- Laplacians and gradients of 3D arrays, lattices with
// compiled axis lengths.
//
// The run-time transforms of tdw_fft.hip (Stockham stages whose radix, span
// and strides are kernel arguments) spend their time on index arithmetic and
// on a ping-pong buffer: 1.9-2.2 TB/s on 48^3.  Here the lengths are
// template arguments and the transforms in place:
//   d_x       x pencils, one lane per pencil, FFT in registers: D_x;
//   d_x2      tiles of x pencils in LDS: D_x and the x derivative;
//   lap_yz    planes in LDS: in T + D_y + D_z, one 2D transform;
//   grad_yz   planes in LDS, per axis: T + D_y + D_z and the y, z derivatives.
// Streams and, in the gradient passes, the LDS stages bound them.  In us, run-
// time form and here: 48^3 x 400 arrays, D_x with gradient 1590 -> 419, the
// planes with gradients 3264 -> 1080; 16^3 x 2000, D_x 36 -> 14, planes 88 ->
// 24, with gradients 154 -> 71 and 444 -> 127.
#include "tdw_axis.hpp"
#include "tdw_fft.hpp"
#include "tdw_internal.hpp"

namespace tdw {

static constexpr int DT = 256;

// T = D_x in; S = points of an x plane, m arrays of LX x S
template <int LX>
__global__ void __launch_bounds__(DT)
d_x(const double2 *in, double2 *T, int m, int S, double kscale)
{
    const long P = (long)blockIdx.x * DT + threadIdx.x;
    if (P >= (long)m * S) return;
    const long a = P / S, base = a * LX * S + (P - a * S);
    double2 r[LX];
#pragma unroll
    for (int i = 0; i < LX; i++) r[i] = in[base + (long)i * S];
    rf::fft<LX, -1, double2>(r);
#pragma unroll
    for (int i = 0; i < LX; i++) {
        const int k = (i < LX / 2) ? i : i - LX;
        r[i] = r[i] * (-kscale * (double)(k * k));
    }
    rf::fft<LX, +1, double2>(r);
#pragma unroll
    for (int i = 0; i < LX; i++) T[base + (long)i * S] = r[i];
}

// T = D_x in and ddx = d_x in; a workgroup takes PX neighbouring pencils
// (pencil q, point i at q + i PX in LDS).  k1 = 2 pi / (Lx LX), k2 = (2 pi /
// Lx)^2 / LX.
template <int LX, int PX>
__global__ void __launch_bounds__(DT)
d_x2(const double2 *in, double2 *T, double2 *ddx, int S, const double2 *__restrict__ twg, double k1, double k2)
{
    constexpr int E = LX * PX, KM = (E + DT - 1) / DT;
    __shared__ double2 A[E], B[E], tw[LX];
    const int tid = threadIdx.x, nb = (S + PX - 1) / PX;
    for (int k = tid; k < LX; k += DT) tw[k] = twg[k];
    const long a = blockIdx.x / nb;
    const int j0 = (int)(blockIdx.x - a * nb) * PX;
    const long base = a * LX * S + j0;
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const int e = tid + k * DT;
        if (E % DT && e >= E) continue;
        const int i = e / PX, q = e - i * PX;
        A[e] = j0 + q < S ? in[base + (long)i * S + q] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    axis_d12<LX, PX, PX, 0, 1, PX, DT, true>(A, B, tw, tid, k1, k2);
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const int e = tid + k * DT;
        if (E % DT && e >= E) continue;
        const int i = e / PX, q = e - i * PX;
        if (j0 + q >= S) continue;
        T[base + (long)i * S + q] = A[e];
        ddx[base + (long)i * S + q] = B[e];
    }
}

// NP planes of LY x LZ points per workgroup, rows LZ + 1 apart in LDS
template <int LY, int LZ, int NP> struct Planes {
    static constexpr int E = LY * LZ, EP = LY * (LZ + 1), TOT = NP * E;
    static __device__ __forceinline__ int slot(int e)
    {
        const int p = NP == 1 ? 0 : e / E, r = e - p * E;
        return p * EP + (r / LZ) * (LZ + 1) + r % LZ;
    }
};

// out = T + D_y in + D_z in (T null: without); np planes in all
template <int LY, int LZ, int NP, int NT>
__global__ void __launch_bounds__(NT)
lap_yz(const double2 *in, const double2 *T, double2 *out, long np, const double2 *__restrict__ twyg,
       const double2 *__restrict__ twzg, double kys, double kzs)
{
    typedef Planes<LY, LZ, NP> P;
    __shared__ double2 A[NP * P::EP], twy[LY], twz[LZ];
    __shared__ double zt[LZ];
    const int tid = threadIdx.x;
    const long p0 = (long)blockIdx.x * NP, g = p0 * P::E;
    const int tot = np - p0 >= NP ? P::TOT : (int)(np - p0) * P::E;
    for (int k = tid; k < LY; k += NT) twy[k] = twyg[k];
    for (int k = tid; k < LZ; k += NT) {
        twz[k] = twzg[k];
        const int m = axis_freq<LZ>(k);
        zt[k] = kzs / LY * (double)(m * m);
    }
#pragma unroll
    for (int e = tid; e < P::TOT; e += NT) A[P::slot(e)] = e < tot ? in[g + e] : make_double2(0.0, 0.0);
    __syncthreads();
    dft_axis<LZ, NP * LY, LY, P::EP, LZ + 1, 1, NT, 1>(A, twz, tid, KsMul{0.0});
    dft_axis<LY, NP * LZ, LZ, P::EP, 1, LZ + 1, NT, 0>(A, twy, tid, YZMul{kys / LZ, zt, LZ});
    dft_axis<LZ, NP * LY, LY, P::EP, LZ + 1, 1, NT, 2>(A, twz, tid, KsMul{0.0});
#pragma unroll
    for (int e = tid; e < P::TOT; e += NT)
        if (e < tot) out[g + e] = T ? T[g + e] + A[P::slot(e)] : A[P::slot(e)];
}

// out = T + D_y in + D_z in, ddy, ddz
template <int LY, int LZ, int NP, int NT>
__global__ void __launch_bounds__(NT)
grad_yz(const double2 *in, const double2 *T, double2 *out, double2 *ddy, double2 *ddz, long np,
        const double2 *__restrict__ twyg, const double2 *__restrict__ twzg, double k1y, double k2y, double k1z,
        double k2z)
{
    typedef Planes<LY, LZ, NP> P;
    constexpr int KM = (P::TOT + NT - 1) / NT;
    extern __shared__ double2 g_lds[];
    __shared__ double2 twy[LY], twz[LZ];
    double2 *A = g_lds, *B = A + NP * P::EP;
    const int tid = threadIdx.x;
    const long p0 = (long)blockIdx.x * NP, g = p0 * P::E;
    const int tot = np - p0 >= NP ? P::TOT : (int)(np - p0) * P::E;
    for (int k = tid; k < LY; k += NT) twy[k] = twyg[k];
    for (int k = tid; k < LZ; k += NT) twz[k] = twzg[k];
    double2 X[KM], O[KM];
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const int e = tid + k * NT;
        X[k] = e < tot ? in[g + e] : make_double2(0.0, 0.0);
        O[k] = e < tot ? T[g + e] : make_double2(0.0, 0.0);
        if (e < P::TOT) A[P::slot(e)] = X[k];
    }
    __syncthreads();
    axis_d12<LZ, NP * LY, LY, P::EP, LZ + 1, 1, NT, true>(A, B, twz, tid, k1z, k2z);
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const int e = tid + k * NT;
        if (e >= P::TOT) continue;
        const int pe = P::slot(e);
        O[k] = O[k] + A[pe];
        if (e < tot) ddz[g + e] = B[pe];
        A[pe] = X[k];
    }
    __syncthreads();
    axis_d12<LY, NP * LZ, LZ, P::EP, 1, LZ + 1, NT, true>(A, B, twy, tid, k1y, k2y);
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const int e = tid + k * NT;
        if (e >= tot) continue;
        const int pe = P::slot(e);
        out[g + e] = O[k] + A[pe];
        ddy[g + e] = B[pe];
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static double k1f(const tdw_ctx *c, int d, int L) { return 2.0 * M_PI / c->Lphys[d] / L; }
static double k2f(const tdw_ctx *c, int d, int L) { return pow(2.0 * M_PI / c->Lphys[d], 2) / L; }

template <int LX> static int run_dx(tdw_ctx *c, int m, const double2 *in, double2 *T)
{
    const long tot = (long)m * c->S;
    hipLaunchKernelGGL(d_x<LX>, dim3((unsigned)((tot + DT - 1) / DT)), dim3(DT), 0, c->stream, in, T, m, c->S,
                       k2f(c, 0, LX));
    return (int)hipGetLastError();
}
template <int LX, int PX> static int run_dx2(tdw_ctx *c, int m, const double2 *in, double2 *T, double2 *ddx)
{
    const long nb = (c->S + PX - 1) / PX;
    hipLaunchKernelGGL((d_x2<LX, PX>), dim3((unsigned)(m * nb)), dim3(DT), 0, c->stream, in, T, ddx, c->S, c->d_tw[0],
                       k1f(c, 0, LX), k2f(c, 0, LX));
    return (int)hipGetLastError();
}

int deriv3d_outer(tdw_ctx *c, int m, const double2 *in, double2 *T, double2 *ddx, int mode, int *done)
{
    *done = 1;
    if (c->dim == 3 && mode == 0) {
        switch (c->nx) {
        case 8: return run_dx<8>(c, m, in, T);
        case 12: return run_dx<12>(c, m, in, T);
        case 16: return run_dx<16>(c, m, in, T);
        case 18: return run_dx<18>(c, m, in, T);
        case 24: return run_dx<24>(c, m, in, T);
        case 32: return run_dx<32>(c, m, in, T);
        case 36: return run_dx<36>(c, m, in, T);
        case 48: return run_dx<48>(c, m, in, T);
        default: break;
        }
    } else if (c->dim == 3) {
        switch (c->nx) {
        case 12: return run_dx2<12, 64>(c, m, in, T, ddx);
        case 16: return run_dx2<16, 64>(c, m, in, T, ddx);
        case 18: return run_dx2<18, 32>(c, m, in, T, ddx);
        case 24: return run_dx2<24, 32>(c, m, in, T, ddx);
        case 32: return run_dx2<32, 32>(c, m, in, T, ddx);
        case 36: return run_dx2<36, 16>(c, m, in, T, ddx);
        case 48: return run_dx2<48, 16>(c, m, in, T, ddx);
        default: break;
        }
    }
    *done = 0;
    return 0;
}

template <int LY, int LZ, int NP, int NT, int NTG>
static int run_yz(tdw_ctx *c, int m, const double2 *in, const double2 *T, double2 *out, double2 *ddy, double2 *ddz,
                  int mode)
{
    const long np = (long)m * c->nx;
    const dim3 g((unsigned)((np + NP - 1) / NP));
    TDW_TIMED(c, mode ? "fft_inner_deriv" : "fft_inner");
    if (mode == 0)
        hipLaunchKernelGGL((lap_yz<LY, LZ, NP, NT>), g, dim3(NT), 0, c->stream, in, T, out, np, c->d_tw[1], c->d_tw[2],
                           k2f(c, 1, LY), k2f(c, 2, LZ));
    else
        hipLaunchKernelGGL((grad_yz<LY, LZ, NP, NTG>), g, dim3(NTG), sizeof(double2) * 2 * NP * LY * (LZ + 1),
                           c->stream, in, T, out, ddy, ddz, np, c->d_tw[1], c->d_tw[2], k1f(c, 1, LY), k2f(c, 1, LY),
                           k1f(c, 2, LZ), k2f(c, 2, LZ));
    return (int)hipGetLastError();
}

int deriv3d_inner(tdw_ctx *c, int m, const double2 *in, const double2 *T, double2 *out, double2 *ddy, double2 *ddz,
                  int mode, int *done)
{
    *done = 1;
    const int ny = c->ny, nz = c->nz;
    if (c->dim == 3 && (mode == 0 || T)) {
        // planes per workgroup: enough points for two to four waves
        if (ny == 12 && nz == 12) return run_yz<12, 12, 4, 192, 192>(c, m, in, T, out, ddy, ddz, mode);
        if (ny == 16 && nz == 16) return run_yz<16, 16, 4, 256, 256>(c, m, in, T, out, ddy, ddz, mode);
        if (ny == 18 && nz == 18) return run_yz<18, 18, 2, 192, 192>(c, m, in, T, out, ddy, ddz, mode);
        if (ny == 24 && nz == 24) return run_yz<24, 24, 2, 192, 384>(c, m, in, T, out, ddy, ddz, mode);
        if (ny == 32 && nz == 32) return run_yz<32, 32, 2, 512, 512>(c, m, in, T, out, ddy, ddz, mode);
        if (ny == 36 && nz == 36) return run_yz<36, 36, 1, 256, 448>(c, m, in, T, out, ddy, ddz, mode);
        if (ny == 48 && nz == 48) return run_yz<48, 48, 1, 384, 384>(c, m, in, T, out, ddy, ddz, mode);
        if (ny == 32 && nz == 96) return run_yz<32, 96, 1, 512, 768>(c, m, in, T, out, ddy, ddz, mode);
    }
    *done = 0;
    return 0;
}

}  // namespace tdw
