// tdw_functional_ad.hpp -- the pointwise SLDA functional over a generic
// scalar (double or Dual<K>), for the adjoint's Jacobian of the potentials.
//
// Same formulas, constants and branch decisions as tdw_functional.hpp
// (pca_edf.h:17-352, tdwslda_functionals.h:47-306, FAST constant-mass mode);
// branches are decided on values, so the dual result is the derivative of
// the branch the forward step took.
#pragma once
#include "tdw_dual.hpp"
#include "tdw_functional.hpp"

namespace tdw {
namespace ad {

template <typename R> struct S;
template <> struct S<double> {
    static __host__ __device__ __forceinline__ double c(double v) { return v; }
};
template <int K> struct S<Dual<K>> {
    static __host__ __device__ __forceinline__ Dual<K> c(double v) { return dconst<K>(v); }
};

template <typename R> __host__ __device__ __forceinline__ R p_reg(const FParams &f, const R &n)
{
    if (val(n) <= f.p_nmin) return S<R>::c(0.0);
    if (val(n) >= f.p_nmax) return S<R>::c(1.0);
    return 0.5 + 0.5 * ad_tanh(TDW_P_ALPHA * ad_tan((M_PI * (n - f.p_nmin)) / (f.p_nmax - f.p_nmin) - M_PI / 2.0));
}
template <typename R> __host__ __device__ __forceinline__ R der_p_reg(const FParams &f, const R &n)
{
    if (val(n) <= f.p_nmin || val(n) >= f.p_nmax) return S<R>::c(0.0);
    R a = (M_PI * (n - f.p_nmin)) / (f.p_nmax - f.p_nmin) - M_PI / 2.0;
    R q = ad_cosh(TDW_P_ALPHA * ad_tan(a)) * ad_cos(a);
    return 0.5 * TDW_P_ALPHA * M_PI / (q * q) / (f.p_nmax - f.p_nmin);
}
template <typename R> __host__ __device__ __forceinline__ R polar(const FParams &f, const R &na, const R &nb)
{
    R pr = p_reg(f, na + nb);
    if (val(pr) == 0.0) return S<R>::c(0.0);
    return pr * (na - nb) / (na + nb);
}
template <typename R>
__host__ __device__ __forceinline__ R der_pol(const FParams &f, const R &na, const R &nb, int wrt_b)
{
    R np = na + nb, pr = p_reg(f, np), dpr = der_p_reg(f, np);
    R r = S<R>::c(0.0);
    if (val(pr) != 0.0) r = r + pr * (wrt_b ? (-2.0 * na) : (2.0 * nb)) / (np * np);
    if (val(dpr) != 0.0) r = r + dpr * (na - nb) / np;
    return r;
}
template <typename R> __host__ __device__ __forceinline__ R funG(const R &p) { return TDW_G0 + TDW_G1 * p * p; }

template <typename R>
__host__ __device__ __forceinline__ R der_funD(const FParams &f, const R &na, const R &nb, int wrt_b)
{
    R p = polar(f, na, nb);
    R base = funG(p) - TDW_A0 * ad_pow((1.0 + p) / 2.0, 5.0 / 3.0) - TDW_A0 * ad_pow((1.0 - p) / 2.0, 5.0 / 3.0);
    R dpol = der_pol(f, na, nb, wrt_b);
    return (1.0 / 2.0) * ad_pow(6.0 * M_PI * M_PI * (na + nb), 2.0 / 3.0) * base +
           (1.0 / (20.0 * M_PI * M_PI)) * ad_pow(6.0 * M_PI * M_PI * (na + nb), 5.0 / 3.0) *
               (2.0 * TDW_G1 * p - (5.0 / 6.0) * TDW_A0 * ad_pow((1.0 + p) / 2.0, 2.0 / 3.0) +
                (5.0 / 6.0) * TDW_A0 * ad_pow((1.0 - p) / 2.0, 2.0 / 3.0)) *
               dpol;
}
template <typename R> __host__ __device__ __forceinline__ R tildeC(const FParams &f, const R &na, const R &nb)
{
    return TDW_A0 * ad_pow(na + nb + f.denseps, 1.0 / 3.0) / (TDW_GAMMA0 * 1.0);
}
template <typename R> __host__ __device__ __forceinline__ R der_tildeC(const FParams &f, const R &na, const R &nb)
{
    return ((1.0 / 3.0) * TDW_A0 * ad_pow(na + nb + f.denseps, -2.0 / 3.0)) / (TDW_GAMMA0 * 1.0);
}

template <typename R> __host__ __device__ __forceinline__ Cx<R> csqrt_real(const R &x)
{
    if (val(x) >= 0.0) return cx<R>(ad_sqrt(x), S<R>::c(0.0));
    return cx<R>(S<R>::c(0.0), ad_sqrt(-x));
}

// the real branch above the band bottom as in tdw_functional.hpp; real: wz
// and p0 are real with zero tangents in their imaginary parts
template <typename R>
__host__ __device__ __forceinline__ bool reg_wz(const FParams &f, const R &t7, double alph_plus, Cx<R> &wz, Cx<R> &p0)
{
    const R z = S<R>::c(0.0), kc2 = (2.0 / alph_plus) * (f.ec + t7), p02 = (2.0 / alph_plus) * t7;
    if (val(t7) >= 0.0 && (f.cubic || val(kc2) >= 0.0)) {
        const R p = ad_sqrt(p02), k = f.cubic ? S<R>::c(M_PI / f.dx) : ad_sqrt(kc2);
        if (val(k) > val(p)) {
            p0 = cx<R>(p, z);
            wz = cx<R>((k - f.R1 * (p * ad_log((k + p) / (k - p)))) * f.R0, z);
            return true;
        }
    }
    p0 = csqrt_real(p02);
    Cx<R> kc = f.cubic ? cx<R>(S<R>::c(M_PI / f.dx), z) : csqrt_real(kc2);
    Cx<R> w = cxlog(cxdiv(kc + p0, kc - p0));
    if (val(w.y) < 0.) w.y = w.y + 2. * M_PI;
    wz = cxscale(kc - cxscale(cxmul(p0, w), f.R1), f.R0);
    return false;
}

// (see mf_corr of tdw_functional.hpp for the form)
template <typename R>
__host__ __device__ __forceinline__ R mf_corr(const FParams &f, const R &p0x, const R &g, const R &lkF, const R &n,
                                              double alph_plus)
{
    R b = p0x / (lkF + 1.0e-12);
    R lx = b * lkF * (f.dx / M_PI);
    if (val(g) < -1.0e-10 && val(lx) > 1.0e-10) {
        R q = 1.0 / ((1.0 - lx) * (1.0 + lx));
        return (-f.R0 * f.R1 / (3. * alph_plus)) * (lkF / n) * b *
               (ad_log((1.0 + lx) * (1.0 + lx) * q) + 2.0 * (lx * q));
    }
    return S<R>::c(0.0);
}

// Transpose of the SLDA potentials at one point: l = dL/d(Va, Vb, Re delta,
// Im delta) to gr = dL/d(na, nb, Re nu, Im nu, ua, ub, Va_prev, Vb_prev).
//
// The 15-step mixing loop reaches its inputs through four of them only: c =
// Va_const + Vb_const, n = na + nb, |nu|^2 and s0 = Va_prev + Vb_prev.  Both
// potentials receive the same X(Va + Vb) per step, so with Y the mixed sum of
// the X, Va = A Va_prev + (1 - A) Va_const + Y with A = (1 - mix)^15, and four
// tangents of Va + Vb, Y and g carry the loop instead of eight of each
// variable.  The loop's values are those of the potentials' own update, so it
// takes the branches that update took.
__host__ __device__ __forceinline__ void slda_vjp(const FParams &f, double na, double nb, double nux, double nuy,
                                                  double ua, double ub, double Va, double Vb, const double (&l)[4],
                                                  double (&gr)[8])
{
    typedef Dual<4> D;
    const double alph_plus = TDW_A0;
    const Dual<2> ea = dvar<2>(na, 0), eb = dvar<2>(nb, 1);
    const Dual<2> fa = der_funD(f, ea, eb, 0), fb = der_funD(f, ea, eb, 1);
    const double Va_const = ua + fa.v, Vb_const = ub + fb.v;
    // tangents: 0 c, 1 n, 2 |nu|^2, 3 s0
    const D dn = dvar<4>(na + nb, 1), z = dconst<4>(0.0);
    const D t3 = der_tildeC(f, dn, z) / alph_plus;
    const D t5 = tildeC(f, dn, z);
    D lkF = z;
    if (f.mf) lkF = ad_pow(3.0 * M_PI * M_PI * dn, 1.0 / 3.0);
    const D nu2 = dvar<4>(nux * nux + nuy * nuy, 2);
    D g = z, Y = z;
    double sd[4] = {0.0, 0.0, 0.0, 1.0};   // of Va + Vb
    double A = 1.0;
    for (int k = 0; k < TDW_UD_SCITERS; k++) {
        D t7;
        t7.v = (f.mu_a - Va + f.mu_b - Vb) / 2.0;
#pragma unroll
        for (int j = 0; j < 4; j++) t7.d[j] = -0.5 * sd[j];
        Cx<D> wz, p0;
        const bool real = reg_wz(f, t7, alph_plus, wz, p0);
        const D d = t5 - wz.x;
        g = real ? alph_plus / d : alph_plus * d / (d * d + wz.y * wz.y);
        const D t7b = (g * g) * nu2;
        D X = -(t3 * t7b);
        if (f.mf) X = X + mf_corr(f, p0.x, g, lkF, dn, alph_plus) * t7b;
        Va = TDW_UD_MIX * (Va_const + X.v) + (1.0 - TDW_UD_MIX) * Va;
        Vb = TDW_UD_MIX * (Vb_const + X.v) + (1.0 - TDW_UD_MIX) * Vb;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            sd[j] = TDW_UD_MIX * (2.0 * X.d[j] + (j == 0 ? 1.0 : 0.0)) + (1.0 - TDW_UD_MIX) * sd[j];
            Y.d[j] = TDW_UD_MIX * X.d[j] + (1.0 - TDW_UD_MIX) * Y.d[j];
        }
        A *= 1.0 - TDW_UD_MIX;
    }
    // delta = -nu g
    const double lY = l[0] + l[1], lg = -(l[2] * nux + l[3] * nuy);
    double w[4];
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = lY * Y.d[j] + lg * g.d[j];
    const double la = l[0] * (1.0 - A) + w[0], lb = l[1] * (1.0 - A) + w[0];
    gr[0] = la * fa.d[0] + lb * fb.d[0] + w[1];
    gr[1] = la * fa.d[1] + lb * fb.d[1] + w[1];
    gr[2] = 2.0 * nux * w[2] - l[2] * g.v;
    gr[3] = 2.0 * nuy * w[2] - l[3] * g.v;
    gr[4] = la;
    gr[5] = lb;
    gr[6] = l[0] * A + w[3];
    gr[7] = l[1] * A + w[3];
}

}  // namespace ad
}  // namespace tdw
