// tdw_functional.hpp -- pointwise SLDA / ASLDA / BdG functional on the device.
//
// Restates hpc-engine/pca_edf.h:17-352 (SLDA with the A0=1 effective mass of
// SLDA_FORCE_A1, pca_settings.h:80-90; ASLDA with the polarization-dependent
// effective mass of tdw_aslda.hpp) and the potential loops of
// tdwslda_functionals.h:47-306 (SLDA, ASLDA) and :373-452 (BdG).
#pragma once
#include "tdw_aslda.hpp"
#include "tdw_sldae.hpp"
#include "tdw_device.hpp"

namespace tdw {

// SLDA constants (pca_settings.h:80-110, 226-239)
#define TDW_A0 1.000
#define TDW_G0 0.357
#define TDW_G1 0.642
#define TDW_P_ALPHA 1.0
#define TDW_GAMMA0 (-11.11)
#define TDW_UD_SCITERS 15
#define TDW_UD_MIX 0.75

struct FParams {
    double p_nmin, p_nmax, denseps;
    double mu_a, mu_b, ec, dx;
    double R0, R1;
    int cubic, mf, bdg, aslda, sldae, a1;
    double sclgth;
    const double *agrid;   // project build: scattering_length() per point (N), or null
};

__device__ __forceinline__ double p_reg(const FParams &f, double n)
{
    if (n <= f.p_nmin) return 0.0;
    if (n >= f.p_nmax) return 1.0;
    return 0.5 + 0.5 * tanh(TDW_P_ALPHA * tan((M_PI * (n - f.p_nmin)) / (f.p_nmax - f.p_nmin) - M_PI / 2.0));
}
__device__ __forceinline__ double der_p_reg(const FParams &f, double n)
{
    if (n <= f.p_nmin || n >= f.p_nmax) return 0.0;
    double a = (M_PI * (n - f.p_nmin)) / (f.p_nmax - f.p_nmin) - M_PI / 2.0;
    double q = cosh(TDW_P_ALPHA * tan(a)) * cos(a);
    return 0.5 * TDW_P_ALPHA * M_PI / (q * q) / (f.p_nmax - f.p_nmin);
}
__device__ __forceinline__ double polar(const FParams &f, double na, double nb)
{
    double pr = p_reg(f, na + nb);
    if (pr == 0.0) return 0.0;
    return pr * (na - nb) / (na + nb);
}
__device__ __forceinline__ double der_pol(const FParams &f, double na, double nb, int wrt_b)
{
    double np = na + nb, pr = p_reg(f, np), dpr = der_p_reg(f, np), r = 0.0;
    if (pr != 0.0) r += pr * (wrt_b ? (-2.0 * na) : (2.0 * nb)) / (np * np);
    if (dpr != 0.0) r += dpr * (na - nb) / np;
    return r;
}
// alpha(p) = A0 for SLDA with A1 = A2 = 0.
__device__ __forceinline__ double alpha_f(double) { return TDW_A0; }
__device__ __forceinline__ double funG(double p) { return TDW_G0 + TDW_G1 * p * p; }

__device__ __forceinline__ double funD(const FParams &f, double na, double nb)
{
    double p = polar(f, na, nb);
    return (1.0 / (20.0 * M_PI * M_PI)) * pow(6.0 * M_PI * M_PI * (na + nb), 5.0 / 3.0) *
           (funG(p) - alpha_f(p) * pow((1.0 + p) / 2.0, 5.0 / 3.0) -
            alpha_f(-1.0 * p) * pow((1.0 - p) / 2.0, 5.0 / 3.0));
}
// x^(1/3), x^(2/3) and x^(5/3), NaN for x < 0 as pow gives: one cbrt instead
// of three pow.  c^2 with c = cbrt(x) rounded is good to 2 units in the last
// place, which is less than pow gives: dD/dn over densities of 1e-8.5 to
// 1e-0.8 had a median relative error of 3.4e-16 with it and 3.0e-16 with pow.
// So c^2 is taken in two parts with the residual x - c^3 put back, c^2 (1 + 2
// (x - c^3) / (3 x)), half a unit in x^(2/3) and one in x^(5/3): 1.3e-16.
struct Thirds {
    double x13, x23, x53;
};
__device__ __forceinline__ Thirds thirds(double x)
{
    // the parts' roundings are what is computed here: no contraction but the
    // fma written
#pragma clang fp contract(off)
    const double c = x < 0.0 ? nan("") : cbrt(x);
    const double p = c * c, pl = fma(c, c, -p);
    const double r = fma(-pl, c, fma(-p, c, x));   // x - c^3
    // (zero and infinity are their own powers; an estimate of 1 / c is enough
    // for a correction in the last place)
    const double t = p > 0.0 && p < 1.0e300 ? fma((2.0 / 3.0) * r, __builtin_amdgcn_rcp(c), pl) : 0.0;
    const double h = p + t;
    return {c, h, fma(x, t - (h - p), x * h)};
}

// What the mixing loop holds fixed at a point: dD/dn_a, dD/dn_b, C~ and its
// derivatives (ccoeff = 1), with alpha(p), alpha(-p), alpha_plus and their
// p-derivatives given (pca_edf.h:232-352).
struct EdfConst {
    double dDa, dDb, C, dCa, dCb;
};
__device__ __forceinline__ EdfConst edf_const(const FParams &f, double n, double p, double dpa, double dpb,
                                              double g0, double g1, double gamma0, double al_p, double al_m,
                                              double dal_p, double dal_m, double alph_plus, double dalph_plus)
{
    EdfConst r;
    const Thirds x = thirds(6.0 * M_PI * M_PI * n), hp = thirds((1.0 + p) / 2.0), hm = thirds((1.0 - p) / 2.0);
    const double base = g0 + g1 * p * p - al_p * hp.x53 - al_m * hm.x53;
    const double s = 2.0 * g1 * p - dal_p * hp.x53 - (5.0 / 6.0) * al_p * hp.x23 - dal_m * hm.x53 +
                     (5.0 / 6.0) * al_m * hm.x23;
    const double d0 = 0.5 * x.x23 * base, d1 = (1.0 / (20.0 * M_PI * M_PI)) * x.x53 * s;
    r.dDa = d0 + d1 * dpa;
    r.dDb = d0 + d1 * dpb;
    const Thirds e = thirds(n + f.denseps);
    const double dce = (1.0 / 3.0) * alph_plus / e.x23;
    r.C = alph_plus * e.x13 / gamma0;
    r.dCa = (dalph_plus * dpa * e.x13 + dce) / gamma0;
    r.dCb = (dalph_plus * dpb * e.x13 + dce) / gamma0;
    return r;
}

// complex helpers on double2 for the regularisation (principal branches, as
// thrust::complex<double>)
__device__ __forceinline__ double2 csqrt_real(double x)
{
    // sqrt(x + 0i)
    return x >= 0.0 ? make_double2(sqrt(x), 0.0) : make_double2(0.0, sqrt(-x));
}
__device__ __forceinline__ double2 cdiv(double2 a, double2 b)
{
    double d = b.x * b.x + b.y * b.y;
    return make_double2((a.x * b.x + a.y * b.y) / d, (a.y * b.x - a.x * b.y) / d);
}
__device__ __forceinline__ double2 clog2(double2 z)
{
    return make_double2(log(hypot(z.x, z.y)), atan2(z.y, z.x));
}

// One evaluation of the regularised coupling (tdwslda_functionals.h:251-265)
// given t7 = mu_+ - V_+ and kscale2 = 2 / alpha_plus for SLDA (p0 =
// sqrt(2 t7 / alpha)), 2 for BdG: wz = R0 (k_c - R1 p0 log((k_c + p0)/(k_c -
// p0))) before the final inversion, and p0 (for the mean-field correction).
__device__ __forceinline__ void reg_wz(const FParams &f, double t7, double kscale2, double2 &wz, double2 &p0)
{
    p0 = csqrt_real(t7 * kscale2);
    const double2 kc = f.cubic ? make_double2(M_PI / f.dx, 0.0) : csqrt_real((f.ec + t7) * kscale2);
    double2 w = clog2(cdiv(kc + p0, kc - p0));
    if (w.y < 0.) w.y += 2. * M_PI;
    wz = (kc - cmul(p0, w) * f.R1) * f.R0;
}
// Re(a / (c - wz)), a and c real
__device__ __forceinline__ double re_inv(double a, double c, double2 wz)
{
    const double d = c - wz.x;
    return wz.y == 0.0 ? a / d : a * d / (d * d + wz.y * wz.y);
}

// Mean-field correction of the regularisation scheme (:268-290), dLam/dn or
// 0.  With b = Re p0 / k_F and lx = b k_F dx / pi the reference's
// (k_F / (3 n alpha)) (Lam0 + dLam0 b dx k_F / pi) is
//   -(k_F / (3 n alpha)) R0 R1 b (log((1 + lx)/(1 - lx)) + 2 lx / (1 - lx^2))
// (its two terms of opposite sign, b R0 / lx, cancel).
struct MfConst {
    double ikF, fx, pre;   // 1 / (k_F + 1e-12), k_F dx / pi, -k_F R0 R1 / (3 n alpha)
};
__device__ __forceinline__ MfConst mf_const(const FParams &f, double n, double alph_plus)
{
    MfConst m;
    const double kF = thirds(3.0 * M_PI * M_PI * n).x13;
    m.ikF = 1.0 / (kF + 1.0e-12);
    m.fx = kF * f.dx / M_PI;
    m.pre = -(kF / (3. * n * alph_plus)) * f.R0 * f.R1;
    return m;
}
__device__ __forceinline__ double mf_corr(const MfConst &m, double p0x, double g)
{
    const double b = p0x * m.ikF, lx = b * m.fx;
    const double q = 1.0 / ((1.0 - lx) * (1.0 + lx));
    const double v = m.pre * b * (log((1.0 + lx) * (1.0 + lx) * q) + 2.0 * lx * q);
    return (g < -1.0e-10 && lx > 1.0e-10) ? v : 0.0;
}

// The same two above the band bottom: p0 = p and k_c real, p < k_c, lx < 1.
// With k_c^2 - p^2 = d (2 ec / alpha, or (pi / dx)^2 - p^2) the logarithm's
// argument is (k_c + p)^2 / d.  Arguments are positive and of order one, so
// short square roots, reciprocals and logarithms do (see tdw_device.hpp).
__device__ __forceinline__ bool reg_real(const FParams &f, const MfConst &m, double t7, double kscale2, double &wz,
                                         double &mfv, double &lx)
{
    const double p2 = t7 * kscale2, kc2 = f.cubic ? (M_PI / f.dx) * (M_PI / f.dx) : (f.ec + t7) * kscale2;
    const double d = f.cubic ? kc2 - p2 : f.ec * kscale2;
    const double p = sqrt_pos(p2), k = f.cubic ? M_PI / f.dx : sqrt_pos(kc2);
    const double b = p * m.ikF;
    lx = b * m.fx;
    const double q = rcp_pos((1.0 - lx) * (1.0 + lx));
    const double l1 = log_pos((k + p) * (k + p) * rcp_pos(d)), l2 = log_pos((1.0 + lx) * (1.0 + lx) * q);
    wz = (k - f.R1 * p * l1) * f.R0;
    mfv = m.pre * b * (l2 + 2.0 * lx * q);
    // small or large arguments, and every other branch, take the general form
    return p2 >= 1.0e-30 && p2 < 1.0e30 && d > 1.0e-10 * kc2 && kc2 < 1.0e30 && lx < 0.999;
}

// The 15 mixing iterations of V_a, V_b and Delta = -nu g
// (tdwslda_functionals.h:236-300) from the previous V_a, V_b: each new V_s is
// V_s,const - e_s Re(Delta* nu) - c_s |Delta|^2 + the mean-field correction.
// g = Re(alpha_+ / (C - wz)), or with REAL_WZ (SLDAE) alpha_+ / (C -
// Re wz).  The two part where wz is complex: below the cutoff's reach (mu_+ -
// V_+ < -ec) and, with the cubic cutoff, above it (p0 > pi / dx).
template <bool REAL_WZ = false>
__device__ __forceinline__ void mix_loop(const FParams &f, double n, double2 nu, double alph_plus, double C,
                                         double Va_const, double Vb_const, double ea, double eb, double ca, double cb,
                                         double &Va, double &Vb, double2 &delta)
{
    // The loop is a chain of fifteen evaluations per point with too few points
    // to hide it: with the general form alone (complex logarithm, five
    // divisions and two logarithms one after the other) it was most of the 25
    // us that k_potentials took on 64 points, and a third of that problem's
    // step.  A wave whose points are all above the band bottom takes reg_real,
    // one straight run in which the two logarithms overlap: 10.7 us.
    const double kscale2 = 2.0 / alph_plus, nu2 = nu.x * nu.x + nu.y * nu.y;
    MfConst m{0.0, 0.0, 0.0};
    if (f.mf) m = mf_const(f, n, alph_plus);
    double g = 0.0;
    for (int k = 0; k < TDW_UD_SCITERS; k++) {
        const double t7 = (f.mu_a - Va + f.mu_b - Vb) / 2.0;
        double wr, mfv, lx, dl = 0.0;
        if (__all(reg_real(f, m, t7, kscale2, wr, mfv, lx))) {
            g = alph_plus / (C - wr);
            dl = (f.mf && g < -1.0e-10 && lx > 1.0e-10) ? mfv : 0.0;
        } else {
            double2 wz, p0;
            reg_wz(f, t7, kscale2, wz, p0);
            g = REAL_WZ ? alph_plus / (C - wz.x) : re_inv(alph_plus, C, wz);
            if (f.mf) dl = mf_corr(m, p0.x, g);
        }
        const double dn = -g * nu2, d2 = g * g * nu2;   // Re(Delta* nu), |Delta|^2
        const double Vanew = Va_const - ea * dn - ca * d2 + dl * d2;
        const double Vbnew = Vb_const - eb * dn - cb * d2 + dl * d2;
        Va = TDW_UD_MIX * Vanew + (1.0 - TDW_UD_MIX) * Va;
        Vb = TDW_UD_MIX * Vbnew + (1.0 - TDW_UD_MIX) * Vb;
    }
    delta = nu * (-1.0 * g);
}

// SLDA potentials at one point (tdwslda_functionals.h:47-306, FAST mode).
__device__ __forceinline__ void slda_point(const FParams &f, double na, double nb, double2 nu,
                                           double ua, double ub, double &Va, double &Vb,
                                           double2 &delta)
{
    const double n = na + nb, p = polar(f, na, nb);
    const EdfConst e = edf_const(f, n, p, der_pol(f, na, nb, 0), der_pol(f, na, nb, 1), TDW_G0, TDW_G1, TDW_GAMMA0,
                                 TDW_A0, TDW_A0, 0.0, 0.0, TDW_A0, 0.0);
    mix_loop(f, n, nu, TDW_A0, e.C, ua + e.dDa, ub + e.dDb, 0.0, 0.0, e.dCa / TDW_A0, e.dCb / TDW_A0, Va, Vb, delta);
}

// ASLDA potentials at one point (tdwslda_functionals.h:47-306 without
// FAST_CONST_EFFECTIVE_MASS_MODE, with CURRENT_CORRECTIONS): V_a, V_b, Delta,
// the effective masses alpha_a, alpha_b and the vector potentials
// A_s = cc f_r(n_s) (1 - alpha_s) j_s / n_s (dim components; cc is the
// current-corrections coefficient).  tau and j are the densities of the same
// half-step.
__device__ __forceinline__ void aslda_point(const FParams &f, double na, double nb, double2 nu, double taua,
                                            double taub, const double *ja, const double *jb, int dim, double cc,
                                            double ua, double ub, double &Va, double &Vb, double2 &delta,
                                            double &ala, double &alb, double *Aa, double *Ab)
{
    const double n = na + nb;
    const double p = polar(f, na, nb);
    const double dpa = der_pol(f, na, nb, 0), dpb = der_pol(f, na, nb, 1);
    const double alph_plus = aslda::alpha_plus(p), alph_minus = aslda::alpha_minus(p);
    const double aA = aslda::alpha(p), aB = aslda::alpha(-p);
    ala = aA;
    alb = aB;
    const double fa = p_reg(f, na) * cc, fb = p_reg(f, nb) * cc;
    double j2a = 0.0, j2b = 0.0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        if (d >= dim) break;
        Aa[d] = fa == 0.0 ? 0.0 : fa * (1. - aA) * ja[d] / na;
        Ab[d] = fb == 0.0 ? 0.0 : fb * (1. - aB) * jb[d] / nb;
        j2a += ja[d] * ja[d];
        j2b += jb[d] * jb[d];
    }
    const double dalphp_dna = aslda::dalpha_plus_dp(p) * dpa, dalphp_dnb = aslda::dalpha_plus_dp(p) * dpb;
    const double dalphm_dna = aslda::dalpha_minus_dp(p) * dpa, dalphm_dnb = aslda::dalpha_minus_dp(p) * dpb;
    double Va_const = ua, Vb_const = ub;
    Va_const += dalphm_dna * (taua - taub) / 2.0;
    Vb_const += dalphm_dnb * (taua - taub) / 2.0;
    Va_const += dalphp_dna * (taua + taub) / 2.0;
    Vb_const += dalphp_dnb * (taua + taub) / 2.0;
    // d alpha(p)/dp and d alpha(-p)/dp as pca_edf.h:245-314 takes them
    const EdfConst e = edf_const(f, n, p, dpa, dpb, aslda::G0, aslda::G1, aslda::GAMMA0, aA, aB,
                                 aslda::dalpha_plus_dp(p) + aslda::dalpha_minus_dp(p),
                                 aslda::dalpha_plus_dp(p) - aslda::dalpha_minus_dp(p), alph_plus,
                                 aslda::dalpha_plus_dp(p));
    Va_const += e.dDa;
    Vb_const += e.dDb;
    if (fa != 0.0) {
        const double t7 = fa * j2a / (2.0 * na);
        Va_const += ((alph_plus + alph_minus - 1.0) / na - (dalphp_dna + dalphm_dna)) * t7;
        Va_const -= cc * der_p_reg(f, na) * (alph_plus + alph_minus - 1.0) * j2a / (2.0 * na);
        Vb_const -= (dalphp_dnb + dalphm_dnb) * t7;
    }
    if (fb != 0.0) {
        const double t7 = fb * j2b / (2.0 * nb);
        Va_const -= (dalphp_dna - dalphm_dna) * t7;
        Vb_const += ((alph_plus - alph_minus - 1.0) / nb - (dalphp_dnb - dalphm_dnb)) * t7;
        Vb_const -= cc * der_p_reg(f, nb) * (alph_plus - alph_minus - 1.0) * j2b / (2.0 * nb);
    }
    mix_loop(f, n, nu, alph_plus, e.C, Va_const, Vb_const, dalphp_dna / alph_plus, dalphp_dnb / alph_plus,
             e.dCa / alph_plus, e.dCb / alph_plus, Va, Vb, delta);
}

// SLDAE potentials at one point (tdwslda_functionals.h:530-812, with
// CURRENT_CORRECTIONS): alpha_a = alpha_b = A(x), x = |a k_F(n)|, the vector
// potentials as in ASLDA, V_s = U_ext + A' (tau_a + tau_b)/2 + beta e_F
// + current terms - (A'/A) Re(Delta* nu) - C~'/A |Delta|^2, and
// Delta = -nu A / (C~ - Lambda) with Lambda = Re of the regularised integral.
__device__ __forceinline__ void sldae_point(const FParams &f, double na, double nb, double2 nu, double taua,
                                            double taub, const double *ja, const double *jb, int dim, double cc,
                                            double ua, double ub, double &Va, double &Vb, double2 &delta,
                                            double &ala, double &alb, double *Aa, double *Ab)
{
    const double n = na + nb;
    const sldae::Local L = sldae::local(n, p_reg(f, n), f.sclgth, f.a1);
    const double af = L.af, af_p = L.af_p;
    ala = af;
    alb = af;
    // SLDA_FORCE_A1: FAST_CONST_EFFECTIVE_MASS_MODE, no current corrections
    const double fa = f.a1 ? 0.0 : p_reg(f, na) * cc, fb = f.a1 ? 0.0 : p_reg(f, nb) * cc;
    double j2a = 0.0, j2b = 0.0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        if (d >= dim) break;
        Aa[d] = fa == 0.0 ? 0.0 : fa * (1. - af) * ja[d] / na;
        Ab[d] = fb == 0.0 ? 0.0 : fb * (1. - af) * jb[d] / nb;
        j2a += ja[d] * ja[d];
        j2b += jb[d] * jb[d];
    }
    double Va_const = ua + af_p * (taua + taub) / 2.;
    double Vb_const = ub + af_p * (taua + taub) / 2.;
    Va_const += L.beta * L.eF;
    Vb_const += L.beta * L.eF;
    if (fa != 0.0) {
        const double t7 = fa * j2a / (2.0 * na);
        Va_const += ((af - 1.0) / na - af_p) * t7;
        Va_const -= cc * der_p_reg(f, na) * (af - 1.0) * j2a / (2.0 * na);
        Vb_const -= af_p * t7;
    }
    if (fb != 0.0) {
        const double t7 = fb * j2b / (2.0 * nb);
        Va_const -= af_p * t7;
        Vb_const += ((af - 1.0) / nb - af_p) * t7;
        Vb_const -= cc * der_p_reg(f, nb) * (af - 1.0) * j2b / (2.0 * nb);
    }
    mix_loop<true>(f, n, nu, af, L.ctilde, Va_const, Vb_const, af_p / af, af_p / af, L.ctilde_p / af, L.ctilde_p / af,
                   Va, Vb, delta);
}

// BdG potentials at one point (tdwslda_functionals.h:373-452).
__device__ __forceinline__ void bdg_point(const FParams &f, double na, double nb, double2 nu,
                                          double ua, double ub, double al_a, double al_b,
                                          double &Va, double &Vb, double2 &delta)
{
    const double alph_plus = 0.5 * (al_a + al_b);
    const double t5 = 1.0 / (4.0 * M_PI * f.sclgth * alph_plus);
    double t7 = (f.mu_a - Va + f.mu_b - Vb) / 2.0;
    double2 wz, p0;
    reg_wz(f, t7, 2.0, wz, p0);
    wz = wz * (1.0 / alph_plus);
    const double g = re_inv(1.0, t5, wz);
    double2 ld = nu * (-1.0 * g);
    double nVa = ua, nVb = ub;
    if (f.mf) {
        const double dl = mf_corr(mf_const(f, na + nb, alph_plus), p0.x, g);
        double t7b = ld.x * ld.x + ld.y * ld.y;
        nVa += dl * t7b;
        nVb += dl * t7b;
    }
    Va = nVa;
    Vb = nVb;
    delta = ld;
}

}  // namespace tdw
