"""The pointwise functional over the whole range of its inputs, through the C
ABI against the CPU oracle: densities from far below the regularisation
threshold to several times the uniform gas, each functional, both
regularisation schemes.  The first test starts the mixing loop from mean fields
on both sides of the band bottom; without an external potential the loop has
left those behind at its end.  The second holds points outside the real range
of the regularisation by an external potential: below the cutoff's reach
(imaginary k_c) and, with the cubic cutoff, above it (p0 > pi / dx)."""
import ctypes as C

import numpy as np
import pytest

from oracle import pyoracle as po
from tests import tdgauss
from tests.test_gpu_parity import cuda, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no HIP device")
    return t


def inputs(N, seed):
    r = np.random.default_rng(seed)
    dens, pots = np.zeros(12 * N), np.zeros(12 * N)
    na = 10.0 ** r.uniform(-8.5, -0.8, N)
    nb = na * np.where(r.random(N) < 0.2, 1.0, r.uniform(0.0, 1.0, N))
    nu = 0.5 * np.sqrt(na * nb) * np.exp(2j * np.pi * r.random(N))
    dens[:2 * N] = nu.view(np.float64)
    dens[2 * N:3 * N], dens[7 * N:8 * N] = na, nb
    for k, n in ((3, na), (8, nb)):
        dens[k * N:(k + 1) * N] = n ** (5 / 3) * r.uniform(0.5, 5.0, N)
        for d in range(1, 4):
            dens[(k + d) * N:(k + d + 1) * N] = n * r.uniform(-0.3, 0.3, N)
    # V from well below to well above mu: the loop starts on either branch
    pots[:2 * N] = r.uniform(-3.0, 3.0, 2 * N)
    pots[2 * N:4 * N] = r.uniform(-0.5, 0.5, 2 * N)
    pots[4 * N:6 * N] = r.uniform(0.9, 1.2, 2 * N)
    return dens, pots


@pytest.mark.parametrize("functional,a1", [(po.SLDA, 0), (po.BDG, 0), (po.ASLDA, 0), (po.SLDAE, 0), (po.SLDAE, 1)])
@pytest.mark.parametrize("reg", [88, 89])
@pytest.mark.parametrize("ec", [4.9, 0.3])
def test_potentials_over_the_input_range(torch, functional, a1, reg, ec):
    from wslda_amd import td
    say("case: potentials functional=%d a1=%d regularization=%d ec=%.1f" % (functional, a1, reg, ec))
    cfg = po.make_cfg(2, 24, 16, 4, dx=1.1, functional=functional, force_a1=a1,
                      sclgth=-0.9 if functional in (po.BDG, po.SLDAE) else 0.0)
    cfg.regularization, cfg.mf_correction = reg, 1
    cfg.mu_a, cfg.mu_b, cfg.ec = 0.25, 0.2, ec
    N = po.npts(cfg)
    dens, pots = inputs(N, 7 + functional + reg)

    def oracle(d, p):
        p = p.copy()
        po.lib().tdwo_potentials(C.byref(cfg), 1, po.ptr(np.ascontiguousarray(d)), po.ptr(p))
        return p

    ref = oracle(dens, pots)
    # what a relative change of the inputs by 1e-13 does to the oracle's own
    # result: the loop amplifies rounding near its resonance C~ = Re wz and
    # near k_c = p0, where no two correct evaluations agree to round-off
    r = np.random.default_rng(1)
    amp = np.zeros_like(ref)
    for _ in range(6):
        amp = np.maximum(amp, np.abs(oracle(dens * (1 + 1e-13 * r.choice([-1, 1], dens.size)),
                                            pots * (1 + 1e-13 * r.choice([-1, 1], pots.size))) - ref))
    prm = tdgauss.to_params(cfg, td.FP64)
    ctx = td.TDContext(prm, 4, 0)
    dd, dp = cuda(torch, dens), cuda(torch, pots)
    ctx.compute_potentials(1, dd, dp)
    ctx.sync()
    got = dp.cpu().numpy()
    ctx.close()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    # every point within ten times that amplification (the results of the
    # point: V_a, V_b and Delta share one loop), plus round-off of the result
    a = np.zeros(N)
    for k in range(12):
        f = amp[k * N:(k + 1) * N] if k not in (2, 3) else amp[2 * N:4 * N].reshape(N, 2).max(1)
        a = np.maximum(a, np.where(np.isnan(f), 0.0, f))
    lim = np.concatenate([np.repeat(a, 2) if k == 2 else a for k in range(12) if k != 3])
    lim = 10.0 * lim + 1e-12 * np.maximum(np.abs(ref), 1.0)
    d = np.abs(got - ref)
    assert (d[ok] <= lim[ok]).all(), (d[ok] / lim[ok]).max()


@pytest.mark.parametrize("functional,a1", [(po.SLDA, 0), (po.BDG, 0), (po.ASLDA, 0), (po.SLDAE, 0), (po.SLDAE, 1)])
@pytest.mark.parametrize("reg", [88, 89])
def test_potentials_outside_the_real_range(torch, functional, a1, reg):
    """A barrier of 8 ec beside a deep well: V_+ - mu_+ at the end of the loop
    runs from beyond -(pi / dx)^2 / 2 over the band bottom to several ec, so the
    last iterations see every branch of the regularisation."""
    from wslda_amd import td
    say("case: potentials in V_ext functional=%d a1=%d regularization=%d" % (functional, a1, reg))
    ec, dx = 0.3, 1.1
    vext = po.gauss_vext([(8.0 * ec, (-7.0, 0.0, 0.0), (-0.03, -0.02, 0.0)),
                          (-7.0, (7.0, 0.0, 0.0), (-0.03, -0.02, 0.0))])
    cfg = po.make_cfg(2, 24, 16, 4, dx=dx, functional=functional, force_a1=a1, vext=vext,
                      sclgth=-0.9 if functional in (po.BDG, po.SLDAE) else 0.0)
    # (the mean-field correction is the logarithm of a negative number above the
    # cubic cutoff)
    cfg.regularization, cfg.mf_correction = reg, int(reg == 88)
    cfg.mu_a, cfg.mu_b, cfg.ec = 0.25, 0.2, ec
    N = po.npts(cfg)
    dens, pots = inputs(N, 31 + functional + reg)
    va, vb = np.zeros(N), np.zeros(N)
    po.lib().tdwo_vext_eval(C.byref(cfg), 1, po.ptr(va), po.ptr(vb))
    # BdG is one evaluation from the V given
    pots[:N] += va
    pots[N:2 * N] += vb

    def oracle(d, p):
        p = p.copy()
        po.lib().tdwo_potentials(C.byref(cfg), 1, po.ptr(np.ascontiguousarray(d)), po.ptr(p))
        return p

    ref = oracle(dens, pots)
    ok = ~np.isnan(ref[:4 * N]).reshape(4, N).any(0)
    # mu_+ - V_+ of the last evaluation, and which branch that is
    last = pots if functional == po.BDG else ref
    al = np.ones(N) if functional == po.BDG else 0.5 * (ref[4 * N:5 * N] + ref[5 * N:6 * N])
    if functional == po.SLDA or a1:
        al = np.ones(N)
    t7 = 0.5 * (cfg.mu_a + cfg.mu_b - last[:N] - last[N:2 * N])
    below = t7 < -ec
    above = 2.0 * t7 / al > (np.pi / dx) ** 2
    inside = (t7 > 0.0) & ~above
    parts = [below, inside, (t7 < 0.0) & ~below] + ([above] if reg == 89 else [])
    for part in parts:
        assert (part & ok).sum() >= 10
    # as in the first test: ten times what a relative change of the inputs by
    # 1e-13 does to the point, plus round-off (of V_ext and mu, of order one,
    # in V; of Delta itself in Delta)
    r = np.random.default_rng(1)
    amp = np.zeros(4 * N)
    for _ in range(6):
        d = oracle(dens * (1 + 1e-13 * r.choice([-1, 1], dens.size)), pots * (1 + 1e-13 * r.choice([-1, 1], pots.size)))
        amp = np.maximum(amp, np.nan_to_num(np.abs(d - ref)[:4 * N]))

    def points(a):   # per point: V_a, V_b, |Delta|
        return np.stack([a[:N], a[N:2 * N], np.hypot(a[2 * N:4 * N:2], a[2 * N + 1:4 * N:2])])

    scale = np.abs(points(np.abs(ref)))
    scale[:2] = np.maximum(scale[:2], 1.0)
    A = points(amp)
    lim = 10.0 * np.maximum(A, scale * (A / scale).max(0)) + 1e-12 * scale
    # the limit is a real one at most points of every branch
    sharp = (lim <= 1e-10 * scale).all(0) & ok
    for part in parts:
        assert sharp[part].mean() > 0.6, (sharp[part].mean(), part.sum())
    prm = tdgauss.to_params(cfg, td.FP64)
    ctx = td.TDContext(prm, 4, 0)
    dd, dp = cuda(torch, dens), cuda(torch, pots)
    ctx.compute_potentials(1, dd, dp)
    ctx.sync()
    got = dp.cpu().numpy()
    ctx.close()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    err = points(np.abs(got - ref)[:4 * N])
    bad = (err > lim) & ok
    assert not bad.any(), (functional, reg, bad.any(0).sum(), (err / lim)[:, ok].max())


def test_mean_field_rounding(torch):
    """V_s = dD/dn_s (no pairing, no external potential, 15 mixing steps of 3/4
    from zero) against extended precision: its powers of 2/3 and 5/3 have to be as good as pow's.  Each
    term of dD/dn is then good to about three units in the last place; the
    limit is four for nine points in ten (dD/dn_b passes through zero)."""
    from wslda_amd import td
    cfg = po.make_cfg(2, 128, 128, 4, dx=1.1)
    cfg.mu_a, cfg.mu_b, cfg.ec, cfg.mf_correction = 0.25, 0.2, 4.9, 1
    N = po.npts(cfg)
    dens, pots = inputs(N, 3)
    dens[:2 * N], pots[:4 * N] = 0.0, 0.0
    ld = np.longdouble
    na, nb = dens[2 * N:3 * N].astype(ld), dens[7 * N:8 * N].astype(ld)
    n, pi = na + nb, ld("3.14159265358979323846264338327950288")
    lo, hi = ld(cfg.p_nmin), ld(cfg.p_nmax)
    far = np.asarray((n > hi) | (n < lo))    # (between them p_reg amplifies rounding)
    on = n > hi
    p = np.where(on, (na - nb) / n, ld(0))
    hp, hm, g0, g1 = (1 + p) / 2, (1 - p) / 2, ld(0.357), ld(0.642)
    t23, t53 = ld(2) / 3, ld(5) / 3
    base = g0 + g1 * p * p - hp ** t53 - hm ** t53
    s = 2 * g1 * p - ld(5) / 6 * (hp ** t23 - hm ** t23)
    x = 6 * pi * pi * n
    prm = tdgauss.to_params(cfg, td.FP64)
    ctx = td.TDContext(prm, 4, 0)
    dd, dp = cuda(torch, dens), cuda(torch, pots)
    ctx.compute_potentials(1, dd, dp)
    ctx.sync()
    got = dp.cpu().numpy()
    ctx.close()
    err = []
    for k, dpol in ((0, 2 * nb / n ** 2), (1, -2 * na / n ** 2)):
        ref = x ** t23 / 2 * base + x ** t53 / (20 * pi * pi) * s * np.where(on, dpol, ld(0))
        ref *= 1 - ld(0.25) ** 15
        err.append(np.asarray(np.abs(got[k * N:(k + 1) * N] - ref) / np.abs(ref), dtype=float)[far])
    q = np.median(np.concatenate(err))
    assert q < np.finfo(float).eps, q
