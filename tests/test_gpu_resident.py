"""The PECE step of lattices whose state fits in LDS, against the CPU oracle:
axes of one to several radix stages, unequal lengths and spacings, transverse
momenta, more and fewer states than CUs, the largest lattice that fits and
the first that does not."""
import ctypes as C

import numpy as np
import pytest

from oracle import pyoracle as po
from tests import tdgauss
from tests.test_gpu_parity import TOL, rel, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no HIP device")
    return t


def problem(dim, shape, n, scheme, functional, seed=5):
    """Smooth random states (a few low modes each) with real occupations."""
    r = np.random.default_rng(seed)
    cfg = po.make_cfg(dim, *shape, dx=1.1, scheme=scheme, functional=functional,
                      sclgth=-0.8 if functional == po.BDG else 0.0)
    cfg.dy, cfg.dz = 0.9, 1.3
    cfg.mu_a, cfg.mu_b, cfg.ec, cfg.dt = 0.21, 0.2, 4.0, 0.01
    cfg.vext = po.gauss_vext([(0.05, (0.5, 0.0, 0.0), (-0.1, -0.1 if dim > 1 else 0.0, -0.1 if dim > 2 else 0.0))])
    N = po.npts(cfg)
    ax = shape[:dim]
    x = [2 * np.pi * np.arange(L) / L for L in ax]
    wf = np.zeros((2 * n, N), dtype=complex)
    for row in wf:
        for _ in range(3):
            f = 1.0
            for L, xx in zip(ax, x):
                f = np.multiply.outer(f, np.exp(1j * r.integers(-(L // 2) + 1, L // 2 + 1) * xx))
            row += r.normal(size=2).view(complex)[0] * f.ravel()
    wf += 1e-2 * (r.normal(size=wf.shape) + 1j * r.normal(size=wf.shape))
    kt = cnt = None
    if dim == 2:
        kt = r.uniform(0.0, 1.0, n) * (r.random(n) < 0.8)
    if dim == 1:
        kt, cnt = r.uniform(-1.0, 1.0, 2 * n), r.integers(1, 5, n).astype(np.int32)
    pots = np.zeros(12 * N)
    pots[:2 * N], pots[2 * N:4 * N:2], pots[4 * N:6 * N] = -0.1, 0.2, 1.0
    return cfg, wf, r.random(n), kt, cnt, pots


CASES = [
    (1, (2, 4, 4), 5), (1, (54, 4, 4), 300), (1, (256, 4, 4), 40), (1, (432, 4, 4), 6),
    (2, (8, 12, 6), 270), (2, (36, 18, 4), 20), (2, (6, 128, 4), 9), (2, (48, 54, 4), 7), (2, (64, 64, 4), 5),
    (2, (32, 32, 4), 300), (2, (32, 64, 4), 6), (2, (64, 32, 4), 6),
    (2, (72, 72, 4), 4),       # the state (166 KB) does not fit: the plane-wise step
    (1, (27, 4, 4), 9), (1, (243, 4, 4), 20), (2, (9, 27, 4), 12), (2, (27, 16, 4), 30), (2, (12, 9, 4), 260),
    (3, (12, 12, 12), 30), (3, (8, 16, 16), 9), (3, (12, 16, 16), 9), (3, (32, 12, 12), 7), (3, (8, 24, 24), 7),
     (3, (8, 6, 4), 600), (3, (16, 16, 16), 6), (3, (4, 18, 24), 12),
]


@pytest.mark.parametrize("dim,shape,n", CASES)
@pytest.mark.parametrize("scheme,functional", [(po.AB5AM5, po.SLDA), (po.AB4AM5, po.BDG), (po.AB3AM4, po.SLDA)])
def test_resident_step_vs_oracle(torch, dim, shape, n, scheme, functional):
    from wslda_amd import td
    say("case: resident step dim=%d shape=%s n=%d scheme=%d functional=%d" % (dim, shape, n, scheme, functional))
    cfg, wf, fb, kt, cnt, pots = problem(dim, shape, n, scheme, functional)
    P = po.Problem(cfg, wf.copy(), fb, kt=kt, cnt=cnt, pots=pots.copy())
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), n, 0)
    ctx.set_states(fb, kt, cnt)
    R = td.TDRun(ctx, wf, pots, fused=dim == 3)
    P.initial_measure()
    R.initial_measure()
    for it in range(6):
        P.step(it, grad_last=it == 5)
        R.step(it, grad_last=it == 5)
        if it >= 4:
            R.finalize()
            d = R.dens.cpu().numpy()
            assert rel(d, P.dens) < TOL, (it, rel(d, P.dens))
            assert rel(R.pots.cpu().numpy(), P.pots) < TOL, it
            assert rel(R.wf.cpu().numpy(), P.wf) < TOL, it
            assert rel(R.qpe.cpu().numpy(), P.qpe) < TOL, it
    ctx.close()


@pytest.mark.parametrize("dim,shape", [(1, (64, 4, 4)), (2, (16, 16, 4)), (2, (12, 18, 4)), (3, (8, 8, 8)),
                                       (3, (12, 12, 12))])
def test_gradient_step_without_its_arrays_is_refused(torch, dim, shape):
    """The return code, and that nothing was written: no kernel is launched."""
    from wslda_amd import td
    n = 3
    cfg, wf, fb, kt, cnt, pots = problem(dim, shape, n, po.AB4AM5, po.SLDA)
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), n, 0)
    ctx.set_states(fb, kt, cnt)
    R = td.TDRun(ctx, wf, pots, fused=dim == 3)
    fn = td.lib().tdw_step_fused if dim == 3 else td.lib().tdw_step
    before, hist = R.wf.clone(), [R.st.f[k] for k in range(5)]
    for name in ("lap", "ddx", "ddy", "ddz")[:dim + 1]:
        keep = getattr(R.st, name)
        setattr(R.st, name, None)
        assert fn(ctx.h, C.byref(R.st), 0, 1) == td.TDW_EINVAL, name
        setattr(R.st, name, keep)
    ctx.sync()
    assert torch.equal(R.wf, before) and hist == [R.st.f[k] for k in range(5)]
    ctx.close()


@pytest.mark.parametrize("dim,shape,n", [c for c in CASES if c[0] < 3 and c[1] not in ((64, 64, 4), (32, 32, 4))])
def test_step_leaves_the_laplacian(torch, dim, shape, n):
    """lap after a step without gradients (not on 32 x 32 and 64 x 64)."""
    from wslda_amd import td
    say("case: lap after a step dim=%d shape=%s n=%d" % (dim, shape, n))
    cfg, wf, fb, kt, cnt, pots = problem(dim, shape, n, po.AB4AM5, po.SLDA)
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), n, 0)
    ctx.set_states(fb, kt, cnt)
    R = td.TDRun(ctx, wf, pots)
    R.initial_measure()
    for it in range(2):
        R.step(it)
    ctx.sync()
    got, y = R.lap.cpu().numpy(), R.wf.cpu().numpy()
    ctx.close()
    ref = np.zeros_like(y)
    po.lib().tdwo_laplace(C.byref(cfg), 2 * n, po.ptr(y), po.ptr(ref))
    # (relative to the largest: the highest modes carry the rounding)
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


@pytest.mark.parametrize("shape", [(36, 18, 4), (18, 36, 4), (24, 36, 4), (48, 54, 4), (16, 16, 4)])
def test_transforms_are_as_exact_as_their_twiddles(torch, shape):
    """The Laplacian that a step leaves, of states with all modes, against
    extended precision: with correctly rounded twiddles its relative error (of
    the 2-norm) is below two units of rounding on axes with factors of 3 as on
    powers of two; radices 6 and 9 whose twiddles are off by three units give
    2.4 to 2.5."""
    from wslda_amd import td
    say("case: transform accuracy shape=%s" % (shape,))
    n, ld = 60, np.longdouble
    nx, ny = shape[:2]
    cfg, wf, fb, kt, cnt, pots = problem(2, shape, n, po.AB4AM5, po.SLDA)
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), n, 0)
    ctx.set_states(fb, kt, cnt)
    R = td.TDRun(ctx, wf, pots)
    R.initial_measure()
    R.step(0)
    ctx.sync()
    got, y = R.lap.cpu().numpy(), R.wf.cpu().numpy()
    ctx.close()
    pi = ld("3.14159265358979323846264338327950288")

    def second(L, dx):   # the operator along an axis, in extended precision
        i = np.arange(L)
        k = 2 * pi * np.where(i < L // 2, i, i - L).astype(ld) / (L * ld(dx))
        c = -(k ** 2 * np.cos(2 * pi * (np.outer(i, i) % L).astype(ld) / L)).sum(1) / L
        return c[(i[:, None] - i[None, :]) % L]

    A = y.astype(np.clongdouble).reshape(2 * n, nx, ny)
    ref = np.tensordot(second(nx, 1.1), A, (1, 1)).transpose(1, 0, 2) + np.tensordot(A, second(ny, 0.9), (2, 1))
    ref = ref.reshape(2 * n, -1)
    err = float(np.sqrt((np.abs(got - ref) ** 2).sum() / (np.abs(ref) ** 2).sum()))
    say("%.2e" % err)
    assert err < 2 * np.finfo(float).eps
