"""Laplacian and derivatives of 3D arrays on lattices with compiled axis
lengths, against numpy's FFT: every length, x lengths whose planes do not fill
the last tile or workgroup, one array and several, out of place and in place.

Tolerance: 1e-12 of the largest value, as for the other building blocks (an
FFT of L points errs by a few eps sqrt(log L) of the spectrum's norm times
k_max^2, here some 1e-14 of the largest value)."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests import tdgauss
from tests.test_gpu_parity import TOL, cuda, rel, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no HIP device")
    return t


def kax(n, d, first=False):
    i = np.arange(n)
    k = 2 * np.pi / (n * d) * np.where(i < n // 2, i, i - n)
    if first:
        k[n // 2] = 0.0
    return k


@pytest.mark.parametrize("shape", [(8, 12, 12), (12, 16, 16), (16, 18, 18), (18, 24, 24), (24, 32, 32), (32, 36, 36),
                                   (36, 12, 12), (48, 48, 48), (18, 18, 18), (6, 32, 96), (48, 8, 12), (36, 6, 8)])
@pytest.mark.parametrize("m", [1, 3])
def test_derivatives_3d_lengths(torch, shape, m):
    from wslda_amd import td
    say("case: derivatives shape=%s m=%d" % (shape, m))
    nx, ny, nz = shape
    cfg = po.make_cfg(3, nx, ny, nz, dx=0.9)
    cfg.dy, cfg.dz = 1.1, 1.3
    N = nx * ny * nz
    r = np.random.default_rng(nx + ny + m)
    a = r.normal(size=(m, N)) + 1j * r.normal(size=(m, N))
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), m, 0)
    f = np.fft.fftn(a.reshape(m, *shape), axes=(1, 2, 3))
    d = (0.9, 1.1, 1.3)
    K = [kax(n, h).reshape([-1 if e == i else 1 for e in range(3)]) for i, (n, h) in enumerate(zip(shape, d))]
    K1 = [kax(n, h, True).reshape([-1 if e == i else 1 for e in range(3)]) for i, (n, h) in enumerate(zip(shape, d))]
    back = lambda g: np.fft.ifftn(g, axes=(1, 2, 3)).reshape(m, N)
    lap = back(-(K[0] ** 2 + K[1] ** 2 + K[2] ** 2) * f)
    t = cuda(torch, a)
    out = torch.zeros_like(t)
    ctx.compute_laplace(t, out)
    ctx.sync()
    assert rel(out.cpu().numpy(), lap) < TOL
    D = [torch.zeros_like(t) for _ in range(3)]
    out.zero_()
    ctx.compute_derivatives(t, D[0], D[1], D[2], out)
    ctx.sync()
    assert rel(out.cpu().numpy(), lap) < TOL
    for i in range(3):
        assert rel(D[i].cpu().numpy(), back(1j * K1[i] * f)) < TOL, i
    assert rel(t.cpu().numpy(), a) == 0.0
    ctx.compute_laplace(t, t)
    ctx.sync()
    assert rel(t.cpu().numpy(), lap) < TOL
    ctx.close()


@pytest.mark.parametrize("shape", [(32, 32), (32, 64), (64, 32), (64, 64)])
@pytest.mark.parametrize("m", [1, 3])
def test_derivatives_2d_planes(torch, shape, m):
    """The one-pass derivatives of 2D planes on the matrix cores."""
    from wslda_amd import td
    say("case: derivatives shape=%s m=%d" % (shape, m))
    nx, ny = shape
    cfg = po.make_cfg(2, nx, ny, 4, dx=0.9)
    cfg.dy = 1.1
    r = np.random.default_rng(nx + ny + m)
    a = r.normal(size=(m, nx * ny)) + 1j * r.normal(size=(m, nx * ny))
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), m, 0)
    f = np.fft.fftn(a.reshape(m, nx, ny), axes=(1, 2))
    k = lambda first: (kax(nx, 0.9, first).reshape(-1, 1), kax(ny, 1.1, first).reshape(1, -1))
    back = lambda g: np.fft.ifftn(g, axes=(1, 2)).reshape(m, nx * ny)
    kx, ky = k(False)
    gx, gy = k(True)
    t = cuda(torch, a)
    D = [torch.zeros_like(t) for _ in range(3)]
    ctx.compute_derivatives(t, D[0], D[1], None, D[2])
    ctx.sync()
    assert rel(D[0].cpu().numpy(), back(1j * gx * f)) < TOL
    assert rel(D[1].cpu().numpy(), back(1j * gy * f)) < TOL
    assert rel(D[2].cpu().numpy(), back(-(kx ** 2 + ky ** 2) * f)) < TOL
    assert rel(t.cpu().numpy(), a) == 0.0
    ctx.close()


@pytest.mark.parametrize("shape", [(32, 32), (32, 64), (64, 32), (64, 64)])
def test_plane_laplacian_has_no_bias(torch, shape):
    """<psi|lap psi> of smooth states: the rounding of the operator's tables is
    the same at every point and in every state, so it does not average out as
    that of the products does.  Against extended precision, the mean over 40
    states: entries rounded as they come are off by 1.4e-16 to 3.8e-16, the
    limit is half of the spacing of doubles at one."""
    from wslda_amd import td
    say("case: bias of the plane Laplacian shape=%s" % (shape,))
    m, ld = 40, np.longdouble
    nx, ny = shape
    cfg = po.make_cfg(2, nx, ny, 4, dx=1.0)
    r = np.random.default_rng(nx + 2 * ny)
    f = np.zeros((m, nx, ny), dtype=complex)
    for i in range(-4, 5):
        for j in range(-4, 5):
            f[:, i, j] = (r.normal(size=m) + 1j * r.normal(size=m)) * np.exp(-(i * i + j * j) / 4)
    a = np.fft.ifft2(f).reshape(m, nx * ny)
    a /= np.linalg.norm(a, axis=1)[:, None]
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), m, 0)
    t = cuda(torch, a)
    out = [torch.zeros_like(t) for _ in range(3)]
    ctx.compute_derivatives(t, out[0], out[1], None, out[2])
    ctx.sync()
    got = out[2].cpu().numpy()
    ctx.close()
    pi = ld("3.14159265358979323846264338327950288")

    def second(L):   # the operator along an axis, in extended precision
        q = np.where(np.arange(L) < L // 2, np.arange(L), np.arange(L) - L).astype(ld)
        c = -((2 * pi * q / L) ** 2 * np.cos(2 * pi * ((np.outer(np.arange(L), np.arange(L)) % L).astype(ld)) / L)).sum(1) / L
        return c[(np.arange(L)[:, None] - np.arange(L)[None, :]) % L]

    A = a.astype(np.clongdouble).reshape(m, nx, ny)
    ref = np.tensordot(second(nx), A, (1, 1)).transpose(1, 0, 2) + np.tensordot(A, second(ny), (2, 1))
    off = (A.conj() * (got.reshape(m, nx, ny) - ref)).sum((1, 2)).real
    say("mean %.2e" % float(off.mean()))
    assert abs(float(off.mean())) < 0.5 * np.finfo(float).eps


@pytest.mark.parametrize("shape", [(16, 16, 16), (16, 16, 18)])
def test_one_timer_record_per_launch(torch, shape):
    """A compiled plane and one without: each launch is recorded once."""
    from wslda_amd import td
    cfg = po.make_cfg(3, *shape, dx=0.9)
    N = int(np.prod(shape))
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), 2, 0)
    t = cuda(torch, np.ones((2, N), dtype=complex))
    D = [torch.zeros_like(t) for _ in range(4)]
    ctx.timing(1)
    ctx.compute_laplace(t, D[3])
    ctx.compute_derivatives(t, *D)
    ctx.sync()
    rep = ctx.timing_report()
    ctx.timing(0)
    ctx.close()
    assert {k: v[1] for k, v in rep.items()} == {"fft_outer": 1, "fft_inner": 1, "fft_outer_deriv": 1,
                                                 "fft_inner_deriv": 1}


@pytest.mark.parametrize("n", [3, 56, 57, 248, 249])
@pytest.mark.parametrize("shape", [(9, 3, 9), (4, 8, 8)])
def test_densities_chunk_counts(torch, shape, n):
    """Densities with gradients over 1, 7, 8, 31 and 32 chunks of states, the
    limits of the forms of the sum over the chunks; points that do and do not
    fill its workgroups."""
    import ctypes as C
    from wslda_amd import td
    say("case: densities over chunks shape=%s n=%d" % (shape, n))
    cfg = po.make_cfg(3, *shape, dx=0.9)
    N = int(np.prod(shape))
    r = np.random.default_rng(n)
    W = [r.normal(size=(2 * n, N)) + 1j * r.normal(size=(2 * n, N)) for _ in range(5)]
    fb = r.random(n)
    ref = np.zeros(12 * N)
    po.lib().tdwo_densities(C.byref(cfg), n, *[po.ptr(w) for w in W], po.ptr(fb), None, None, po.ptr(ref), 1)
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), n, 0)
    ctx.set_states(fb)
    dens = torch.zeros(12 * N, dtype=torch.float64, device="cuda:0")
    ctx.calculate_densities(*[cuda(torch, w) for w in W], dens, 1)
    ctx.sync()
    got = dens.cpu().numpy()
    ctx.close()
    # (a sum of n terms of either sign, each of order one)
    assert np.abs(got - ref).max() < 1e-14 * n
