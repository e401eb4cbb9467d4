"""The matrix-core yz passes of FP64 planes of 24 and 32 points a side (the
ASLDA Hamiltonian and the densities with gradients) against transforms of the
same fields: planes thicker and thinner than their x axis, spacings that
differ along y and z, and numbers of states around the chunks of the density
pass.

Bound: a derivative's rounding is a few times L eps k_max^2 of the field, the
spectral form's as much; 1e-12 of the largest value is above both.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests import tdgauss

pytestmark = pytest.mark.gpu

SPACING = (1.1, 0.9, 1.3)
TOL = 1e-12


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no HIP device")
    return t


def context(shape, n, functional):
    from wslda_amd import td
    cfg = po.make_cfg(3, *shape, dx=SPACING[0], functional=functional)
    cfg.dy, cfg.dz = SPACING[1], SPACING[2]
    cfg.mu_a, cfg.mu_b = 0.3, 0.25
    return td.TDContext(tdgauss.to_params(cfg), n, 0), cfg


def spectral(torch, shape):
    """d(f, axis, order) along the last three dimensions, Nyquist mode of the
    first derivative zero."""
    def d(f, ax, order):
        L = shape[ax]
        k = 2 * np.pi * torch.fft.fftfreq(L, SPACING[ax], dtype=torch.float64, device=f.device)
        if order == 1:
            k[L // 2] = 0.0
        m = (1j * k) ** order
        v = [1] * f.dim()
        v[f.dim() - 3 + ax] = L
        return torch.fft.ifft(torch.fft.fft(f, dim=f.dim() - 3 + ax) * m.view(v), dim=f.dim() - 3 + ax)
    return d


def states(torch, shape, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda: torch.randn((2, n) + shape, dtype=torch.float64, device="cuda", generator=g)
    return torch.complex(r(), r()) * 0.05


SHAPES = [(24, 24, 24), (12, 24, 24), (32, 32, 32), (16, 32, 32)]


def close(a, b):
    return float((a - b).abs().max() / b.abs().max()) < TOL


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [1, 5])
def test_h(torch, shape, n):
    print("case: H in two passes, %s, %d states" % (shape, n), flush=True)
    ctx, cfg = context(shape, n, po.ASLDA)
    N = po.npts(cfg)
    psi = states(torch, shape, n, 3)
    d = spectral(torch, shape)
    g = torch.Generator(device="cuda").manual_seed(9)
    rnd = lambda: torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)
    V, D = [0.1 * rnd(), 0.1 * rnd()], torch.complex(0.2 + 0.05 * rnd(), 0.03 * rnd())
    al, A = [1 + 0.1 * rnd(), 1 + 0.1 * rnd()], [[0.05 * rnd() for _ in range(3)] for _ in range(2)]
    pots = torch.cat([V[0].ravel(), V[1].ravel(), torch.view_as_real(D).ravel(), al[0].ravel(), al[1].ravel()] +
                     [x.ravel() for s in A for x in s])
    W = psi.reshape(2 * n, N).contiguous()
    out, z = torch.zeros_like(W), [torch.zeros_like(W) for _ in range(4)]
    q = torch.zeros(n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.apply_hamiltonian_full(0, W, out, z[0], z[1], z[2], z[3], None, pots, qpe=q)
    ctx.sync()
    ctx.close()
    ref = []
    for c, (mu, sg) in enumerate(((0.3, 1.0), (0.25, -1.0))):
        w, o = psi[c], psi[1 - c]
        a = al[c]
        cpl = lambda f: f.to(torch.complex128)
        lap = sum(d(cpl(a), x, 2) for x in range(3)).real
        div = sum(d(cpl(A[c][x]), x, 1) for x in range(3)).real
        h = sg * (V[c] - mu + 0.25 * lap) * w - 0.5j * div * w + (D if c == 0 else D.conj()) * o
        for x in range(3):
            h = h - sg * 0.25 * (a * d(w, x, 2) + d(a * w, x, 2)) - 1j * A[c][x] * d(w, x, 1)
        ref.append(h)
    ref = torch.stack(ref)
    e = (psi.conj() * ref).real.sum(dim=(0, 2, 3, 4))
    dv = SPACING[0] * SPACING[1] * SPACING[2]
    got = out.reshape(psi.shape)
    e_dv = (e * dv).view(1, n, 1, 1, 1)
    assert close(q, e * dv)
    assert close(got, ref - e_dv * psi)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [1, 3, 65])
def test_densities(torch, shape, n):
    print("case: densities with gradients in the passes, %s, %d states" % (shape, n), flush=True)
    ctx, cfg = context(shape, n, po.SLDA)
    N = po.npts(cfg)
    psi = states(torch, shape, n, 5)
    d = spectral(torch, shape)
    fb = np.random.default_rng(n).uniform(0.0, 1.0, n)
    ctx.set_states(fb, None, None)
    dens = torch.zeros(12 * N, dtype=torch.float64, device="cuda")
    W = psi.reshape(2 * n, N).contiguous()
    torch.cuda.synchronize()
    ctx.calculate_densities(W, None, None, None, None, dens, 1)
    ctx.sync()
    ctx.close()
    f = torch.as_tensor(fb, device="cuda").view(n, 1, 1, 1)
    got = dens.view(12, N)
    for c, w in ((0, f), (1, 1.0 - f)):
        x = psi[c]
        lap = sum((x.conj() * d(x, a, 2)).real for a in range(3))
        j = [(x.conj() * d(x, a, 1)).imag for a in range(3)]
        b = 2 + 5 * c
        assert close(got[b], (w * x.abs() ** 2).sum(0).ravel())   # (3D: no transverse length)
        assert close(got[b + 1], (w * lap).sum(0).ravel())
        sj = 1.0 if c == 0 else -1.0
        for a in range(3):
            assert close(got[b + 2 + a], sj * (w * j[a]).sum(0).ravel())
