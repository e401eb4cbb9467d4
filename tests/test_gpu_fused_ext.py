"""tdw_step_fused on lattices with 18, 36 or 48 points along an axis, whose
arrays are complete after every step, against the CPU oracle."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests import tdgauss
from tests.test_gpu_parity import TOL, rel, say
from tests.test_gpu_resident import problem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    if not t.cuda.is_available():
        pytest.skip("no HIP device")
    return t


@pytest.mark.parametrize("shape,n", [((18, 18, 18), 7), ((36, 36, 36), 2), ((48, 24, 24), 3), ((18, 48, 48), 2),
                                     ((48, 48, 48), 1), ((36, 12, 12), 5), ((24, 36, 36), 2), ((48, 8, 12), 6)])
@pytest.mark.parametrize("scheme,functional", [(po.AB5AM5, po.SLDA), (po.AB4AM5, po.BDG), (po.AB3AM4, po.SLDA)])
def test_extended_fused_step_vs_oracle(torch, shape, n, scheme, functional):
    from wslda_amd import td
    say("case: extended fused step shape=%s n=%d scheme=%d functional=%d" % (shape, n, scheme, functional))
    cfg, wf, fb, kt, cnt, pots = problem(3, shape, n, scheme, functional)
    P = po.Problem(cfg, wf.copy(), fb, kt=kt, cnt=cnt, pots=pots.copy())
    prm = tdgauss.to_params(cfg, td.FP64)
    ctx = td.TDContext(prm, n, 0)
    assert td.lib().tdw_fused_supported(ctx.h) == 0
    ctx.set_states(fb, kt, cnt)
    R = td.TDRun(ctx, wf, pots, fused=True)
    P.initial_measure()
    R.initial_measure()
    # Hpsi of these states is of the order of the lattice's kinetic energy
    emax = 3 * 0.5 * (np.pi / 0.9) ** 2 * np.abs(P.wf).max()
    for it in range(6):
        grad = it in (2, 5)
        P.step(it, grad_last=grad)
        R.step(it, grad_last=grad)
        ctx.sync()
        assert rel(R.wf.cpu().numpy(), P.wf) < TOL, it
        assert rel(R.dens.cpu().numpy(), P.dens) < TOL, it
        assert rel(R.pots.cpu().numpy(), P.pots) < TOL, it
        assert rel(R.qpe.cpu().numpy(), P.qpe) < TOL, it
        assert np.abs(R.history()[0].cpu().numpy() - P.history()[0]).max() < TOL * emax, it
    ctx.close()
    # the split form of these lattices stays refused
    prm.precision = td.SPLIT
    ctx = td.TDContext(prm, n, 0)
    ctx.set_states(fb, kt, cnt)
    R = td.TDRun(ctx, wf, pots, fused=True)
    with pytest.raises(td.TDWError):
        R.step(0)
    ctx.close()


@pytest.mark.parametrize("shape,n", [((18, 18, 18), 7), ((36, 36, 36), 2), ((48, 24, 24), 3), ((24, 36, 36), 2),
                                     ((48, 8, 12), 6)])
def test_extended_fused_step_takes_the_masses_given(torch, shape, n):
    """alpha_a, alpha_b of the potential block enter H as the caller gives
    them, along x too: different for the components, varying in space."""
    from wslda_amd import td
    say("case: extended fused step with masses, shape=%s n=%d" % (shape, n))
    cfg, wf, fb, kt, cnt, pots = problem(3, shape, n, po.AB4AM5, po.SLDA)
    N = po.npts(cfg)
    X = np.meshgrid(*[2 * np.pi * np.arange(L) / L for L in shape], indexing="ij")
    w = (np.sin(X[0]) * np.cos(X[1]) + 0.5 * np.cos(X[2])).ravel()
    pots[4 * N:5 * N], pots[5 * N:6 * N] = 1.1 + 0.1 * w, 0.9 - 0.1 * w
    P = po.Problem(cfg, wf.copy(), fb, kt=kt, cnt=cnt, pots=pots.copy())
    ctx = td.TDContext(tdgauss.to_params(cfg, td.FP64), n, 0)
    ctx.set_states(fb, kt, cnt)
    R = td.TDRun(ctx, wf, pots, fused=True)
    P.initial_measure()
    R.initial_measure()
    emax = 3 * 0.5 * (np.pi / 0.9) ** 2 * np.abs(P.wf).max()
    for it in range(4):
        P.step(it, grad_last=it == 2)
        R.step(it, grad_last=it == 2)
        ctx.sync()
        assert rel(R.wf.cpu().numpy(), P.wf) < TOL, it
        assert rel(R.dens.cpu().numpy(), P.dens) < TOL, it
        assert rel(R.qpe.cpu().numpy(), P.qpe) < TOL, it
        assert np.abs(R.history()[0].cpu().numpy() - P.history()[0]).max() < TOL * emax, it
    ctx.close()
