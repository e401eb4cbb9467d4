"""The transpose of the potentials in the forms of the functional: gradients
of the particle number in an interval against central differences with both
cut-offs, with and without the mean-field correction, and with a barrier above
the chemical potential (where the momenta of the regularisation turn
imaginary).

Bound: central differences of step 1e-6 are good to about 1e-12 (third
derivative) plus 1e-16 / 1e-6 = 1e-10 of the observable, whose gradient is
1e-4 of it or more: 1e-5 of the largest component."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cubic", [False, True])
@pytest.mark.parametrize("mf", [0, 1])
@pytest.mark.parametrize("amp", [0.15, 2.5])
def test_gradient(cubic, mf, amp):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from wslda_amd import adjoint, problems, td
    print("case: adjoint, cubic %d mf %d barrier %.2f eF" % (cubic, mf, amp), flush=True)
    s = problems.uniform_start(2, (16, 12, 8), n_states=40, scheme=45)
    p = s["params"]
    p.regularization = td.CUBIC_CUTOFF if cubic else td.SPHERICAL_CUTOFF
    p.mf_correction = mf
    L = p.nx * p.dx
    base = np.array([amp * 0.5, 0.12 * L, -0.08 * L, 2.0, -0.05, -0.1 * L, 0.15 * L, 2.5])
    w = adjoint.disk_weights(p, (0.0, 0.0, 0.0), 0.3 * L)
    prob = adjoint.AdjointProblem(p, s["wf"], s["pots"], s["fbeta"], s["kt"], s["cnt"], nsteps=14, K=6, dens_grad=w)

    def vext(k=None, name=None, h=0.0):
        v = adjoint.beams_vext(base)
        for j in range(v.ngauss):
            v.wz[j] = 0.0
        if name:
            getattr(v, name)[k] += h
        return v

    def value(v):
        prob.set_vext(v)
        prob.forward(keep_checkpoints=False)
        return prob.observable()

    prob.set_vext(vext())
    prob.forward()
    g = prob.backward()
    got, ref = [], []
    for k in range(2):
        for q, name in ((0, "amp"), (1, "cx"), (2, "cy"), (4, "wx"), (5, "wy")):
            got.append(g[k, q])
            ref.append((value(vext(k, name, 1e-6)) - value(vext(k, name, -1e-6))) / 2e-6)
    prob.close()
    got, ref = np.array(got), np.array(ref)
    assert np.isfinite(got).all() and np.abs(ref).max() > 0
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
