"""Timed workloads of the td step: what a run of this framework spends its time on.

A case is one stretch of a user's time loop, through the public entry points
of wslda_amd.td and wslda_amd.adjoint:

  step      `steps` PECE steps of a run (TDRun.step), the last one a
            measurement step (gradients, tau, j), and the energies that a
            run logs after it;
  kernels   the same step called kernel by kernel (TDContext), as the driver
            of the reference calls its kernel interface;
  adjoint   the gradient of a final-time observable: the forward run with
            checkpoints and the backward sweep (AdjointProblem).

The start is a set of plane-wave BdG states (chemical potential 0.6 eF above
the mean field, Delta = 0.5 eF, temperature 0.05 eF, kF = 1) with seeded
phases and noise, under a Gaussian and (optionally) a harmonic trap.
"""
import math

import numpy as np
import torch

from wslda_amd import adjoint, td

PI = math.pi
EF = 0.5
MU, V0, DELTA0, TEMP = 0.2, -0.1, 0.5 * EF, 0.05 * EF
FUNC = {"slda": td.SLDA, "aslda": td.ASLDA, "bdg": td.BDG}
SCHEME = {"ab3am4": td.AB3AM4, "ab4am5": td.AB4AM5, "ab5am5": td.AB5AM5}
NHIST = {"ab3am4": 3, "ab4am5": 4, "ab5am5": 5}
PRED = {"ab3am4": (23 / 12, -16 / 12, 5 / 12), "ab4am5": (55 / 24, -59 / 24, 37 / 24, -9 / 24),
        "ab5am5": (1901 / 720, -2774 / 720, 2616 / 720, -1274 / 720, 251 / 720)}
CORR = {"ab3am4": (9 / 24, (19 / 24, -5 / 24, 1 / 24)),
        "ab4am5": (251 / 720, (646 / 720, -264 / 720, 106 / 720, -19 / 720)),
        "ab5am5": (251 / 720, (646 / 720, -264 / 720, 106 / 720, -19 / 720))}
SCLGTH = -1.0     # BdG coupling, in 1/kF


def _case(kind, dim, shape, n, functional="slda", scheme="ab5am5", precision="fp64", steps=10, spinsym=False,
          trap=False):
    return dict(kind=kind, dim=dim, nx=shape[0], ny=shape[1], nz=shape[2], n=n, functional=functional,
                scheme=scheme, precision=precision, steps=steps, spinsym=spinsym, trap=trap)


def listed():
    L = []

    def add(name, *a, **k):
        L.append(dict(_case(*a, **k), name=name))

    # the 1D run of the test configurations: 64 points, 128 states; every
    # step is a few dozen microseconds of work, so launches are what it costs
    add("1d-64", "step", 1, (64, 4, 4), 128, steps=20)
    # a small 2D run on a lattice that is neither square nor a power of two
    add("2d-36x18", "step", 2, (36, 18, 8), 300, scheme="ab3am4", steps=10)
    # the reference's testsuite size in 3D (12^3, 1781 states, AB4AM5)
    add("3d-12", "step", 3, (12, 12, 12), 1781, scheme="ab4am5", steps=10)
    # the 2D beam workload's lattice and transverse box (its gradient is the
    # adjoint case below)
    add("2d-64", "step", 2, (64, 64, 8), 1024, steps=10)
    # the plain 3D uniform workload: a quarter of its 16308 states (one of
    # four GPUs), in FP64 and in split precision
    add("3d-24-fp64", "step", 3, (24, 24, 24), 4096, steps=10)
    add("3d-24-split", "step", 3, (24, 24, 24), 4096, precision="split", steps=10)
    # the trapped gas on 32^3 in split precision
    add("3d-32-split", "step", 3, (32, 32, 32), 1536, precision="split", trap=True, steps=10)
    # the elongated tube's lattice in FP64
    add("3d-tube-fp64", "step", 3, (32, 32, 96), 320, steps=5)
    # ASLDA: derivatives on every half-step, effective mass and currents in H
    add("3d-24-aslda", "step", 3, (24, 24, 24), 2048, functional="aslda", steps=5)
    # 48^3, the smallest lattice of the reference's published cost tables
    # that the FFT plans take; outside the lattices with fused passes
    add("3d-48", "step", 3, (48, 48, 48), 200, steps=4)
    # the gradient of a final-time observable in the beam parameters
    add("adjoint-2d-64", "adjoint", 2, (64, 64, 8), 192, steps=20)
    # the kernel interface, one call per kernel, with gradients every step
    add("kernels-16", "kernels", 3, (16, 16, 16), 1000, steps=2)
    return L


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["1d", "2d", "3d", "3d", "3d", "aslda", "odd3d", "kernels", "adjoint"])
    scheme = rng.choice(["ab3am4", "ab4am5", "ab5am5", "ab5am5"])
    func = rng.choice(["slda", "slda", "bdg"])
    ss = rng.random() < 0.2
    if kind == "1d":
        nx = rng.choice([24, 32, 48, 54, 64, 72, 96, 108, 128, 192, 256])
        return _case("step", 1, (nx, 4, 4), _log_int(rng, 40, 1200), rng.choice(["slda", "slda", "aslda"]), scheme,
                     steps=rng.randint(8, 20), spinsym=ss)
    if kind == "2d":
        f = rng.choice(["slda", "bdg", "aslda"])
        if rng.random() < 0.5:
            nx = ny = rng.choice([8, 12, 16, 24, 32, 64])
        else:
            nx, ny = rng.choice([8, 12, 18, 24, 36, 48, 54]), rng.choice([8, 12, 16, 18, 24, 32, 48])
        n = _log_int(rng, 60, min(4000, (1 << 23) // (nx * ny)))
        return _case("step", 2, (nx, ny, 8), n, f, scheme, steps=rng.randint(4, 10), spinsym=ss)
    if kind in ("3d", "aslda"):
        shape = rng.choice([(12, 12, 12), (16, 16, 16), (24, 24, 24), (32, 32, 32), (16, 24, 24), (32, 16, 16),
                            (12, 32, 32)] + ([(8, 8, 8), (12, 8, 12), (32, 32, 96)] if kind == "3d" else []))
        N = shape[0] * shape[1] * shape[2]
        n = _log_int(rng, 50, min(4000, (1 << (25 if kind == "3d" else 24)) // N))
        if kind == "aslda":
            func = "aslda"
        return _case("step", 3, shape, n, func, scheme, rng.choice(["fp64", "split"]), rng.randint(3, 8), ss,
                     rng.random() < 0.3)
    if kind == "odd3d":
        shape = rng.choice([(48, 48, 48), (36, 36, 36), (18, 18, 18), (24, 32, 32), (48, 24, 24),
                            (36, 16, 18), (16, 48, 32), (54, 12, 36)])
        N = shape[0] * shape[1] * shape[2]
        return _case("step", 3, shape, _log_int(rng, 30, (1 << 24) // N), func, scheme, steps=rng.randint(2, 4),
                     spinsym=ss)
    if kind == "kernels":
        shape = rng.choice([(12, 12, 12), (16, 16, 16), (24, 24, 24), (18, 12, 16), (32, 32, 32)])
        N = shape[0] * shape[1] * shape[2]
        return _case("kernels", 3, shape, _log_int(rng, 30, (1 << 22) // N), func, scheme, steps=rng.randint(1, 3))
    nx = rng.choice([16, 24, 32, 64])
    return _case("adjoint", 2, (nx, nx, 8), _log_int(rng, 24, 192), "slda", scheme, steps=rng.randint(10, 20))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _shape(case):
    return (case["nx"], case["ny"], case["nz"])[:case["dim"]]


def _params(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dperp = 2.5 if case["dim"] == 1 else 1.0
    w = -0.5 / (4.0 * 4.0)
    ww = [w if d < case["dim"] else 0.0 for d in range(3)]
    vext = td.gauss_vext([(0.1 * EF, (1.0, 0.5, -0.5), tuple(ww))], omega=0.05 * EF if case["trap"] else 0.0)
    return td.make_params(case["dim"], nx, ny, nz, dx=1.0, dy=1.0 if case["dim"] >= 2 else dperp,
                          dz=1.0 if case["dim"] == 3 else dperp, functional=FUNC[case["functional"]],
                          mf_correction=1, scheme=SCHEME[case["scheme"]], mu_a=MU, mu_b=MU, ec=0.5 * PI * PI,
                          dt=0.005 / EF, vext=vext, sclgth=SCLGTH if case["functional"] == "bdg" else 0.0,
                          precision=td.SPLIT if case["precision"] == "split" else td.FP64,
                          spinsymmetry=int(case["spinsym"]))


def _kaxis(n):
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    return 2 * PI / n * torch.where(i < n // 2, i, i - n)


def _inputs(case, seed):
    """wf [2n, N], occupations, transverse momenta, degeneracies, potentials (12 N)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (seed + 1) + 7)
    n, dim, shape = case["n"], case["dim"], _shape(case)
    N = int(np.prod(shape))
    rand = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64, device="cuda")
    # lattice momenta drawn uniformly (spacing 1/kF)
    m = torch.stack([torch.floor(rand(n) * L) for L in shape])
    k = torch.stack([_kaxis(L)[m[d].long()] for d, L in enumerate(shape)])
    kt = cnt = None
    k2 = (k * k).sum(0)
    if dim == 2:
        kz = 2 * PI / case["nz"] * torch.floor(rand(n) * (case["nz"] // 2 + 1))
        kt, k2 = kz, k2 + kz * kz
    if dim == 1:
        q = 2 * PI / (4 * 2.5) * torch.floor(rand(2, n) * 3)
        kt, k2 = q.reshape(-1), k2 + (q * q).sum(0)
        cnt = 1 + torch.floor(rand(n) * 4).to(torch.int32)
    eta = 0.5 * k2 + V0 - MU
    E = torch.sqrt(eta * eta + DELTA0 ** 2)
    up = rand(n) < 0.5
    v2 = DELTA0 ** 2 / ((eta + E) ** 2 + DELTA0 ** 2)
    u, v = torch.sqrt(1 - v2), torch.sqrt(v2)
    U, V = torch.where(up, u, -v), torch.where(up, v, u)
    fb = 1.0 / (1.0 + torch.exp(torch.where(up, E, -E) / TEMP))
    r = torch.meshgrid(*[torch.arange(L, dtype=torch.float64, device="cuda") for L in shape], indexing="ij")
    r = torch.stack([x.reshape(-1) for x in r])
    wf = torch.empty((2 * n, N), dtype=torch.complex128, device="cuda")
    one = torch.ones(1, dtype=torch.float64, device="cuda")
    chunk = max(1, (1 << 25) // N)
    for a in range(0, n, chunk):
        b = min(n, a + chunk)
        ph = k[:, a:b].T @ r + 2 * PI * rand(b - a, 1)
        e = torch.polar(one, ph) / math.sqrt(N)
        wf[a:b], wf[n + a:n + b] = e * U[a:b, None], e * V[a:b, None]
        for c in (0, n):
            wf[c + a:c + b] += torch.polar(one * (0.02 / math.sqrt(N)), 2 * PI * rand(b - a, N))
    pots = torch.zeros(12 * N, dtype=torch.float64, device="cuda")
    pots[:2 * N] = V0
    pots[2 * N:4 * N:2] = DELTA0
    pots[4 * N:6 * N] = 1.094 if case["functional"] == "aslda" else 1.0
    return wf, fb, kt, cnt, pots


def _disk(params):
    return adjoint.disk_weights(params, (0.0, 0.0), 0.2 * params.nx)


def prepare(case, seed):
    wf, fb, kt, cnt, pots = _inputs(case, seed)
    p = _params(case)
    host = lambda t: None if t is None else t.cpu().numpy()
    if case["kind"] == "adjoint":
        P = adjoint.AdjointProblem(p, wf, host(pots), host(fb), host(kt), host(cnt), nsteps=case["steps"], K=5,
                                   dens_grad=_disk(p), taped_segments=2)
        return dict(case=case, problem=P)
    ctx = td.TDContext(p, case["n"], 0)
    ctx.set_states(host(fb), host(kt), host(cnt))
    R = td.TDRun(ctx, wf, host(pots), fused=case["dim"] == 3)
    R.initial_measure()
    ctx.sync()
    return dict(case=case, run=R, it=0)


def _kernel_step(R, it, f):
    """One PECE step through the kernel interface, with derivatives and the
    full densities of the corrected state (pca.c:1401-1570)."""
    c = R.ctx
    c.abm_step1(R.wf, f)
    c.normalize_wf(R.wf)
    c.compute_laplace(R.wf, R.lap)
    c.calculate_densities(R.wf, None, None, None, R.lap, R.dens, False)
    c.compute_potentials(it + 1, R.dens, R.pots)
    c.apply_hamiltonian(it + 1, R.wf, R.ddx, R.lap, R.pots, qpe=R.qpe)
    c.abm_step4(R.ddx, R.wf, f[-1])
    c.normalize_wf(R.wf)
    c.compute_derivatives(R.wf, R.ddx, R.ddy, R.ddz, R.lap)
    c.calculate_densities(R.wf, R.ddx, R.ddy, R.ddz, R.lap, R.dens, True)
    c.density_caculate_tau(R.dens)
    c.compute_potentials(it + 1, R.dens, R.pots)
    c.apply_hamiltonian(it + 1, R.wf, f[-1], R.lap, R.pots, qpe=R.qpe)
    return [f[-1]] + f[:-1]


def run(state):
    case = state["case"]
    if case["kind"] == "adjoint":
        P = state["problem"]
        R = P.forward()
        grad = P.backward()
        return dict(grad=grad[:1], observable=P.observable(R), dens=R.dens, lambda_y0=P.lambda_y0)
    R, it, steps = state["run"], state["it"], case["steps"]
    state["it"] = it + steps
    if case["kind"] == "kernels":
        f = state.get("hist") or R.f[:NHIST[case["scheme"]]]
        for k in range(steps):
            f = _kernel_step(R, it + k, f)
        state["hist"] = f
    else:
        for k in range(steps):
            R.step(it + k, grad_last=k == steps - 1)
        f = R.history()
    e = R.energy(it + steps)
    return dict(wf=R.wf, f=f[0], dens=R.dens, pots=R.pots, qpe=R.qpe, energy=e)


# ---------------------------------------------------------------------------
# the least work, and how far off another correct implementation may be
# ---------------------------------------------------------------------------
def work(case):
    """A PECE step cannot do without reading y and the history, writing the
    prediction and the partial corrector, reading them back with the new
    state as the result, and the new history entry (13 state arrays for
    AB5AM5; the history and the entry in FP32 in split precision).  The
    adjoint's backward step reads and writes about as much again, for the
    state, its history and their adjoints."""
    N, n, h = int(np.prod(_shape(case))), case["n"], NHIST[case["scheme"]]
    S = 32.0 * N * n
    if case["precision"] == "split":
        per = (2.0 + 0.5 * h + 0.5) + (1.0 + 0.5 + 1.0) + 1.0
    else:
        per = (1.0 + h + 2.0) + 3.0 + 2.0
    # transforms per half-step: one forward and one inverse; with a varying
    # mass also the three gradients and those of alpha psi
    ffts = 2 if case["functional"] != "aslda" else 7
    flops = 2.0 * n * N * (2 * ffts * 5.0 * math.log2(N) + 150.0)
    if case["kind"] == "adjoint":
        per, flops = per + 3.0 * h + 8.0, 3.0 * flops
    return {"bytes": case["steps"] * per * S, "flops": case["steps"] * flops}


def tolerance(case):
    # measured against exact(): at most 1.4e-14 in FP64 (f = H psi - <H> psi
    # of nearly stationary states loses two digits) and 6.1e-7 in split
    # precision (f again; the state and the densities stay within 3e-8)
    if case["precision"] == "split":
        return {"rel": 2.5e-6, "max": 2.5e-4}
    return {"rel": 1e-13, "max": 1e-11}


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch
# ---------------------------------------------------------------------------
P_NMIN, P_NMAX, DENSEPS = 1.0e-7, 1.0e-5, 1.0e-8


def _preg(n):
    x = torch.clamp(n, P_NMIN * 1.0001, P_NMAX * 0.9999)
    mid = 0.5 + 0.5 * torch.tanh(torch.tan(PI * (x - P_NMIN) / (P_NMAX - P_NMIN) - PI / 2))
    return torch.where(n <= P_NMIN, 0.0 * n, torch.where(n >= P_NMAX, torch.ones_like(n), mid))


def _dpreg(n):
    x = torch.clamp(n, P_NMIN * 1.0001, P_NMAX * 0.9999)
    a = PI * (x - P_NMIN) / (P_NMAX - P_NMIN) - PI / 2
    q = torch.cosh(torch.tan(a)) * torch.cos(a)
    d = 0.5 * PI / (q * q) / (P_NMAX - P_NMIN)
    return torch.where((n <= P_NMIN) | (n >= P_NMAX), 0.0 * n, d)


class _Functional:
    """Mean fields of SLDA (alpha = 1), ASLDA and BdG: constants of the
    reference's pca_settings.h, formulas of pca_edf.h and
    tdwslda_functionals.h."""
    G0, G1, GAMMA0 = 0.357, 0.642, -11.11

    def __init__(self, kind, dx):
        self.kind, self.dx = kind, dx
        self.A0, self.A1, self.A2 = (1.094, 0.156, -0.532) if kind == "aslda" else (1.0, 0.0, 0.0)

    def alpha(self, p):
        return (self.A0 + self.A1 * p * (1 - 2 / 3 * p ** 2 + p ** 4 / 5)
                + self.A2 * p ** 2 * (1 - p ** 2 + p ** 4 / 3))

    def dalpha(self, p):
        return self.A1 * (1 - 2 * p ** 2 + p ** 4) + self.A2 * (2 * p - 4 * p ** 3 + 2 * p ** 5)

    def plus(self, p):
        return 0.5 * (self.alpha(p) + self.alpha(-p))

    def polar(self, na, nb):
        n, r = na + nb, _preg(na + nb)
        p = r * (na - nb) / n
        d = _dpreg(n) * (na - nb) / n
        return p, r * 2 * nb / n ** 2 + d, -r * 2 * na / n ** 2 + d

    def base(self, p):
        return (self.G0 + self.G1 * p * p - self.alpha(p) * ((1 + p) / 2) ** (5 / 3)
                - self.alpha(-p) * ((1 - p) / 2) ** (5 / 3))

    def D(self, na, nb):
        n, p = na + nb, self.polar(na, nb)[0]
        return (6 * PI * PI * n) ** (5 / 3) / (20 * PI * PI) * self.base(p)

    def dD(self, n, p, dp):
        s = (2 * self.G1 * p - self.dalpha(p) * ((1 + p) / 2) ** (5 / 3)
             - 5 / 6 * self.alpha(p) * ((1 + p) / 2) ** (2 / 3) + self.dalpha(-p) * ((1 - p) / 2) ** (5 / 3)
             + 5 / 6 * self.alpha(-p) * ((1 - p) / 2) ** (2 / 3))
        return (0.5 * (6 * PI * PI * n) ** (2 / 3) * self.base(p)
                + (6 * PI * PI * n) ** (5 / 3) / (20 * PI * PI) * s * dp)

    def reg(self, t7, al):
        ec = 0.5 * PI * PI
        p0 = torch.sqrt((2 * t7 / al).to(torch.complex128))
        kc = torch.sqrt((2 * (ec + t7) / al).to(torch.complex128))
        w = torch.log((kc + p0) / (kc - p0))
        w = torch.where(w.imag < 0, w + 2j * PI, w)
        return kc * (1 - p0 / kc * 0.5 * w) / (2 * PI * PI), p0

    def mf(self, p0, g, n, al):
        lkF = (3 * PI * PI * n) ** (1 / 3)
        b = p0.real / (lkF + 1e-12)
        lx = b * lkF * self.dx / PI
        on = (g < -1e-10) & (lx > 1e-10)
        x = torch.where(on, lx, torch.full_like(lx, 0.5))
        R0 = 1 / (2 * PI * PI)
        lam = b * R0 / x * (1 - 0.5 * x * torch.log((1 + x) / (1 - x)))
        dlam = -b * R0 / (1 - x * x) - b * R0 / (x * x)
        v = lkF / (3 * n * al) * (lam + dlam * b * self.dx * lkF / PI)
        return torch.where(on, v, torch.zeros_like(v))

    def potentials(self, d, pt, ext):
        """(V_a, V_b, Delta, alpha_a, alpha_b, A) from the densities d and the previous potentials pt."""
        na, nb, nu = d["na"], d["nb"], d["nu"]
        n = na + nb
        if self.kind == "bdg":
            al = 0.5 * (pt["la"] + pt["lb"])
            wz, p0 = self.reg(MU - 0.5 * (pt["Va"] + pt["Vb"]), torch.ones_like(al))
            g = (1 / (1 / (4 * PI * SCLGTH * al) - wz / al)).real
            De = -nu * g
            V = ext + self.mf(p0, g, n, al) * De.abs() ** 2
            return dict(pt, Va=V, Vb=V, De=De)
        p, dpa, dpb = self.polar(na, nb)
        ap = self.plus(p)
        dap, dam = 0.5 * (self.dalpha(p) - self.dalpha(-p)), 0.5 * (self.dalpha(p) + self.dalpha(-p))
        Ca, Cb = ext + self.dD(n, p, dpa), ext + self.dD(n, p, dpb)
        out = dict(pt)
        if self.kind == "aslda":
            out["la"], out["lb"] = self.alpha(p), self.alpha(-p)
            am = 0.5 * (self.alpha(p) - self.alpha(-p))
            fa, fb = _preg(na), _preg(nb)
            out["Aa"] = [fa * (1 - out["la"]) * j / na for j in d["ja"]]
            out["Ab"] = [fb * (1 - out["lb"]) * j / nb for j in d["jb"]]
            j2a, j2b = sum(j * j for j in d["ja"]), sum(j * j for j in d["jb"])
            ta, tb = d["ta"], d["tb"]
            qa, qb = fa * j2a / (2 * na), fb * j2b / (2 * nb)
            Ca = Ca + dam * dpa * (ta - tb) / 2 + dap * dpa * (ta + tb) / 2
            Cb = Cb + dam * dpb * (ta - tb) / 2 + dap * dpb * (ta + tb) / 2
            Ca = Ca + ((ap + am - 1) / na - (dap + dam) * dpa) * qa - _dpreg(na) * (ap + am - 1) * j2a / (2 * na)
            Cb = Cb - (dap + dam) * dpb * qa
            Ca = Ca - (dap - dam) * dpa * qb
            Cb = Cb + ((ap - am - 1) / nb - (dap - dam) * dpb) * qb - _dpreg(nb) * (ap - am - 1) * j2b / (2 * nb)
        ne = n + DENSEPS
        C = ap * ne ** (1 / 3) / self.GAMMA0
        dC = [(dap * dp * ne ** (1 / 3) + ap * ne ** (-2 / 3) / 3) / self.GAMMA0 for dp in (dpa, dpb)]
        Va, Vb = pt["Va"], pt["Vb"]
        for _ in range(15):
            wz, p0 = self.reg(MU - 0.5 * (Va + Vb), ap)
            g = (ap / (C - wz)).real
            De = -nu * g
            t6, t7 = De.real * nu.real + De.imag * nu.imag, De.real ** 2 + De.imag ** 2
            m = self.mf(p0, g, n, ap) * t7
            Va = 0.75 * (Ca - dap * dpa / ap * t6 - dC[0] / ap * t7 + m) + 0.25 * Va
            Vb = 0.75 * (Cb - dap * dpb / ap * t6 - dC[1] / ap * t7 + m) + 0.25 * Vb
        out.update(Va=Va, Vb=Vb, De=De)
        return out


class _Exact:
    """The PECE run in complex128 with torch.fft (pca.c:1397-1571)."""

    def __init__(self, case, seed, theta=None):
        self.case, self.shape, self.dim = case, _shape(case), case["dim"]
        self.N, self.n = int(np.prod(self.shape)), case["n"]
        wf, self.fb, kt, cnt, pots = _inputs(case, seed)
        N, n = self.N, self.n
        self.dt = 0.005 / EF
        self.tr = {1: 100.0, 2: float(case["nz"]), 3: 1.0}[self.dim]
        self.VE = self.tr
        self.w = torch.ones(n, dtype=torch.float64, device="cuda")
        self.k2t = torch.zeros(n, dtype=torch.float64, device="cuda")
        if self.dim == 2:
            self.k2t = kt * kt
            self.w = torch.where(kt.abs() < 1e-12, self.w, 2 * self.w)
        if self.dim == 1:
            self.k2t = kt[:n] ** 2 + kt[n:] ** 2
            self.w = cnt.to(torch.float64)
        ks = torch.meshgrid(*[_kaxis(L) for L in self.shape], indexing="ij")
        self.k2 = sum(k * k for k in ks)
        self.ik = []
        for d, L in enumerate(self.shape):
            one = _kaxis(L)
            if L % 2 == 0:
                one[L // 2] = 0.0
            self.ik.append(1j * one.reshape([-1 if e == d else 1 for e in range(self.dim)]))
        x = torch.meshgrid(*[torch.arange(L, dtype=torch.float64, device="cuda") - L // 2 for L in self.shape],
                           indexing="ij")
        self.x = [t.reshape(-1) for t in x]
        self.x += [torch.zeros_like(self.x[0])] * (3 - self.dim)
        c = (1.0, 0.5, -0.5)
        w0 = -0.5 / 16.0
        if theta is None:
            ww = [w0 if d < self.dim else 0.0 for d in range(3)]
            theta = torch.tensor([0.1 * EF, *c, *ww], dtype=torch.float64, device="cuda")
        g = theta[0] * torch.exp(sum(theta[4 + d] * (self.x[d] - theta[1 + d]) ** 2 for d in range(3)))
        om = 0.05 * EF if case["trap"] else 0.0
        self.ext = g + 0.5 * om * om * sum(t * t for t in self.x)
        self.F = _Functional(case["functional"], 1.0)
        self.pt = dict(Va=pots[:N], Vb=pots[N:2 * N], De=torch.complex(pots[2 * N:4 * N:2], pots[2 * N + 1:4 * N:2]),
                       la=pots[4 * N:5 * N], lb=pots[5 * N:6 * N], Aa=[pots[6 * N:7 * N]] * 3,
                       Ab=[pots[9 * N:10 * N]] * 3)
        self.y = self.normal(wf)
        self.f = [torch.zeros_like(self.y) for _ in range(NHIST[case["scheme"]])]
        self.chunk = max(1, (1 << 25) // N)

    def normal(self, y):
        s = 1.0 / torch.sqrt((y.real ** 2 + y.imag ** 2).sum(1))
        n = self.n
        s = 1.0 / torch.sqrt(1 / s[:n] ** 2 + 1 / s[n:] ** 2)
        return y * torch.cat([s, s])[:, None]

    def spec(self, a, mul):
        """F^-1 mul F of the rows of a."""
        ax = tuple(range(-self.dim, 0))
        return torch.fft.ifftn(torch.fft.fftn(a.reshape(-1, *self.shape), dim=ax) * mul, dim=ax).reshape(a.shape)

    def rows(self, n):
        return [slice(a, min(n, a + self.chunk)) for a in range(0, n, self.chunk)]

    def densities(self, y, grad):
        n = self.n
        zero = torch.zeros(self.N, dtype=torch.float64, device="cuda")
        d = dict(na=zero, nb=zero, nu=zero + 0j, ta=zero, tb=zero, ja=[zero] * 3, jb=[zero] * 3)
        for s in self.rows(n):
            u, v = y[:n][s], y[n:][s]
            f, fm = (self.fb * self.w)[s, None], ((1 - self.fb) * self.w)[s, None]
            d["na"] = d["na"] + (f * (u.conj() * u).real).sum(0)
            d["nb"] = d["nb"] + (fm * (v.conj() * v).real).sum(0)
            d["nu"] = d["nu"] + (0.5 * (fm - f) * u * v.conj()).sum(0)
            if grad:
                k2 = self.k2t[s, None]
                d["ta"] = d["ta"] + (f * (u.conj() * (self.spec(u, -self.k2) - k2 * u)).real).sum(0)
                d["tb"] = d["tb"] + (fm * (v.conj() * (self.spec(v, -self.k2) - k2 * v)).real).sum(0)
                for e in range(self.dim):
                    d["ja"] = d["ja"][:e] + [d["ja"][e] + (f * (u.conj() * self.spec(u, self.ik[e])).imag).sum(0)] + d["ja"][e + 1:]
                    d["jb"] = d["jb"][:e] + [d["jb"][e] - (fm * (v.conj() * self.spec(v, self.ik[e])).imag).sum(0)] + d["jb"][e + 1:]
        for k in ("na", "nb", "nu", "ta", "tb"):
            d[k] = d[k] / self.tr
        d["ja"], d["jb"] = [j / self.tr for j in d["ja"]], [j / self.tr for j in d["jb"]]
        if self.case["spinsym"]:
            d["nu"] = 2 * d["nu"]
            for a, b in (("na", "nb"), ("ta", "tb")):
                d[a] = d[b] = d[a] + d[b]
            d["ja"] = d["jb"] = [p + q for p, q in zip(d["ja"], d["jb"])]
        if grad:
            for t, r in (("ta", "na"), ("tb", "nb")):
                lap = self.spec(d[r] + 0j, -self.k2).real
                d[t] = torch.clamp(0.5 * lap - d[t], min=0.0)
        return d

    def hpsi(self, y):
        """(H - <H>) psi and <H>."""
        n, p = self.n, self.pt
        hu, hv = [], []
        vm = self.case["functional"] == "aslda"
        if vm:
            la, lb = (self.spec(p[k] + 0j, -self.k2).real for k in ("la", "lb"))
            da, db = (sum(self.spec(p[k][e] + 0j, self.ik[e]).real for e in range(self.dim)) for k in ("Aa", "Ab"))
        for s in self.rows(n):
            u, v, k2 = y[:n][s], y[n:][s], self.k2t[s, None]
            for c, x, o, al, V, sg in ((hu, u, v, p["la"], p["Va"], 1.0), (hv, v, u, p["lb"], p["Vb"], -1.0)):
                if self.case["functional"] == "bdg":
                    al = torch.ones_like(al)
                h = sg * (V - MU + 0.5 * al * k2) * x + (p["De"] if sg > 0 else p["De"].conj()) * o
                if not vm:
                    h = h - 0.5 * sg * al * self.spec(x, -self.k2)
                else:
                    A, lal, div = (p["Aa"], la, da) if sg > 0 else (p["Ab"], lb, db)
                    h = h - 0.25 * sg * (al * self.spec(x, -self.k2) + self.spec(al * x, -self.k2) - lal * x)
                    h = h - 0.5j * div * x - 1j * sum(A[e] * self.spec(x, self.ik[e]) for e in range(self.dim))
                c.append(h)
        h = torch.cat(hu + hv)
        e = (y.conj() * h).real.sum(1)
        e = e[:n] + e[n:]
        return h - torch.cat([e, e])[:, None] * y, e

    def step(self, grad):
        vm = self.case["functional"] == "aslda"
        sch = self.case["scheme"]
        a0, ac = CORR[sch]
        yp = self.y - 1j * self.dt * sum(b * f for b, f in zip(PRED[sch], self.f))
        c = self.y - 1j * self.dt * sum(a * f for a, f in zip(ac, self.f))
        yp = self.normal(yp)
        self.pt = self.F.potentials(self.densities(yp, vm), self.pt, self.ext)
        self.y = self.normal(c - 1j * self.dt * a0 * self.hpsi(yp)[0])
        del yp, c
        self.d = self.densities(self.y, vm or grad)
        self.pt = self.F.potentials(self.d, self.pt, self.ext)
        self.f.pop()
        h, self.e = self.hpsi(self.y)
        self.f.insert(0, h)

    def pots(self):
        p, out = self.pt, torch.zeros(12 * self.N, dtype=torch.float64, device="cuda")
        N = self.N
        out[:N], out[N:2 * N], out[2 * N:4 * N] = p["Va"], p["Vb"], torch.view_as_real(p["De"]).reshape(-1)
        out[4 * N:5 * N], out[5 * N:6 * N] = p["la"], p["lb"]
        if self.case["functional"] == "aslda":
            for e in range(self.dim):
                out[(6 + e) * N:(7 + e) * N], out[(9 + e) * N:(10 + e) * N] = p["Aa"][e], p["Ab"][e]
        return out

    def dens(self):
        d, z = self.d, self.d["na"]
        return torch.cat([torch.view_as_real(d["nu"]).reshape(-1), d["na"], d["ta"], *d["ja"], z * 0 + d["nb"],
                          d["tb"], *d["jb"]])

    def energy(self):
        d, p, F, VE = self.d, self.pt, self.F, self.VE
        na, nb = d["na"], d["nb"]
        qa, qb = (_preg(n) * sum(j * j for j in js) / n for n, js in ((na, d["ja"]), (nb, d["jb"])))
        ta, tb = d["ta"] - qa, d["tb"] - qb
        if self.case["functional"] == "bdg":
            la, lb, pot = p["la"], p["lb"], 0.0 * na
        else:
            po = F.polar(na, nb)[0]
            la, lb, pot = F.alpha(po), F.alpha(-po), F.D(na, nb)
        L = [torch.zeros((), dtype=torch.float64, device="cuda")] * 2
        if self.dim >= 2:
            L = [(self.x[0] * j[1] - self.x[1] * j[0]).sum() for j in (d["ja"], d["jb"])]
        z = torch.zeros((), dtype=torch.float64, device="cuda")
        e = [(0.5 * (la * ta + lb * tb)).sum(), pot.sum(), -(p["De"].conj() * d["nu"]).real.sum(),
             (0.5 * (qa + qb)).sum(), ((na + nb) * self.ext).sum(), z, z, na.sum(), nb.sum(), L[0], L[1]]
        return (torch.stack(e) * VE).cpu().numpy()


def exact(case, seed):
    if case["kind"] == "adjoint":
        if case["n"] * case["nx"] * case["ny"] * case["steps"] > 18 << 20:
            return None
        w = -0.5 / 16.0
        theta = torch.tensor([0.1 * EF, 1.0, 0.5, -0.5, w, w, 0.0], dtype=torch.float64, device="cuda",
                             requires_grad=True)
        X = _Exact(case, seed, theta)
        y0 = X.y.clone().requires_grad_(True)
        X.y = y0
        for _ in range(case["steps"]):
            X.step(False)
        g = torch.as_tensor(_disk_exact(case), device="cuda")
        O = (g * (X.d["na"] + X.d["nb"])).sum()
        O.backward()
        grad = theta.grad.cpu().numpy().reshape(1, 7)
        with torch.no_grad():
            return dict(grad=grad, observable=float(O.detach()), dens=X.dens().detach(), lambda_y0=y0.grad)
    with torch.no_grad():
        X = _Exact(case, seed)
        for k in range(case["steps"]):
            X.step(k == case["steps"] - 1 or case["kind"] == "kernels")
        return dict(wf=X.y, f=X.f[0], dens=X.dens(), pots=X.pots(), qpe=X.e, energy=X.energy())


def _disk_exact(case):
    x, y = np.meshgrid(np.arange(case["nx"]) - case["nx"] // 2, np.arange(case["ny"]) - case["ny"] // 2,
                       indexing="ij")
    return ((x ** 2 + y ** 2 < (0.2 * case["nx"]) ** 2) * float(case["nz"])).ravel()
