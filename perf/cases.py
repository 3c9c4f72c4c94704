"""Workloads by which the speed of this framework is judged.

Each case is one call, or a short chain of calls, that a program using the package makes:
propagating one Wigner function over some steps (Lie and Strang schemes, the damping models,
Gross-Pitaevskii, every kind of potential), an ensemble of them, the 16-plane Wigner-Dirac
state, the gradient of a control problem (forward and adjoint), and the plain axis transforms.
`listed()` names twelve of them, `draw()` gives more of the same ranges: sides are the powers of
two that the library accepts, X and P drawn apart, step counts odd and even.

A program keeps the plan and the initial state; `run()` clones the state and propagates the
clone, which is what comes back together with the per-step record.  The record of a complex64
run is taken in single precision, as the state it was summed from.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

DEVICE = "cuda:0"
HBAR, MASS = 1.0, 1.0

# potentials: C strings for the library, and torch functions of (t, x) for V and dV/dx at t = 0.
#   well     the damped double well of the benchmark        (polynomial coefficient rows)
#   quartic  the quartic oscillator of the benchmark        (polynomial coefficient rows)
#   trap     harmonic trap, as the Gross-Pitaevskii and ODM notebooks use
#   driven   harmonic trap with a field cos(t) x            (one coefficient row per time index)
#   soft     soft Coulomb                                   (tabulated once on the host)
#   pulsed   double well with a Gaussian sin(t) pulse       (program evaluated per cell and step)
POTENTIALS = {
    "well": ("0.1*pow(x,4) - pow(x,2)", "0.4*pow(x,3) - 2.0*x",
             lambda t, x: 0.1 * x ** 4 - x ** 2, lambda x: 0.4 * x ** 3 - 2.0 * x),
    "quartic": ("0.5*pow(x,2) + 0.1*pow(x,4)", "x + 0.4*pow(x,3)",
                lambda t, x: 0.5 * x ** 2 + 0.1 * x ** 4, lambda x: x + 0.4 * x ** 3),
    "trap": ("0.5*pow(x,2)", "x", lambda t, x: 0.5 * x ** 2, lambda x: x),
    "driven": ("0.5*pow(x,2) - 0.3*cos(t)*x", "x - 0.3*cos(t)",
               lambda t, x: 0.5 * x ** 2 - 0.3 * math.cos(t) * x, lambda x: x - 0.3),
    "soft": ("-2.0/sqrt(x*x + 1.0)", "2.0*x/pow(x*x + 1.0, 1.5)",
             lambda t, x: -2.0 / torch.sqrt(x * x + 1.0), lambda x: 2.0 * x / (x * x + 1.0) ** 1.5),
    "pulsed": ("0.1*pow(x,4) - pow(x,2) + 0.05*sin(t)*exp(-x*x)",
               "0.4*pow(x,3) - 2.0*x - 0.1*x*sin(t)*exp(-x*x)",
               lambda t, x: 0.1 * x ** 4 - x ** 2 + 0.05 * math.sin(t) * torch.exp(-x * x),
               lambda x: 0.4 * x ** 3 - 2.0 * x),
}
# friction f(p) of the damping models: C string and torch function
FRICTION = {"CaldeiraLeggett": ("fabs(p)", torch.abs),
            "ODM": ("p*p/sqrt(p*p + 0.5)", lambda p: p * p / torch.sqrt(p * p + 0.5))}
GAMMA = {"none": 0.0, "CaldeiraLeggett": 0.1, "ODM": 0.07 / 4.0}
D_THETA = {"none": 0.0, "CaldeiraLeggett": 0.1, "ODM": 0.0}
L_MATERIAL = 3.0


# ---------------------------------------------------------------------------------- the cases
def wigner(X, P, steps, *, scheme="lie", damping="none", gp=0.0, potential="well", precision="fp64"):
    # the absorbing edge mask is on, as in the reference's kernels
    return {"kind": "wigner", "X": X, "P": P, "steps": steps, "scheme": scheme, "damping": damping, "gp": gp,
            "potential": potential, "precision": precision, "amp": 12.0 if max(X, P) > 256 else 10.0, "dt": 0.005}


def ensemble(members, least, most, steps, precision, mix):
    return {"kind": "ensemble", "members": members, "least": least, "most": most, "steps": steps,
            "precision": precision, "mix": mix, "dt": 0.01}


def dirac(X, P, steps, *, damping="none", potential="soft", precision="fp64"):
    return {"kind": "dirac", "X": X, "P": P, "steps": steps, "damping": damping, "potential": potential,
            "precision": precision, "dt": 0.002}


def control(side, steps, terms, keep):
    return {"kind": "control", "X": side, "P": side, "steps": steps, "terms": terms, "keep": keep, "dt": 0.01}


def axes(X, P, precision):
    return {"kind": "axes", "X": X, "P": P, "precision": precision}


def listed():
    return [
        # a few steps between two saved frames on the smallest grid: launches and fixed work per call
        dict(wigner(128, 128, 21, damping="CaldeiraLeggett"), name="frame_128"),
        # a notebook's run with a time-dependent potential that is no polynomial, sides apart
        dict(wigner(512, 256, 101, scheme="strang", potential="pulsed"), name="pulsed_256x512"),
        # the notebooks' usual 512^2 grid, damped, in the complex64 form
        dict(wigner(512, 512, 150, damping="CaldeiraLeggett", potential="driven", precision="fp32"), name="damped_512_c64"),
        # Gross-Pitaevskii, Strang scheme with friction, as its notebook
        dict(wigner(512, 512, 60, scheme="strang", damping="CaldeiraLeggett", gp=0.5, potential="trap"), name="gp_512"),
        # the ODM Lindblad dissipator
        dict(wigner(512, 512, 60, damping="ODM", potential="trap"), name="odm_512"),
        # the benchmark's damped double well
        dict(wigner(1024, 1024, 100, damping="CaldeiraLeggett"), name="damped_1024"),
        # the largest single grid, without damping
        dict(wigner(2048, 2048, 50, potential="quartic"), name="plain_2048"),
        # a parameter scan: uneven members in the complex64 form, one launch per sweep for all
        dict(ensemble(64, 128, 1024, 40, "fp32", 11), name="scan_uneven_c64"),
        # many grids at once in complex128, far beyond the caches
        dict(ensemble(32, 1024, 1024, 20, "fp64", 12), name="batch_1024"),
        # the 16-plane Wigner-Dirac state of the notebooks
        dict(dirac(512, 512, 40), name="dirac_512"),
        # gradient of a control field: forward, recomputation and adjoint
        dict(control(512, 100, 64, 25), name="control_512"),
        # the plan/exec calls that replace cuFFT's: both axes, both directions
        dict(axes(1024, 512, "fp64"), name="axes_512x1024"),
    ]


def _side(rng, least, most):
    return 2 ** rng.randint(int(math.log2(least)), int(math.log2(most)))


def _steps(rng, least, most):
    return int(round(math.exp(rng.uniform(math.log(least), math.log(most)))))


def draw(rng: random.Random):
    kind = rng.choices(["wigner", "ensemble", "dirac", "control", "axes"], [8, 3, 2, 1, 1])[0]
    if kind == "wigner":
        X, P = _side(rng, 128, 2048), _side(rng, 128, 2048)
        scheme, damping = rng.choice(["lie", "strang"]), rng.choice(["none", "CaldeiraLeggett", "CaldeiraLeggett", "ODM"])
        gp = rng.choice([0.0, 0.5]) if scheme == "strang" else 0.0
        if damping == "ODM" or gp:
            X, P = min(X, 1024), min(P, 1024)
        steps = _steps(rng, 8, max(16.0, min(300.0, 2.0e8 / (X * P))))
        return wigner(X, P, steps, scheme=scheme, damping=damping, gp=gp,
                      potential=rng.choice(["trap", "driven"] if damping == "ODM" or gp else sorted(POTENTIALS)),
                      precision=rng.choice(["fp64", "fp64", "fp32"]))
    if kind == "ensemble":
        least = _side(rng, 128, 1024)
        most = _side(rng, least, 1024)
        members = max(3, min(rng.randint(5, 96), 24 * 1024 ** 2 // (most * most)))
        return ensemble(members, least, most, _steps(rng, 8, 25), rng.choice(["fp64", "fp32"]), rng.randrange(1000))
    if kind == "dirac":
        X, P = _side(rng, 128, 1024), _side(rng, 128, 1024)
        return dirac(X, P, _steps(rng, 4, max(6.0, min(60.0, 8.0e6 / (X * P)))),
                     damping=rng.choice(["none", "CaldeiraLeggett"]), potential=rng.choice(["soft", "trap"]),
                     precision=rng.choice(["fp64", "fp32"]))
    if kind == "control":
        side = _side(rng, 128, 512)
        return control(side, _steps(rng, 20, 110), rng.choice([8, 32, 64]), rng.choice([20, 25, 50]))
    return axes(_side(rng, 64, 2048), _side(rng, 64, 2048), rng.choice(["fp64", "fp32"]))


def _members(case):
    """[(side, a, b)] of an ensemble: V = a x^4 - b x^2 on a square grid."""
    rng = random.Random(case["mix"])
    lo, hi = int(math.log2(case["least"])), int(math.log2(case["most"]))
    return [(2 ** rng.randint(lo, hi), rng.uniform(0.05, 0.2), rng.uniform(0.5, 2.0)) for _ in range(case["members"])]


# ---------------------------------------------------------------------------------- the inputs
def _axis(n, step):
    """Coordinates of n FFT-ordered indices."""
    k = torch.arange(n, dtype=torch.float64, device=DEVICE)
    return step * (torch.remainder(k + n // 2, n) - n // 2)


def _linspaced(n, amp):
    """The same coordinates as a notebook's linspace gives them: the ODM tables take the sign of
    p +/- hbar lambda/2, which at p = lambda = 0 is that of linspace's rounding."""
    return torch.from_numpy(np.fft.fftshift(np.linspace(-amp, amp - 2.0 * amp / n, n))).to(DEVICE)


def _grid(X, P, x_amp, p_amp):
    """x [1, X], p [P, 1] and their conjugates lambda [1, X], theta [P, 1]; dx, dp."""
    dx, dp = 2.0 * x_amp / X, 2.0 * p_amp / P
    return (_axis(X, dx)[None, :], _axis(P, dp)[:, None], _axis(X, math.pi / x_amp)[None, :],
            _axis(P, math.pi / p_amp)[:, None], dx, dp)


def _cat(x, p, dx, dp, rng):
    """Superposition of two Gaussians with its interference term, normalised."""
    a, s, p0, phi = rng.uniform(1.0, 2.5), rng.uniform(0.8, 1.25), rng.uniform(-1.0, 1.0), rng.uniform(0.0, 2.0 * np.pi)
    fall = torch.exp(-(s * (p - p0)) ** 2)
    W = fall * (torch.exp(-((x - a) / s) ** 2) + torch.exp(-((x + a) / s) ** 2)
                + 2.0 * torch.exp(-(x / s) ** 2) * torch.cos(2.0 * a * (p - p0) + phi))
    return W / (W.sum() * dx * dp)


def _spinor(x, theta, dx, dp, rng):
    """[4, 4, P, X]: Wigner matrix of a positive-energy Gaussian spinor."""
    x0, px, s = rng.uniform(-3.0, -1.0), rng.uniform(4.0, 7.0), rng.uniform(0.9, 1.2)
    up, down = math.sqrt(px * px + 1.0) + 1.0, px

    def psi(y):
        rho = torch.exp(1j * px * y) * torch.exp(-0.5 * ((y - x0) / s) ** 2)
        return [rho * up, None, None, rho * down]

    left, right = psi(x - 0.5 * theta), psi(x + 0.5 * theta)
    W = torch.zeros((4, 4, theta.shape[0], x.shape[1]), dtype=torch.complex128, device=DEVICE)
    for i in (0, 3):
        for j in (0, 3):
            W[i, j] = torch.fft.ifft(left[i] * right[j].conj(), dim=0)
    return W / (torch.einsum("iipx->", W).real * dx * dp)


def _initial(case, seed):
    """The states a case starts from, complex128 on the GPU."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "wigner":
        x, p, _, _, dx, dp = _grid(case["X"], case["P"], case["amp"], case["amp"])
        return [_cat(x, p, dx, dp, rng).to(torch.complex128)]
    if case["kind"] == "ensemble":
        out = []
        for side, _, _ in _members(case):
            x, p, _, _, dx, dp = _grid(side, side, 10.0, 10.0)
            out.append(_cat(x, p, dx, dp, rng).to(torch.complex128))
        return out
    if case["kind"] == "dirac":
        x, p, _, theta, dx, dp = _grid(case["X"], case["P"], 18.0, 16.0)
        return [_spinor(x, theta, dx, dp, rng)]
    if case["kind"] == "control":
        x, p, _, _, dx, dp = _grid(case["X"], case["P"], 10.0, 10.0)
        return [_cat(x + 0.5, p, dx, dp, rng).to(torch.complex128)]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    return [torch.randn((case["P"], case["X"]), dtype=torch.complex128, device=DEVICE, generator=g)]


def _control_inputs(case, seed):
    """Fourier coefficients of the field (N(0, 0.1), as the benchmark's), the target, the still part of V."""
    rng = np.random.default_rng(seed + 1)
    params = torch.tensor(rng.normal(0.0, 0.1, case["terms"]), dtype=torch.float64, device=DEVICE)
    x, p, _, _, _, _ = _grid(case["X"], case["P"], 10.0, 10.0)
    target = torch.exp(-((x - rng.uniform(1.0, 2.5)) ** 2) - p ** 2) / math.pi
    base = np.zeros(9)
    base[4], base[2] = 0.25, -1.0
    return params, target, base


def _state_type(precision):
    return torch.complex128 if precision == "fp64" else torch.complex64


def prepare(case, seed):
    W0 = _initial(case, seed)
    kind = case["kind"]
    if kind == "wigner":
        from pywignercuda_amd.wigner2d import Wigner2D

        v, dv, _, _ = POTENTIALS[case["potential"]]
        damping = case["damping"]
        plan = Wigner2D(case["X"], case["P"], case["amp"], case["amp"], HBAR, MASS, case["dt"], potential=v,
                        dpotential=dv, scheme=case["scheme"], gamma=GAMMA[damping], D_theta=D_THETA[damping],
                        damping=None if damping == "none" else damping,
                        fp_damping=None if damping == "none" else FRICTION[damping][0],
                        L_material=L_MATERIAL if damping == "ODM" else None, gp_coeff=case["gp"],
                        precision=case["precision"], time_rows=case["steps"] + 2, device=DEVICE)
        return {"case": case, "plan": plan, "W0": W0[0].to(plan.dtype)}
    if kind == "ensemble":
        from pywignercuda_amd.wigner2d import WignerEnsemble

        members = []
        for side, a, b in _members(case):
            table = np.zeros((1, 9))
            table[0, 4], table[0, 2] = a, -b
            members.append(dict(X=side, P=side, X_amp=10.0, P_amp=10.0, potential=f"{a!r}*pow(x,4) - {b!r}*pow(x,2)",
                                dpotential=f"{4 * a!r}*pow(x,3) - {2 * b!r}*x", pot_table=table, mask=False))
        plan = WignerEnsemble(members, HBAR, MASS, case["dt"], scheme="lie", precision=case["precision"], device=DEVICE)
        return {"case": case, "plan": plan, "W0": [w.to(plan.dtype) for w in W0]}
    if kind == "dirac":
        from pywignercuda_amd.dirac import WignerDirac4x4

        damped = case["damping"] != "none"
        plan = WignerDirac4x4(case["X"], case["P"], 18.0, 16.0, 1.0, 1.0, case["dt"],
                              potentials=(POTENTIALS[case["potential"]][0], "0.", "0.", "0."),
                              gamma=0.05 if damped else 0.0, damping="CaldeiraLegget" if damped else None,
                              D_theta=0.01 if damped else 0.0, truncate_constants=False,
                              precision=case["precision"], device=DEVICE)
        return {"case": case, "plan": plan, "W0": plan.to_device(W0[0])}
    if kind == "control":
        from pywignercuda_amd.wigner2d import Wigner2D

        params, target, base = _control_inputs(case, seed)
        plan = Wigner2D(case["X"], case["P"], 10.0, 10.0, HBAR, MASS, case["dt"],
                        potential="0.25*pow(x,4) - pow(x,2)", dpotential="pow(x,3) - 2*x", mask=False,
                        pot_table=np.tile(base, (case["steps"] + 2, 1)), device=DEVICE)
        return {"case": case, "plan": plan, "W0": W0[0].requires_grad_(), "params": params.requires_grad_(),
                "target": target, "base": base}
    from pywignercuda_amd import cufft_wrapper as cw

    shape = (case["P"], case["X"])
    double = case["precision"] == "fp64"
    return {"case": case, "W0": W0[0].to(_state_type(case["precision"])),
            "axis0": (cw.Plan_Z2Z_2D_Axis0 if double else cw.Plan_C2C_2D_Axis0)(shape),
            "axis1": (cw.Plan_Z2Z_2D_Axis1 if double else cw.Plan_C2C_2D_Axis1)(shape)}


# ---------------------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind, n = case["kind"], case.get("steps")
    if kind in ("wigner", "dirac"):
        W = state["W0"].clone()
        record = state["plan"].run(W, n)
        return {"W": W, "record": record if W.dtype == torch.complex128 else record.float()}
    if kind == "ensemble":
        Ws = [w.clone() for w in state["W0"]]
        record = state["plan"].run(Ws, n)
        # the members as one tensor: a scan's result is saved as a whole
        return {"W": torch.cat([w.reshape(-1) for w in Ws]),
                "record": record if Ws[0].dtype == torch.complex128 else record.float()}
    if kind == "control":
        from pywignercuda_amd.adjoint import fourier_control_table, propagate

        table = fourier_control_table(state["params"], n, case["dt"], 20.0, state["base"])
        W = propagate(state["plan"], table, state["W0"], n, checkpoint_every=case["keep"])
        plan = state["plan"]
        loss = 1.0 - 2.0 * math.pi * plan.dX * plan.dP * (W * state["target"]).sum()
        g_params, g_W0 = torch.autograd.grad(loss, (state["params"], state["W0"]))
        return {"loss": loss.detach(), "W": W.detach(), "g_params": g_params, "g_W0": g_W0}
    from pywignercuda_amd import cufft_wrapper as cw

    W = state["W0"].clone()
    cw.fft_Z2Z(W, W, state["axis1"])
    cw.fft_Z2Z(W, W, state["axis0"])
    V = state["W0"].clone()
    cw.ifft_Z2Z_normalized(V, V, state["axis0"])
    cw.ifft_Z2Z(V, V, state["axis1"])
    return {"forward": W, "inverse": V}


# ---------------------------------------------------------------------------------- its size
def work(case):
    """Bytes: the state in and out once per step (every step couples all rows and then all columns),
    or once per transform.  Flops: 5 N log2 N per complex transform, 6 per complex product."""
    size = 16 if case.get("precision", "fp64") == "fp64" else 8

    def grid(X, P, transforms, products, scale=1.0):
        lx, lp = math.log2(X), math.log2(P)
        return X * P * scale * (transforms[0] * 5.0 * lx + transforms[1] * 5.0 * lp + 6.0 * products)

    kind = case["kind"]
    if kind == "ensemble":
        cells = sum(s * s for s, _, _ in _members(case))
        flops = sum(grid(s, s, (2, 2), 2) for s, _, _ in _members(case))
        return {"bytes": 2.0 * size * cells * case["steps"], "flops": flops * case["steps"]}
    cells = case["X"] * case["P"]
    if kind == "axes":
        return {"bytes": 2.0 * size * cells * 4, "flops": grid(case["X"], case["P"], (2, 2), 0)}
    steps = case["steps"]
    if kind == "dirac":
        along_p = 6 if case["damping"] != "none" else 2
        return {"bytes": 2.0 * 16 * size * cells * steps,
                "flops": grid(case["X"], case["P"], (2, along_p), 6, 16.0) * steps}
    if kind == "control":
        # forward, recomputation, and the adjoint (which reads the forward state too)
        return {"bytes": 16.0 * cells * steps * (2 + 2 + 3),
                "flops": grid(case["X"], case["P"], (6, 7), 7) * steps}
    along_x, along_p, products = 2, 2, 2
    if case["scheme"] == "strang" and (case["gp"] or case["damping"] != "none"):
        along_p += 2
    if case["damping"] == "CaldeiraLeggett":
        along_p, products = along_p + 6, products + 3
    if case["damping"] == "ODM":
        along_x, along_p, products = along_x + 4, along_p + 3, products + 6
    if case["gp"]:
        products += 2
    return {"bytes": 2.0 * size * cells * steps,
            "flops": grid(case["X"], case["P"], (along_x, along_p), products) * steps}


# ---------------------------------------------------------------------------------- in 64 bits
def _rows(W, x, p, dv, v0, d, raw):
    """Record row of a normalised state: moments, <dV/dx> family, energy, negative area, norms."""
    r = W.real
    mean = lambda A: d * (r * A).sum()  # noqa: E731
    zero = torch.zeros((), dtype=torch.float64, device=DEVICE)
    return torch.stack([mean(x), mean(x * x), mean(p), mean(p * p), mean(x * p), mean(dv), mean(p * dv),
                        mean(x * dv), mean(p * p / (2.0 * MASS) + v0), d * torch.clamp(r, max=0.0).sum(),
                        d * r.sum(), raw.real, raw.imag, zero, zero, zero])


class _Exact:
    """The steps of one Wigner function in torch's complex128."""

    def __init__(self, X, P, amp, dt, V, dV, scheme="lie", damping="none", gp=0.0, mask=True):
        self.x, self.p, self.lam, self.th, self.dx, self.dp = _grid(X, P, amp, amp)
        self.dt, self.V, self.scheme, self.damping, self.gp = dt, V, scheme, damping, gp
        self.d = self.dx * self.dp
        self.frac = 1.0 if scheme == "lie" else 0.5
        self.K = torch.exp(-1j * dt * self.lam * self.p / MASS)
        self.r = torch.exp(-self.frac * D_THETA[damping] * self.th ** 2 * dt)
        if mask:
            xm, w2 = self.dx * (X - 1.0) / 2.0, (10.0 * self.dx) ** 2
            self.r = self.r * (1.0 - torch.exp(-((self.x - xm) ** 2) / w2)) * (1.0 - torch.exp(-((self.x + xm) ** 2) / w2))
        self.dv = dV(self.x) * torch.ones_like(self.x)
        self.v0 = V(0.0, self.x)
        if damping == "CaldeiraLeggett":
            f = FRICTION[damping][1](self.p)
            self.sigma = torch.where(self.p >= 0.0, f, -f)
        if damping == "ODM":
            g = lambda q: torch.sqrt(L_MATERIAL * FRICTION["ODM"][1](q.abs() + HBAR / (2.0 * L_MATERIAL)))  # noqa: E731
            p, lam = _linspaced(P, amp)[:, None], _linspaced(X, math.pi / amp * X / 2.0)[None, :]
            qp, qm = p + 0.5 * HBAR * lam, p - 0.5 * HBAR * lam
            self.g = g(qp), g(qm), g(qp) * torch.sign(qp), g(qm) * torch.sign(qm)
            xp, xm = self.x + 0.5 * HBAR * self.th, self.x - 0.5 * HBAR * self.th
            self.h = torch.cos(xp), torch.cos(xm), torch.sin(xp), torch.sin(xm)

    def kinetic(self, W):
        return torch.fft.ifft(torch.fft.fft(W, dim=1) * self.K, dim=1)

    def density(self, W):
        return W.real.sum(0) * self.dp

    def potential(self, W, t, rho=None):
        u = 0.5 * HBAR * self.th
        phase = (self.V(t, self.x - u) - self.V(t, self.x + u)) / HBAR
        if rho is not None:
            f = torch.fft.fft(rho.to(torch.complex128))[None, :]
            shift = torch.exp(0.5j * self.lam * self.th)
            phase = phase + self.gp / HBAR * (torch.fft.ifft(f / shift, dim=1) - torch.fft.ifft(f * shift, dim=1)).real
        return torch.fft.ifft(torch.fft.fft(W, dim=0) * self.r * torch.exp(-1j * self.frac * self.dt * phase), dim=0)

    def friction(self, W):
        a = 1j * self.dt * GAMMA["CaldeiraLeggett"]
        D = lambda Y: torch.fft.ifft(self.th * torch.fft.fft(self.sigma * Y, dim=0), dim=0)  # noqa: E731
        L = W + (2.0 / 3.0) * a * D(W)
        L = L + a * D(L)
        return W + 2.0 * a * D(L)

    def lindblad(self, W):
        (gp, gm, gsp, gsm), (cp, cm, sp, sm) = self.g, self.h
        F = torch.fft.fft(W, dim=1)
        term = lambda g: torch.fft.fft(torch.fft.ifft(F * g, dim=1), dim=0)  # noqa: E731
        L = term(gp * gm) * (cp * cm) + 1j * term(gp * gsm) * (cm * sp) - 1j * term(gsp * gm) * (sm * cp)
        L = L + term(gsp * gsm) * (sp * sm) + term(-0.5 * gp ** 2) + term(-0.5 * gm ** 2)
        return W + 2.0 * self.dt * GAMMA["ODM"] * torch.fft.ifft(L, dim=0)

    def row(self, W, raw):
        return _rows(W, self.x, self.p, self.dv, self.v0, self.d, raw)

    def run(self, W, n):
        raw = W.sum() * self.d
        W = W / raw
        rows = [self.row(W, raw)] if self.scheme == "lie" else []
        for k in range(n):
            t, prob = k * self.dt, None
            if self.scheme == "lie":
                W = self.potential(self.kinetic(W), t)
            else:
                W = self.kinetic(self.potential(W, t, self.density(W) if self.gp else None))
                rho = self.density(W) if self.gp else None
                if self.gp:
                    prob = (rho * rho).sum() * self.dx
                W = self.potential(W, t, rho)
            if self.damping == "CaldeiraLeggett":
                W = self.friction(W)
            if self.damping == "ODM":
                W = self.lindblad(W)
            raw = W.sum() * self.d
            if self.damping != "none":
                W = W / raw
            rows.append(self.row(W, raw))
            if prob is not None:
                rows[-1][13] = prob
        if self.scheme != "lie":
            rows.append(torch.zeros(16, dtype=torch.float64, device=DEVICE))
        return W, torch.stack(rows)


def _exact_dirac(case, W):
    x, p, lam, th, dx, dp = _grid(case["X"], case["P"], 18.0, 16.0)
    dt, d, n, mh = case["dt"], dx * dp, case["steps"], 0.5
    V, dV = POTENTIALS[case["potential"]][2:]
    damped = case["damping"] != "none"

    def kinetic(q, sign):
        s = torch.sqrt(mh * mh + q * q)
        c, f = torch.cos(dt * s), sign * torch.sin(dt * s) / s
        return torch.complex(c, -mh * f), torch.complex(torch.zeros_like(f), -q * f), torch.complex(c, mh * f)

    K, R = kinetic(p + 0.5 * lam, 1.0), kinetic(p - 0.5 * lam, -1.0)
    F, u = mh * dt, 0.5 * th
    phase = dt * (V(0.0, x - u) - V(0.0, x + u))
    j = torch.arange(case["X"], dtype=torch.float64, device=DEVICE)
    edge = (1.0 - torch.exp(-(((j - case["X"] // 2) / 24.0) ** 2)))[None, :]
    fall = torch.exp(-dt * (0.01 if damped else 0.0) * th ** 2)
    pots = {m: fall * torch.exp(-1j * (phase + m)) for m in (0.0, 2.0 * F, -2.0 * F)}
    e2 = 2.0 * torch.sqrt(1.0 + p * p)
    aa, bb, dd = (0.5 - 1.0 / e2)[:, 0], (-p / e2)[:, 0], (0.5 + 1.0 / e2)[:, 0]
    dv = dV(x)
    D = lambda Y: torch.fft.ifft(th * torch.fft.fft(p * Y, dim=0), dim=0)  # noqa: E731
    a = 1j * dt * 0.05

    def row(W):
        tr, a1 = W[0, 0] + W[1, 1] + W[2, 2] + W[3, 3], W[0, 3] + W[1, 2] + W[2, 1] + W[3, 0]
        pairs = [tr * x, tr * p, tr * x * p, tr * x * x, tr * p * p, a1, tr * dv, tr * x * dv, tr * p * dv, a1 * p, a1 * x]
        out = torch.zeros(32, dtype=torch.float64, device=DEVICE)
        out[:22] = torch.view_as_real(torch.stack([d * v.sum() for v in pairs])).reshape(-1)
        out[24] = d * torch.clamp(tr.real, max=0.0).sum()
        out[25] = d * torch.where((x > 10.0).expand(tr.shape), tr.real, torch.zeros_like(tr.real)).sum()
        line = W.real.sum(-1)
        out[26] = d * (aa * (line[0, 0] + line[1, 1]) + dd * (line[2, 2] + line[3, 3])
                       + bb * (line[0, 3] + line[1, 2] + line[2, 1] + line[3, 0])).sum()
        out[27] = d * tr.real.sum()
        return out

    rows = [row(W)]
    rows[0][28] = rows[0][27]
    for _ in range(n):
        new = torch.empty_like(W)
        for r1, r2 in ((0, 3), (1, 2)):
            for c1, c2 in ((0, 3), (1, 2)):
                w = [torch.fft.fft(W[i, k], dim=1) for i in (r1, r2) for k in (c1, c2)]
                y = [K[0] * w[0] + K[1] * w[2], K[0] * w[1] + K[1] * w[3], K[1] * w[0] + K[2] * w[2], K[1] * w[1] + K[2] * w[3]]
                z = [y[0] * R[0] + y[1] * R[1], y[0] * R[1] + y[1] * R[2], y[2] * R[0] + y[3] * R[1], y[2] * R[1] + y[3] * R[2]]
                for (i, k), v in zip(((r1, c1), (r1, c2), (r2, c1), (r2, c2)), z):
                    new[i, k] = torch.fft.ifft(v, dim=1)
        for i in range(4):
            for k in range(4):
                m = 2.0 * F * ((i < 2) - (k < 2))
                w = torch.fft.ifft(torch.fft.fft(new[i, k], dim=0) * pots[m], dim=0)
                if damped:
                    w = w + 2.0 * a * D(w + a * D(w))
                new[i, k] = w * edge
        raw = d * torch.einsum("iipx->", new).real
        W = new / raw
        rows.append(row(W))
        rows[-1][28] = raw
    return W, torch.stack(rows)


def _exact_control(case, seed):
    params, target, base = _control_inputs(case, seed)
    W0, n, dt = _initial(case, seed)[0], case["steps"], case["dt"]
    params.requires_grad_()
    W0.requires_grad_()
    x, p, lam, th, dx, dp = _grid(case["X"], case["P"], 10.0, 10.0)
    K = torch.exp(-1j * dt * lam * p / MASS)
    xm, xp = x - 0.5 * HBAR * th, x + 0.5 * HBAR * th
    still = 0.25 * (xm ** 4 - xp ** 4) - (xm ** 2 - xp ** 2)
    half = case["terms"] // 2
    j = torch.arange(1, half + 1, dtype=torch.float64, device=DEVICE)
    W = W0
    for k in range(n):
        arg = 2.0 * math.pi * (k * dt) * j / 20.0
        field = torch.cos(arg) @ params[:half] + torch.sin(arg) @ params[half:]
        phase = (still - field * (xm - xp)) * (dt / HBAR)
        W = torch.fft.ifft(torch.fft.fft(W, dim=1) * K, dim=1)
        W = torch.fft.ifft(torch.fft.fft(W, dim=0) * torch.exp(-1j * phase), dim=0)
    loss = 1.0 - 2.0 * math.pi * dx * dp * (W.real * target).sum()
    g_params, g_W0 = torch.autograd.grad(loss, (params, W0))
    return {"loss": loss.detach(), "W": W.real.detach(), "g_params": g_params, "g_W0": g_W0}


def exact(case, seed):
    kind = case["kind"]
    if kind == "control":
        return _exact_control(case, seed)
    W0 = _initial(case, seed)
    if kind != "axes":  # what the run starts from: the state as its precision holds it
        W0 = [w.to(_state_type(case["precision"])).to(torch.complex128) for w in W0]
    if kind == "wigner":
        V, dV = POTENTIALS[case["potential"]][2:]
        W, record = _Exact(case["X"], case["P"], case["amp"], case["dt"], V, dV, case["scheme"], case["damping"],
                           case["gp"]).run(W0[0], case["steps"])
        return {"W": W, "record": record}
    if kind == "ensemble":
        done = [_Exact(side, side, 10.0, case["dt"], lambda t, x, a=a, b=b: a * x ** 4 - b * x ** 2,
                       lambda x, a=a, b=b: 4.0 * a * x ** 3 - 2.0 * b * x, mask=False).run(w, case["steps"])
                for w, (side, a, b) in zip(W0, _members(case))]
        return {"W": torch.cat([w.reshape(-1) for w, _ in done]), "record": torch.stack([r for _, r in done])}
    if kind == "dirac":
        W, record = _exact_dirac(case, W0[0])
        return {"W": W.reshape(16, case["P"], case["X"]), "record": record}
    W = W0[0].to(_state_type(case["precision"])).to(torch.complex128)
    return {"forward": torch.fft.fft2(W), "inverse": torch.fft.ifft2(W) * case["X"]}
