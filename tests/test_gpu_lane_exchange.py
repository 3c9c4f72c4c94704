"""GPU: single sweeps whose last transform pass exchanges its inputs between lanes in registers
(v_permlane32_swap / v_permlane16_swap), and their neighbours that exchange through LDS, against
complex128 torch transforms of the same random complex state.

Bounds: a transform of length N rounds each element about log2 N times; two transforms and one
product in FP64 stay below 2 * 3 * log2(2048) * 2^-53 < 1e-14 in the 2-norm, taken as 5e-14.  The
complex64 states add one rounding per sweep (and one per LDS exchange in the throughput forms),
2^-24 each at most: five of them give 3e-7."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUND = {"fp64": 5e-14, "fp32": 3e-7}
SIDES = (128, 256, 512, 1024, 2048)


def plan(cuda, X, P, precision):
    from pywignercuda_amd.wigner2d import Wigner2D

    return Wigner2D(X, P, 9.0, 7.0, 0.8, 1.3, 0.02, potential="0.5*pow(x,2)+0.02*pow(x,4)", dpotential="x",
                    mask=False, precision=precision, device=cuda, variants=(-1, -1, -1))


def state(cuda, p, seed):
    import torch

    g = torch.Generator(device=cuda).manual_seed(seed)
    return torch.randn((p.P, p.X), dtype=torch.complex128, device=cuda, generator=g).to(p.dtype)


def rel(W, ref):
    import torch

    return float(torch.linalg.norm(W.to(torch.complex128) - ref) / torch.linalg.norm(ref))


def axis(n, step, cuda):
    import torch

    k = (np.arange(n) + n // 2) % n - n // 2
    return torch.tensor(k * step, dtype=torch.float64, device=cuda)


def variants(table):
    from pywignercuda_amd import _lib

    return range(_lib.lib().wh_variant_info(table, -1, None, None))


def try_variant(p, **kw):
    from pywignercuda_amd import _lib

    try:
        p.set_variants(**kw)
        return True
    except _lib.WignerHipInvalidValue:
        return False  # this variant does not cover the size


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N", SIDES)
def test_x_sweep(cuda, N, precision):
    import torch

    p = plan(cuda, N, 128, precision)
    W = state(cuda, p, N)
    lam, mom = axis(N, np.pi / 9.0, cuda)[None, :], axis(128, 14.0 / 128, cuda)[:, None]
    ref = torch.fft.ifft(torch.fft.fft(W.to(torch.complex128), dim=1) * torch.exp(-1j * 0.02 * lam * mom / 1.3), dim=1)
    done = 0
    for v in variants(0):
        if not try_variant(p, xvar=v):
            continue
        Y = W.clone()
        p.kinetic(Y)
        assert rel(Y, ref) < BOUND[precision], (N, v)
        done += 1
    assert done >= 1


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N", SIDES)
def test_p_sweep(cuda, N, precision):
    import torch

    p = plan(cuda, 128, N, precision)
    W = state(cuda, p, N + 1)
    x, th = axis(128, 18.0 / 128, cuda)[None, :], axis(N, np.pi / 7.0, cuda)[:, None]
    V = lambda y: 0.5 * y ** 2 + 0.02 * y ** 4  # noqa: E731
    phase = 0.02 / 0.8 * (V(x - 0.4 * th) - V(x + 0.4 * th))
    ref = torch.fft.ifft(torch.fft.fft(W.to(torch.complex128), dim=0) * torch.exp(-1j * phase), dim=0)
    # the phase itself is a polynomial of some 1e5 rad at the corners: its rounding joins the bound
    bound = BOUND[precision] + 4.0 * float(phase.abs().max()) * 2.0 ** -53
    done = 0
    for v in variants(1):
        if not try_variant(p, pvar=v):
            continue
        Y = W.clone()
        p.potential(Y)
        assert rel(Y, ref) < bound, (N, v)
        done += 1
    assert done >= 1


@pytest.mark.parametrize("X,P", [(128, 128), (256, 512), (128, 1024)])
def test_friction_without_diffusion(cuda, X, P):
    """Caldeira-Leggett friction with D_theta = 0 (no decay table from the caller) in every p variant,
    record rows included, against the oracle: 4 steps, the FP64 bar of the parity tests (1e-10)."""
    from oracle import wigner2d as ow
    from pywignercuda_amd.wigner2d import Wigner2D

    args = (X, P, 9.0, 7.0, 0.8, 1.3, 0.01)
    kw = dict(scheme="lie", gamma=0.1, damping="CaldeiraLeggett", mask=True)
    p = Wigner2D(*args, potential="0.5*pow(x,2)+0.02*pow(x,4)", dpotential="x+0.08*pow(x,3)", fp_damping="fabs(p)",
                 device=cuda, variants=(-1, -1, -1), **kw)
    o = ow.Wigner2DOracle(*args, potential=lambda t, x: 0.5 * x ** 2 + 0.02 * x ** 4,
                          dpotential=lambda t, x: x + 0.08 * x ** 3, fp_damping=np.abs, **kw)
    W0 = ow.gaussian_wigner(o.g, x0=1.0, p0=-0.5, s=1.1)
    ref, obs_ref, _ = o.run(W0, 3)
    done = 0
    for v in variants(2):
        if not try_variant(p, pclvar=v):
            continue
        W = p.to_device(W0)
        obs = p.run(W, 4).cpu().numpy()
        assert np.linalg.norm(W.cpu().numpy() - ref) < 1e-10 * np.linalg.norm(ref), v
        assert abs(obs[3, 0] - obs_ref["X"][3]) < 1e-10 and abs(obs[3, 9] - obs_ref["neg"][3]) < 1e-10, v
        done += 1
    assert done >= 1
