"""GPU: Wigner-Dirac steps in complex128 against the same steps in 80-bit arithmetic on the CPU.

Bound.  A step has four transforms of log2 N stages and about ten more roundings a cell (two products with
2 x 2 blocks, phase, edge, norm): n steps move W by sqrt(n (4 log2 N + 10)) 2^-53 |W|_2 where they change
with the values.  Four factors a step are rounded alike in every step, by 0.4 2^-53 each: 0.8 n 2^-53.
A quarter above both together.  A constant of the butterflies rounded alike goes beyond it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

XA, PA, DT = 18.0, 16.0, 0.002
L, C = np.longdouble, np.clongdouble


def axes(N):
    ax = lambda step: L(step) * (((np.arange(N) + N // 2) % N) - N // 2).astype(L)  # noqa: E731
    return ax(2 * XA / N)[None, :], ax(2 * PA / N)[:, None], ax(np.pi / XA)[None, :], ax(np.pi / PA)[:, None]


def spinor(N):
    """Wigner matrix of a Gaussian spinor of positive energy."""
    x, _, _, th = axes(N)
    px = L(5.3)
    up = {0: np.sqrt(px * px + 1) + 1, 3: px}
    rho = lambda y: np.exp(C(1j) * px * y - ((y + L(2.1)) / L(1.05)) ** 2 / 2)  # noqa: E731
    both = rho(x - th / 2) * rho(x + th / 2).conj()
    W = np.zeros((4, 4, N, N), complex)
    for a in up:
        for b in up:
            W[a, b] = np.fft.ifft((up[a] * up[b] * both).astype(complex), axis=0)
    return W / (np.einsum("iipx->", W).real * (2 * XA / N) * (2 * PA / N))


def exact(N, steps, W0):
    import scipy.fft as sf

    x, p, lam, th = axes(N)
    dt, d, mh, i = L(DT), L(2 * XA / N) * L(2 * PA / N), L(0.5), C(1j)

    def kinetic(q, sign):
        s = np.sqrt(mh * mh + q * q)
        c, f = np.cos(dt * s), sign * np.sin(dt * s) / s
        return c - i * mh * f, -i * q * f, c + i * mh * f

    K, R = kinetic(p + lam / 2, 1), kinetic(p - lam / 2, -1)
    V = lambda y: -2 / np.sqrt(y * y + 1)  # noqa: E731
    phase = dt * (V(x - th / 2) - V(x + th / 2))
    edge = (1 - np.exp(-(((np.arange(N).astype(L) - N // 2) / 24) ** 2)))[None, :]
    pot = {k: np.exp(-i * (phase + 2 * k * mh * dt)) for k in (-1, 0, 1)}
    W = W0.astype(C)
    for _ in range(steps):
        new = np.empty_like(W)
        for r in ((0, 3), (1, 2)):
            for c in ((0, 3), (1, 2)):
                w = [sf.fft(W[a, b], axis=1) for a in r for b in c]
                y = [K[0] * w[0] + K[1] * w[2], K[0] * w[1] + K[1] * w[3],
                     K[1] * w[0] + K[2] * w[2], K[1] * w[1] + K[2] * w[3]]
                z = [y[0] * R[0] + y[1] * R[1], y[0] * R[1] + y[1] * R[2],
                     y[2] * R[0] + y[3] * R[1], y[2] * R[1] + y[3] * R[2]]
                for (a, b), v in zip(((a, b) for a in r for b in c), z):
                    new[a, b] = sf.ifft(v, axis=1)
        for a in range(4):
            for b in range(4):
                k = int(a < 2) - int(b < 2)
                new[a, b] = sf.ifft(sf.fft(new[a, b], axis=0) * pot[k], axis=0) * edge
        W = new / (d * np.einsum("iipx->", new).real)
    return W.astype(complex)


@pytest.mark.parametrize("N,steps", [(128, 40), (256, 20)])
def test_state(cuda, N, steps):
    from pywignercuda_amd.dirac import WignerDirac4x4

    W0 = spinor(N)
    plan = WignerDirac4x4(N, N, XA, PA, 1.0, 1.0, DT, potentials=("-2.0/sqrt(x*x + 1.0)", "0.", "0.", "0."), gamma=0.0,
                          damping=None, D_theta=0.0, truncate_constants=False, device=cuda)
    W = plan.to_device(torch.from_numpy(W0).to(cuda))
    plan.run(W, steps)
    ref = exact(N, steps, W0)
    bound = 1.25 * np.hypot(np.sqrt(steps * (4 * np.log2(N) + 10)), 0.8 * steps) * 2.0**-53
    assert np.linalg.norm(W.cpu().numpy().ravel() - ref.ravel()) < bound * np.linalg.norm(ref.ravel())
