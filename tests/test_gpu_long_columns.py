"""GPU: <p^2> over many steps on long columns, against the same steps in 80-bit arithmetic on the CPU.

Plans of few cells transform P = 1024 and 2048 with radix 8.  A rounded constant in its butterflies acts
in every pass and both directions alike: it leaves W a residue at the edges of p, which <p^2> weighs
with p^2 and which grows with the steps.

Bound.  Rounding that changes with the values: 288 transforms of 72 steps move W by sqrt(288 log2 P)
2^-53 |W|_2, spread over all cells; weighed with p^2 and over <p^2> = 1/2, with |W|_2^2 = 1 / (2 pi dx dp):
sqrt(dx dp / (2 pi)) 54 2^-53 p_max^2 / sqrt(5) / (1/2) = 2.1e-14 at 1024.  A fixed relative error of 7e-17 in
a quarter of each butterfly's terms, 6 passes a step, leaves about 1e-12.  2e-13 lies between them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

AMP, DT, STEPS = 12.0, 0.005, 72


def exact(X, P, W0):
    """<p^2> of each step, Lie scheme, V = x^2/2, no mask."""
    import scipy.fft as sf

    L = np.longdouble
    axis = lambda n, step: L(step) * (((np.arange(n) + n // 2) % n) - n // 2).astype(L)  # noqa: E731
    x, p = axis(X, 2 * AMP / X)[None, :], axis(P, 2 * AMP / P)[:, None]
    lam, th = axis(X, np.pi / AMP)[None, :], axis(P, np.pi / AMP)[:, None]
    i = np.clongdouble(1j)
    K = np.exp(-i * L(DT) * lam * p)
    V = lambda y: y * y / 2  # noqa: E731
    M = np.exp(-i * L(DT) * (V(x - th / 2) - V(x + th / 2)))
    W, out = W0.astype(np.clongdouble), []
    for k in range(STEPS + 1):
        r = W.real
        out.append(float((r * p * p).sum() / r.sum()))
        if k < STEPS:
            W = sf.ifft(sf.fft(W, axis=1) * K, axis=1)
            W = sf.ifft(sf.fft(W, axis=0) * M, axis=0)
    return np.array(out)


@pytest.mark.parametrize("P", [1024, 2048])
def test_second_moment_of_p(cuda, P):
    from pywignercuda_amd.wigner2d import Wigner2D

    X = 128
    plan = Wigner2D(X, P, AMP, AMP, 1.0, 1.0, DT, potential="0.5*pow(x,2)", dpotential="x", mask=False, device=cuda)
    x, p = plan.x_host[None, :], plan.p_host[:, None]
    W0 = np.exp(-((x - 1.3) ** 2) - (p - 0.7) ** 2) / np.pi
    W = plan.to_device(W0)
    got = plan.run(W, STEPS).cpu().numpy()[: STEPS + 1, 3]
    ref = exact(X, P, W0.astype(complex))
    assert np.abs(got / ref - 1.0).max() < 2e-13
