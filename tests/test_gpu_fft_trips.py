"""GPU: the second moment of a Gaussian after 72 forward and inverse complex128 axis transforms.

Bound.  Rounding that changes with the values: 144 transforms of log2 N stages move a line by
sqrt(144 log2 N) 2^-53 |g|_2, spread over its N cells; weighed with q^2 (|q| < 12) and over sum g q^2, with
g = exp(-(q - 1.1)^2), |g|_2^2 = sqrt(pi / 2) / dq and sum g q^2 = sqrt(pi) (1.1^2 + 1/2) / dq, that is
sqrt(144 log2 N) 2^-53 sqrt(dq) 23.8: 2.1e-14 (N = 512) to 3.6e-14 (128).  5e-14 leaves it some room.  A
constant of the butterflies rounded by 7e-17 leaves about 1e-13 in every line."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("N", [128, 256, 512])
def test_second_moment(cuda, N, axis):
    from pywignercuda_amd import cufft_wrapper as cw

    shape = (N, 64) if axis == 0 else (64, N)
    plan = (cw.Plan_Z2Z_2D_Axis0 if axis == 0 else cw.Plan_Z2Z_2D_Axis1)(shape)
    q = np.longdouble(24.0 / N) * (np.arange(N) - N // 2)
    q = q[:, None] if axis == 0 else q[None, :]
    g0 = np.ascontiguousarray(np.broadcast_to(np.exp(-((q - 1.1) ** 2)), shape)).astype(complex)
    W = torch.from_numpy(g0).to(cuda)
    for _ in range(72):
        cw.fft_Z2Z(W, W, plan)
        cw.ifft_Z2Z_normalized(W, W, plan)
    g = W.cpu().numpy().real.astype(np.longdouble)
    moment = lambda a: (a * q * q).sum(axis) / a.sum(axis)  # noqa: E731
    assert np.abs(moment(g) / moment(g0.real.astype(np.longdouble)) - 1.0).max() < 5e-14
