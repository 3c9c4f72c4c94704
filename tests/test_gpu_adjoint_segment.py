"""GPU: the backward pass of a segment in one call, on rectangular grids at the edges of the tiles,
against autograd of the torch reference and against the single adjoint steps.

Bounds: the states are exact to about 1e-14 and the gradient terms of a_k are sums of products of
two of them, compared per coefficient with that coefficient's largest gradient: 1e-9 (the terms
cancel by up to five digits on these grids).  A segment runs the sweeps of the single steps: equal
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def setup(cuda, X, P, n, precision="fp64"):
    import torch

    from oracle import wigner2d as ow
    from pywignercuda_amd.wigner2d import Wigner2D

    base = np.array([0.0, 0.1, 0.4, -0.02, 0.03, 0.002, 0.001, 1e-4, 1e-5])
    prop = Wigner2D(X, P, 6.0, 7.0, 0.9, 1.1, 0.02, potential="0.4*pow(x,2)", dpotential="0.8*x", mask=False,
                    device=cuda, pot_table=np.tile(base, (n + 2, 1)), precision=precision)
    table = torch.tensor(np.tile(base, (n + 2, 1)), dtype=torch.float64, device=cuda)
    table[:, 1] += 0.05 * torch.cos(torch.arange(n + 2, device=cuda, dtype=torch.float64))
    W0 = torch.tensor(ow.gaussian_wigner(ow.Grid(X, P, 6.0, 7.0), x0=0.5, p0=-0.3), device=cuda).to(prop.dtype)
    weight = torch.tensor(ow.gaussian_wigner(ow.Grid(X, P, 6.0, 7.0), x0=-0.5, p0=0.4, s=1.2), device=cuda)
    return prop, table, W0, weight


@pytest.mark.parametrize("n,keep", [(5, 2), (3, 3), (1, 4)])
@pytest.mark.parametrize("X,P", [(128, 128), (128, 512), (256, 1024), (128, 2048), (1024, 128)])
def test_gradients_against_torch(cuda, X, P, n, keep):
    import torch

    from pywignercuda_amd.adjoint import propagate, reference_propagate_torch

    prop, table, W0, weight = setup(cuda, X, P, n)
    out = []
    for f in (lambda t, w: propagate(prop, t, w, n, checkpoint_every=keep),
              lambda t, w: reference_propagate_torch(t, w, X, P, 6.0, 7.0, 0.9, 1.1, 0.02, n)):
        t, w = table.clone().requires_grad_(), W0.clone().requires_grad_()
        out.append(torch.autograd.grad((f(t, w) * weight).sum(), (t, w)))
    (gt, gw), (rt, rw) = out
    assert float(torch.linalg.norm(gw - rw)) < 1e-10 * float(torch.linalg.norm(rw))
    for k in range(9):
        assert float((gt[:, k] - rt[:, k]).abs().max()) <= 1e-9 * max(float(rt[:, k].abs().max()), 1e-12), k


@pytest.mark.parametrize("precision", ["fp64", "fp32fast"])
@pytest.mark.parametrize("X,P", [(256, 128), (128, 2048)])
def test_segment_equals_single_steps(cuda, X, P, precision):
    import torch

    prop, table, W0, weight = setup(cuda, X, P, 4, precision)
    prop.set_potential(table)
    W, Lam = W0.clone(), weight.to(prop.dtype)
    states = []
    for k in range(4):
        prop.kinetic(W)
        prop.potential(W, k)
        states.append(W.clone())
    one = Lam.clone()
    grads = torch.zeros((4, 9), dtype=torch.float64, device=cuda)
    for k in reversed(range(4)):
        prop.adjoint_step(one, states[k], k, grads[k])
    room = torch.empty((4, P, X), dtype=prop.dtype, device=cuda)
    both, rows = Lam.clone(), torch.zeros_like(grads)
    prop.adjoint_segment(W0, room, both, 0, rows)
    assert torch.equal(room, torch.stack(states)) and torch.equal(both, one) and torch.equal(rows, grads)
    last = W0.clone()
    prop.steps(last, last, 4)
    assert torch.equal(last, states[-1])
