"""GPU: Gross-Pitaevskii runs, whose density comes from the p sweep's column sums and tile partials
(before the first half step) and from the x sweep's partial sums (before the second), against the
oracle at every side of the grid, and an uneven ensemble against its members run alone.

Bounds: the FP64 bar of the parity tests (relative L2 1e-10, records 1e-10)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

V, DV = "0.5*pow(x,2)", "x"


def pair(cuda, X, P, scheme, gamma):
    from oracle import wigner2d as ow
    from pywignercuda_amd.wigner2d import Wigner2D

    args = (X, P, 9.0, 8.0, 0.9, 1.0, 0.01)
    damping = "CaldeiraLeggett" if gamma else None
    p = Wigner2D(*args, potential=V, dpotential=DV, scheme=scheme, gamma=gamma, damping=damping,
                 fp_damping="fabs(p)" if gamma else None, gp_coeff=0.6, device=cuda)
    o = ow.Wigner2DOracle(*args, potential=lambda t, x: 0.5 * x ** 2, dpotential=lambda t, x: x, scheme=scheme,
                          gamma=gamma, damping=damping, fp_damping=np.abs, gp_coeff=0.6)
    return p, o, ow.gaussian_wigner(o.g, x0=1.0, p0=-0.5, s=1.1, hbar=0.9) * (1.0 + 0.1 * np.cos(o.g.x_host))


@pytest.mark.parametrize("gamma", [0.0, 0.1])
@pytest.mark.parametrize("scheme", ["lie", "strang"])
@pytest.mark.parametrize("X,P", [(128, 128), (256, 128), (512, 256), (1024, 128), (2048, 128), (128, 2048)])
def test_density_against_oracle(cuda, X, P, scheme, gamma):
    if gamma and P == 2048:
        # theta p gamma dt reaches 3.2 at the grid's corner: the order-3 composite without diffusion
        # amplifies rounding 34-fold per step there, and the oracle itself ends 1.1e-10 off the same
        # steps in long double (the library 9.8e-11, as before its density came from the sweeps)
        pytest.skip("the oracle is less exact than the bar on this input")
    p, o, W0 = pair(cuda, X, P, scheme, gamma)
    n = 4
    ref, obs_ref, extra = o.run(W0, n - 1)
    W = p.to_device(W0)
    obs = p.run(W, n).cpu().numpy()
    assert np.linalg.norm(W.cpu().numpy() - ref) < 1e-10 * np.linalg.norm(ref)
    np.testing.assert_allclose(obs[:n, 0], obs_ref["X"], atol=1e-10)
    np.testing.assert_allclose(obs[:n, 9], obs_ref["neg"], atol=1e-10)
    if scheme == "strang":
        np.testing.assert_allclose(obs[:n, 13], extra["ProbabilitySquare"], atol=1e-10)


@pytest.mark.parametrize("scheme", ["lie", "strang"])
def test_uneven_ensemble_and_graph(cuda, scheme):
    """35 steps (the middle ones replayed from a graph): three uneven members in one plan against
    each alone with direct launches."""
    from oracle import wigner2d as ow
    from pywignercuda_amd.wigner2d import Wigner2D, WignerEnsemble

    sides = [(128, 256), (512, 128), (256, 256)]
    W0 = [ow.gaussian_wigner(ow.Grid(x, p, 9.0, 8.0), x0=0.5 * k, s=1.0) for k, (x, p) in enumerate(sides)]
    ens = WignerEnsemble([dict(X=x, P=p, X_amp=9.0, P_amp=8.0, potential=V, dpotential=DV) for x, p in sides],
                         1.0, 1.0, 0.01, scheme=scheme, gp_coeff=0.6, device=cuda)
    Ws = ens.states_to_device(W0)
    rows = ens.run(Ws, 35).cpu().numpy()
    for k, (x, p) in enumerate(sides):
        one = Wigner2D(x, p, 9.0, 8.0, 1.0, 1.0, 0.01, potential=V, dpotential=DV, scheme=scheme, gp_coeff=0.6,
                       mask=False, device=cuda)
        W = one.to_device(W0[k])
        obs = one.run(W, 35, use_graph=False).cpu().numpy()
        assert np.linalg.norm((W - Ws[k]).cpu().numpy()) < 1e-10 * np.linalg.norm(W.cpu().numpy())
        np.testing.assert_allclose(rows[k], obs, atol=1e-10)
