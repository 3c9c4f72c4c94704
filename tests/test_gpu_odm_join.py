"""GPU: ODM runs whose iterations share a launch (the last sweep of one, the observables and the
next kinetic step), at the edges of the tiles, with one and two channels, against the oracle.

Bounds: the FP64 bar of the parity tests (relative L2 1e-10, records 1e-10)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 2, 5])
@pytest.mark.parametrize("scheme,weights", [("lie", None), ("lie", (1.0, 0.9)), ("strang", None)])
@pytest.mark.parametrize("X,P", [(128, 128), (512, 128), (1024, 256), (2048, 128), (128, 2048)])
def test_steps_against_oracle(cuda, X, P, scheme, weights, steps):
    from oracle import wigner2d as ow
    from pywignercuda_amd.wigner2d import Wigner2D

    args = (X, P, 11.0, 10.0, 1.0, 1.0, 0.005)
    kw = dict(scheme=scheme, gamma=0.02, damping="ODM", L_material=3.0, odm_weights=weights)
    p = Wigner2D(*args, potential="0.5*pow(x,2)-0.3*cos(t)*x", dpotential="x-0.3*cos(t)",
                 fp_damping="p*p/sqrt(p*p+0.5)", time_rows=steps + 2, device=cuda, **kw)
    o = ow.Wigner2DOracle(*args, potential=lambda t, x: 0.5 * x ** 2 - 0.3 * np.cos(t) * x,
                          dpotential=lambda t, x: x - 0.3 * np.cos(t), time_dependent=True,
                          fp_damping=lambda q: q * q / np.sqrt(q * q + 0.5), **kw)
    W0 = ow.gaussian_wigner(o.g, x0=0.5, p0=2.0, s=1.0)
    ref, obs_ref, _ = o.run(W0, steps - 1)
    W = p.to_device(W0)
    obs = p.run(W, steps).cpu().numpy()
    assert np.linalg.norm(W.cpu().numpy() - ref) < 1e-10 * np.linalg.norm(ref)
    for col, key in ((0, "X"), (2, "P"), (3, "P2"), (4, "XP"), (7, "XdV"), (8, "H"), (9, "neg")):
        np.testing.assert_allclose(obs[:steps, col], obs_ref[key], atol=1e-10, err_msg=key)
