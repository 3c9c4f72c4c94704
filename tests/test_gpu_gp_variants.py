"""GPU: the x variants that a Gross-Pitaevskii plan takes.  Its own choice depends on the side; the
default variant (index 0, what every such plan was created with before) is accepted at every side
and gives the same steps; any other is refused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(cuda, X, P, variants, after=None):
    from pywignercuda_amd.wigner2d import Wigner2D

    p = Wigner2D(X, P, 8.0, 8.0, 1.0, 1.0, 0.005, potential="0.5*pow(x,2)", dpotential="x", scheme="strang",
                 gp_coeff=0.5, variants=variants, device=cuda)
    if after is not None:
        p.set_variants(*after)
    x, pp = p.x_host[None, :], p.p_host[:, None]
    W = p.to_device(np.exp(-((x - 1.0) ** 2) - pp ** 2) / np.pi)
    obs = p.run(W, 21)
    return W.cpu().numpy(), obs.cpu().numpy()


# every side's own choice: radix 4 (128, 256), 8 (512, 2048), 16 (1024)
@pytest.mark.parametrize("X,P", [(128, 256), (256, 128), (512, 128), (1024, 128), (2048, 128)])
def test_default_x_variant_is_accepted(cuda, X, P):
    W, obs = _run(cuda, X, P, None)
    for variants, after in (((0, 0, 0), None), (None, (0, -1, -1)), ((0, -1, -1), (0, 0, -1))):
        V, o = _run(cuda, X, P, variants, after)
        # other radices round otherwise: 21 steps of four transforms each, a few eps per transform
        tol = 21 * 4 * 8 * 2.3e-16
        assert np.linalg.norm(V - W) <= tol * np.linalg.norm(W)
        assert np.abs(o - obs).max() <= 100 * tol * np.abs(obs).max()


def test_other_x_variants_stay_refused(cuda):
    from pywignercuda_amd import _lib
    from pywignercuda_amd.wigner2d import Wigner2D

    p = Wigner2D(512, 256, 8.0, 8.0, 1.0, 1.0, 0.005, potential="0.5*pow(x,2)", dpotential="x", gp_coeff=0.5, device=cuda)
    own = 1  # radix 8 at 512
    for v in range(int(_lib.lib().wh_variant_info(0, -1, None, None))):
        if v in (0, own):
            p.set_variants(v, -1, -1)
        else:
            with pytest.raises(_lib.WignerHipError):
                p.set_variants(v, -1, -1)
