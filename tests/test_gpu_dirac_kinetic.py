"""The kinetic and filter sweeps of the Wigner-Dirac step at every grid side: their factors are
evaluated once per row at q = p + lambda/2 and read backwards for the other side, with an entry of
its own for the bin N/2 that has no mirror image, and up to 1024 one block holds the four plane
groups of a row.  A random state fills every bin (a smooth one is zero there)."""
import numpy as np
import pytest

from oracle.dirac4x4 import Dirac4x4Oracle, gaussian_spinor_particle_up, wigner_from_spinor
from tests.test_gpu_dirac import CASES, check_obs, rel_l2, run_both, zero

pytestmark = pytest.mark.gpu

# two transforms of <= 11 passes of two at 1.1e-16 each, plus the factors: under 1e-14 in
# complex128; complex64 planes are rounded to 6e-8 at the load and the store, and FP32 transforms
# add a rounding per pass (22 of 6e-8, as a random walk under 1e-6)
BOUND = {"fp64": 1e-13, "fp32": 3e-7, "fp32fast": 2e-6}


@pytest.mark.parametrize("kvn", [False, True])
@pytest.mark.parametrize("X,precision", [(128, "fp64"), (256, "fp64"), (512, "fp64"), (1024, "fp64"), (2048, "fp64"),
                                         (128, "fp32"), (512, "fp32"), (1024, "fp32fast"), (256, "fp32fast")])
def test_kinetic_sweep_every_bin(cuda, X, precision, kvn):
    import torch

    from pywignercuda_amd.dirac import WignerDirac4x4

    P = 128
    vs, vf, dvf = CASES["ramp"]
    hip = WignerDirac4x4(X, P, 18.0, 16.0, 1.0, 1.0, 0.01, potentials=(vs, "0.", "0.", "0."), kvn=kvn,
                         precision=precision, device=cuda)
    orc = Dirac4x4Oracle(X, P, 18.0, 16.0, 1.0, 1.0, 0.01, [vf, zero, zero, zero], dpotential0=dvf, kvn=kvn)
    rng = np.random.default_rng(X)
    W0 = rng.standard_normal((4, 4, P, X)) + 1j * rng.standard_normal((4, 4, P, X))
    W = hip.to_device(W0)
    hip.kinetic(W)
    torch.cuda.synchronize()
    ref = orc.lambda_to_x(orc.kinetic_step(orc.x_to_lambda(W0)))
    err = rel_l2(W.cpu().numpy().reshape(4, 4, P, X), ref)
    print(f"{X} {precision} kvn {kvn}: rel L2 {err:.2e}")
    assert err < BOUND[precision]


@pytest.mark.parametrize("X", [256, 1024, 2048])
def test_step_filter_sides(cuda, X):
    from pywignercuda_amd.dirac import WignerDirac4x4

    vs, vf, dvf = CASES["ramp"]
    hip = WignerDirac4x4(X, 128, 18.0, 16.0, 1.0, 1.0, 0.01, potentials=(vs, "0.", "0.", "0."), D_theta=0.01,
                         energy=True, step_filter=True, device=cuda)
    orc = Dirac4x4Oracle(X, 128, 18.0, 16.0, 1.0, 1.0, 0.01, [vf, zero, zero, zero], dpotential0=dvf,
                         D_theta=0.01, compute_energy=True, step_filter=True)
    W0 = wigner_from_spinor(lambda Xg: gaussian_spinor_particle_up(-2.0, 3.0, 1.0, Xg, 1.0, 1.0), orc)
    W, obs, W_ref, rec = run_both(hip, orc, W0, 4)
    assert rel_l2(W, W_ref) < 1e-10
    check_obs(obs, rec)
