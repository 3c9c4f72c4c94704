"""The potential sweep of the Wigner-Dirac step at every grid side: up to P = 512 a column's team lies
in one wave (the lanes change teams at the first exchange and back before the store), above it a team
spans several; two mass classes per block share their multipliers; with friction the column's p and
theta come from LDS.  A random state fills every bin."""
import numpy as np
import pytest

from oracle.dirac4x4 import Dirac4x4Oracle, gaussian_spinor_particle_up, wigner_from_spinor
from tests.test_gpu_dirac import CASES, check_obs, rel_l2, run_both, zero

pytestmark = pytest.mark.gpu

# up to six transforms of <= 11 passes of two at 1.1e-16 each: under 1e-14 in complex128; complex64
# planes are rounded to 6e-8 at the load and the store, FP32 transforms add a rounding per pass
# (66 of 6e-8, as a random walk under 1e-6; the friction's p theta amplifies some of them by up to 5)
BOUND = {"fp64": 1e-13, "fp32": 3e-7, "fp32fast": 5e-6}


def pair(cuda, case, P, X=128, gamma=0.0, D_theta=0.02, precision="fp64"):
    from pywignercuda_amd.dirac import WignerDirac4x4

    vs, vf, dvf = CASES[case]
    damping = "CaldeiraLegget" if gamma else None
    hip = WignerDirac4x4(X, P, 18.0, 16.0, 1.0, 1.0, 0.01, potentials=(vs, "0.", "0.", "0."), gamma=gamma,
                         damping=damping, D_theta=D_theta, energy=True, precision=precision, device=cuda)
    orc = Dirac4x4Oracle(X, P, 18.0, 16.0, 1.0, 1.0, 0.01, [vf, zero, zero, zero], dpotential0=dvf, gamma=gamma,
                         damping=damping, D_theta=D_theta, compute_energy=True)
    return hip, orc


@pytest.mark.parametrize("gamma", [0.0, 0.05])
@pytest.mark.parametrize("P,case,precision", [(128, "klein", "fp64"), (256, "ramp", "fp64"), (512, "klein", "fp64"),
                                              (1024, "ramp", "fp64"), (2048, "klein", "fp64"), (128, "ramp", "fp32"),
                                              (512, "ramp", "fp32"), (256, "klein", "fp32fast"),
                                              (1024, "klein", "fp32fast")])
def test_potential_sweep_every_bin(cuda, P, case, precision, gamma):
    import torch

    hip, orc = pair(cuda, case, P, gamma=gamma, precision=precision)
    rng = np.random.default_rng(P)
    W0 = rng.standard_normal((4, 4, P, 128)) + 1j * rng.standard_normal((4, 4, P, 128))
    W = hip.to_device(W0)
    hip.potential(W, step=3)
    torch.cuda.synchronize()
    ref = orc.theta_to_p(orc.potential_step(orc.p_to_theta(W0), orc.dt * 3))
    if gamma:
        ref = orc.cl_order2(ref)
    ref = ref * orc.absorber()
    err = rel_l2(W.cpu().numpy().reshape(4, 4, P, 128), ref)
    print(f"{P} {case} {precision} gamma {gamma}: rel L2 {err:.2e}")
    assert err < BOUND[precision]


@pytest.mark.parametrize("P", [256, 512, 1024, 2048])
def test_record_sides(cuda, P):
    """Column sums of both layouts: the whole record over a few steps."""
    hip, orc = pair(cuda, "ramp", P, gamma=0.05)
    W0 = wigner_from_spinor(lambda Xg: gaussian_spinor_particle_up(-2.0, 3.0, 1.0, Xg, 1.0, 1.0), orc)
    W, obs, W_ref, rec = run_both(hip, orc, W0, 3)
    assert rel_l2(W, W_ref) < 1e-10
    check_obs(obs, rec)
