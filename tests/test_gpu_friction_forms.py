"""GPU: the friction p sweep in every form (radix 16 and 8, tables in registers and read per operator)
at every side, all precisions, against the oracle.

Bounds.  complex128: the FP64 bar of the parity tests (1e-10).  complex64 states with FP64 arithmetic:
one rounding (2^-24) for each of the 8 sweeps of 4 steps and one for the initial state, 9 * 6e-8 =
5.4e-7, taken as 6e-7; the exchanges are in FP64 in every form.  FP32 arithmetic: 10 transforms per
step of log2(2048) = 11 roundings each, 4 * 10 * 11 * 2^-24 = 2.7e-5, taken as 3e-5.  gamma keeps the
composite's largest factor below 2 at P = 2048 (dt gamma p theta = 0.3), so that nothing is amplified."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUND = {"fp64": 1e-10, "fp32": 6e-7, "fp32fast": 3e-5}


@pytest.mark.parametrize("precision", sorted(BOUND))
@pytest.mark.parametrize("P", [128, 256, 512, 1024, 2048])
def test_friction_forms(cuda, P, precision):
    from oracle import wigner2d as ow
    from pywignercuda_amd import _lib
    from pywignercuda_amd.wigner2d import Wigner2D

    args = (128, P, 9.0, 7.0, 0.8, 1.3, 0.01)
    kw = dict(scheme="lie", gamma=0.01, damping="CaldeiraLeggett", D_theta=1e-4, mask=True)
    p = Wigner2D(*args, potential="0.5*pow(x,2)", dpotential="x", fp_damping="fabs(p)", precision=precision, device=cuda,
                 **kw)
    o = ow.Wigner2DOracle(*args, potential=lambda t, x: 0.5 * x ** 2, dpotential=lambda t, x: x, fp_damping=np.abs, **kw)
    W0 = ow.gaussian_wigner(o.g, x0=1.0, p0=-0.5, s=1.1)
    ref, _, _ = o.run(W0, 3)
    done = 0
    for v in range(_lib.lib().wh_variant_info(2, -1, None, None)):
        try:
            p.set_variants(-1, -1, v)
        except _lib.WignerHipInvalidValue:
            continue  # this form does not cover the size
        W = p.to_device(W0)
        p.run(W, 4)
        err = np.linalg.norm(W.cpu().numpy().astype(complex) - ref) / np.linalg.norm(ref)
        assert err < BOUND[precision], (v, err)
        done += 1
    assert done >= 2
