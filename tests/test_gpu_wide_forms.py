"""GPU: every launch variant of the sweeps in the block width that its table names.  A plan of few cells
takes 64- or 128-lane blocks in place of 256-lane ones of radix 4 and 8 (narrow_variants), so that an
ensemble of 2^19 cells and more, a 256-lane block of radix 8 for each of the 256 CUs, is needed to
launch them.  Against the oracle, first and last member, 4 steps; and against the member alone, whose
blocks are narrow.

Bounds.  complex128: the FP64 bar of the parity tests (1e-10).  complex64 states: one rounding (2^-24) per
sweep and one for the initial state, and in the throughput forms of the plain sweeps one per exchange
(at most 3 per transform, 2 transforms per sweep): 9 + 8 * 6 = 57 * 6e-8 = 3.4e-6, taken as 4e-6.
Narrow against wide: 4 steps whose norms differ in the order of their partial sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUND = {"fp64": 1e-10, "fp32": 4e-6}
ALONE = {"fp64": 1e-13, "fp32": 1e-6}
CUS, LANES = 256, 256


def forms(table):
    """(index, radix, lanes) of a table's variants."""
    import ctypes

    from pywignercuda_amd import _lib

    out = []
    for v in range(_lib.lib().wh_variant_info(table, -1, None, None)):
        r, n = ctypes.c_int(), ctypes.c_int()
        assert _lib.lib().wh_variant_info(table, v, ctypes.byref(r), ctypes.byref(n)) == 0
        out.append((v, r.value, n.value))
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("damped", [False, True])
@pytest.mark.parametrize("X,P", [(N, 128) for N in (128, 256, 512, 1024, 2048)] + [(128, N) for N in (256, 512, 1024, 2048)])
def test_forms_in_filled_ensembles(cuda, X, P, damped, precision):
    from oracle import wigner2d as ow
    from pywignercuda_amd import _lib
    from pywignercuda_amd.wigner2d import Wigner2D, WignerEnsemble

    members = (1 << 19) // (X * P) + 1
    model = dict(scheme="lie", gamma=0.01, damping="CaldeiraLeggett") if damped else dict(scheme="lie")
    own = dict(fp_damping="fabs(p)", D_theta=1e-4) if damped else {}
    args, pot = (X, P, 9.0, 7.0), dict(potential="0.5*pow(x,2)", dpotential="x", mask=True)
    many = WignerEnsemble([dict(X=X, P=P, X_amp=9.0, P_amp=7.0, **pot, **own)] * members, 0.8, 1.3, 0.01,
                          precision=precision, device=cuda, **model)
    one = Wigner2D(*args, 0.8, 1.3, 0.01, precision=precision, device=cuda, **pot, **own, **model)
    okw = dict(fp_damping=np.abs, D_theta=1e-4) if damped else {}
    orc = ow.Wigner2DOracle(*args, 0.8, 1.3, 0.01, potential=lambda t, x: 0.5 * x ** 2, dpotential=lambda t, x: x,
                            mask=True, **okw, **model)
    W0 = ow.gaussian_wigner(orc.g, x0=1.0, p0=-0.5, s=1.1)
    ref, _, _ = orc.run(W0, 3)
    done = 0
    for table in (0, 2) if damped else (0, 1):
        for v, R, lanes in forms(table):
            choice = [-1, -1, -1]
            choice[table] = v
            try:
                many.set_variants(*choice)
            except _lib.WignerHipInvalidValue:
                continue  # this form does not cover the size
            if R < 16 and lanes == LANES:  # the width stays
                assert members * X * P // (R * lanes) >= CUS
            one.set_variants(*choice)
            A, B = one.to_device(W0), many.states_to_device([W0] * members)
            one.run(A, 4)
            many.run(B, 4)
            a = A.cpu().numpy().astype(complex)
            for i in (0, members - 1):
                b = B[i].cpu().numpy().astype(complex)
                assert np.linalg.norm(b - ref) < BOUND[precision] * np.linalg.norm(ref), (table, v, i)
                assert np.linalg.norm(b - a) < ALONE[precision] * np.linalg.norm(a), (table, v, i)
            done += 1
    assert done >= 4
