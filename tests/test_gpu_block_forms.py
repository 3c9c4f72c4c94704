"""Narrow and wide blocks give the same states: a plan of few cells takes blocks of 64 or 128 lanes, the
same grid in an ensemble with a block for every CU takes 256.  Radix and arithmetic are the same, so
that only the order of the norm's partial sums differs (a rounding or two per step)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

POT = dict(potential="0.1*pow(x,4) - pow(x,2)", dpotential="0.4*pow(x,3) - 2.0*x")


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("damped", [False, True])
@pytest.mark.parametrize("X,P,members", [(128, 128, 64), (256, 128, 40), (128, 256, 40), (512, 256, 9)])
def test_member_alone_and_in_an_ensemble(cuda, X, P, members, damped, precision):
    import torch

    from pywignercuda_amd.wigner2d import Wigner2D, WignerEnsemble

    cl = dict(fp_damping="fabs(p)", D_theta=0.1) if damped else {}
    model = dict(gamma=0.1, damping="CaldeiraLeggett") if damped else {}
    variants = (1, 2, 1)  # radix 8 throughout
    one = Wigner2D(X, P, 10.0, 10.0, 1.0, 1.0, 0.005, precision=precision, variants=variants, device=cuda, mask=True,
                   **POT, **cl, **model)
    many = WignerEnsemble([dict(X=X, P=P, X_amp=10.0, P_amp=10.0, mask=True, **POT, **cl)] * members, 1.0, 1.0, 0.005,
                          precision=precision, variants=variants, device=cuda, **model)
    x, p = one.x_host[None, :], one.p_host[:, None]
    W0 = np.exp(-((x - 1.0) ** 2) - p ** 2) / np.pi
    A, B = one.to_device(W0), many.states_to_device([W0] * members)
    ra, rb = one.run(A, 20), many.run(B, 20)
    torch.cuda.synchronize()
    # 20 steps of a factor that differs by a few 1.1e-16; complex64 states round differently where
    # that moves a value over a rounding boundary (6e-8, rarely)
    tol = 1e-13 if precision == "fp64" else 1e-6
    for i in (0, members - 1):
        assert float(torch.linalg.vector_norm(A - B[i]) / torch.linalg.vector_norm(A)) < tol
        torch.testing.assert_close(rb[i][:20], ra[:20], rtol=max(tol, 1e-12), atol=max(tol, 1e-12))


@pytest.mark.parametrize("steps", [1, 2, 17, 33, 34])
def test_dirac_record_at_run_lengths(cuda, steps):
    """The record rides on the next x sweep, the first and last rows do not: run lengths around the
    graph's 16 iterations, replayed and launched, row sums alternating between two buffers."""
    import torch

    from tests.test_gpu_dirac import check_obs, make_pair

    hip, orc, W0 = make_pair(cuda, "coulomb")
    _, rec = orc.run(W0, steps)
    Wa, Wb = hip.to_device(W0), hip.to_device(W0)
    oa = hip.run(Wa, steps, use_graph=False)
    ob = hip.run(Wb, steps, use_graph=True)
    torch.cuda.synchronize()
    assert torch.equal(Wa, Wb) and torch.equal(oa, ob)
    check_obs(oa.cpu().numpy(), rec)
