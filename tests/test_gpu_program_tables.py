"""GPU: potentials given as programs, whose table of a time index lies in one of two slots (even and
odd indices) and is evaluated for half of the theta rows: runs cut at odd and even indices against
one run, and against the same potential as coefficient rows.

Bounds: cutting a run changes nothing but the merging of two half steps (rounding, taken as 1e-12);
against coefficient rows the FP64 bar of the parity tests, 1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("X,P", [(128, 128), (256, 1024), (2048, 128)])
@pytest.mark.parametrize("scheme", ["lie", "strang"])
def test_cut_runs_and_coefficient_rows(cuda, X, P, scheme):
    from oracle import wigner2d as ow
    from pywignercuda_amd.wigner2d import Wigner2D

    args = (X, P, 9.0, 8.0, 1.0, 1.0, 0.01)
    W0 = ow.cat_state_wigner(ow.Grid(X, P, 9.0, 8.0), a=1.5)
    # the same function: a program (Heaviside keeps it from being a polynomial) and rows
    prog = Wigner2D(*args, potential="0.5*x*x+0.1*sin(40*t)*x*x*x*Heaviside(x*x+1)", dpotential="x", scheme=scheme,
                    device=cuda)
    rows = Wigner2D(*args, potential="0.5*x*x+0.1*sin(40*t)*x*x*x", dpotential="x", scheme=scheme, time_rows=60,
                    device=cuda)
    W = prog.to_device(W0)
    prog.run(W, 45, use_graph=True)
    R = rows.to_device(W0)
    rows.run(R, 45)
    norm = float((R.abs() ** 2).sum()) ** 0.5
    assert float(((W - R).abs() ** 2).sum()) ** 0.5 < 1e-10 * norm
    C = prog.to_device(W0)
    done = 0
    for n in (3, 1, 4, 37):
        prog.run(C, n, first_step=done, normalize_initial=done == 0, use_graph=False)
        done += n
    assert float(((W - C).abs() ** 2).sum()) ** 0.5 < 1e-12 * norm
