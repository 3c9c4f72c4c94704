"""The axis transforms at the edges of their blocks: row counts that leave a block partly empty (a
block holds up to eight rows), and the smallest column counts (one or a few tiles), between guard
rows that must stay as they are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# multiples that the column plans ask for
COLUMNS = {64: 64, 128: 32, 256: 16, 512: 8, 1024: 4, 2048: 2}


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", sorted(COLUMNS))
@pytest.mark.parametrize("direction", [-1, 1])
def test_partly_filled_blocks(cuda, prec, n, direction):
    import torch

    from pywignercuda_amd import cufft_wrapper as cw

    rng = np.random.default_rng(n)
    dt = torch.complex128 if prec == "fp64" else torch.complex64
    ft = cw.CUFFT_Z2Z if prec == "fp64" else cw.CUFFT_C2C
    # 11 passes of two roundings at most, 1.1e-16 or 6e-8 each, and complex64's input rounding
    tol = 1e-14 if prec == "fp64" else 2e-6
    fwd = direction < 0
    for axis, other in [(1, 1), (1, 3), (1, 9), (0, COLUMNS[n]), (0, 3 * COLUMNS[n])]:
        shape = (other, n) if axis == 1 else (n, other)
        a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
        whole = torch.full((shape[0] + 2, shape[1]), 7.0 - 3.0j, dtype=dt, device=cuda)
        t = whole[1:-1]
        t.copy_(torch.tensor(a, dtype=dt))
        plan = (cw.Plan_Z2Z_2D_Axis1 if axis == 1 else cw.Plan_Z2Z_2D_Axis0)(shape, fft_type=ft)
        (cw.fft_Z2Z if fwd else cw.ifft_Z2Z_normalized)(t, t, plan)
        torch.cuda.synchronize()
        ref = np.fft.fft(a, axis=axis) if fwd else np.fft.ifft(a, axis=axis)
        err = np.linalg.norm(t.cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err < tol, (axis, other, err)
        assert torch.all(whole[0] == 7.0 - 3.0j) and torch.all(whole[-1] == 7.0 - 3.0j), (axis, other)
