"""GPU: axis transforms on both sides of the batch sizes from which the wide blocks are taken, with
ragged last blocks, against torch's complex128 transforms.

Bounds (relative 2-norm): a transform of length N rounds each element about log2 N times by 2^-53 on
either side (complex128), or by 2^-24 on ours (complex64)."""
import math

import pytest

pytestmark = pytest.mark.gpu


def check(cuda, N, batch, axis, precision, seed):
    import torch

    from pywignercuda_amd import cufft_wrapper as cw

    dtype = torch.complex128 if precision == "fp64" else torch.complex64
    shape = (batch, N) if axis == 1 else (N, batch)
    names = {("fp64", 0): cw.Plan_Z2Z_2D_Axis0, ("fp64", 1): cw.Plan_Z2Z_2D_Axis1, ("fp32", 0): cw.Plan_C2C_2D_Axis0,
             ("fp32", 1): cw.Plan_C2C_2D_Axis1}
    plan = names[precision, axis](shape)
    g = torch.Generator(device=cuda).manual_seed(seed)
    A = torch.randn(shape, dtype=dtype, device=cuda, generator=g)
    bound = 2 * math.log2(N) * 2.0 ** -53 if precision == "fp64" else math.log2(N) * 2.0 ** -24
    for inverse in (False, True):
        W = A.clone()
        if inverse:
            cw.ifft_Z2Z_normalized(W, W, plan)
        else:
            cw.fft_Z2Z(W, W, plan)
        # transformed along contiguous rows, in parts, so that no reference is larger than the data
        X, Y = (A, W) if axis == 1 else (A.t(), W.t())
        err = ref2 = 0.0
        for lo in range(0, batch, 1 << 20):
            x = X[lo:lo + (1 << 20)].to(torch.complex128).contiguous()
            r = torch.fft.ifft(x, dim=1) if inverse else torch.fft.fft(x, dim=1)
            err += float((Y[lo:lo + (1 << 20)].to(torch.complex128) - r).abs().square().sum())
            ref2 += float(r.abs().square().sum())
        assert math.sqrt(err / ref2) < bound, (N, batch, axis, precision, inverse)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N", [64, 128, 256, 512])
def test_columns_around_the_wide_blocks(cuda, N, precision):
    wide = 256 // (N // 16)  # columns of a wide block
    for blocks in (1, 255, 256, 261):
        check(cuda, N, blocks * wide, 0, precision, N + blocks)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N", [64, 128, 256, 512, 1024, 2048])
def test_rows_around_the_wide_blocks(cuda, N, precision):
    wide = max(1, 256 // (N // 16))  # rows of a wide block
    for rows in (1, 256 * wide - 1, 256 * wide, 256 * wide + 1, 300 * wide + wide // 2 + 1):
        check(cuda, N, rows, 1, precision, N + rows)


def test_columns_of_64_around_512_mib(cuda):
    for cols in ((1 << 19) - 64, 1 << 19, (1 << 19) + 64):
        check(cuda, 64, cols, 0, "fp64", cols)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N", [64, 512, 1024, 2048])
def test_rows_around_512_mib(cuda, N, precision):
    rows = (512 << 20) // (N * (16 if precision == "fp64" else 8))
    for r in (rows - 1, rows, rows + 3):
        check(cuda, N, r, 1, precision, N)
