"""Column transforms of batches whose array spans more than 2^32 bytes per team of lanes.

CPU: the element index that the kernels use (wh_index.hpp, compiled for the host) against Python
integers, at batches above and below the point where a 32-bit byte offset wraps.
GPU: a batch above that point, against torch.fft on some of its columns; the others stay zero."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "pywignercuda_amd" / "csrc"
# (row, columns, column): last row of a team's lanes at its length, first and last columns
PLACES = [(row, X, col) for row in (0, 1, 7, 15, 31, 63, 127, 1920, 2047)
          for X in (64, 8521760, 8521792, 4260864, 4260896, 38404096, 2 ** 31 - 64) for col in (0, X // 2 + 1, X - 1)]


def test_column_element_indices(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("needs g++")
    src, exe = tmp_path / "index.cpp", tmp_path / "index"
    src.write_text('#include "wh_index.hpp"\n#include <cstdio>\nint main() {\n'
                   + "".join(f'  std::printf("%zu\\n", wh::col_element({r}, {X}, {c}));\n' for r, X, c in PLACES) + "}\n")
    subprocess.run([cxx, "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    got = [int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]
    assert got == [r * X + c for r, X, c in PLACES]


def test_where_byte_offsets_fit_32_bits(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("needs g++")
    cases = [(rows, X, size) for rows in (4, 8, 32, 64, 128) for size in (8, 16)
             for X in (64, 2 ** 32 // (rows * size) - 1, 2 ** 32 // (rows * size), 2 ** 32 // (rows * size) + 1, 2 ** 31 - 64)]
    src, exe = tmp_path / "fit.cpp", tmp_path / "fit"
    src.write_text('#include "wh_index.hpp"\n#include <cstdio>\nint main() {\n' + "".join(
        f'  std::printf("%d\\n", int(wh::offsets_fit_32({r}, {X}, {s})));\n' for r, X, s in cases) + "}\n")
    subprocess.run([cxx, "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    got = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    # the largest offset is that of the last element of row rows - 1
    assert got == [str(int((r * X - 1) * s < 2 ** 32)) for r, X, s in cases]


@pytest.mark.gpu
@pytest.mark.parametrize("n,X", [(64, 38404096), (1024, 4325376)])
def test_columns_beyond_four_gigabytes_per_team(cuda, n, X):
    """complex128: the byte offset of the last of eight lane rows (39 GB), and of the last of the 64 lane
    rows of length 1024 (71 GB, the kernels with 64-bit offsets), passes 2^32."""
    import torch

    from pywignercuda_amd import cufft_wrapper as cw

    if torch.cuda.mem_get_info()[0] < (n * X * 16 >> 30) + 20 << 30:
        pytest.skip("needs that much free device memory")
    cols = [0, 1, 63, 55960, X // 2, X - 65, X - 1]
    W = torch.zeros((n, X), dtype=torch.complex128, device=cuda)
    try:
        g = torch.Generator(device="cpu").manual_seed(3)
        a = torch.randn((n, len(cols)), dtype=torch.complex128, generator=g)
        for i, c in enumerate(cols):
            W[:, c] = a[:, i].to(cuda)
        plan = cw.Plan_Z2Z_2D_Axis0((n, X))
        cw.fft_Z2Z(W, W, plan)
        ref = np.fft.fft(a.numpy(), axis=0)
        got = np.stack([W[:, c].cpu().numpy() for c in cols], axis=1)
        # one transform's rounding: eps log2(n) on each side, relative to the largest element
        assert np.abs(got - ref).max() <= 2.3e-16 * np.log2(n) * 4 * np.abs(ref).max()
        for c in cols:
            W[:, c] = 0
        for row in W:  # (row by row: no second array of this size)
            assert int(torch.count_nonzero(torch.view_as_real(row))) == 0
    finally:
        del W
        torch.cuda.empty_cache()
