"""What Wigner2D.adjoint_segment and wh_wigner2d_steps / _adjoint_segment refuse before any launch.

CPU: the Python checks, on a plan and tensors that only carry what is checked; the library is
replaced by one that fails the test when it is called.  GPU: misaligned addresses."""
import ctypes

import pytest
import torch

X, P, N = 128, 256, 3


class _Tensor:
    """A device tensor's metadata."""

    def __init__(self, shape, dtype, device="cuda:0", contiguous=True):
        self.shape, self.dtype, self.device, self._contiguous = shape, dtype, torch.device(device), contiguous
        self.is_cuda = self.device.type == "cuda"

    def is_contiguous(self):
        return self._contiguous

    def __getitem__(self, i):
        if not -self.shape[0] <= i < self.shape[0]:
            raise IndexError(i)
        return _Tensor(self.shape[1:], self.dtype, str(self.device))


def _state(n=None, **kw):
    return _Tensor((P, X) if n is None else (n, P, X), torch.complex128, **kw)


@pytest.fixture
def plan(monkeypatch):
    from pywignercuda_amd import _lib
    from pywignercuda_amd.wigner2d import Wigner2D

    def called():
        raise AssertionError("the library was called")

    monkeypatch.setattr(_lib, "lib", called)
    p = object.__new__(Wigner2D)
    p.X, p.P, p.dtype, p._plan = X, P, torch.complex128, None
    return p


BAD_GRADS = [_Tensor((N, 9), torch.float32), _Tensor((N, 9), torch.complex64), _Tensor((N, 9), torch.float64, "cpu"),
             _Tensor((N, 9), torch.float64, "cuda:1"), _Tensor((N, 9), torch.float64, contiguous=False),
             _Tensor((N, 8), torch.float64), _Tensor((N + 1, 9), torch.float64)]


@pytest.mark.parametrize("grads", BAD_GRADS)
def test_gradient_rows_that_the_kernels_cannot_write(plan, grads):
    with pytest.raises(ValueError, match="grads"):
        plan.adjoint_segment(_state(), _state(N), _state(), 0, grads)


def test_no_steps_and_scattered_states(plan):
    with pytest.raises(ValueError, match="no step"):
        plan.adjoint_segment(_state(), _state(0), _state(), 0, _Tensor((0, 9), torch.float64))
    with pytest.raises(ValueError, match="states"):
        plan.adjoint_segment(_state(), _state(N, contiguous=False), _state(), 0, _Tensor((N, 9), torch.float64))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32fast"])
def test_misaligned_addresses(cuda, precision):
    from pywignercuda_amd import _lib
    from pywignercuda_amd.wigner2d import Wigner2D

    p = Wigner2D(128, 128, 8.0, 8.0, 1.0, 1.0, 0.01, potential="0.5*pow(x,2)", dpotential="x", precision=precision,
                 device=cuda)
    W = torch.zeros((4, 128, 128), dtype=p.dtype, device=cuda)
    g = torch.zeros((4, 9), dtype=torch.float64, device=cuda)
    L, addr, half = _lib.lib(), int(W.data_ptr()), W.element_size() // 2
    ptr, odd, gp, godd = (ctypes.c_void_p(a) for a in (addr, addr + half, int(g.data_ptr()), int(g.data_ptr()) + 4))
    unaligned = 9  # WH_UNALIGNED_DATA
    for a, b in ((odd, ptr), (ptr, odd)):
        assert L.wh_wigner2d_steps(p._plan, a, b, 0, 1, None) == unaligned
    for first, states, lam, grads in ((odd, ptr, ptr, gp), (ptr, odd, ptr, gp), (ptr, ptr, odd, gp), (ptr, ptr, ptr, godd)):
        assert L.wh_wigner2d_adjoint_segment(p._plan, first, states, lam, 0, 1, grads, None) == unaligned
