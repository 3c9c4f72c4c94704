"""What Wigner2D.adjoint_segment refuses before the library is called.

On a plan and tensors that only carry what is checked; the library is replaced by one that fails
the test when it is called."""
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
