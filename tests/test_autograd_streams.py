"""logdet_quad on a device that is not the current one: the factor works on its own stream, so
what it reads and overwrites must be waited for on the tensors' device.  On the CPU, with
stand-ins that record who waits for what."""
from types import SimpleNamespace

import pytest

from swcholesky_amd import autograd


class _Device:
    """Device ``cuda:k``: whether work is queued on its stream."""

    def __init__(self):
        self.busy = {0: False, 1: False}

    def stream(self, device=None):
        k = 0 if device is None else int(device[-1])  # cuda:0 is current

        def synchronize():
            self.busy[k] = False
        return SimpleNamespace(synchronize=synchronize)


class _Tensor:
    is_cuda, device, shape = True, "cuda:1", (3,)

    def __init__(self, dev):
        self.dev = dev

    def _kernel(self, *_):
        self.dev.busy[1] = True
        return _Tensor(self.dev)

    to = contiguous = clone = __mul__ = __rmul__ = _kernel

    def detach(self):
        return self


class _Factor:
    n, bcsc = 3, SimpleNamespace(nnz=5)

    def __init__(self, dev):
        self.dev, self.calls = dev, []

    def _idle(self, what):
        assert not self.dev.busy[1], f"{what} starts before the tensors' values are there"
        self.calls.append(what)

    def factor(self, values):
        self._idle("factor")
        return 0

    def solve_device(self, x):
        self._idle("solve")
        return x

    def gradient(self, x, alpha, beta, out):
        self._idle("gradient")

    def logdet(self):
        return 0.0


@pytest.fixture
def world(monkeypatch):
    dev = _Device()
    fake = SimpleNamespace(float64="f64", dot=lambda a, b: 0.0, tensor=lambda v, dtype, device: v,
                           empty=lambda n, dtype, device: _Tensor(dev),
                           cuda=SimpleNamespace(is_available=lambda: True, current_stream=dev.stream))
    monkeypatch.setattr(autograd, "torch", fake)
    return dev, _Factor(dev)


def test_waits_on_the_tensors_device(world):
    dev, factor = world
    ctx = SimpleNamespace(save_for_backward=lambda *t: setattr(ctx, "saved_tensors", t))
    autograd._LogdetQuad.forward(ctx, _Tensor(dev), _Tensor(dev), factor, 1.0, 1.0)
    dev.busy[1] = True  # the caller goes on using the device
    autograd._LogdetQuad.backward(ctx, _Tensor(dev))
    assert factor.calls == ["factor", "solve", "gradient"]
