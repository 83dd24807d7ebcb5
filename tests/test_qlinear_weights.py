"""QLinear.forward goes through its weight's own matmul_t: a subclass of QTensor
that overrides it (to count, log or place calls), or any object with shape(),
device and matmul_t.  No device is needed."""
from types import SimpleNamespace

import torch

from xn_amd import QLinear, QTensor


def product(w, mkn, lhs, dst):
    m, k, n = mkn
    dst.copy_((lhs.reshape(m, k) @ w.t()).view(dst.shape))


def test_any_object_with_matmul_t():
    class Weight:
        device = torch.device("cpu")

        def __init__(self, w):
            self.w = w

        def shape(self):
            return tuple(self.w.shape)

        def matmul_t(self, mkn, lhs, dst):
            product(self.w, mkn, lhs, dst)

    w, x = torch.randn(5, 8), torch.randn(2, 3, 8)
    assert torch.allclose(QLinear(Weight(w)).forward(x), x @ w.t(), atol=1e-6)


def test_a_subclass_that_overrides_matmul_t():
    class Counting(QTensor):
        calls = 0

        def matmul_t(self, mkn, lhs, dst):
            self.calls += 1
            product(self.w, mkn, lhs, dst)

    qt = object.__new__(Counting)
    qt.w = torch.randn(5, 8)
    qt._shape, qt.storage = (5, 8), SimpleNamespace(device=torch.device("cpu"), _h=None, handle=None)
    x = torch.randn(4, 8)
    assert torch.allclose(QLinear(qt, torch.ones(5)).forward(x), x @ qt.w.t() + 1, atol=1e-6)
    assert qt.calls == 1
