"""What the learned network's Python calls hand to the library, with a recording
stand-in for it: gradients of the wrong size are refused before any call."""
from __future__ import annotations

import pytest
import torch

from cube2_amd import _lib, learned


class Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return _lib.OK
        return call

    def names(self):
        return [n for n, _ in self.calls]


@pytest.fixture
def net(monkeypatch):
    rec = Recorder()
    monkeypatch.setattr(_lib, "lib", lambda: rec)
    net = learned.LearnedPP(seed=3, device="cpu")
    net.rec = rec
    return net


@pytest.mark.parametrize("D", [9, 10, 12])
@pytest.mark.parametrize("shape", [(2, 1), (2, 2, 2, 1, 3), (2, 40, 3), (1, 0)])
def test_backward_refuses_a_gradient_of_another_size(net, D, shape):
    net.forward(torch.zeros(2, D, D, D, 4))
    net.rec.calls.clear()
    with pytest.raises(RuntimeError):
        net.backward(torch.zeros(shape))
    assert net.rec.calls == []


@pytest.mark.parametrize("D", [9, 10])
def test_backward_takes_any_shape_of_the_right_size(net, D):
    net.forward(torch.zeros(2, D, D, D, 4))
    net.rec.calls.clear()
    grads = net.backward(torch.zeros(2, (D - 8) ** 3 * 3))
    assert net.rec.names() == ["cube2_cnn_net_backward_dev"] and len(grads) == 4
