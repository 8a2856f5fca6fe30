"""What the learned network's Python calls hand to the library, with a recording
stand-in for it: gradients of the wrong size are refused before any call, and a
step given some layers' gradients moves those layers."""
from __future__ import annotations

import ctypes as C

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


def _grads(net, n):
    return [(torch.ones_like(w), torch.ones_like(b)) for w, b in zip(net.W, net.b)][:n]


def test_step_of_all_layers_is_one_call_with_eight_gradients(net):
    net.rec.calls.clear()
    grads = _grads(net, 4)
    net.step(grads)
    (name, args), = net.rec.calls
    assert name == "cube2_cnn_net_adam_dev" and net.t == 1
    assert list(args[1]) == [g.data_ptr() for g in [dW for dW, _ in grads] + [db for _, db in grads]]
    assert all(len(a) == 8 for a in args[:4]) and all(len(a) == 4 for a in args[4:6])


@pytest.mark.parametrize("n", [0, 1, 3])
def test_step_of_some_layers_moves_those(net, n):
    net.rec.calls.clear()
    grads = _grads(net, n)
    net.step(grads, lr=2e-3)
    adam = [a for name, a in net.rec.calls if name == "cube2_cnn_adam_dev"]
    assert "cube2_cnn_net_adam_dev" not in net.rec.names()
    want = [x for l in range(n) for x in ((net.W[l], grads[l][0]), (net.b[l], grads[l][1]))]
    assert [(a[0], a[1], a[5]) for a in adam] == [(w.data_ptr(), g.data_ptr(), w.numel()) for w, g in want]
    assert all(a[6:] == (2e-3, 0.9, 0.999, 1e-8, 1) for a in adam)
    # every layer's packed weights are refreshed after it
    assert net.rec.names()[2 * n:] == ["cube2_cnn_conv_pack_dev"] * 4
    assert isinstance(learned._ps(net.W), C.Array) and net.t == 1
