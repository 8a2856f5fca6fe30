"""The network's one-call backward and Adam step (training patches) against
the im2col products and the per-tensor Adam kernel they stand in for."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net_and_input(B, D, seed):
    import torch
    from cube2_amd.learned import LearnedPP
    net = LearnedPP(seed=seed)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn((B, D, D, D, 4), generator=g, device="cuda")
    dout = torch.randn((B, D - 8, D - 8, D - 8, 3), generator=g, device="cuda")
    return net, x, dout


@pytest.mark.parametrize("B,D", [(1, 10), (5, 10), (257, 10), (600, 10), (1, 9), (300, 9)])
def test_patch_backward_matches_im2col(monkeypatch, B, D):
    """Same BF16 operands and per-tap products; the weight gradients' FP32 sums
    over n = B (D - 2)^3 positions at most run in another order, each with an
    error of about 2^-24 sqrt(n / 2) of their norm (3e-5 at n = 3e5)."""
    from cube2_amd import learned
    net, x, dout = _net_and_input(B, D, 31 + B)
    net.forward(x)
    print(f"net backward B={B} D={D}", flush=True)
    got = net.backward(dout)
    monkeypatch.setattr(learned, "PATCH", 0)
    want = net.backward(dout)
    for l, ((gw, gb), (ww, wb)) in enumerate(zip(got, want)):
        for name, a, b in (("dW", gw, ww), ("db", gb, wb)):
            err = float((a.double() - b.double()).norm() / b.double().norm())
            assert err < 3e-5, (l, name, err)


def test_net_adam_equals_the_tensor_kernels():
    import torch
    from cube2_amd import _lib
    net, x, dout = _net_and_input(4, 10, 5)
    L, p = _lib.lib(), lambda t: t.data_ptr()  # noqa: E731
    w = [t.clone() for t in net.W + net.b]
    m, v = [torch.zeros_like(t) for t in w], [torch.zeros_like(t) for t in w]
    for step in (1, 2, 3):
        net.forward(x)
        grads = net.backward(dout)
        net.step(grads, lr=3e-3)
        g = [a for a, _ in grads] + [b for _, b in grads]
        for q in range(8):
            wb = torch.empty(w[q].shape, dtype=torch.int16, device="cuda")
            _lib.check(L.cube2_cnn_adam_dev(p(w[q]), p(g[q]), p(m[q]), p(v[q]), p(wb), w[q].numel(),
                                            3e-3, 0.9, 0.999, 1e-8, step))
            if q < 4:
                cin, cout = (4, 32, 32, 32, 3)[q:q + 2]
                wp = torch.empty_like(net.Wp[q])
                _lib.check(L.cube2_cnn_conv_pack_dev(p(w[q]), p(wp), cin, cout))
                assert torch.equal(net.Wb[q], wb) and torch.equal(net.Wp[q], wp)
        assert all(np.array_equal(a.cpu().numpy(), b.cpu().numpy()) for a, b in zip(net.W + net.b, w))


def test_larger_patches_are_refused_by_the_one_call_backward():
    import ctypes as C
    from cube2_amd import _lib
    net, x, dout = _net_and_input(1, 11, 6)
    net.forward(x)
    ps = lambda ts: (C.c_void_p * len(ts))(*[t.data_ptr() for t in ts])  # noqa: E731
    rc = _lib.lib().cube2_cnn_net_backward_dev(ps(net.acts), ps(net.Wb), dout.data_ptr(), 1, 11,
                                               ps(net.mW), ps(net.mb))
    assert rc == _lib.ERR_CAPACITY
    assert len(net.backward(dout)) == 4      # the general path


@pytest.mark.parametrize("D,l", [(10, 1), (10, 3), (9, 0), (9, 1), (9, 2), (9, 3)])
def test_patch_backward_keeps_infinities_where_they_belong(monkeypatch, D, l):
    """An infinite activation in the last row of layer l's input reaches the
    weight gradients of the taps that read it and no others, as with im2col:
    the rows that pad the positions to fours are no terms of the sum."""
    import torch
    from cube2_amd import learned
    net, x, dout = _net_and_input(3, D, 40 + l)
    net.forward(x)
    d = D - 2 * l
    net.acts[l] = net.acts[l].clone()
    net.acts[l][1, 1, d - 1, 2, 3] = float("inf")
    got = net.backward(dout)
    monkeypatch.setattr(learned, "PATCH", 0)
    want = net.backward(dout)
    for k, ((gw, gb), (ww, wb)) in enumerate(zip(got, want)):
        for a, b in ((gw, ww), (gb, wb)):
            ok = torch.isfinite(b)
            assert torch.equal(torch.isfinite(a), ok), (k, int(ok.sum()), int(torch.isfinite(a).sum()))
            assert float((a - b)[ok].double().norm()) <= 3e-5 * float(b[ok].double().norm())
    assert not torch.isfinite(want[l][0]).all() and torch.isfinite(want[l][0]).any()


@pytest.mark.parametrize("D,l", [(10, 3), (10, 1), (9, 2)])
def test_patch_backward_keeps_infinite_weights_off_the_border(monkeypatch, D, l):
    """An infinite weight of a tap that no output uses at the only position where
    its input channel is active: the gradients stay finite, as with im2col."""
    import torch
    from cube2_amd import learned
    net, x, dout = _net_and_input(3, D, 50 + l)
    net.forward(x)
    c, cout = 5, (4, 32, 32, 32, 3)[l + 1]
    net.acts[l] = net.acts[l].clone()
    net.acts[l][..., c] = 0.0
    net.acts[l][:, -1, -1, -1, c] = 1.0
    net.Wb[l].view(27, 32, cout)[0, c, 1] = 0x7f80  # (tap 0 reaches the inputs 0 .. P - 1 alone)
    got = net.backward(dout)
    monkeypatch.setattr(learned, "PATCH", 0)
    want = net.backward(dout)
    for k, ((gw, gb), (ww, wb)) in enumerate(zip(got, want)):
        for a, b in ((gw, ww), (gb, wb)):
            assert torch.isfinite(b).all() and torch.isfinite(a).all(), k
            assert float((a - b).double().norm()) <= 3e-5 * float(b.double().norm())
