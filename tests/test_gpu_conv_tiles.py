"""The convolution's tile shapes: 16, 8 or 4 positions along x of 1, 2 or 4
grids side by side, with remainders in x, in the rows of y, in the group of
grids and in z.  Integer operands, so that every result is exact."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_learned import _bf16_round, _conv_ref, _pack_and_conv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,D", [(8, 6), (5, 6), (3, 5), (7, 4), (9, 3), (2, 10), (3, 9), (1, 10),
                                 (1, 18), (1, 19), (2, 26), (3, 27), (1, 34), (5, 12)])
@pytest.mark.parametrize("cin,cout,xb,yb", [(4, 32, 0, 0), (4, 32, 0, 1), (32, 32, 0, 0),
                                            (32, 32, 1, 1), (32, 3, 0, 0), (32, 3, 1, 0)])
def test_conv3_tile_shapes(B, D, cin, cout, xb, yb):
    import torch
    from cube2_amd import _lib
    rng = np.random.default_rng(B * 1000 + D * 10 + cin + cout)
    X = rng.integers(-3, 4, (B, D, D, D, cin)).astype(np.float64)
    W = rng.integers(-2, 3, (27 * cin, cout)).astype(np.float64)
    b = rng.integers(-4, 5, cout).astype(np.float64)
    print(f"conv3 tiles B={B} D={D} {cin}->{cout} x_bf16={xb} y_bf16={yb}", flush=True)
    got = _pack_and_conv(torch, _lib, X, W, b, cin, cout, int(cout == 32), x_bf16=bool(xb),
                         y_bf16=bool(yb))
    want = _conv_ref(X, W, b, cout == 32)
    assert np.array_equal(got, _bf16_round(want) if yb else want)


@pytest.mark.parametrize("cin,cout,xb,yb", [(4, 32, 0, 0), (4, 32, 0, 1), (32, 32, 0, 0), (32, 32, 1, 1),
                                            (32, 3, 0, 0), (32, 3, 1, 0)])
def test_conv3_on_views_that_begin_at_any_element(cin, cout, xb, yb):
    """Activations one element past a 16-byte boundary: the same bits."""
    import torch
    from cube2_amd import _lib
    B, D = 3, 13
    P, L = D - 2, _lib.lib()
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    tx, ty = (torch.bfloat16 if b else torch.float32 for b in (xb, yb))
    x = torch.randn(B * D ** 3 * cin, generator=g, device="cuda").to(tx)
    W = torch.randn((27 * cin, cout), generator=g, device="cuda")
    bias = torch.randn(cout, generator=g, device="cuda")
    Wp = torch.empty((27 if cin == 32 else 32) * (16 if cout == 3 else 32) * cin, dtype=torch.int16, device="cuda")
    _lib.check(L.cube2_cnn_conv_pack_dev(W.data_ptr(), Wp.data_ptr(), cin, cout))
    out = []
    for off in (0, 1):
        xv = torch.empty(x.numel() + 8, dtype=tx, device="cuda")[off:off + x.numel()].copy_(x)
        y = torch.empty(B * P ** 3 * cout + 8, dtype=ty, device="cuda")[off:off + B * P ** 3 * cout]
        assert xv.data_ptr() % 16 == off * (2 if xb else 4) and y.data_ptr() % 16 == off * (2 if yb else 4)
        _lib.check(L.cube2_cnn_conv3_dev(xv.data_ptr(), xb, Wp.data_ptr(), bias.data_ptr(), y.data_ptr(), yb,
                                         B, D, cin, cout, 1))
        out.append(y.clone())
    assert torch.equal(out[0], out[1])
