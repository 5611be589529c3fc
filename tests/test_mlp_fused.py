"""The one-launch forward and backward of the MLP against a launch per layer: the same outputs bit for bit, the
gradients within the rounding of float32 sums in another order (GPU)."""

import numpy as np
import pytest
import torch

from maxichem_amd.learned import MLP, pad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in, n_out, width, depth, rows", [
    (120, 71, 256, 4, 64), (120, 71, 256, 4, 1500), (3, 1, 64, 1, 1), (200, 130, 192, 2, 1088), (64, 256, 128, 3, 640),
    (70, 9, 64, 0, 200), (16, 4, 64, 2, 32769),
])  # fmt: skip
def test_one_launch_equals_a_launch_per_layer(n_in, n_out, width, depth, rows):
    g = torch.Generator(device="cuda").manual_seed(rows)
    net = MLP(n_in, n_out, "cuda", width=width, depth=depth, seed=1)
    assert net.fused
    M = pad(rows)
    x = torch.zeros(M, net.dims[0], device="cuda")
    x[:rows, :n_in] = torch.randn(rows, n_in, generator=g, device="cuda")
    X, T = net.to_bf16(x), torch.randn(rows, n_out, generator=g, device="cuda")
    w = torch.linspace(0.5, 2.0, n_out, device="cuda")
    got = []
    for fused in (True, False):
        net.fused = fused
        plain = net.forward(X)
        Y = net.forward(X, keep=True)
        assert torch.equal(plain, Y)
        kept = [a.clone() for a in (*net._acts, *net._pre)]
        for ly in net.layers:  # every entry is written
            ly.gw.fill_(float("nan"))
            ly.gb.fill_(float("nan"))
        net.backward(net.loss_grad(Y, T, w, rows))
        got.append((Y, kept, [ly.gw.clone() for ly in net.layers], [ly.gb.clone() for ly in net.layers]))
    (y0, k0, gw0, gb0), (y1, k1, gw1, gb1) = got
    assert torch.equal(y0, y1) and all(torch.equal(a, b) for a, b in zip(k0, k1))
    for a, b in zip(gw0 + gb0, gw1 + gb1):
        # two float32 sums of M terms: each within M u of the terms' absolute sum, in practice sqrt(M) u of its size
        assert float((a - b).abs().max()) <= 4.0 * np.sqrt(M) * 2.0**-24 * np.sqrt(M) * float(b.abs().max())
        assert torch.isfinite(a).all()
