"""Node and edge features that start inside a larger array (not 16-byte aligned)
train as their aligned copies do, bit for bit: forward and backward take them."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from cabanadem_amd import surrogate as S
from test_gpu_gnn import bf, radius_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,offset", [(40, 2), (400, 2), (400, 6)])
def test_feature_views(gpu_lib, n, offset):
    g, _ = radius_graph(n, seed=1)
    assert g.E > 0
    rng = np.random.default_rng(2)
    xn, xe = (bf(rng.normal(size=(k, 32))).cuda() for k in (g.N, g.E))
    d_out = torch.from_numpy(rng.normal(size=(g.N, 3)).astype(np.float32)).cuda()
    net = S.Network(n_layers=2, seed=3, residual_scale=0.5)

    def view(t):
        a = torch.zeros(t.numel() + 8, dtype=t.dtype, device=t.device)
        v = a[offset:offset + t.numel()].view(t.shape)
        assert v.data_ptr() % 16 == 2 * offset
        return v.copy_(t)

    out = []
    for f in (lambda t: t, view):
        y = net.forward(g, f(xn), f(xe), train=True).clone()
        net.grad.fill_(7.)
        net.backward(g, f(xn), f(xe), d_out)
        out.append((y, net.grad.clone()))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert out[0][1].abs().max() > 0
