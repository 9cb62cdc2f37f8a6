"""Parameter gradients of gnn_mlp_grads equal gnn_weight_grad's over 64 chunks
bit for bit: the same products added in the same order, whatever the shape
(rows around a step of 32 and a chunk, one chunk and 64, gathered sources)."""
from __future__ import annotations

import pytest
import torch

from cabanadem_amd import surrogate as S
from test_gpu_gnn import make_mlp
from test_gpu_gnn_grads import BF, fused, rnd, separate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 31, 33, 2047, 2049, 9241, 20011])
@pytest.mark.parametrize("kind", ["node", "edge", "decoder", "encoder"])
def test_same_bits(gpu_lib, kind, M):
    gen = torch.Generator(device="cuda").manual_seed(M + 1)
    K, nout = {"node": (256, 128), "edge": (384, 128), "decoder": (128, 3), "encoder": (32, 128)}[kind]
    m, fl, _ = make_mlp(K, nout, seed=M)
    hid = torch.relu(rnd(gen, M, 128)).to(BF)
    dY = rnd(gen, M, nout)
    add = idx = None
    if kind == "edge":
        h = rnd(gen, 57, 128).to(BF)
        pick = lambda: torch.randint(0, 57, (M,), device="cuda", generator=gen).to(torch.int32)
        add, idx, send, e = rnd(gen, 57, 128), pick(), pick(), rnd(gen, M, 128).to(BF)
        io = S.io(M, (e, None), (h, idx), (h, send))
        _, gb = fused(m, fl, io, hid, dY.clone(), add, idx, [None] * 3, 0)[1:]
        dY = dY + add[idx.long()]
    else:
        xs = [rnd(gen, M, min(K, 128)).to(BF) for _ in range(2 if kind == "node" else 1)]
        io = S.io(M, *[(x, None) for x in xs])
        _, gb = fused(m, fl, io, hid, dY, None, None, [None] * 3, 0)[1:]
    _, ga = separate(m, fl, io, hid, dY, [None] * 3, 0)
    for a, b in zip(m.views(ga), m.views(gb)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("M", [1, 97, 5003])
@pytest.mark.parametrize("parts", ["dY", "add", "both"])
def test_residual_into_another_buffer(gpu_lib, parts, M):
    """accumulate bit 3 writes what the in-place form writes, from the same dY."""
    gen = torch.Generator(device="cuda").manual_seed(M)
    m, fl, _ = make_mlp(128, 128, seed=M)
    x, hid = rnd(gen, M, 128).to(BF), torch.relu(rnd(gen, M, 128)).to(BF)
    dY = rnd(gen, M, 128) if parts != "add" else None
    add = rnd(gen, 9, 128) if parts != "dY" else None
    idx = torch.randint(0, 9, (M,), device="cuda", generator=gen).to(torch.int32)
    a = rnd(gen, M, 128) if dY is None else dY.clone()
    b = rnd(gen, M, 128)
    io = S.io(M, (x, None))
    ra = fused(m, fl, io, hid, None if dY is None else a, add, idx, [a, None, None], 1)
    rb = fused(m, fl, io, hid, dY, add, idx, [b, None, None], 8)
    assert torch.equal(a, b)
    for p, q in zip(ra, rb):
        assert torch.equal(p[:m.end], q[:m.end])
