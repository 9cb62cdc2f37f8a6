"""The fused MLP gradients (gnn_mlp_grads, gnn_edge_hidden_grad_to_nodes)
against the single-purpose entry points they stand for (gnn_broadcast_add,
gnn_mlp_backward, gnn_weight_grad, gnn_edge_grad_to_nodes), which
test_gpu_gnn.py pins to FP32 autograd.

Row quantities (dH, dX, node sums) take the same products in the same order,
so they are equal bit for bit.  Parameter gradients are FP32 sums over M rows
in another order: random rounding of M terms stays near sqrt(M) 2^-24 of the
sum's own norm (1.6e-5 at 70,001 rows if every partial sum were as large as
the total), so 2e-5 normwise."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from cabanadem_amd import surrogate as S
from test_gpu_gnn import make_mlp, rel

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def rnd(gen, *s):
    return torch.randn(s, device="cuda", generator=gen)


def separate(m, fl, io, hid, dY, dX, acc):
    """dH, grad slot of the MLP from the single-purpose kernels; dX filled."""
    L, s, M = S.glib(), S.stream(), io.M
    dH = torch.empty((M, 128), dtype=BF, device="cuda")
    part = torch.empty(64 * 3 * 128 * 128, device="cuda")
    bpart = torch.empty(64 * 128, device="cuda")
    grad = torch.zeros(m.end, device="cuda")
    g = lambda o: C.c_void_p(grad.data_ptr() + 4 * o)
    # W2 first: dY may be a dX target
    assert L.gnn_weight_grad(S.io(M, (hid, None)), None, S.ptr(dY), m.nout, m.NP, S.ptr(part), S.ptr(bpart), 64,
                             g(m.o_W2), g(m.o_b2), 0, s) == 0
    p = (C.c_void_p * 3)(*[None if d is None else d.data_ptr() for d in dX])
    assert L.gnn_mlp_backward(io, m.weights(fl), S.ptr(dY), S.ptr(hid), S.ptr(dH), p, acc, 0, s) == 0
    assert L.gnn_weight_grad(io, S.ptr(dH), None, 128, 128, S.ptr(part), S.ptr(bpart), 64, g(m.o_W1), g(m.o_b1),
                             0, s) == 0
    return dH, grad


def fused(m, fl, io, hid, dY, add, idx, dX, acc):
    L, s, M = S.glib(), S.stream(), io.M
    dH = torch.empty((M, 128), dtype=BF, device="cuda")
    dYb = torch.empty((M, m.NP), dtype=BF, device="cuda")
    work = torch.empty(S.GRAD_WORK_FLOATS, device="cuda")
    grad = torch.full((m.end,), 7.0, device="cuda")
    p = (C.c_void_p * 3)(*[None if d is None else d.data_ptr() for d in dX])
    assert L.gnn_mlp_grads(io, m.weights(fl), S.ptr(dY), S.ptr(add), S.ptr(idx), S.ptr(hid), p, acc, S.ptr(dH),
                           S.ptr(dYb), S.ptr(work), S.GRAD_WORK_FLOATS, S.ptr(grad), s) == 0
    return dH, dYb, grad


@pytest.mark.parametrize("M", [1, 15, 129, 4133, 70001])
@pytest.mark.parametrize("kind", ["node", "decoder", "encoder"])
def test_mlp_grads(gpu_lib, kind, M):
    gen = torch.Generator(device="cuda").manual_seed(M)
    K, nout = {"node": (256, 128), "decoder": (128, 3), "encoder": (32, 128)}[kind]
    m, fl, _ = make_mlp(K, nout, seed=M)
    xs = [rnd(gen, M, min(K, 128)).to(BF) for _ in range(2 if kind == "node" else 1)]
    hid = torch.relu(rnd(gen, M, 128)).to(BF)
    dY = rnd(gen, M, nout)
    io = S.io(M, *[(x, None) for x in xs])
    if kind == "node":  # the residual source accumulates into dY itself
        ya, yb = dY.clone(), dY.clone()
        da, db = torch.empty_like(dY), torch.empty_like(dY)
        dHa, ga = separate(m, fl, io, hid, ya, [ya, da, None], 1)
        dHb, dYb, gb = fused(m, fl, io, hid, yb, None, None, [yb, db, None], 1)
        assert torch.equal(ya, yb) and torch.equal(da, db)
    elif kind == "decoder":
        da, db = (torch.empty((M, 128), device="cuda") for _ in range(2))
        dHa, ga = separate(m, fl, io, hid, dY, [da, None, None], 0)
        dHb, dYb, gb = fused(m, fl, io, hid, dY, None, None, [db, None, None], 0)
        assert torch.equal(da, db)
    else:
        dHa, ga = separate(m, fl, io, hid, dY, [None] * 3, 0)
        dHb, dYb, gb = fused(m, fl, io, hid, dY, None, None, [None] * 3, 0)
    assert torch.equal(dHa, dHb)
    assert torch.equal(dYb[:, :nout], dY.to(BF)) and not dYb[:, nout:].any()
    for a, b in zip(m.views(ga), m.views(gb)):
        assert rel(b.cpu(), a.cpu()) < 2e-5


@pytest.mark.parametrize("N,last", [(1, False), (17, False), (300, True), (5003, False)])
def test_edge_grads(gpu_lib, N, last):
    """Edge MLP over gathered sources, rows of 0 to 40 edges: d_agg[recv] added
    to dY on the way in (alone, for the last layer), and the node sums."""
    rng = np.random.default_rng(N)
    gen = torch.Generator(device="cuda").manual_seed(N)
    deg = rng.integers(0, 14, size=N)
    deg[::7] = 0
    deg[N // 2] = 40
    row = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    E = int(row[-1])
    recv = torch.from_numpy(np.repeat(np.arange(N, dtype=np.int32), deg)).cuda()
    send = torch.from_numpy(rng.integers(0, N, size=E).astype(np.int32)).cuda()
    rev = torch.from_numpy(rng.permutation(E).astype(np.int32)).cuda()
    row_d = torch.from_numpy(row).cuda()
    m, fl, _ = make_mlp(384, 128, seed=N + 1)
    e, h = rnd(gen, E, 128).to(BF), rnd(gen, N, 128).to(BF)
    hid = torch.relu(rnd(gen, E, 128)).to(BF)
    d_agg, d_e = rnd(gen, N, 128), rnd(gen, E, 128)
    dh = rnd(gen, N, 128)
    if last:
        d_e.zero_()
    io = S.io(E, (e, None), (h, recv), (h, send))
    L, s = S.glib(), S.stream()
    ea, ha = d_e.clone(), dh.clone()
    hi, hj = torch.empty_like(d_e), torch.empty_like(d_e)
    assert L.gnn_broadcast_add(S.ptr(d_agg), S.ptr(recv), E, S.ptr(ea), s) == 0
    dHa, ga = separate(m, fl, io, hid, ea, [ea, hi, hj], 1)
    assert L.gnn_edge_grad_to_nodes(S.ptr(hi), S.ptr(hj), S.ptr(row_d), S.ptr(rev), N, S.ptr(ha), s) == 0
    eb, hb = d_e.clone(), dh.clone()
    if last:
        eb.fill_(7.0)  # not read: dY is null
    dHb, _, gb = fused(m, fl, io, hid, None if last else eb, d_agg, recv, [eb, None, None], 1)
    assert L.gnn_edge_hidden_grad_to_nodes(N, S.ptr(dHb), S.ptr(row_d), S.ptr(rev), m.weights(fl), S.ptr(hb),
                                           s) == 0
    assert torch.equal(dHa, dHb) and torch.equal(ea, eb) and torch.equal(ha, hb)
    for a, b in zip(m.views(ga), m.views(gb)):
        assert rel(b.cpu(), a.cpu()) < 2e-5


def test_mlp_grads_refuses_other_shapes(gpu_lib):
    m, fl, _ = make_mlp(256, 128, seed=1)
    M = 8
    x = torch.zeros((M, 256), dtype=BF, device="cuda")
    f = torch.zeros((M, 128), device="cuda")
    b = torch.zeros((M, 128), dtype=BF, device="cuda")
    work, grad = torch.empty(S.GRAD_WORK_FLOATS, device="cuda"), torch.empty(m.end + 4, device="cuda")
    none = (C.c_void_p * 3)()

    def call(io, dY=f, wf=S.GRAD_WORK_FLOATS, g=grad):
        return S.glib().gnn_mlp_grads(io, m.weights(fl), S.ptr(dY), None, None, S.ptr(b), none, 0, S.ptr(b),
                                      S.ptr(b), S.ptr(work), wf, S.ptr(g), S.stream())

    ok = S.io(M, (x[:, :128].contiguous(), None), (x[:, 128:].contiguous(), None))
    assert call(S.io(M, (x, None))) == -1           # one 256-wide source
    assert call(ok, dY=None) == -1
    assert call(ok, wf=100) == -1
    assert call(ok, g=grad[1:]) == -1               # not 16-byte aligned
