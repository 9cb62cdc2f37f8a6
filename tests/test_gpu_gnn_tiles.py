"""A layer's forward over the first rows of a graph equals the same rows of the
whole graph bit for bit: how tiles are dealt to blocks and waves, and the node
pass's two shapes (up to eight tiles a CU, and more), change no value."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from cabanadem_amd import surrogate as S
from test_gpu_gnn import make_mlp
from test_gpu_gnn_grads import BF, rnd

pytestmark = pytest.mark.gpu

N_ALL = 33500  # 2,094 tiles: more than eight for each of 256 CUs


@pytest.fixture(scope="module")
def graph(gpu_lib):
    rng = np.random.default_rng(1)
    deg = rng.integers(0, 12, size=N_ALL)
    row = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    E = int(row[-1])
    gen = torch.Generator(device="cuda").manual_seed(1)
    g = dict(row_h=row, E=E, row=torch.from_numpy(row).cuda(),
             recv=torch.from_numpy(np.repeat(np.arange(N_ALL, dtype=np.int32), deg)).cuda(),
             send=torch.from_numpy(rng.integers(0, N_ALL, size=E).astype(np.int32)).cuda(),
             h=rnd(gen, N_ALL, 128).to(BF), e=rnd(gen, E, 128).to(BF), P=rnd(gen, N_ALL, 128))
    g["edge"], g["node"] = make_mlp(384, 128, seed=2), make_mlp(256, 128, seed=3)
    return g


def forward(g, n, from_p):
    L, s, E = S.glib(), S.stream(), int(g["row_h"][n])
    m, fl, _ = g["edge"]
    k, fk, _ = g["node"]
    new = lambda r: torch.empty((max(r, 1), 128), dtype=BF, device="cuda")
    eh, eo, agg, nh, ho = new(E), new(E), new(n), new(n), new(n)
    p = S.ptr
    assert L.gnn_edge_mlp_forward(E, p(g["e"]), p(g["recv"]), p(g["send"]), p(g["P"]) if from_p else None,
                                  p(g["h"]), m.weights(fl), p(eh), p(eo), 0, s) == 0
    assert L.gnn_node_layer_forward(n, p(g["h"]), p(eo), p(g["row"]), k.weights(fk), p(agg), p(nh), p(ho), None,
                                    None, s) == 0
    return [t[:r] for t, r in ((eh, E), (eo, E), (agg, n), (nh, n), (ho, n))]


@pytest.mark.parametrize("from_p", [False, True])
@pytest.mark.parametrize("n", [1, 17, 700, 4097, 9240, 32768, 32769])
def test_prefix(graph, n, from_p):
    whole = forward(graph, N_ALL, from_p)
    for a, b in zip(whole, forward(graph, n, from_p)):
        assert torch.equal(a[:b.shape[0]], b)
