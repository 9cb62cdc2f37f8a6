"""Parameter gradients of gnn_mlp_grads over more rows than 64 chunks of 32 steps
hold evenly: gnn_weight_grad's bit for bit, as at smaller sizes."""
from __future__ import annotations

import pytest

from test_gpu_gnn_grad_order import test_same_bits as same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["node", "edge", "decoder", "encoder"])
@pytest.mark.parametrize("M", [65537, 70001])
def test_same_bits_many_rows(gpu_lib, kind, M):
    same_bits(gpu_lib, kind, M)
