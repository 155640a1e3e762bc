"""The tiled GEMMs at few tokens of a small hidden size (two tokens and more at
H <= 1024, I >= 3584): one token still streams, the routed and the two-phase
call agree bit for bit, and the layer meets the fp64 golden."""

from __future__ import annotations

import pytest
import torch

from oracle import op1_ref
from tests.test_gpu_op1 import REL_L2_TOL, _forward_and_golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,budget", [(1, 8), (2, 8), (2, 2), (17, 3), (65, 8)])
def test_small_hidden_layer(t, budget):
    from treemoe_spec_amd.kernels import op1_tree_moe as m

    print(f"small hidden t={t} B={budget}", flush=True)
    h, i = 1024, 3584
    assert m.uses_tiled_gemms(t, budget, 8, i, h) == (t >= 2)
    out, golden, inputs, _ = _forward_and_golden(t, 8, h, i, budget, 5 + t)
    assert op1_ref.rel_l2(out.cpu().float(), golden) <= REL_L2_TOL
    x, w1, w2, w3, router, accept = [a.cuda() for a in inputs]
    out = out.clone()
    routing = m.route_experts(x, router, accept, budget, i)
    again = m.tree_moe_forward(x, w1, w2, w3, router, accept, budget, routing=routing)
    assert torch.equal(out, again)
