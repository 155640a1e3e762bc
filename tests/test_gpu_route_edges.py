"""Routing at the token counts where its launches change: one fused launch up to
16 logits, one token per lane up to 64 tokens and 8 experts, one workgroup, and
from 1024 tokens several launches (whose workgroups take 512 tokens).  Every
output is bit-exact against the C oracle; buffers are poisoned first, so an
entry that no launch writes shows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle_c
from tests.conftest import bf16_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,e", [
    (1, 8), (2, 8), (3, 8), (8, 2), (9, 2), (4, 5), (3, 5), (1, 16), (63, 8), (64, 8), (64, 3),
    (65, 8), (64, 16), (1023, 8), (1024, 8), (1025, 6), (1536, 8), (1537, 16), (4097, 64)])
@pytest.mark.parametrize("objective", ["mass", "critical_path"])
def test_routing_bit_exact_at_launch_edges(t, e, objective):
    from treemoe_spec_amd import _capi
    from treemoe_spec_amd.kernels import op1_tree_moe as m

    h = 512
    g = torch.Generator().manual_seed(31 * t + e)
    x = torch.randn(t, h, generator=g).to(torch.bfloat16)
    router = (torch.randn(e, h, generator=g) * 0.1).to(torch.bfloat16)
    router[e - 1] = router[0]              # exact ties go to the lower expert
    accept = torch.rand(t, generator=g)
    accept[::5] = 0.01                     # below tau: the second pick is dropped
    gates = oracle_c.router_gates(bf16_bits(x), bf16_bits(router))
    xd, rd, ad = x.cuda(), router.cuda(), accept.cuda()
    for budget in sorted({2, (e + 2) // 2, e}):
        for bm in (16, 32):
            print(f"route edges t={t} E={e} B={budget} BM={bm} {objective}", flush=True)
            mb = m.compact_block_capacity(2 * t, budget, bm)
            mt = m.compact_block_limit(2 * t, budget, 64)
            ref = oracle_c.route_bucket(gates, accept.numpy(), budget, objective=objective,
                                        block_m=bm)
            i32, i64, f32 = torch.int32, torch.int64, torch.float32
            o = [torch.full((n,), -77, dtype=d, device="cuda") for n, d in (
                (t * e, f32), (2 * t, i64), (2 * t, f32), (mb * bm, i64), (mb, i64), (2 * t, i64),
                (e, f32), (e + 1, i32), (2 * t, i32), (2 * t, i32), (4 * mt, i32))]
            _capi.call("tm_op1_route", xd.data_ptr(), rd.data_ptr(), ad.data_ptr(), t, h, e,
                       budget, 0.05, _capi.TM_OBJECTIVE[objective], bm, mb, mt,
                       *[v.data_ptr() for v in o], _capi.TM_DTYPE_BF16, _capi.stream_of(0))
            got = [v.cpu().numpy() for v in o]
            want = [np.asarray(gates, dtype=np.float32).reshape(-1), ref.topk_ids, ref.gates_flat,
                    ref.padded_slots, ref.block_expert_ids, ref.slot_to_row, ref.demand,
                    ref.expert_offsets, ref.sorted_slots, ref.slot_pos, ref.tiles]
            for k, (a, b) in enumerate(zip(got, want)):
                b = np.ascontiguousarray(b).reshape(-1)
                assert a.shape == b.shape and a.dtype.itemsize == b.dtype.itemsize, k
                assert np.array_equal(a.view(f"u{a.dtype.itemsize}"),
                                      b.view(f"u{b.dtype.itemsize}")), (k, budget, bm)
