"""Tree attention where only some of a workgroup's four 32-row waves hold query
rows, over chunk counts on both sides of what the four combining waves take in
one trip: against the float32 oracle, at the bound of the other attention tests
(bf16 probabilities and output, 2^-8 relative each, fp16 partials)."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_attn import _case, _check, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,hq,kvh", [(1, 32, 8), (8, 32, 8), (9, 32, 8), (24, 32, 8),
                                      (25, 32, 8), (33, 32, 8), (40, 4, 4)])
def test_partial_waves_and_chunk_counts(n, hq, kvh):
    from treemoe_spec_amd.kernels.tree_attention import tree_attention

    # chunks of 64: none, 1 + 1, 2 + 1, 3 + 1, 4 + 1, 17 + 1
    for seq_len in (0, 64, 128, 190, 256, 1030):
        print(f"attention edges n={n} seq={seq_len}", flush=True)
        kv, q, k, v, mask = _case(n, hq, kvh, seq_len, 16, 7 * n + seq_len)
        qc, kc, vc, mc = q.cuda(), k.cuda(), v.cuda(), mask.cuda()
        want = _oracle(kv, q, k, v, mask, 1)
        _check(tree_attention(qc, kc, vc, kv, 1, mc, chunk_keys=64), want)
        _check(tree_attention(qc, kc, vc, kv, -1, mc), want)


def test_layer_out_of_range_is_refused():
    from treemoe_spec_amd.kernels.tree_attention import tree_attention

    kv, q, k, v, mask = _case(4, 8, 2, 20, 16, 3)
    with pytest.raises(IndexError):
        tree_attention(q.cuda(), k.cuda(), v.cuda(), kv, 2, mask.cuda())


@pytest.mark.parametrize("n,hq,kvh", [(72, 32, 8), (73, 32, 8), (80, 32, 8), (81, 32, 8),
                                      (97, 32, 32), (33, 64, 64)])
def test_combine_with_many_units(n, hq, kvh):
    """On both sides of the unit count (KV heads x 32-row groups x 16) from which one wave merges
    a unit's chunks; the last row group partly empty."""
    from treemoe_spec_amd.kernels.tree_attention import tree_attention

    for seq_len in (64, 190, 1030):
        print(f"attention combine n={n} hq={hq} kvh={kvh} seq={seq_len}", flush=True)
        kv, q, k, v, mask = _case(n, hq, kvh, seq_len, 16, 5 * n + seq_len)
        want = _oracle(kv, q, k, v, mask, 1)
        _check(tree_attention(q.cuda(), k.cuda(), v.cuda(), kv, 1, mask.cuda(), chunk_keys=64),
               want)
