"""Tree attention captured in a HIP graph, and on two streams: later eager calls
with longer contexts and other masks neither free nor overwrite what a graph's
replays read, a replay packs the mask as it then is, and two streams do not
share chunk partials."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_attn import _case, _check, _oracle

pytestmark = pytest.mark.gpu


def _capture(fn):
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _on_gpu(n, seq_len, seed, hq=32, kvh=8):
    kv, q, k, v, mask = _case(n, hq, kvh, seq_len, 16, seed)
    return kv, q.cuda(), k.cuda(), v.cuda(), mask.cuda()


def test_replays_after_longer_contexts_and_many_masks():
    from treemoe_spec_amd.kernels.tree_attention import tree_attention

    print("attention capture, longer contexts and many masks", flush=True)
    kv, q, k, v, mask = _on_gpu(27, 700, 1)
    att = lambda: tree_attention(q, k, v, kv, 0, mask, chunk_keys=64)
    want = att().clone()
    graph, out = _capture(att)
    for r in range(3):
        # more masks than are kept, and a longer context than any before
        for j in range(20):
            m = mask.clone()
            tree_attention(q, k, v, kv, 0, m, chunk_keys=64)
        lkv, lq, lk, lv, lmask = _on_gpu(64, 2000 * (r + 1), 2 + r)
        tree_attention(lq, lk, lv, lkv, 0, lmask, chunk_keys=64)
        # whatever was freed is taken and filled
        junk = [torch.full((1 << s,), 0x7f, dtype=torch.uint8, device="cuda")
                for s in range(9, 24) for _ in range(3)]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), r
        assert all(bool((j == 0x7f).all()) for j in junk), r
        assert torch.equal(att(), want), r


def test_mask_first_packed_in_a_capture_and_changed_in_place():
    from treemoe_spec_amd.kernels.tree_attention import tree_attention

    print("attention capture, mask packed inside", flush=True)
    kv, q, k, v, mask = _on_gpu(40, 300, 5)
    other = torch.eye(40, dtype=torch.bool, device="cuda")
    att = lambda m: tree_attention(q, k, v, kv, 0, m)
    want, want_other = att(mask.clone()).clone(), att(other).clone()
    assert not torch.equal(want, want_other)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = att(mask)
    # the capture recorded the pack and did not run it: eager calls pack their own
    with torch.cuda.stream(s):
        assert torch.equal(att(mask), want)
    assert torch.equal(att(mask), want)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    mask.copy_(other)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want_other)
    assert torch.equal(att(mask), want_other)


def test_two_streams_have_their_own_partials():
    from treemoe_spec_amd.kernels.tree_attention import tree_attention

    print("attention on two streams", flush=True)
    cases = [_on_gpu(33, 1500, 11), _on_gpu(33, 1500, 12)]
    want = []
    for kv, q, k, v, mask in cases:
        want.append(tree_attention(q, k, v, kv, 0, mask, chunk_keys=64).clone())
    _check(want[0], _oracle(cases[0][0], *(t.cpu() for t in cases[0][1:]), 0))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in cases]
    got = [[], []]
    for _ in range(40):
        for j, (kv, q, k, v, mask) in enumerate(cases):
            with torch.cuda.stream(streams[j]):
                got[j].append(tree_attention(q, k, v, kv, 0, mask, chunk_keys=64))
    torch.cuda.synchronize()
    for j in range(2):
        assert all(torch.equal(o, want[j]) for o in got[j]), j


def test_two_threads_on_one_stream():
    """A call's two launches may have another thread's between them."""
    import threading

    from treemoe_spec_amd.kernels.tree_attention import tree_attention

    print("attention from two threads", flush=True)
    cases = [_on_gpu(33, 1500, 21), _on_gpu(33, 1500, 22)]
    want = [tree_attention(q, k, v, kv, 0, mask, chunk_keys=64).clone()
            for kv, q, k, v, mask in cases]
    torch.cuda.synchronize()
    got = [[], []]

    def work(j):
        kv, q, k, v, mask = cases[j]
        for _ in range(60):
            got[j].append(tree_attention(q, k, v, kv, 0, mask, chunk_keys=64))

    threads = [threading.Thread(target=work, args=(j,)) for j in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for j in range(2):
        assert len(got[j]) == 60 and all(torch.equal(o, want[j]) for o in got[j]), j
