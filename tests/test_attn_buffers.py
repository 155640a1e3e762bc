"""CPU: which device buffers tree attention keeps between calls.  The packed mask
words and the chunk partials belong to one stream (the partials to one thread
too), and a graph capture gets its own."""

from __future__ import annotations

import threading

import pytest
import torch

from treemoe_spec_amd.kernels import tree_attention as ta

CPU = torch.device("cpu")


@pytest.fixture()
def packs(monkeypatch):
    """The (stream, capture) under which masks are packed, and the packs done."""
    state = {"stream": 0, "capture": 0, "done": []}
    monkeypatch.setattr(ta, "_mask_cache", {})
    monkeypatch.setattr(ta, "call", lambda name, *a: state["done"].append((name, a[-1])))
    monkeypatch.setattr(ta._capi, "stream_of", lambda dev: state["stream"])
    monkeypatch.setattr(ta, "_capture_id", lambda stream: state["capture"], raising=False)
    return state


def test_mask_words_are_packed_per_stream_and_capture(packs):
    mask = torch.eye(3, dtype=torch.bool)
    first = ta.pack_tree_mask(mask)
    assert ta.pack_tree_mask(mask) is first and len(packs["done"]) == 1
    packs["stream"] = 7
    second = ta.pack_tree_mask(mask)
    assert second is not first and packs["done"][-1] == ("tm_tree_mask_pack", 7)
    # inside a capture: packed again by the capture, once for all its layers
    packs["capture"] = 1
    captured = ta.pack_tree_mask(mask)
    assert captured is not second and len(packs["done"]) == 3
    assert ta.pack_tree_mask(mask) is captured and len(packs["done"]) == 3
    packs["capture"] = 2
    assert ta.pack_tree_mask(mask) is not captured
    # and eager calls go on with their own
    packs["capture"] = 0
    assert ta.pack_tree_mask(mask) is second and len(packs["done"]) == 4
    mask[2, 0] = True
    assert ta.pack_tree_mask(mask) is not second


def test_workspace_belongs_to_a_stream_and_a_thread(monkeypatch):
    monkeypatch.setattr(ta, "_ws_cache", {})
    a = ta._workspace(100, CPU, 1, 0)
    assert ta._workspace(60, CPU, 1, 0) is a          # reused in stream order
    assert ta._workspace(100, CPU, 2, 0) is not a
    other = []
    t = threading.Thread(target=lambda: other.append(ta._workspace(100, CPU, 1, 0)))
    t.start()
    t.join()
    assert other[0] is not a
    assert ta._workspace(200, CPU, 1, 0).numel() == 200      # grown
    assert ta._workspace(0, CPU, 1, 0) is None


def test_workspace_of_a_capture_is_not_kept(monkeypatch):
    monkeypatch.setattr(ta, "_ws_cache", {})
    kept = ta._workspace(100, CPU, 1, 0)
    inside = ta._workspace(100, CPU, 1, 5)
    assert inside is not kept and ta._workspace(100, CPU, 1, 5) is not inside
    assert ta._workspace(100, CPU, 1, 0) is kept


def test_kept_workspaces_are_bounded(monkeypatch):
    monkeypatch.setattr(ta, "_ws_cache", {})
    for stream in range(1, 200):
        ta._workspace(16, CPU, stream, 0)
    assert len(ta._ws_cache) <= 32


@pytest.mark.parametrize("foreign", [False, True])
def test_block_table_keeps_its_device_buffer_as_the_sequence_grows(foreign):
    """A captured graph holds the table's address: growing the sequence must fill the same
    buffer, not put a new one in its place."""
    from tests.ref_layout_cache import RefLayoutKVCache
    from treemoe_spec_amd.kv_cache import MixtralConfig, PagedKVCache, device_tables_of

    if foreign:
        kv, page = RefLayoutKVCache(1, 2, 8, 12, device="cpu"), 64
    else:
        cfg = MixtralConfig(num_layers=1, num_kv_heads=2, head_dim=8, num_heads=2)
        kv, page = PagedKVCache(cfg, 12, device="cpu", page_size=16, tree_size=8), 16
    empty, scratch = device_tables_of(kv, "cpu")
    address = empty.data_ptr()
    for pages in (1, 3, 10):
        kv._ensure_capacity(pages * page)
        table, pages_again = device_tables_of(kv, "cpu")
        assert table.tolist() == kv.block_table and table.data_ptr() == address
        assert pages_again is scratch
    # another mapping of the same length
    kv.block_table.reverse()
    if not foreign:
        kv._dev_table_len = -1
    assert device_tables_of(kv, "cpu")[0].tolist() == kv.block_table


class _OnGpu(torch.Tensor):
    """A CPU tensor that says it is on the GPU, to reach the launch arguments."""

    is_cuda = property(lambda self: True)


def test_layer_is_looked_up_in_both_caches(monkeypatch):
    """K and V are addressed by their own layer counts: a V cache with fewer layers than K's is
    refused where it ends, as indexing it is."""
    from treemoe_spec_amd.kv_cache import MixtralConfig, PagedKVCache

    cfg = MixtralConfig(num_layers=3, num_kv_heads=2, head_dim=128, num_heads=4)
    kv = PagedKVCache(cfg, 4, device="cpu", page_size=16, tree_size=8)
    kv._ensure_capacity(16)
    kv.seq_len = 16
    seen = {}
    monkeypatch.setattr(ta, "_mask_cache", {})
    monkeypatch.setattr(ta, "_fast", None)
    monkeypatch.setattr(ta, "call", lambda name, *a: seen.update({name: a}))
    monkeypatch.setattr(ta._capi, "stream_of", lambda dev: 0)
    q = torch.zeros(4, 4, 128, dtype=torch.bfloat16).as_subclass(_OnGpu)
    k = torch.zeros(4, 2, 128, dtype=torch.bfloat16)
    att = lambda layer: ta.tree_attention(q, k, k, kv, layer, torch.eye(4, dtype=torch.bool))
    for layer in (0, 2, -1, -3):
        att(layer)
        assert seen["tm_tree_attention"][5:7] == (kv.k[layer].data_ptr(), kv.v[layer].data_ptr())
    for layer in (3, -4):
        with pytest.raises(IndexError):
            att(layer)
    kv.v = kv.v[:2]
    att(1)
    assert seen["tm_tree_attention"][6] == kv.v[1].data_ptr()
    for layer in (2, -3):
        with pytest.raises(IndexError):
            att(layer)
