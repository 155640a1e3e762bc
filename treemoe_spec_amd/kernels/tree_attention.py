"""Tree attention of the verification forward on the paged KV cache.

Drop-in for the tree branch of the reference's ``MixtralForward._attention``
(treemoe/model/mixtral.py:208-250), which runs

    kv.write_tree(layer, k, v)                         # kv_cache.py:80-86
    full_k, full_v = kv.gather_with_tail(layer, k, v)  # kv_cache.py:125-145
    mask = [ones(N, seq_len) | tree_mask]              # mixtral.py:211-218
    o = F.scaled_dot_product_attention(q, full_k, full_v, mask,
                                       scale=hd**-0.5, enable_gqa=True)

as one HIP launch (plus a chunk combine at long contexts): the prefix is read
in place through the block table, the tree rows come from ``k``/``v`` and are
stored into the scratch pages by the same kernel.  The context comes back as
[N, Hq * hd], the layout ``o_proj`` takes (mixtral.py:251-254).
"""

from __future__ import annotations

import ctypes
import operator
import threading
import weakref

import torch

from treemoe_spec_amd import _capi
from treemoe_spec_amd._capi import call, check, ptr
from treemoe_spec_amd.kv_cache import device_tables_of, scratch_pages_of

# Called once per layer of every forward: the C ABI goes through the CPython
# binding where it is built, and a layer's cache is addressed by its offset
# instead of through a tensor view.  Host time of a call 14-17 -> 8 us, which
# is what bounded the short contexts (27 nodes over 333 positions: 10.5 us on
# the device).
_fast = _capi.fast_binding()

_mask_cache: dict = {}
_CACHE_ENTRIES = 16


def _capture_id(stream: int) -> int:
    """0, or the identity of the graph capture under way on a raw stream (the
    default stream, 0, cannot be captured)."""
    if stream == 0:
        return 0
    if _fast is not None:
        rc, cid = _fast.stream_capture_id(stream)
        check(rc, "tm_stream_capture_id")
        return cid
    out = ctypes.c_uint64()
    call("tm_stream_capture_id", stream, ctypes.byref(out))
    return out.value


def pack_tree_mask(tree_mask: torch.Tensor) -> torch.Tensor:
    """[N, N] bool device mask -> [N, ceil(N/64)] int64 bit words (bit j of row
    i = tree_mask[i, j]), packed on the current stream of the mask's device.
    Kept per live mask tensor and its version counter, since the engine reuses
    one mask for every layer of a step."""
    stream = _capi.stream_of(tree_mask.device)
    return _packed_mask(tree_mask, stream, _capture_id(stream))


def _packed_mask(tree_mask: torch.Tensor, stream: int, capture: int) -> torch.Tensor:
    """pack_tree_mask for a raw stream and the capture under way on it.  The
    words are used on the stream that packed them only, which orders both, and
    inside a capture only where that capture packed them: words from before it
    could be freed or become stale under the graph, and words packed inside it
    hold nothing until a replay."""
    key = (id(tree_mask), stream, capture)
    hit = _mask_cache.get(key)
    if hit is not None and hit[0]() is tree_mask and hit[1] == tree_mask._version:
        return hit[2]
    n = tree_mask.shape[0]
    if tree_mask.dim() != 2 or tree_mask.shape[1] != n or tree_mask.stride(1) != 1:
        raise ValueError("tree_mask must be [N, N] with unit stride along columns")
    m = tree_mask if tree_mask.dtype in (torch.bool, torch.uint8) else tree_mask.bool()
    bits = torch.empty(n, (n + 63) // 64, dtype=torch.int64, device=tree_mask.device)
    call("tm_tree_mask_pack", ptr(m), n, m.stride(0), ptr(bits), stream)
    if len(_mask_cache) > _CACHE_ENTRIES:
        _mask_cache.clear()
    _mask_cache[key] = (weakref.ref(tree_mask), tree_mask._version, bits)
    return bits


def tree_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, kv, layer: int,
                   tree_mask: torch.Tensor, scale: float | None = None,
                   out: torch.Tensor | None = None, write_tree: bool = True,
                   chunk_keys: int = 0) -> torch.Tensor:
    """q [N, Hq, hd] (after RoPE), k/v [N, kvh, hd] (k after RoPE) for the tree
    nodes; ``kv`` a paged cache with ``seq_len`` committed positions.  Returns
    the attention context [N, Hq * hd] bf16.  ``write_tree`` also stores k/v
    in the scratch pages, as the reference's write_tree does."""
    if not q.is_cuda:
        raise RuntimeError("treemoe_spec_amd tree attention runs on ROCm devices only; "
                           "got a CPU tensor")
    n, hq, hd = q.shape
    kshape = k.shape
    if kshape[0] != n or v.shape != kshape or len(kshape) != 3:
        raise ValueError("k and v must be [N, kv_heads, head_dim] like q's N")
    kvh = kshape[1]
    if hq % kvh != 0:
        raise ValueError("num_heads must be a multiple of num_kv_heads")
    qs, ks, vs = q.stride(), k.stride(), v.stride()
    for name, t, st in (("q", q, qs), ("k", k, ks), ("v", v, vs)):
        if t.dtype != torch.bfloat16:
            raise ValueError(f"{name} must be bfloat16")
        if st[2] != 1 or st[1] != hd:
            raise ValueError(f"{name} must have contiguous heads")
    if ks[0] != vs[0]:
        raise ValueError("k and v must share the node stride")
    kc, vc = kv.k, kv.v
    cshape = kc.shape
    if kc.dtype != torch.bfloat16 or cshape[3] != kvh or cshape[4] != hd:
        raise ValueError("cache layout must be [L, pages, page, kv_heads, head_dim] bf16")
    layer = operator.index(layer)
    layers, vlayers = cshape[0], vc.shape[0]  # refused where indexing either refuses it
    if not (-layers <= layer < layers and -vlayers <= layer < vlayers):
        raise IndexError(f"layer {layer} is out of range for a cache of "
                         f"{min(layers, vlayers)} layers")
    if tuple(tree_mask.shape) != (n, n):
        raise ValueError("tree_mask must be [N, N]")
    dev = q.device
    if scale is None:
        scale = hd ** -0.5
    stream = _capi.stream_of(dev)
    capture = _capture_id(stream) if stream else 0
    bits = _packed_mask(tree_mask, stream, capture)
    pages = scratch_pages_of(kv)
    page = kv.block_size
    if write_tree and len(pages) * page < n:
        raise ValueError("tree larger than the KV scratch pages")
    table, scratch = device_tables_of(kv, dev)
    seq_len = kv.seq_len
    if _fast is not None:
        rc, nbytes = _fast.attn_workspace(n, hq, kvh, hd, seq_len, page, chunk_keys)
        check(rc, "tm_tree_attention_plan")
    else:
        chunks = ctypes.c_int64()
        wbytes = ctypes.c_int64()
        call("tm_tree_attention_plan", n, hq, kvh, hd, seq_len, page, chunk_keys,
             ctypes.byref(chunks), ctypes.byref(wbytes))
        nbytes = wbytes.value
    ws = _workspace(nbytes, dev, stream, capture)
    if out is None:
        out = torch.empty(n, hq * hd, dtype=torch.bfloat16, device=dev)
    elif out.shape != (n, hq * hd) or out.dtype != torch.bfloat16 or not out.is_contiguous():
        raise ValueError("out must be a contiguous [N, Hq * hd] bf16 tensor")
    cs, vcs = kc.stride(), vc.stride()
    args = (q.data_ptr(), qs[0], k.data_ptr(), v.data_ptr(), ks[0],
            kc.data_ptr() + 2 * cs[0] * (layer % layers),
            vc.data_ptr() + 2 * vcs[0] * (layer % vlayers), cs[1], cs[2],
            page, table.data_ptr(), max(1, len(kv.block_table)), seq_len, scratch.data_ptr(),
            len(pages), 1 if write_tree else 0, bits.data_ptr(), n, hq, kvh, hd, float(scale),
            out.data_ptr(), hq * hd, chunk_keys, 0 if ws is None else ws.data_ptr(), nbytes,
            stream)
    if _fast is not None:
        check(_fast.tree_attention(*args), "tm_tree_attention")
    else:
        call("tm_tree_attention", *args)
    return out


_ws_cache: dict = {}


def _workspace(nbytes: int, device, stream: int, capture: int) -> torch.Tensor | None:
    """Chunk partials, written by a call's first launch and read by its second.
    One buffer per (device, stream, calling thread), grown on demand: calls of
    one thread on one stream reuse it in stream order, while calls of other
    streams or threads may come between the two launches.  Under a graph capture
    the buffer comes from the graph's pool and is not kept, so that no later
    call can free or overwrite what the replays use."""
    if nbytes == 0:
        return None
    if capture:
        return torch.empty(nbytes, dtype=torch.uint8, device=device)
    key = (device, stream, threading.get_ident())
    buf = _ws_cache.get(key)
    if buf is None or buf.numel() < nbytes:
        if buf is None and len(_ws_cache) >= _CACHE_ENTRIES:
            _ws_cache.clear()
        buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
        _ws_cache[key] = buf
    return buf
