"""CPU: the chunk counts that the tree-attention planner picks."""

from __future__ import annotations

import ctypes

import pytest


@pytest.mark.parametrize("n,hq,kvh,seq_len,chunks", [
    (64, 32, 8, 4096, 14),
    (1, 32, 8, 7777, 32),
    (27, 32, 8, 333, 7),
    (60, 32, 8, 5860, 32),
    # three row blocks: nine chunks of five stages, not 21 of two on shared CUs
    (72, 32, 8, 2500, 9),
    (90, 32, 8, 2500, 9),
    (90, 32, 8, 4096, 17),
])
def test_chunks(n, hq, kvh, seq_len, chunks):
    from treemoe_spec_amd import _capi

    got, nbytes = ctypes.c_int64(), ctypes.c_int64()
    _capi.call("tm_tree_attention_plan", n, hq, kvh, 128, seq_len, 16, 0, ctypes.byref(got),
               ctypes.byref(nbytes))
    assert got.value == chunks
