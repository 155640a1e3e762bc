"""CPU: the tile that the tiled GEMMs take.  The 256-row tile has half as many jobs as
the 128-row one, so a layer too narrow to fill the GPU with them takes the latter."""

from __future__ import annotations

import ctypes

import pytest


def tiles(t, h, i, e, split, budget=None):
    from treemoe_spec_amd import _capi
    from treemoe_spec_amd.kernels import op1_tree_moe as m

    gate_up, down = ctypes.c_int64(), ctypes.c_int64()
    max_tiles = m.compact_block_limit(2 * t, budget or e, m.TILE_M)
    _capi.call("tm_op1_prefill_tiles", max_tiles, split, t, h, i, e, ctypes.byref(gate_up),
               ctypes.byref(down))
    return gate_up.value, down.value


@pytest.mark.parametrize("t,h,i,e,split,want", [
    # wide layers: from 112 rows per expert on (T = 447 is below it)
    (447, 4096, 14336, 8, 2, (128, 128)),
    (517, 4096, 14336, 8, 2, (256, 256)),
    (2048, 4096, 14336, 8, 2, (256, 256)),
    (6011, 4096, 14336, 8, 2, (256, 256)),
    (4800, 2048, 1536, 64, 2, (256, 256)),
    # narrow ones: where the 128-row jobs fit one round over the CUs
    (700, 4096, 1792, 8, 2, (128, 256)),
    (1200, 4096, 1792, 8, 2, (256, 256)),
    (700, 512, 2048, 8, 4, (128, 128)),
    (700, 1024, 3584, 8, 4, (256, 128)),
    (3000, 512, 2048, 8, 2, (256, 256)),
    # few rows per expert, few jobs
    (64, 4096, 14336, 8, 2, (64, 128)),
    (64, 1024, 3584, 8, 4, (64, 64)),
])
def test_tile_follows_jobs(t, h, i, e, split, want):
    assert tiles(t, h, i, e, split) == want


def test_active_experts_come_from_the_tile_list():
    # two of eight experts hold all rows: 2 x 448 rows are 14 M-tiles of 128 at most 28 columns
    assert tiles(448, 1024, 3584, 8, 4, budget=2)[0] == 128
    assert tiles(448, 4096, 14336, 8, 2, budget=2)[0] == 256


def test_bad_sizes_are_refused():
    with pytest.raises(RuntimeError):
        tiles(64, 1024, 3584, 1, 2, budget=2)
    with pytest.raises(RuntimeError):
        tiles(64, 1024, 3584, 8, 0)
