"""SwiGLU of the tiled gate/up over the whole range of the gate's pre-activation,
against float64, on each of its tiles.

A token's first feature is its pre-activation a and the w3 rows scale the second
to b, so a and b are exact.  h = silu(a) b carries, relative to |h|: the rounding
to 16 bits (2^-9 in bf16, 2^-12 in fp16, plus half its smallest subnormal) and
the fp32 exponential, sum, division and product.  The exponential's error is
that of a log2(e) rounded to fp32, at most |a| 2^-24 relative, plus one unit
(2^-23) of the instruction; the other three operations round once, 2^-24 each.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# e^-a overflows fp32 below this: silu is then -0
OVERFLOW = -88.72
# rows of the tile, experts, tile-list length, hidden, intermediate size
TILES = [(256, 2, 14, 256, 6144), (128, 8, 14, 64, 256), (64, 8, 52, 64, 256)]


def _gate_up(tile, experts, max_tiles, h, a, c, b, dtype):
    """(h, a, c per row): experts 0 and 1 hold every token, the others none."""
    from treemoe_spec_amd import _capi

    dev = torch.device("cuda")
    t, i = a.numel(), b.numel()
    rows = 2 * t
    taken = ctypes.c_int64()
    _capi.call("tm_op1_prefill_tiles", max_tiles, 1, t, h, i, experts, ctypes.byref(taken),
               ctypes.byref(ctypes.c_int64()))
    assert taken.value == tile
    x = torch.zeros(t, h)
    x[:, 0], x[:, 1] = a, c
    w1, w3 = torch.zeros(experts, i, h), torch.zeros(experts, i, h)
    w1[:, :, 0], w3[:, :, 1] = 1.0, b
    slots = torch.cat([torch.arange(0, rows, 2), torch.arange(1, rows, 2)]).to(torch.int32)
    offsets = torch.tensor([0, t] + [rows] * (experts - 1), dtype=torch.int32)
    tiles = [[e, e * t + r, min(64, t - r), 0] for e in range(2) for r in range(0, t, 64)]
    assert len(tiles) <= max_tiles
    tiles = torch.tensor(tiles + [[-1, 0, 0, 0]] * (max_tiles - len(tiles)), dtype=torch.int32)
    xd, w1d, w3d = (v.to(device=dev, dtype=dtype) for v in (x, w1, w3))
    sd, od, td = slots.to(dev), offsets.to(dev), tiles.to(dev)
    hd = torch.empty(rows, i, dtype=dtype, device=dev)
    _capi.call("tm_op1_prefill_gemm1", xd.data_ptr(), w1d.data_ptr(), w3d.data_ptr(),
               hd.data_ptr(), sd.data_ptr(), od.data_ptr(), td.data_ptr(), max_tiles, t, h, i,
               experts, _capi.TM_DTYPE_BF16 if dtype == torch.bfloat16 else _capi.TM_DTYPE_F16,
               _capi.stream_of(dev))
    token = slots.long() >> 1
    return hd.cpu(), x[token, 0].double()[:, None], x[token, 1].double()[:, None]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile,experts,max_tiles,hidden,inter", TILES)
def test_swiglu_range_matches_float64(tile, experts, max_tiles, hidden, inter, dtype):
    print(f"swiglu {tile} rows {dtype}", flush=True)
    a = torch.cat([torch.arange(-100.0, 100.25, 0.5), torch.zeros(1)])   # exact in 16 bits
    # b over the powers of two that the type holds
    powers = [-60, -10, 0, 8, 30, 60, 90, 120] if dtype == torch.bfloat16 else [-8, -4, -1, 0, 1, 4]
    b = torch.tensor([2.0 ** powers[n % len(powers)] for n in range(inter)])
    h, av, _ = _gate_up(tile, experts, max_tiles, hidden, a, torch.ones_like(a), b, dtype)
    out = h.double()
    ref = av * torch.sigmoid(av) * b.double()
    info = torch.finfo(dtype)
    assert ref.abs().max() < info.max
    half_ulp = info.eps / 2
    tol = (half_ulp + (av.abs() + 5.0) * 2.0 ** -24) * ref.abs() + info.smallest_normal * half_ulp
    tol = torch.where(av < OVERFLOW, ref.abs(), tol)
    bad = (out - ref).abs() > tol
    assert not bad.any(), (av.expand_as(ref)[bad][:4], out[bad][:4], ref[bad][:4])


@pytest.mark.parametrize("tile,experts,max_tiles,hidden,inter", TILES)
def test_fp16_h_is_rounded_once(tile, experts, max_tiles, hidden, inter):
    """fp16 h where silu(a) = a exactly (e^-a below half a unit of 1) and b is a product of two
    11-bit values: the 33-bit product a b rounded once to fp16, not to fp32 first."""
    print(f"fp16 rounding {tile} rows", flush=True)
    g = torch.Generator().manual_seed(5)
    a = (18.0 + 40.0 * torch.rand(402, generator=g)).half().float()
    c = (1.0 + torch.rand(402, generator=g)).half().float()
    b = (1.0 + torch.rand(inter, generator=g)).half().float()
    h, av, cv = _gate_up(tile, experts, max_tiles, hidden, a, c, b, torch.float16)
    exact = (av * cv * b.double()).numpy()
    once = torch.from_numpy(exact.astype("float16"))
    twice = torch.from_numpy(exact.astype("float32").astype("float16"))
    assert (once != twice).sum() >= 8      # the values that tell the two apart
    assert torch.equal(h, once), ((h != once).sum(), (h != twice).sum())
