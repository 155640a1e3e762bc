"""The 256-row tile of the tiled expert GEMMs at its edges: experts that end on
either side of every 64-row part, and step counts of every remainder modulo the
five operand buffers its K loop rotates through (and fewer steps than buffers).

Every product is compared with float64 torch on the same 16-bit operands.  A
GEMM sums K terms in fp32 (relative error at most K 2^-24 of the sum of the
magnitudes); h is then rounded to 16 bits (2^-9 relative in bf16), y is not.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

COUNTS = [1, 63, 64, 65, 128, 129, 192, 193, 255, 256, 257, 321]


def _layout(dev, g):
    offsets, tiles = [0], []
    for k, c in enumerate(COUNTS):
        tiles += [[k, offsets[k] + r0, min(64, c - r0), 0] for r0 in range(0, c, 64)]
        offsets.append(offsets[-1] + c)
    slots = torch.randperm(offsets[-1], generator=g).to(torch.int32)
    as_dev = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    return offsets, slots, as_dev(offsets), slots.to(dev), as_dev(tiles), len(tiles)


def _tiles(max_tiles, split, t, h, i, e):
    from treemoe_spec_amd import _capi

    out = (ctypes.c_int64 * 2)()
    _capi.call("tm_op1_prefill_tiles", max_tiles, split, t, h, i, e, ctypes.byref(out),
               ctypes.byref(out, 8))
    return tuple(out)


@pytest.mark.parametrize("steps", [4, 5, 6, 7, 8, 9])
def test_tile256_gemms_match_float64(steps):
    from treemoe_spec_amd import _capi

    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(steps)
    e, rows = len(COUNTS), sum(COUNTS)
    t, h, i = rows // 2, 64 * steps, 2048
    print(f"tile256 steps={steps}", flush=True)
    offsets, slots, off_d, slots_d, tiles_d, nt = _layout(dev, g)
    assert rows % 2 == 0 and _tiles(nt, 1, t, h, i, e)[0] == 256
    draw = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    x, w1, w3 = draw(t, h), draw(e, i, h) * 0.1, draw(e, i, h) * 0.1
    xd, w1d, w3d = x.to(dev), w1.to(dev), w3.to(dev)
    hd = torch.full((rows + 1, i), 7.0, dtype=torch.bfloat16, device=dev)
    st = _capi.stream_of(dev)
    _capi.call("tm_op1_prefill_gemm1", xd.data_ptr(), w1d.data_ptr(), w3d.data_ptr(),
               hd.data_ptr(), slots_d.data_ptr(), off_d.data_ptr(), tiles_d.data_ptr(), nt, t, h,
               i, e, _capi.TM_DTYPE_BF16, st)
    out = hd.double().cpu()
    assert torch.all(out[rows] == 7.0)
    for k in range(e):
        r = slice(offsets[k], offsets[k + 1])
        xf = x[slots[r].long() >> 1].double()
        a, b = xf @ w1[k].double().T, xf @ w3[k].double().T
        ref = a * torch.sigmoid(a) * b
        # one bf16 rounding, plus the fp32 sums' share where a and b cancel
        tol = 2.0 ** -8 * ref.abs() + 1e-5 * (1.0 + a.abs()) * (1.0 + b.abs())
        assert torch.all((out[r] - ref).abs() <= tol), (steps, COUNTS[k])

    # down: K = 64 * steps per segment, two segments
    ki, n = 128 * steps, 2048
    assert _tiles(nt, 2, t, n, ki, e)[1] == 256
    hm, w2 = draw(rows, ki), draw(e, n, ki) * 0.1
    gates = torch.rand(rows, generator=g)
    hmd, w2d, gd = hm.to(dev), w2.to(dev), gates.to(dev)
    y = torch.full((2, rows, n), 7.0, device=dev)
    _capi.call("tm_op1_prefill_gemm2", hmd.data_ptr(), w2d.data_ptr(), y.data_ptr(),
               gd.data_ptr(), slots_d.data_ptr(), off_d.data_ptr(), tiles_d.data_ptr(), nt, 2, t,
               n, ki, e, _capi.TM_DTYPE_BF16, st)
    out = y.double().cpu()
    half = ki // 2
    for k in range(e):
        r = slice(offsets[k], offsets[k + 1])
        for s in range(2):
            a, w = hm[r, s * half:(s + 1) * half].double(), w2[k, :, s * half:(s + 1) * half].double()
            gate = gates[slots[r].long()].double()[:, None]
            ref, mag = gate * (a @ w.T), gate * (a.abs() @ w.abs().T)
            tol = (half + 2) * 2.0 ** -24 * mag
            assert torch.all((out[s, r] - ref).abs() <= tol), (steps, COUNTS[k], s)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,masked,i", [
    ([0, 300, 0, 257, 1, 0, 512, 64, 0, 130, 0], (), 4096),    # empty first, last and between
    ([200, 300, 256, 257, 1, 255, 513, 64], (0, 2, 7), 3072),  # masked, as exclude_experts does
    ([0, 400, 401, 0, 399, 400], (2,), 3072),
])
def test_tile256_empty_and_masked_experts(counts, masked, i, dtype):
    """Empty experts have no M-tiles; a masked one keeps its tiles in the job order and leaves its
    rows of h and y alone."""
    from treemoe_spec_amd import _capi

    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(sum(counts))
    e, rows = len(counts), sum(counts)
    t, h, split = rows // 2, 256, 2
    offsets, tiles = [0], []
    for k, c in enumerate(counts):
        tiles += [[-1 if k in masked else k, offsets[k] + r0, min(64, c - r0), 0]
                  for r0 in range(0, c, 64)]
        offsets.append(offsets[-1] + c)
    nt = len(tiles)
    assert rows % 2 == 0 and _tiles(nt, 1, t, h, i, e)[0] == 256
    assert _tiles(nt, split, t, i, 2 * h, e)[1] == 256
    print(f"tile256 empty/masked {counts} {masked} {dtype}", flush=True)
    code = _capi.TM_DTYPE_BF16 if dtype == torch.bfloat16 else _capi.TM_DTYPE_F16
    half_ulp = torch.finfo(dtype).eps / 2
    as_dev = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    slots = torch.randperm(rows, generator=g).to(torch.int32)
    draw = lambda *s: torch.randn(*s, generator=g).to(dtype)
    x, w1, w3 = draw(t, h), draw(e, i, h) * 0.1, draw(e, i, h) * 0.1
    xd, w1d, w3d, sd, od, td = (x.to(dev), w1.to(dev), w3.to(dev), slots.to(dev),
                                as_dev(offsets), as_dev(tiles))
    hd = torch.full((rows, i), 7.0, dtype=dtype, device=dev)
    st = _capi.stream_of(dev)
    _capi.call("tm_op1_prefill_gemm1", xd.data_ptr(), w1d.data_ptr(), w3d.data_ptr(),
               hd.data_ptr(), sd.data_ptr(), od.data_ptr(), td.data_ptr(), nt, t, h, i, e, code, st)
    out = hd.double().cpu()
    # down: i output columns, two segments of K = 256
    hm, w2, gates = draw(rows, 2 * h), draw(e, i, 2 * h) * 0.1, torch.rand(rows, generator=g)
    hmd, w2d, gd = hm.to(dev), w2.to(dev), gates.to(dev)
    y = torch.full((split, rows, i), 7.0, device=dev)
    _capi.call("tm_op1_prefill_gemm2", hmd.data_ptr(), w2d.data_ptr(), y.data_ptr(),
               gd.data_ptr(), sd.data_ptr(), od.data_ptr(), td.data_ptr(), nt, split, t, i, 2 * h,
               e, code, st)
    yo = y.double().cpu()
    for k in range(e):
        r = slice(offsets[k], offsets[k + 1])
        if k in masked:
            assert torch.all(out[r] == 7.0) and torch.all(yo[:, r] == 7.0), k
            continue
        xf = x[slots[r].long() >> 1].double()
        a, b = xf @ w1[k].double().T, xf @ w3[k].double().T
        ref = a * torch.sigmoid(a) * b
        tol = 2 * half_ulp * ref.abs() + 1e-5 * (1.0 + a.abs()) * (1.0 + b.abs())
        assert torch.all((out[r] - ref).abs() <= tol), k
        for s in range(split):
            p, w = hm[r, s * h:(s + 1) * h].double(), w2[k, :, s * h:(s + 1) * h].double()
            gate = gates[slots[r].long()].double()[:, None]
            ref, mag = gate * (p @ w.T), gate * (p.abs() @ w.abs().T)
            assert torch.all((yo[s, r] - ref).abs() <= (h + 2) * 2.0 ** -24 * mag), (k, s)


@pytest.mark.parametrize("counts", [[16] * 8, [1, 15, 64, 65, 3, 0, 28, 0], [2, 2], [128, 0, 0, 0]])
def test_narrow_down_tile_matches_float64(counts):
    """Down with too few 128-row jobs for the chip (64-row tiles, 128 columns)."""
    from treemoe_spec_amd import _capi

    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(len(counts))
    e, rows = len(counts), sum(counts)
    t, n, ki = rows // 2, 1024, 768
    offsets, tiles = [0], []
    for k, c in enumerate(counts):
        tiles += [[k, offsets[k] + r0, min(64, c - r0), 0] for r0 in range(0, c, 64)]
        offsets.append(offsets[-1] + c)
    assert _tiles(len(tiles), 4, t, n, ki, e)[1] == 64
    print(f"narrow down {counts}", flush=True)
    draw = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    hm, w2, gates = draw(rows, ki), draw(e, n, ki) * 0.1, torch.rand(rows, generator=g)
    slots = torch.randperm(rows, generator=g).to(torch.int32)
    as_dev = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    hmd, w2d, gd, sd, od, td = (hm.to(dev), w2.to(dev), gates.to(dev), slots.to(dev),
                                as_dev(offsets), as_dev(tiles))
    y = torch.full((4, rows + 1, n), 7.0, device=dev)
    seg = ki // 4
    _capi.call("tm_op1_prefill_gemm2", hmd.data_ptr(), w2d.data_ptr(), y.data_ptr(),
               gd.data_ptr(), sd.data_ptr(), od.data_ptr(), td.data_ptr(), len(tiles), 4, t, n, ki,
               e, _capi.TM_DTYPE_BF16, _capi.stream_of(dev))
    out = y.double().cpu().reshape(-1)
    assert torch.all(out[4 * rows * n:] == 7.0)      # nothing past the [4, rows, n] partials
    out = out[:4 * rows * n].reshape(4, rows, n)
    for k, c in enumerate(counts):
        r = slice(offsets[k], offsets[k + 1])
        for s in range(4):
            a, w = (v[..., s * seg:(s + 1) * seg].double() for v in (hm[r], w2[k]))
            gate = gates[slots[r].long()].double()[:, None]
            ref, mag = gate * (a @ w.T), gate * (a.abs() @ w.abs().T)
            assert torch.all((out[s, r] - ref).abs() <= (seg + 2) * 2.0 ** -24 * mag), (k, s)
