"""The sampling walk's entry-to-thread map at its edges: vocabularies that end
inside a group of four, at a whole round of 1024 groups (4096 entries) and at
the register and tile limits, aligned and unaligned rows.  A root whose only
child is rejected or accepted by construction, then the exponential race: the
accepted path, the bonus and the residual against float64 torch."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 3, 4, 5, 4095, 4096, 4097, 8192, 8193, 16384, 16385, 32000,
                                   32767, 32768, 32769, 36865, 65536, 65537])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_walk_and_race_at_vocabulary_edges(vocab, dtype):
    from treemoe_spec_amd import _capi

    print(f"sampling edges V={vocab} {dtype}", flush=True)
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(vocab)
    code = _capi.TM_DTYPE_F32 if dtype == torch.float32 else _capi.TM_DTYPE_BF16
    for pad in (0, 1):                       # row stride: aligned, and one element more
        stride = (vocab + 7) // 8 * 8 + pad
        logits = torch.zeros(2, stride, dtype=dtype)
        logits[:, :vocab] = (torch.randn(2, vocab, generator=g) * 2).to(dtype)
        q = torch.zeros(2, stride)
        q[:, :vocab] = torch.softmax(torch.randn(2, vocab, generator=g), -1)
        e = torch.empty(vocab).exponential_(1.0, generator=g)
        for tok in sorted({0, vocab // 2, vocab - 1}):
            for accept in (False, True):
                p0 = torch.softmax(logits[0, :vocab].double(), -1)
                ratio = min(1.0, float(p0[tok] / max(float(q[1, tok]), 1e-20)))
                uni = torch.tensor([0.0, ratio * 0.5 if accept else 0.5 + ratio * 0.5])
                if not accept and ratio > 0.999:
                    continue                 # nothing rejects it
                if accept:
                    want = torch.softmax(logits[1, :vocab].double(), -1)
                else:
                    want = (p0 - q[1, :vocab].double()).clamp(min=0)
                    want = want / want.sum().clamp(min=1e-20)
                i32, i64 = torch.int32, torch.int64
                d = lambda t: t.to(dev)
                ld, qd, ud, ed = d(logits), d(q), d(uni), d(e)
                toks = d(torch.tensor([0, tok], dtype=i64))
                csr = d(torch.tensor([0, 1, 1, 0, 1], dtype=i32))
                res = torch.full((vocab + 8,), 7.0, device=dev)
                out = torch.full((2 + 2 + 3,), -9, dtype=i64, device=dev)
                _capi.call("tm_op4_sample_walk", ld.data_ptr(), code, 2, vocab, stride,
                           qd.data_ptr(), stride, toks.data_ptr(), csr.data_ptr(),
                           csr.data_ptr() + 8, csr.data_ptr() + 16, 1, ud.data_ptr(),
                           ed.data_ptr(), 1.0, res.data_ptr(), out.data_ptr(),
                           out.data_ptr() + 16, out.data_ptr() + 32, _capi.stream_of(dev))
                got, o = res.double().cpu(), out.cpu()
                assert torch.all(got[vocab:] == 7.0)
                assert o[0] == (1 if accept else -1) and o[5] == int(accept), (tok, accept)
                # fp32 softmax and one renormalisation: a few 2^-24 of a probability, and of
                # p and q where they cancel
                assert torch.all((got[:vocab] - want).abs() <= 2e-6 * (want + p0.max()) + 1e-9)
                race = want / e.double()
                top = race.max()
                bonus = int(o[4])
                assert 0 <= bonus < vocab and race[bonus] >= top * (1 - 1e-4) - 1e-9
