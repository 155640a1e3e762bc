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


@pytest.mark.parametrize("vocab", [4, 5, 4095, 4096, 4097, 32767, 32768, 32769, 65537])
def test_second_child_meets_the_updated_residual(vocab):
    """The first child is rejected, so the second, at either end of the vocabulary or a group
    of four, is tested against max(p - q_1, 0) renormalised: accepted just below its ratio there,
    and rejected above it, which updates the residual once more."""
    from treemoe_spec_amd import _capi

    print(f"sampling second child V={vocab}", flush=True)
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(vocab)
    stride = (vocab + 3) // 4 * 4
    logits = torch.zeros(3, stride)
    logits[:, :vocab] = torch.randn(3, vocab, generator=g) * 2
    e = torch.empty(vocab).exponential_(1.0, generator=g)
    p0 = torch.softmax(logits[0, :vocab].double(), -1)
    d = lambda t: t.to(dev)
    for tok1 in sorted({0, vocab - 1}):
        for tok2 in sorted({0, 3, vocab // 2, vocab - 1, min(4096, vocab - 1)}):
            for accept in (False, True):
                # the draft overrates a token that is to be rejected
                raw = torch.randn(3, vocab, generator=g)
                q = torch.zeros(3, stride)
                raw[1, tok1] = torch.logsumexp(raw[1], 0) + 0.5
                if not accept:
                    raw[2, tok2] = torch.logsumexp(raw[2], 0) + 0.5
                q[:, :vocab] = torch.softmax(raw, -1)
                q1, q2 = q[1, :vocab].double(), q[2, :vocab].double()
                r1 = (p0 - q1).clamp(min=0)
                r1 = r1 / r1.sum().clamp(min=1e-20)
                first = min(1.0, float(p0[tok1] / q1[tok1]))
                second = min(1.0, float(r1[tok2] / q2[tok2]))
                if first > 0.95 or (second < 1e-3 if accept else second > 0.95):
                    continue
                if accept:
                    want = torch.softmax(logits[2, :vocab].double(), -1)
                else:
                    want = (r1 - q2).clamp(min=0)
                    want = want / want.sum().clamp(min=1e-20)
                uni = torch.tensor([0.0, 0.5 + 0.5 * first,
                                    0.98 * second if accept else 0.05 + 0.95 * second])
                i32, i64 = torch.int32, torch.int64
                ld, qd, ud, ed = d(logits), d(q), d(uni), d(e)
                toks = d(torch.tensor([0, tok1, tok2], dtype=i64))
                csr = d(torch.tensor([0, 2, 2, 2, 0, 0, 1, 2], dtype=i32))  # starts|counts|list
                res = torch.full((vocab + 8,), 7.0, device=dev)
                out = torch.full((3 + 3 + 3,), -9, dtype=i64, device=dev)
                _capi.call("tm_op4_sample_walk", ld.data_ptr(), _capi.TM_DTYPE_F32, 3, vocab,
                           stride, qd.data_ptr(), stride, toks.data_ptr(), csr.data_ptr(),
                           csr.data_ptr() + 12, csr.data_ptr() + 24, 2, ud.data_ptr(),
                           ed.data_ptr(), 1.0, res.data_ptr(), out.data_ptr(),
                           out.data_ptr() + 24, out.data_ptr() + 48, _capi.stream_of(dev))
                got, o = res.double().cpu(), out.cpu()
                assert o[0] == (2 if accept else -1) and o[7] == int(accept), (tok1, tok2, accept)
                assert torch.all(got[vocab:] == 7.0)
                # two renormalisations divide by what is left of the sum: a few 2^-24 of p and
                # q over it
                left = float((p0 - q1).clamp(min=0).sum()) * (
                    1.0 if accept else float((r1 - q2).clamp(min=0).sum()))
                tol = 2e-6 * (want + 1.0 / max(left, 1e-3)) + 1e-9
                assert torch.all((got[:vocab] - want).abs() <= tol), (tok1, tok2, accept)
                race = want / e.double()
                assert race[int(o[6])] >= race.max() * (1 - 1e-3) - 1e-6 / max(left, 1e-3)
