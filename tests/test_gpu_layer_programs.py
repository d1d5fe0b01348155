"""The layer programs of csrc/lfm25_layer.hip at the edges of their position
blocks: attention_context_cache against attention_context and
append_attention_cache (which the oracle holds elsewhere), and its context
inside the interval derived from the oracle's algorithm, which a position
more or less leaves."""

from __future__ import annotations

import pytest
import torch

from parity_helpers import attention_interval

pytestmark = pytest.mark.gpu


def inputs(gpu, past):
    g = torch.Generator(device=gpu)
    g.manual_seed(past)
    normal = lambda *s: torch.randn(s, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    return normal(3072), normal(8 * 2 * past * 64)


def by_parts(lab, gpu, qkv, cache, past):
    tail = torch.empty(2048, dtype=torch.bfloat16, device=gpu)
    nxt = torch.empty(8 * 2 * (past + 1) * 64, dtype=torch.bfloat16, device=gpu)
    lab.ops.attention_context(qkv[:2048], cache, tail[1024:])
    lab.ops.append_attention_cache(qkv[:2048], cache, nxt)
    tail[:1024].copy_(qkv[2048:])
    return tail, nxt


@pytest.mark.parametrize("past", [1, 2, 62, 63, 64, 65, 127, 511, 512, 513, 1023, 3000, 4095])
def test_context_cache_at_block_edges(lab, gpu, past):
    qkv, cache = inputs(gpu, past)
    tail = torch.full((2048,), float("nan"), dtype=torch.bfloat16, device=gpu)
    nxt = torch.full((8 * 2 * (past + 1) * 64,), float("nan"), dtype=torch.bfloat16, device=gpu)
    lab.ops.attention_context_cache(qkv, cache, tail, nxt, past_length=past)
    want_tail, want_next = by_parts(lab, gpu, qkv, cache, past)
    assert torch.equal(nxt, want_next)
    assert torch.equal(tail[:1024], want_tail[:1024])
    # the same scores; the two FP32 sums (z, the context) in another order: a
    # probability or the result may round to the neighbouring BF16 value
    a, b = tail[1024:].double(), want_tail[1024:].double()
    v = nxt.view(8, 2, past + 1, 64)[:, 1].double().abs().amax(dim=(1, 2)).repeat_interleave(128)
    assert bool(((a - b).abs() <= 2.0 ** -8 * b.abs() + 2.0 ** -16 * v).all() | (past > 64) &
                ((a - b).abs() <= 2.0 ** -7 * b.abs().clamp_min(b.abs().mean())).all())
    # FP32 roundings on one path: a lane's passes of 512 positions, five over
    # the lanes, sixteen waves; the sum of the probabilities has fewer
    rows = nxt.view(8, 2, past + 1, 64).float().cpu().numpy()
    lo, hi = attention_interval(qkv[:1024].view(16, 64).float().cpu().numpy(), rows[:, 0], rows[:, 1],
                                24 + (past + 1) // 512)
    got = tail[1024:].double().cpu().numpy()
    assert ((got >= lo) & (got <= hi)).all()


def test_context_cache_of_a_misaligned_cache(lab, gpu):
    """Outputs that are not 16-byte aligned take the separate calls, bit for bit."""
    past = 70
    qkv, cache = inputs(gpu, past)
    store = torch.zeros(8 * 2 * (past + 1) * 64 + 1, dtype=torch.bfloat16, device=gpu)
    tail = torch.empty(2048, dtype=torch.bfloat16, device=gpu)
    lab.ops.attention_context_cache(qkv, cache, tail, store[1:], past_length=past)
    want_tail, want_next = by_parts(lab, gpu, qkv, cache, past)
    assert torch.equal(store[1:], want_next) and torch.equal(tail, want_tail) and float(store[0]) == 0


def test_context_cache_scores_of_infinity(lab, gpu):
    """A key whose scores are -inf adds nothing, +inf makes its head NaN, as in attention_context."""
    past = 130
    qkv, cache = inputs(gpu, past)
    qkv[:2048] = qkv[:2048].abs() + 0.1
    rows = cache.view(8, 2, past, 64)
    rows[0, 0, 5] = -float("inf")
    rows[1, 0, 100] = float("inf")
    rows[2, 0, 64:128] = -float("inf")  # a whole block of positions
    tail = torch.empty(2048, dtype=torch.bfloat16, device=gpu)
    nxt = torch.empty(8 * 2 * (past + 1) * 64, dtype=torch.bfloat16, device=gpu)
    lab.ops.attention_context_cache(qkv, cache, tail, nxt, past_length=past)
    want, _ = by_parts(lab, gpu, qkv, cache, past)
    heads, ref = tail[1024:].view(8, 128), want[1024:].view(8, 128)
    assert torch.equal(torch.isnan(heads), torch.isnan(ref))
    fine = ~torch.isnan(ref)
    assert torch.allclose(heads[fine].float(), ref[fine].float(), rtol=2.0 ** -7, atol=2.0 ** -7)
