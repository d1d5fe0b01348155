"""The prompt pass's attention and gated conv alone (attention_probe.py's
weights), every row against the oracle: at the edges of query and key tiles,
across runs and earlier positions, with every cache row that the pass has not
written a NaN."""

from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

import attention_probe as A
from oracle import lfm25 as O
from parity_helpers import attention_interval

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
EDGES = (0, 1, 15, 16, 31, 32, 63)  # of the query tiles


def decoder(capacity, ck):
    bd = importlib.import_module("ryzenai-npu-lab_amd.batch").BatchDecoder(3, capacity, weights=ck)
    for cache in (bd.keys, bd.values):
        cache.fill_(float("nan"))
    return bd


def prompt_pass(lab, bd, runs, ids, gpu):
    flat = torch.from_numpy(np.concatenate(ids).astype(np.int32)).to(gpu)
    table = np.asarray(runs, np.int32)
    ws = torch.full((lab._lib.load().lfm25_prompt_workspace_bytes(int(table[:, 2].sum())),), 0xff, dtype=torch.uint8,
                    device=gpu)
    lab._lib.call("lfm25_prompt_pass", bd._desc, flat.data_ptr(), table.ctypes.data, len(runs), None, None,
                  ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert bd._status() == 0


def run(lab, bd, before, runs, tokens, gpu):
    """`tokens[s]` of each sequence: the first before[s] in one pass, then the runs."""
    for s, n in before.items():
        prompt_pass(lab, bd, [(s, 0, n)], [tokens[s][:n]], gpu)
    prompt_pass(lab, bd, runs, [tokens[s][pos:pos + n] for s, pos, n in runs], gpu)


def read(bd, s, att, rows) -> np.ndarray:
    """Dimensions 0 .. 511 of the residual stream of the first `rows` positions."""
    return bd.kv(s, att, rows - 1)[1].transpose(1, 0, 2).reshape(rows, A.PICK)


# ------------------------------------------------------------------ attention


@pytest.mark.parametrize("capacity,before,runs", [
    (64, {}, [(0, 0, 1)]),
    (96, {0: 3, 1: 1}, [(1, 1, 16), (0, 3, 17), (2, 0, 15)]),   # around a 16-query tile
    (256, {0: 62}, [(2, 0, 63), (0, 62, 3), (1, 0, 65)]),       # key counts 63, 64, 65 both ways
    (300, {2: 64}, [(2, 64, 129), (1, 0, 64), (0, 0, 2)]),
    (1100, {1: 7}, [(0, 0, 1031), (1, 7, 33)]),                 # 32 queries a block
    (2200, {1: 100}, [(1, 100, 2050), (0, 0, 31)]),             # 64 queries a block
])
def test_attention_rows(lab, gpu, capacity, before, runs):
    rng = np.random.default_rng(capacity)
    sign = lambda heads: rng.choice([-1.0, 1.0], (A.TOKENS, heads, A.DIM))  # noqa: E731
    q, k, v = sign(A.HEADS), sign(A.KV_HEADS), A.bf(rng.standard_normal((A.TOKENS, A.KV_HEADS, A.DIM)) / 128)
    gq, gk = np.full(A.DIM, 2.0), np.ones(A.DIM)
    bd = decoder(capacity, A.attention_checkpoint(lab, q, k, v, gq, gk))
    tokens = rng.integers(0, A.TOKENS, (3, capacity))
    run(lab, bd, before, runs, tokens, gpu)
    for s, pos, n in runs:
        end = pos + n
        ids = tokens[s][:end]
        keys, values = bd.kv(s, 0, end - 1)
        kr = A.norm_rope(k[ids], gk, np.arange(end)).transpose(1, 0, 2)
        assert np.array_equal(keys, kr) and np.array_equal(values, v[ids].transpose(1, 0, 2))
        got = read(bd, s, 1, end)
        rows = {p for p in range(pos, end) if n <= 70 or (p - pos) // 64 % 4 == 0 and (p - pos) % 64 in EDGES}
        rows |= {p for p in range(pos, end) if p >= end - 2 or p in (63, 64, 65, 127, 128)}
        qr = A.norm_rope(q[ids], gq, np.arange(end))
        for p in sorted(rows):
            # FP32 roundings on one path: the sum of the probabilities takes a
            # lane's 16 per tile, a tile at a time, then the four lanes; the
            # context 32 keys a product
            lo, hi = attention_interval(qr[p], kr[:, :p + 1], values[:, :p + 1], 64 + (p + 1) // 32)
            inside = (got[p] >= lo[A.picked()]) & (got[p] <= hi[A.picked()])
            assert inside.all(), (s, p, np.flatnonzero(~inside)[:4], got[p][~inside][:4])


@pytest.mark.parametrize("gamma", [2.0, 2.0 ** 55])
@pytest.mark.parametrize("rows", [70, 1500, 4096])
def test_uniform_scores(lab, gpu, rows, gamma):
    """Every key the same, in the dimension pair that RoPE leaves alone over
    4,096 positions, so the p of the query at position n - 1 is bf16(1 / n)
    whatever the scores are (up to +-256 before their scale, or +-2^116): the
    FP32 quotient is within B of 1 / n, B from the sum of n equal terms (15
    additions in a tile, one a tile, two over the lanes) and three more
    roundings."""
    rng = np.random.default_rng(3)
    slow, fast = 31, 5  # a pair of lowest and one of high frequency: k has none of the latter
    c = rng.uniform(0.2, 1.0, (A.TOKENS, A.HEADS)) * rng.choice([-1, 1], (A.TOKENS, A.HEADS))
    q = np.zeros((A.TOKENS, A.HEADS, A.DIM))
    q[:, :, slow], q[:, :, fast] = A.bf(8 * c), A.bf(8 * np.sqrt(1 - c * c))
    k = np.zeros((A.TOKENS, A.KV_HEADS, A.DIM))
    k[:, :, slow] = 8
    v = np.full((A.TOKENS, A.KV_HEADS, A.DIM), 1 / 64)
    g = np.full(A.DIM, gamma)
    bd = decoder(rows, A.attention_checkpoint(lab, q, k, v, g, g))
    run(lab, bd, {}, [(0, 0, rows)], rng.integers(0, A.TOKENS, (1, rows)), gpu)
    got = read(bd, 0, 1, rows)
    n = np.arange(1, rows + 1, dtype=np.float64)[:, None]
    bound = (15 + (n + 63) // 64 + 2 + 3) * U
    # n equal products of p and 1 / 64 add up exactly (20 bits)
    lo, hi = (A.bf(n * A.bf(1 / n * (1 + d)).astype(np.float64) / 64) for d in (-bound, bound))
    bad = ~((got >= lo) & (got <= hi))
    i, j = np.argwhere(bad)[0] if bad.any() else (0, 0)
    assert not bad.any(), (int(bad.any(axis=1).sum()), int(n[i, 0]), j, float(got[i, j]), float(lo[i, 0]), float(hi[i, 0]))


# ------------------------------------------------------------------ gated conv


@pytest.mark.parametrize("before,runs", [
    ({}, [(0, 0, 1)]),
    ({0: 3, 2: 1}, [(1, 0, 2), (0, 3, 1), (2, 1, 3)]),       # runs of one, two and three rows
    ({1: 2}, [(2, 0, 4), (1, 2, 2), (0, 0, 70)]),
    ({1: 65}, [(1, 65, 1), (0, 0, 2), (2, 0, 301)]),
])
def test_conv_rows(lab, gpu, before, runs):
    """Layer 0's conv gate, bit for bit (the oracle rounds at the same points
    and every sum is exact or in the same order), and the state it leaves."""
    rng = np.random.default_rng(len(runs))
    b, x = (A.bf(rng.standard_normal((A.TOKENS, A.HIDDEN)) / 2) for _ in range(2))
    c = A.bf(rng.standard_normal((A.TOKENS, A.HIDDEN)) / 128)
    taps = A.bf(rng.standard_normal((A.HIDDEN, 3)) / 2)
    ck = A.checkpoint(lab)
    ck["model.layers.0.conv.in_proj.weight"] = A.columns(np.concatenate([b, c, x], axis=1))
    ck["model.layers.0.conv.conv.weight"] = A.bits(taps).reshape(A.HIDDEN, 1, 3)
    out = np.zeros((A.HIDDEN, A.HIDDEN), np.uint16)
    out[np.arange(A.PICK), 2 * np.arange(A.PICK)] = A.bits(1.0)
    ck["model.layers.0.conv.out_proj.weight"] = out
    A.read_back(ck, 2)
    bd = decoder(400, ck)
    tokens = rng.integers(0, A.TOKENS, (3, 400))
    run(lab, bd, before, runs, tokens, gpu)
    for s, pos, n in runs:
        state, want = np.zeros((A.HIDDEN, 3), np.float32), []
        for t in tokens[s][:pos + n]:
            y, state = O.conv_gate(b[t], c[t], x[t], taps, state)
            want.append(y[::2])
        assert np.array_equal(read(bd, s, 0, pos + n), np.stack(want)), s
        assert np.array_equal(bd.conv_state(s, 0), state), s
