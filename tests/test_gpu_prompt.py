"""The prompt pass (lfm25_prompt_pass) against the batched pass
(lfm25_batch_pass, which the oracle holds elsewhere) on the same rows: both
round at the same points and sum in different FP32 orders, so hidden states,
conv states and KV rows agree within the bound that holds each of them to the
oracle, twice (16 BF16 ulps of the vector's scale each)."""

from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

VOCAB = 1024


@pytest.fixture(scope="module")
def batch(gpu):
    return importlib.import_module("ryzenai-npu-lab_amd.batch")


@pytest.fixture(scope="module")
def ck(lab):
    return lab.weights.synthetic_checkpoint(5, vocab=VOCAB)


def scale_ulps(got, want) -> float:
    s = float(np.max(np.abs(want)))
    return float(np.max(np.abs(got - want))) / 2.0 ** (np.floor(np.log2(s)) - 7) if s > 0 else float(np.max(np.abs(got)))


def by_passes(bd, runs, ids):
    """The runs' rows through lfm25_batch_pass, 64 at a time; the last rows' hidden states."""
    last = []
    for (s, pos, n), t in zip(runs, ids):
        for i in range(0, n, 64):
            _, h = bd.run_rows([(int(t[j]), s, pos + j) for j in range(i, min(i + 64, n))], hidden=True)
        last.append(h[-1])
    return np.stack(last)


def by_prompt_pass(lab, bd, runs, ids, gpu):
    flat = torch.from_numpy(np.concatenate(ids).astype(np.int32)).to(gpu)
    table = np.asarray(runs, np.int32)
    rows = int(table[:, 2].sum())
    ws = torch.full((lab._lib.load().lfm25_prompt_workspace_bytes(rows),), 0xff, dtype=torch.uint8, device=gpu)
    h = torch.empty(len(runs), 1024, dtype=torch.bfloat16, device=gpu)
    tok = torch.full((len(runs),), -1, dtype=torch.int32, device=gpu)
    lab._lib.call("lfm25_prompt_pass", bd._desc, flat.data_ptr(), table.ctypes.data, len(runs), tok.data_ptr(),
                  h.data_ptr(), ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert bd._status() == 0
    return h.float().cpu().numpy(), tok.cpu().numpy()


@pytest.mark.parametrize("capacity,before,runs", [
    (64, {}, [(0, 0, 1)]),                                            # one row
    (64, {0: 3}, [(1, 0, 2), (0, 3, 1), (2, 0, 3)]),                  # runs of one, two and three rows
    (64, {1: 1}, [(0, 0, 17), (1, 1, 16), (2, 0, 15)]),               # around a 16-query attention tile
    (256, {0: 65}, [(2, 0, 63), (0, 65, 64), (1, 0, 65)]),            # around a key tile
    (320, {2: 40}, [(2, 40, 257), (1, 0, 5)]),                        # 250-odd rows: 32 x 64 and 64 x 64 tiles
    (1100, {}, [(0, 0, 1031)]),                                       # 32 queries a block
    (2200, {1: 100}, [(1, 100, 2050), (0, 0, 31)]),                   # 64 queries a block, 256-row tiles
])
def test_prompt_pass_matches_the_batched_pass(lab, gpu, batch, ck, capacity, before, runs):
    a = batch.BatchDecoder(3, capacity, weights=ck)
    b = batch.BatchDecoder(3, capacity, share=a)
    rng = np.random.default_rng(capacity)
    for bd in (a, b):
        g = np.random.default_rng(7)
        for s, n in before.items():
            by_passes(bd, [(s, 0, n)], [g.integers(0, VOCAB, n)])
        # rows past the prompts' ends hold junk: none of it may be read
        bd.keys.view(3, 6, 8, capacity, 64)[:, :, :, -1] = float("nan") if capacity == 64 else 0
    ids = [rng.integers(0, VOCAB, n) for _, _, n in runs]
    want = by_passes(a, runs, ids)
    got, tok = by_prompt_pass(lab, b, runs, ids, gpu)
    assert scale_ulps(got, want) <= 32
    table = torch.from_numpy(ck["model.embed_tokens.weight"].view(np.int16)).to(gpu).view(torch.bfloat16).double()
    gamma = torch.from_numpy(ck["model.embedding_norm.weight"].view(np.int16)).to(gpu).view(torch.bfloat16).double()
    for r, (s, pos, n) in enumerate(runs):
        for c in range(8):
            assert scale_ulps(b.conv_state(s, c), a.conv_state(s, c)) <= 32, (s, c)
        for l in range(6):
            for x, y in zip(b.kv(s, l, pos + n - 1), a.kv(s, l, pos + n - 1)):
                assert scale_ulps(x, y) <= 32, (s, l)
        # the selection is a maximum of its own hidden state's logits, within a BF16 step
        x = torch.from_numpy(got[r]).to(gpu).double()
        logits = table @ (x / torch.sqrt((x * x).mean() + 1e-5) * gamma)
        assert float(logits[int(tok[r])]) >= float(logits.max()) - 2.0 ** -6 * abs(float(logits.max()))


def test_prompt_pass_repeats_bitwise_and_keeps_runs_apart(lab, gpu, batch, ck):
    """Two calls give the same bits, and a run's do not depend on the runs beside it."""
    runs = [(0, 0, 70), (1, 0, 33), (2, 0, 9)]
    ids = [np.random.default_rng(i).integers(0, VOCAB, n) for i, (_, _, n) in enumerate(runs)]
    outs = []
    for pick in ([0, 1, 2], [0, 1, 2], [1]):
        bd = batch.BatchDecoder(3, 128, weights=ck)
        h, _ = by_prompt_pass(lab, bd, [runs[i] for i in pick], [ids[i] for i in pick], gpu)
        outs.append((h[pick.index(1)], bd.conv_state(1, 7), *bd.kv(1, 5, 32)))
    for other in outs[1:]:
        for x, y in zip(outs[0], other):
            assert np.array_equal(x, y)


def test_prompt_pass_rejects_bad_runs(lab, gpu, batch, ck):
    bd = batch.BatchDecoder(2, 64, weights=ck)
    ids = torch.zeros(64, dtype=torch.int32, device=gpu)
    ws = torch.empty(lab._lib.load().lfm25_prompt_workspace_bytes(64), dtype=torch.uint8, device=gpu)
    for runs in ([(2, 0, 4)], [(0, 0, 4), (0, 4, 4)], [(0, 60, 5)], [(0, -1, 4)], [(0, 0, 0)]):
        table = np.asarray(runs, np.int32)
        with pytest.raises(ValueError):
            lab._lib.call("lfm25_prompt_pass", bd._desc, ids.data_ptr(), table.ctypes.data, len(runs), None, None,
                          ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
