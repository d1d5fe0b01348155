"""The encoder attention's two splits of the work (blocks of 16 queries up to
eight sequences, two blocks per sequence and head above) against the oracle,
at masks on either side of a wave's 32 keys."""

import numpy as np
import pytest
import torch

from test_gpu_parakeet import T, P, _qkv_fields, dev, host, layer0, pk, scale_ulps, stream  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("valid", [1, 32, 33, 127, 128])
@pytest.mark.parametrize("batch", [1, 8, 9])
def test_attention_splits(lab, gpu, pk, layer0, batch, valid):  # noqa: F811
    distinct = min(batch, 2)
    qkv, bd, delta = _qkv_fields(layer0, distinct, 53 + valid)
    pick = [0] * (batch - 1) + [distinct - 1]
    table = pk.pack_layer(*layer0)["pos"]
    qd, pd, dd = dev(qkv[pick], gpu), dev(table, gpu), dev(delta, gpu)
    od = torch.zeros(batch * T * 1024, dtype=torch.bfloat16, device=gpu)
    lab._lib.call("lfm25_pk_attention", qd.data_ptr(), pd.data_ptr(), dd.data_ptr(), od.data_ptr(), batch, T, valid,
                  stream())
    got = host(od, (batch, T, 1024))
    assert all(np.array_equal(got[b], got[0]) for b in range(batch - 1))
    for b in {0, batch - 1}:
        want = P.attention(qkv[pick[b]], bd[pick[b]], delta, valid)
        for h in range(8):
            sl = slice(128 * h, 128 * (h + 1))
            assert scale_ulps(got[b][:, sl], want[:, sl]) <= 2.0, (b, h)


@pytest.mark.parametrize("batch", [1, 9])
def test_large_values_do_not_overflow(lab, gpu, batch):
    """Equal scores over 128 values of 2^122: their mean is 2^122, their sum
    past FP32's range."""
    qkv = torch.zeros(batch, T, 3, 1024, dtype=torch.bfloat16, device=gpu)
    qkv[:, :, 2] = 2.0 ** 122
    pos = torch.zeros(8, 2 * T, 128, dtype=torch.bfloat16, device=gpu)
    delta = torch.zeros(8, 128, dtype=torch.bfloat16, device=gpu)
    out = torch.zeros(batch, T, 1024, dtype=torch.bfloat16, device=gpu)
    lab._lib.call("lfm25_pk_attention", qkv.data_ptr(), pos.data_ptr(), delta.data_ptr(), out.data_ptr(), batch, T, T,
                  stream())
    assert bool((out == 2.0 ** 122).all())
