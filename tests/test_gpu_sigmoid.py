"""The sigmoid gates of csrc/lfm25_gemm.h (over_one_plus_exp), which the
encoder's Swish, its GLU and the prompt pass's SiLU share: what infinities and
NaN give where the gated value is not the gate, and the FP32 error."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def test_glu_keeps_nan_and_infinities(lab, gpu):
    """Every pair of a value and a gate among NaN, the infinities and ordinary
    numbers, a channel each, in one frame of lfm25_pk_conv with the taps
    (0, .., 1, .., 0): out = swish(bf16(value * sigmoid(gate)))."""
    values, gates = [NAN, INF, -INF, 0.0, 1.5, -2.0], [NAN, INF, -INF, 300.0, -300.0, 0.25]
    frames, at = 128, 64
    c = torch.ones(frames, 2048, dtype=torch.float64)
    for i, v in enumerate(values):
        for j, g in enumerate(gates):
            c[at, len(gates) * i + j] = v
            c[at, 1024 + len(gates) * i + j] = g
    taps = torch.zeros(1024, 9, dtype=torch.bfloat16)
    taps[:, 4] = 1
    cd, wd = c.bfloat16().to(gpu), taps.to(gpu)
    bias = torch.zeros(1024, dtype=torch.bfloat16, device=gpu)
    out = torch.zeros(frames, 1024, dtype=torch.bfloat16, device=gpu)
    lab._lib.call("lfm25_pk_conv", cd.data_ptr(), wd.data_ptr(), bias.data_ptr(), out.data_ptr(), 1, frames, frames,
                  torch.cuda.current_stream().cuda_stream)
    sigmoid = lambda x: torch.sigmoid(x.float()).double()  # noqa: E731  (of -300: 0 in FP32, and 0 times an infinity a NaN)
    glu = (c[:, :1024] * sigmoid(c[:, 1024:])).bfloat16().double()
    pad = torch.nn.functional.pad(glu, (0, 0, 4, 4))
    y = sum(pad[j:j + frames] * taps[:, j].double() for j in range(9))  # (0 times a NaN or an infinity is a NaN)
    want, got = y * sigmoid(y), out.double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    finite = torch.isfinite(want)
    assert torch.equal(got[~finite & ~torch.isnan(want)], want[~finite & ~torch.isnan(want)])
    # a gate value next to a BF16 boundary may round either way, and the result once more
    assert bool(((got - want).abs()[finite] <= 2.0 ** -7 * want.abs()[finite]).all())


def test_sigmoid_error_in_fp32(lab, gpu):
    """Swish of 3.6 million FP32 numbers (hi + 2^e (lo + lo2) from a product
    with exact sums, 24 bits each) against 64 bits. The FP32 value is within 7
    x 2^-24 of the exact one (a unit in the last place each, that is 2 x
    2^-24, for the exponential and the reciprocal, a rounding each for the
    correction, the sum and the final product), so the BF16 result is within
    half a step and that of it."""
    rows, cols = [], []
    for e in range(-3, 4):
        for hi in range(128, 256):
            rows += [(sign * hi * 2.0 ** (e - 7), 2.0 ** e) for sign in (1, -1)]
    g = torch.Generator().manual_seed(5)
    lo2 = torch.randint(0, 256, (2048,), generator=g)
    a = torch.zeros(len(rows), 64)
    a[:, :2] = torch.tensor(rows)
    a[:, 2] = a[:, 1]
    b = torch.zeros(2048, 64)
    b[:, 0] = 1
    b[:, 1] = (torch.arange(2048) % 256) * 2.0 ** -15
    b[:, 2] = lo2 * 2.0 ** -23
    ad, bd = a.bfloat16().to(gpu), b.bfloat16().to(gpu)
    assert torch.equal(ad.cpu().float(), a) and torch.equal(bd.cpu().float(), b)
    c = torch.empty(len(rows), 2048, dtype=torch.bfloat16, device=gpu)
    lab._lib.call("lfm25_pk_gemm", ad.data_ptr(), 64, bd.data_ptr(), 64, None, c.data_ptr(), 2048, len(rows), 2048, 64,
                  2, 1, None, torch.cuda.current_stream().cuda_stream)
    x = ad.double() @ bd.double().T.contiguous()
    want = x / (1 + torch.exp(-x))
    step = torch.ldexp(torch.ones_like(x), torch.frexp(want.abs())[1] - 8)
    excess = ((c.double() - want).abs() - step / 2) / want.abs() * 2.0 ** 24
    print(f"largest excess over half a step {float(excess.max()):.2f} x 2^-24, "
          f"{int((c != want.to(torch.bfloat16)).sum())} values off the nearest")
    assert float(excess.max()) <= 7
