"""The matrix-core tile product (csrc/lfm25_gemm.h) behind lfm25_pk_gemm at
the sizes where its tile shapes, its rectangles of tiles per XCD and its
remainders change over. Operands are small integers, so every product and
partial sum is exact in FP32 and the result has one correct BF16 value."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def ints(seed, shape, gpu):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    return torch.randint(-2, 3, shape, generator=g, device=gpu).to(torch.bfloat16)


@pytest.mark.parametrize("m,n,k,lda,ldc,splits", [
    (31, 128, 64, 64, 128, 1),              # one 32-row tile, a row short; one K step (fewer than stages)
    (33, 4096, 192, 200, 4096, 1),          # 32 x 64 tiles
    (300, 2048, 320, 320, 2052, 1),         # 64 x 64; rows that allow 8-byte stores only
    (640, 3072, 128, 128, 3072, 1),         # 64 x 128, whole tiles
    (577, 3072, 448, 448, 3080, 1),         # 64 x 128, ragged
    (1025, 2048, 256, 256, 2048, 1),        # 128 x 128
    (2049, 3072, 192, 192, 3072, 1),        # 256 x 128, one row in the last tile
    (3900, 3072, 128, 128, 3072, 1),        # 128 x 128, two blocks per CU
    (4100, 1024, 1088, 1088, 1024, 1),      # 256 x 128 in rectangles (17 x 8 tiles)
    (2177, 1152, 1024, 1032, 1152, 1),      # 128 x 128 in rectangles (18 x 9 tiles)
    (130, 1024, 1024, 1024, 1024, 4),       # split K
    (3, 256, 128, (1 << 22) + 8, 256, 1),   # rows beyond a tile's 32-bit offsets
    (3, 256, 128, (1 << 22) + 8, 256, 2),
])
def test_every_tile_shape_is_exact(lab, gpu, m, n, k, lda, ldc, splits):
    a = torch.zeros(m, lda, dtype=torch.bfloat16, device=gpu)
    a[:, :k] = ints(1, (m, k), gpu)
    b = ints(2, (n, k), gpu)
    bias = ints(3, (n,), gpu)
    c = torch.full((m, ldc), float("nan"), dtype=torch.bfloat16, device=gpu)
    ws = torch.full((splits * m * n,), float("nan"), dtype=torch.float32, device=gpu)
    lab._lib.call("lfm25_pk_gemm", a.data_ptr(), lda, b.data_ptr(), k, bias.data_ptr(), c.data_ptr(), ldc, m, n, k, 1,
                  splits, ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
    want = (a[:, :k].double() @ b.double().T.contiguous() + bias.double()).to(torch.bfloat16)
    assert torch.equal(c[:, :n], want)
    assert bool(torch.isnan(c[:, n:]).all())  # nothing written beyond n


def test_swish_epilogue_over_the_whole_range(lab, gpu):
    """Every finite BF16 value, both infinities and a NaN through the Swish
    epilogue (an identity product), against x / (1 + exp(-x)) in 64 bits: the
    epilogue's FP32 error is a few 2^-24, so the rounded value is the nearest
    BF16 or, next to a rounding boundary, its neighbour."""
    x = torch.arange(1 << 16, device=gpu, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = x[torch.isfinite(x)]
    special = torch.tensor([float("inf"), -float("inf"), float("nan")], device=gpu).bfloat16()
    x = torch.cat([x, special, torch.zeros(-(x.numel() + 3) % 128, device=gpu).bfloat16()])
    n = x.numel()
    a = torch.zeros(1, 64, dtype=torch.bfloat16, device=gpu)
    a[0, 0] = 1
    b = torch.zeros(n, 64, dtype=torch.bfloat16, device=gpu)
    b[:, 0] = x
    c = torch.empty(n, dtype=torch.bfloat16, device=gpu)
    lab._lib.call("lfm25_pk_gemm", a.data_ptr(), 64, b.data_ptr(), 64, None, c.data_ptr(), n, 1, n, 64, 2, 1, None,
                  torch.cuda.current_stream().cuda_stream)
    v = x.double()
    want = v / (1 + torch.exp(-v))
    nearest = want.to(torch.bfloat16)
    same = (c == nearest) | (torch.isnan(c) & torch.isnan(v / (1 + torch.exp(-v))))
    # denormal products: the epilogue may flush below the smallest normal number
    tiny = want.abs() < 2.0 ** -126
    step = torch.ldexp(torch.ones_like(v), torch.frexp(want.abs().clamp_min(2.0 ** -126))[1] - 8)
    close = (c.double() - want).abs() <= 0.5001 * step
    assert bool((same | close | (tiny & (c.double().abs() < 2.0 ** -126))).all())
    assert int((~same & ~tiny).sum()) <= 64  # ~3 of 2^24 per value off a boundary


@pytest.mark.parametrize("m,n,k,splits", [
    (130, 128, 8192, 1),    # 32 x 64 tiles
    (130, 128, 8192, 8),
    (700, 1280, 192, 1),    # 128 x 128 tiles, ragged
    (700, 1280, 256, 2),
])
def test_far_rows_take_the_tiles_and_the_splits(lab, gpu, m, n, k, splits):
    """Rows of A and then of B farther apart than a tile's 32-bit offsets
    reach: exact, beside rows that hold NaN past k, and (where the product
    itself is what takes the time) in about the time of near rows; an output
    per thread took 26 times as long."""
    far = (1 << 22) + 8

    def run(a, lda, b, ldb):
        c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
        ws = torch.full((splits * m * n,), float("nan"), dtype=torch.float32, device=gpu)
        times = []
        for _ in range(6):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            lab._lib.call("lfm25_pk_gemm", a.data_ptr(), lda, b.data_ptr(), ldb, bias.data_ptr(), c.data_ptr(), n, m, n,
                          k, 1, splits, ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        assert torch.equal(c, want)
        return min(times)

    def spread(x):
        y = torch.empty(x.shape[0], far, dtype=torch.bfloat16, device=gpu)
        y[:, :k] = x
        y[:, k:k + 64] = float("nan")
        return y

    a, b, bias = ints(6, (m, k), gpu), ints(7, (n, k), gpu), ints(8, (n,), gpu)
    want = (a.double() @ b.double().T.contiguous() + bias.double()).to(torch.bfloat16)
    near = run(a, k, b, k)
    times = run(spread(a), far, b, k), run(a, k, spread(b), far)
    assert k < 8192 or max(times) <= 5 * near
