"""Attention without (T, T) matrices in workgroups of 128 rows: calls of more than 1024 keys, or more blocks of 32 rows than those of
32 rows take."""

import numpy as np
import pytest

from oracle import ref_gemm as O
from tests.test_flash_gpu import test_flash_attention as check

pytestmark = pytest.mark.gpu


# Every width class of a head (16, 32, 64, 96, 128; above 64 with one buffer a tensor), both directions, packed and not.
@pytest.mark.parametrize("dtype,B,T,H,hd,packed", [
    # 1405 blocks of 32 rows in 562 workgroups: whole rounds of 256, the second dealt out backwards, and a part of one
    ("bf16", 1, 150, 281, 16, False), ("f16", 1, 150, 281, 32, False), ("bf16", 1, 150, 281, 64, False), ("f16", 1, 150, 281, 64, True),
    ("bf16", 1, 150, 281, 80, True), ("f16", 1, 150, 281, 128, False),
    # more than 1024 keys; with 15 heads and more, also too many blocks of 32 rows for the backward form of those
    ("f16", 1, 1100, 1, 16, True), ("bf16", 1, 1100, 15, 32, True), ("bf16", 1, 1040, 17, 56, False), ("f16", 1, 1100, 15, 96, False),
    ("bf16", 1, 1100, 1, 128, True)])
def test_both_directions_of_every_width(B, T, H, hd, packed, dtype):
    check(B, T, H, hd, packed, dtype)


@pytest.mark.parametrize("gap", [60.0, 7.0, 0.0])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_lse_of_rows_whose_first_tile_is_far_below(dev, gap, dtype):
    """The row's reference point follows its maximum: held relative to a first tile 60 (base 2) below the rest, a sum has the
    exponent 2^60, and its logarithm six bits fewer."""
    from vkgrad_amd.tkernels import make_transformer_kernels
    TK, T, hd, log2e = make_transformer_kernels(dev, dtype), 1088, 64, np.log2(np.e)
    scale = 1.0 / 8.0
    rng = np.random.default_rng(3)
    q, k = rng.standard_normal((T, hd)) * 0.25, rng.standard_normal((T, hd)) * 0.25
    q[:, 0], k[:, 0] = 8.0, rng.standard_normal(T) * 0.5
    k[:64, 0] -= gap / log2e
    qkv = O.round_to(np.concatenate([q, k, k], 1).astype(np.float32), dtype)
    bqkv, b16, blse = dev.buffer(qkv.nbytes, "device"), dev.buffer(T * hd * 2, "device"), dev.buffer(T * 4, "device")
    bqkv.upload(qkv.view(np.uint16))
    TK["flash_fwd"]([bqkv, None, b16, None, blse], 1, T, 1, hd, scale)
    lse = blse.download(np.float32, (T,))
    for b in (bqkv, b16, blse):
        b.destroy()
    w = O.widen(qkv, dtype).astype(np.float64)
    s = w[:, :hd] @ w[:, hd:2 * hd].T * (scale * log2e)
    s[np.triu_indices(T, 1)] = -np.inf
    m = s.max(1, keepdims=True)
    want = (m[:, 0] + np.log2(np.exp2(s - m).sum(1)))
    rows = slice(66, 320)       # sums of 2 to 256 terms above the first tile's: lse below 16
    assert np.abs(want[rows]).max() < 16
    # roundings of exponents, sum, logarithm and result are each spread over an ulp of a value below 16 (2^-20), a few of them; relative
    # to the first tile the logarithm alone has an ulp of 2^-17
    assert np.sqrt(np.mean((lse[rows] - want[rows]) ** 2)) <= 2.0 ** -20
