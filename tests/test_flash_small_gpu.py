"""Attention without (T, T) matrices on both sides of the line between 32 and 128 rows a workgroup, and at the edges of the
key ranges that the smaller form is built for (128, 256, 512, 1024 keys); the oracle and its bounds are those of test_flash_gpu."""

import numpy as np
import pytest

from oracle import ref_gemm as O
from tests.test_flash_gpu import test_flash_attention as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("B,T,H,hd,packed", [
    (1, 128, 1, 64, True), (1, 256, 2, 16, False), (1, 257, 1, 64, True), (1, 512, 1, 80, False), (1, 513, 1, 32, True),
    (1, 1025, 1, 64, False), (1, 160, 1, 128, True),     # 1025 keys and heads of 128 backward: 128 rows a workgroup
    (4, 97, 32, 16, False), (3, 97, 43, 16, True),       # 512 and 516 blocks of 32 rows: backward changes over
    (8, 97, 32, 8, False), (5, 129, 41, 8, True)])       # 1024 and 1025: forward does
def test_both_sides_of_the_rules(B, T, H, hd, packed, dtype):
    check(B, T, H, hd, packed, dtype)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("B,T,H,hd", [
    (1, 64, 2, 64), (2, 200, 1, 96), (1, 333, 2, 128), (1, 1024, 1, 64),   # 32 rows forward, and (but 128) backward
    (1, 128, 150, 32),                                                     # 32 rows forward, 128 backward
    (1, 1100, 1, 64), (1, 1030, 1, 80)])                                   # 128 rows forward
def test_backward_rebuilds_the_p_of_the_forward_pass(dev, B, T, H, hd, dtype):
    """Narrowed P, read off both passes: with V one-hot on a window of keys the output is a block of P, with dOut one-hot on a
    window of queries dV is.  The row term cancels in the gradients only if the two are the same."""
    from vkgrad_amd.tkernels import make_transformer_kernels
    TK, D, scale = make_transformer_kernels(dev, dtype), H * hd, 1.0 / np.sqrt(hd)
    rng = np.random.default_rng(T + hd)
    q0 = T - hd
    for k0 in sorted({0, q0}):
        qkv = (rng.standard_normal((B, T, 3, H, hd)) * 2).astype(np.float32)
        qkv[:, :, 2] = 0
        dout = np.zeros((B, T, H, hd), np.float32)
        for i in range(hd):
            qkv[:, k0 + i, 2, :, i] = dout[:, q0 + i, :, i] = 1
        qkv, dout = O.round_to(qkv.reshape(B * T, 3 * D), dtype), O.round_to(dout.reshape(B * T, D), dtype)
        bqkv, bg, b16, b32, blse, bds, bdq = (dev.buffer(n, "device") for n in (qkv.nbytes, dout.nbytes, dout.nbytes, 2 * dout.nbytes,
                                                                               4 * B * H * T, 4 * B * H * T, qkv.nbytes))
        bqkv.upload(qkv.view(np.uint16))
        bg.upload(dout.view(np.uint16))
        TK["flash_fwd"]([bqkv, None, b16, b32, blse], B, T, H, hd, scale)
        TK["flash_bwd"]([bqkv, None, bg, b32, blse, bds, bdq], B, T, H, hd, scale)
        out = O.widen(b16.download(np.uint16, (B, T, H, hd)).view(qkv.dtype), dtype)
        dv = O.widen(bdq.download(np.uint16, (B, T, 3, H, hd)).view(qkv.dtype), dtype)[:, :, 2]
        for b in (bqkv, bg, b16, b32, blse, bds, bdq):
            b.destroy()
        forward, backward = out[:, q0:].transpose(0, 2, 1, 3), dv[:, k0:k0 + hd].transpose(0, 2, 3, 1)   # (B, H, query, key)
        assert forward.any() and np.array_equal(forward, backward)


@pytest.mark.parametrize("T,H,hd", [(64, 256, 80), (128, 128, 96), (96, 170, 64), (64, 256, 64)])   # 510 and 512 blocks of 32 rows
def test_backward_of_many_short_rows_is_no_slower_than_that_of_more(dev, T, H, hd):
    """Workgroups of 32 rows took up to 512 blocks of any width and length: 28.6 us for 256 heads of 64 x 80, 21.5 for 260."""
    from vkgrad_amd.tkernels import make_transformer_kernels
    TK = make_transformer_kernels(dev, "bf16")

    def us(H):
        n, D = T, H * hd
        sizes = (n * 3 * D * 2, n * D * 2, n * D * 4, 4 * H * n, 4 * H * n, n * 3 * D * 2)
        bqkv, bg, b32, blse, bds, bdq = bufs = [dev.buffer(x, "device") for x in sizes]
        for b in bufs:
            b.upload(np.zeros(b.size, np.uint8))
        g = dev.graph("backward")
        for _ in range(8):
            TK["flash_bwd"]([bqkv, None, bg, b32, blse, bds, bdq], 1, T, H, hd, 0.1, graph=g)
        g.finish()
        g.time(3)
        t = float(np.median(g.time(15))) * 1e6 / 8
        g.destroy()
        for b in bufs:
            b.destroy()
        return t
    assert us(H) <= 1.15 * us(H + 4)
