"""Softmax cross-entropy of the LM head (mg_tk_softmax_ce) at the edges of its row splits: a wavefront, 256 or 1024 threads a
row, whole and partial groups of loads, the loss alone and with its gradients."""

import numpy as np
import pytest

from oracle import ref_gemm as O
from oracle import ref_transformer as RT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,stride,ncls", [(1, 1, 1), (7, 64, 64), (5, 1024, 1024), (6, 1028, 1025), (3, 1090, 1027),
                                              (2, 4096, 4096), (2, 16384, 16383), (2, 16384, 16384), (1, 16500, 16389)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_loss_with_and_without_gradients(dev, rows, stride, ncls, dtype):
    from vkgrad_amd.tkernels import make_transformer_kernels
    TK = make_transformer_kernels(dev, dtype)
    rng = np.random.default_rng(rows + stride)
    logits = (rng.standard_normal((rows, stride)) * 3).astype(np.float32)
    logits[:, ncls:] = 1e4                                   # padding is masked
    labels = rng.integers(0, ncls, rows).astype(np.uint32)
    labels[-1] = ncls - 1
    w = rng.uniform(0.5, 2.0, rows).astype(np.float32)
    w[0] = 0 if rows > 1 else w[0]
    bufs = [dev.buffer(n, "device") for n in (logits.nbytes, 4 * rows, 4 * rows, 2 * rows * stride, 4 * rows * stride, 4 * rows)]
    bl, by, bw, b16, b32, bloss = bufs
    for b, a in ((bl, logits), (by, labels), (bw, w)):
        b.upload(a)
    ulp = 2.0 ** -10 if dtype == "f16" else 2.0 ** -7
    for weights in (None, w):
        loss, dl16, dl32 = RT.softmax_ce_rows(logits, labels, ncls, weights, dtype)
        for out16, out32 in ((b16, b32), (b16, None), (None, None)):
            bloss.upload(np.full(rows, np.nan, np.float32))
            b16.upload(np.full(rows * stride, 0x7bad, np.uint16))
            b32.upload(np.full(rows * stride, np.nan, np.float32))
            if weights is None:
                TK["softmax_ce"]([bl, by, out16, out32, bloss], rows, stride, ncls)
            else:
                TK["softmax_ce_w"]([bl, by, bw, out16, bloss], rows, stride, ncls)
            # f32 sums of up to 16384 terms, exponentials of one ulp or two
            assert np.allclose(bloss.download(np.float32, (rows,)), loss, rtol=1e-5, atol=1e-5)
            raw = b16.download(np.uint16, (rows, stride))
            if out16 is None:
                assert (raw == 0x7bad).all()
            else:
                got = O.widen(raw.view(np.float16) if dtype == "f16" else raw, dtype)
                want = O.widen(dl16, dtype)
                assert (np.abs(got - want) <= ulp * np.maximum(np.abs(want), 2.0 ** -14) + 1e-6).all()
                assert not got[:, ncls:].any()
            if weights is None and out32 is not None:
                assert np.abs(b32.download(np.float32, (rows, stride)) - dl32).max() <= 1e-6
    for b in bufs:
        b.destroy()


@pytest.mark.parametrize("ncls,more", [(96, 700), (2000, 9000), (20000, 30000)])   # a wavefront, 256 and 1024 threads a row
def test_impossible_classes_change_no_bit(dev, ncls, more):
    """A thread adds its exponentials up one after the other, however many of its loads travel together: the sum, and so the loss,
    does not depend on what follows a class."""
    from vkgrad_amd.tkernels import make_transformer_kernels
    TK, rows = make_transformer_kernels(dev, "bf16"), 64
    rng = np.random.default_rng(ncls)
    logits = np.full((rows, more), -np.inf, np.float32)
    logits[:, :ncls] = rng.standard_normal((rows, ncls)) - np.log(ncls)
    labels = rng.integers(0, ncls, rows).astype(np.uint32)
    logits[np.arange(rows), labels] = 0                      # losses of about 1: their last bit is that of the sum
    losses = []
    for n in (ncls, more):
        bl, by, bloss = dev.buffer(4 * rows * n, "device"), dev.buffer(4 * rows, "device"), dev.buffer(4 * rows, "device")
        bl.upload(np.ascontiguousarray(logits[:, :n]))
        by.upload(labels)
        TK["softmax_ce"]([bl, by, None, None, bloss], rows, n, n)
        losses.append(bloss.download(np.float32, (rows,)))
        for b in (bl, by, bloss):
            b.destroy()
    assert np.isfinite(losses[0]).all() and np.array_equal(*losses)
