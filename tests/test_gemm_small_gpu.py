"""Products of a few tiles whose K slices meet in LDS (gemm_small_kernel.h): the oracle, and the bits that
the same slices have where they meet in the workspace, at the edges of 32 x 32 blocks, of K-blocks and of the rule that takes them."""

import numpy as np
import pytest

from oracle import ref_gemm as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,split,nt", [(33, 512, 784, 5, False), (128, 10, 512, 4, False), (1, 8, 128, 2, False), (65, 72, 1000, 8, True),
                                            (31, 40, 520, 3, True), (32, 33, 264, 2, False), (7, 5, 776, 7, True), (96, 64, 4096, 8, False),
                                            (128, 128, 640, 2, True), (500, 512, 512, 2, False)])   # (the last: more blocks than CUs)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_slices_in_one_workgroup(dev, m, n, k, split, nt, dtype):
    from vkgrad_amd.kernels import Matmul
    rng = np.random.default_rng(m + n + k)
    a = O.round_to(rng.standard_normal((m, k)).astype(np.float32), dtype)
    b = O.round_to(rng.standard_normal((n, k) if nt else (k, n)).astype(np.float32), dtype)
    bias, c0 = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    ba, bb, bbias, bc, by = (dev.buffer(x + 64, "device") for x in (a.nbytes, b.nbytes, 4 * n, 4 * m * n, 2 * m * n))
    for buf, arr in ((ba, a), (bb, b), (bbias, bias)):
        buf.upload(arr)
    mm = Matmul(dev, trans_b=nt, dtype=dtype, tile=4, split_k=split)
    want = O.widen(a, dtype).astype(np.float64) @ (O.widen(b, dtype).T if nt else O.widen(b, dtype)).astype(np.float64) + bias

    def run(which, **kw):
        bc.upload(c0)
        which(ba, bb, bc, m, n, k, bias=bbias, **kw)
        return bc.download(np.float32, (m, n))
    got = run(mm)
    # f32 sums of up to 4096 products of N(0, 1) values
    assert np.abs(got - want).max() <= 2.0 ** -22 * k
    assert np.array_equal(got, run(mm))
    assert np.abs(run(mm, accumulate=True) - (want + c0)).max() <= 2.0 ** -22 * k
    assert np.array_equal(run(mm, act="relu", y16=by), got)
    y = by.download(np.uint16, (m, n))
    y = O.widen(y.view(np.float16) if dtype == "f16" else y, dtype)
    assert np.array_equal(y, O.widen(O.round_to(np.maximum(got, 0), dtype), dtype))
    # a larger result with the same rows and columns first takes the slices to the workspace: the same bits
    big = 32 * (dev.compute_units // -(-n // 32) + 1)
    a2 = np.zeros((big, k), a.dtype)
    a2[:m] = a
    ba2, bc2 = dev.buffer(a2.nbytes + 64, "device"), dev.buffer(4 * big * n, "device")
    ba2.upload(a2)
    assert mm.statistics(big, n, k)["workgroupThreads"] == 256
    mm(ba2, bb, bc2, big, n, k, bias=bbias)
    assert np.array_equal(bc2.download(np.float32, (big, n))[:m], got)
    for buf in (ba, bb, bbias, bc, by, ba2, bc2):
        buf.destroy()


@pytest.mark.parametrize("m,n,k,split,nt,lda,ldb,ldc,ldy", [
    (33, 40, 200, 2, True, 208, 203, 43, 45), (70, 37, 256, 2, True, 264, 257, 40, 48),    # NT, B element by element
    (33, 40, 264, 2, False, 272, 48, 44, 56), (65, 37, 328, 3, False, 336, 41, 37, 39),    # NN, pieces and elements
    (64, 72, 520, 3, True, 528, 536, 80, 80), (32, 32, 128, 2, True, 136, 136, 33, 32)])   # NT, pieces
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_padded_pitches(dev, m, n, k, split, nt, lda, ldb, ldc, ldy, dtype):
    """Integers, exact in any order; NaN between the rows of the operands, what lies between those of the results stays."""
    from vkgrad_amd.kernels import Matmul
    rng = np.random.default_rng(m + k)
    a, b = rng.integers(-3, 4, (m, k)).astype(np.float32), rng.integers(-3, 4, (n, k) if nt else (k, n)).astype(np.float32)
    bias, c0 = rng.integers(-9, 10, n).astype(np.float32), rng.integers(-9, 10, (m, ldc)).astype(np.float32)

    def padded(x, pitch):
        p = np.full((x.shape[0], pitch), np.nan, np.float32)
        p[:, :x.shape[1]] = x
        return O.round_to(p, dtype)
    mm = Matmul(dev, trans_b=nt, dtype=dtype, tile=4, split_k=split)
    assert mm.statistics(m, n, k, lda=lda, ldb=ldb, ldc=ldc)["workgroupThreads"] == 64 * split
    pa, pb, y0 = padded(a, lda), padded(b, ldb), np.full((m, ldy), 7, np.uint16)
    ba, bb, bbias, bc, by = bufs = [dev.buffer(x.nbytes, "device") for x in (pa, pb, bias, c0, y0)]
    for buf, x in zip(bufs, (pa, pb, bias, c0, y0)):
        buf.upload(x)
    want = a @ (b.T if nt else b) + bias
    mm(ba, bb, bc, m, n, k, bias=bbias, accumulate=True, lda=lda, ldb=ldb, ldc=ldc)
    got = bc.download(np.float32, (m, ldc))
    assert np.array_equal(got[:, :n], want + c0[:, :n]) and np.array_equal(got[:, n:], c0[:, n:])
    mm(ba, bb, bc, m, n, k, bias=bbias, lda=lda, ldb=ldb, ldc=ldc, act="relu", y16=by, ldy=ldy)
    got, y = bc.download(np.float32, (m, ldc)), by.download(np.uint16, (m, ldy))
    assert np.array_equal(got[:, :n], want) and np.array_equal(got[:, n:], c0[:, n:]) and (y[:, n:] == 7).all()
    assert np.array_equal(y[:, :n], O.round_to(np.maximum(want, 0), dtype).view(np.uint16))
    for buf in bufs:
        buf.destroy()


@pytest.mark.parametrize("m,n,k,split,odd,taken", [
    (128, 512, 784, 5, "", True), (128, 10, 512, 4, "", True),          # the hidden and the last layer of the MNIST model
    (300, 768, 1536, 3, "", False), (128, 512, 1024, 4, "", False),     # eight and four K-blocks a slice
    (128, 512, 640, 2, "", True), (128, 512, 768, 2, "", True), (128, 512, 832, 2, "", False),
    (64, 2048, 4096, 8, "", False), (64, 2048, 1024, 8, "", True),
    (128, 37, 1536, 3, "", True), (128, 37, 1536, 6, "", True), (128, 37, 1920, 6, "", False),     # B element by element
    (64, 512, 768, 3, "nt", True), (64, 512, 960, 3, "nt", False), (64, 512, 1024, 8, "nt", True),
    (64, 512, 256, 2, "nt odd", True), (64, 512, 384, 2, "nt odd", False), (64, 512, 512, 8, "nt odd", True)])
def test_slices_of_many_k_blocks_stay_workgroups(dev, m, n, k, split, odd, taken):
    """A wavefront asks for four K-blocks at a time: 64 x 2048 x 4096 in eight slices of eight took 19.9 us and 10.9 as workgroups."""
    from vkgrad_amd.kernels import Matmul
    st = Matmul(dev, trans_b="nt" in odd, dtype="f16", tile=4, split_k=split).statistics(m, n, k, ldb=k + 1 if "odd" in odd else None)
    assert st["workgroupThreads"] == (64 * split if taken else 256)
