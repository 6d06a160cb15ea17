"""Column sums of one chunk of rows and of several, two matrices to a launch, and staging copies from host memory: at the edges of
their row batches, columns and pieces.  Integers: exact in any order."""

import ctypes as C

import numpy as np
import pytest

from oracle import ref_gemm as O
from vkgrad_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrow,ncol", [(1, 1), (513, 15), (1000, 16), (1024, 2049), (769, 33), (512, 64), (2000, 70)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_column_sums(dev, nrow, ncol, accumulate):
    from vkgrad_amd.tkernels import make_transformer_kernels
    TK = make_transformer_kernels(dev, "bf16")
    rng = np.random.default_rng(nrow + ncol)
    a, b = (rng.integers(-4, 5, (nrow, ncol)).astype(np.float32) for _ in range(2))
    s0 = rng.integers(-9, 10, ncol).astype(np.float32)
    b32, ba, bb, sa, sb = (dev.buffer(n, "device") for n in (a.nbytes, a.nbytes // 2, a.nbytes // 2, 4 * ncol, 4 * ncol))
    b32.upload(a)
    ba.upload(O.round_to(a, "bf16"))
    bb.upload(O.round_to(b, "bf16"))
    keep = s0 if accumulate else 0
    for s in (sa, sb):
        s.upload(s0)
    assert dev._lib.mg_ew_col_sum(dev._ctx, b32.ptr, sa.ptr, ncol, nrow, int(accumulate)) == L.MG_OK
    assert np.array_equal(sa.download(np.float32, (ncol,)), a.sum(0) + keep)
    sa.upload(s0)
    TK["col_sum16_pair"]([ba, sa, bb, sb], ncol, nrow, accumulate)
    assert np.array_equal(sa.download(np.float32, (ncol,)), a.sum(0) + keep)
    assert np.array_equal(sb.download(np.float32, (ncol,)), b.sum(0) + keep)
    for x in (b32, ba, bb, sa, sb):
        x.destroy()


@pytest.mark.parametrize("kind", ["shared", "device"])
@pytest.mark.parametrize("sizes", [(1,), (15, 16, 17), (16384, 262144), (262145, 5), (3000001, 4098)])
def test_staging_copies(dev, sizes, kind):
    rng = np.random.default_rng(sum(sizes))
    data = [rng.integers(0, 256, n, dtype=np.uint8) for n in sizes]
    src, dst = [dev.buffer(n + 16, kind) for n in sizes], [dev.buffer(n + 16, "device") for n in sizes]
    for s, d, x in zip(src, dst, data):
        s.upload(np.concatenate([x, np.full(16, 7, np.uint8)]))
        d.upload(np.full(x.size + 16, 9, np.uint8))
    n = len(sizes)
    rc = dev._lib.mg_ew_copy_multi(dev._ctx, (C.c_void_p * n)(*[d.ptr for d in dst]), (C.c_void_p * n)(*[s.ptr for s in src]),
                                   (C.c_int64 * n)(*sizes), n)
    assert rc == L.MG_OK
    for d, x in zip(dst, data):
        got = d.download(np.uint8, (x.size + 16,))
        assert np.array_equal(got[:x.size], x) and (got[x.size:] == 9).all()   # not a byte more
    for b in src + dst:
        b.destroy()


def test_staging_form_follows_the_source(dev):
    """The few workgroups that suit a long aligned host buffer are not what other copies get: 3 MB that is aligned to 4 bytes took
    four times as long as aligned 3 MB with them (241 and 61 us, 64 without), 6 MB in HBM three times (18.7 and 5.5 us)."""
    def us(calls):
        def launch():
            for dst, src, n in calls:
                one = (C.c_void_p * 1)(dst), (C.c_void_p * 1)(src), (C.c_int64 * 1)(n)
                assert dev._lib.mg_ew_copy_multi(dev._ctx, *one, 1) == L.MG_OK
        g = dev.graph("copies")
        g.record(launch, [])
        g.finish()
        g.time(3)
        t = float(np.median(g.time(15))) * 1e6 / len(calls)
        g.destroy()
        return t
    n = 3 << 20
    host, hbm, dst = dev.buffer(n + 64, "shared"), dev.buffer(2 * n, "device"), dev.buffer(2 * n, "device")
    aligned, odd = (us([(dst.ptr + off, host.ptr + off, n)] * 8) for off in (0, 4))
    inside = us([(dst.ptr, hbm.ptr, 2 * n)] * 8)
    few = us([(dst.ptr, hbm.ptr, 1024)] * 8)
    for b in (host, hbm, dst):
        b.destroy()
    assert odd <= 2 * aligned
    assert inside - few <= 6     # 12 MB moved: 2 us at 6 TB/s, 13 in the form that walks
