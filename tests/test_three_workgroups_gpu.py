"""The 128 x 128 tile with K-blocks of 32 in its form for three workgroups a CU, which products of more than two
workgroups for a CU run: integer operands, so that every sum is exact, against the same product in 64 x 64 tiles and a CPU product."""

import ctypes as C

import numpy as np
import pytest

from oracle import ref_gemm as O
from vkgrad_amd import _lib as L
from vkgrad_amd.kernels import Matmul, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["plain", "accumulate", "res", "gelu", "relu", "narrow", "grad", "split", "split_sum"])
@pytest.mark.parametrize("layout,m,n,k", [("nn", 3001, 2936, 72), ("nt", 2945, 3000, 96), ("tn", 3008, 2952, 33), ("nn", 4096, 2176, 64)])
def test_same_as_small_tiles(dev, layout, m, n, k, form):
    if layout == "tn" and form in ("gelu", "relu", "narrow", "grad"):
        pytest.skip("no fused 16-bit output in this layout")
    if form.startswith("split"):
        m, n, k = m // 2 // 8 * 8, n // 2 // 8 * 8, 32 * (24 if form == "split_sum" else 8) + k
    slices = {"split": 4, "split_sum": 6}.get(form, 1)   # (six of these tiles: from there on sums have a launch of their own)
    assert -(-m // 128) * -(-n // 128) * slices > 2 * dev.compute_units   # or it is the form for two
    dtype = "f16" if k % 64 else "bf16"
    rng = np.random.default_rng(m + n)
    a, b = rng.integers(-3, 4, (m, k)).astype(np.float32), rng.integers(-3, 4, (k, n)).astype(np.float32)
    z, bias = rng.standard_normal((m, n)).astype(np.float32), rng.integers(-9, 10, n).astype(np.float32)
    ta, tb = layout == "tn", layout == "nt"
    pad = lambda x: np.pad(x, ((0, 0), (0, -x.shape[1] % 8)))     # whole 16-byte pieces
    ah, bh = pad(np.ascontiguousarray(a.T) if ta else a), pad(np.ascontiguousarray(b.T) if tb else b)
    bufs = {}
    for name, x in (("a", O.round_to(ah, dtype)), ("b", O.round_to(bh, dtype)), ("z", z), ("bias", bias)):
        bufs[name] = dev.buffer(x.nbytes + 16, "device")
        bufs[name].upload(x)
    kw = dict(plain={}, accumulate=dict(accumulate=True), res=dict(res=bufs["z"]), split={}, split_sum={})
    out = []
    for tile in (14, 3, 4):   # (tile 3: with the fused outputs the same kernel)
        c, y = dev.buffer(m * n * 4, "device"), dev.buffer(m * n * 2, "device")
        c.upload(np.full((m, n), 5, np.float32))
        y.upload(np.zeros((m, n), np.uint16))
        extra = kw.get(form) or dict(gelu=dict(act="gelu", y16=y), relu=dict(act="relu", y16=y), narrow=dict(y16=y),
                                     grad=dict(act="gelu_grad", z=bufs["z"], y16=y)).get(form, {})
        extra = dict(bias=None if form == "grad" else bufs["bias"], accumulate=False, lda=ah.shape[1], ldb=bh.shape[1], ldc=n) | extra
        mm = Matmul(dev, trans_a=ta, trans_b=tb, dtype=dtype, tile=tile, split_k=slices if tile != 4 else 1)
        ga = mm._args(bufs["a"], bufs["b"], c, m, n, k, 1, (0, 0, 0), **extra)
        assert tile != 14 or mm.plan(m, n, k, lda=ah.shape[1], ldb=bh.shape[1])[:2] == (14, slices)
        # slices that meet in the workgroup that is last, or in a launch of their own
        ga.flags = ga.flags & ~L.MG_FLAG_SPLITK_SUM if form == "split" else ga.flags | L.MG_FLAG_SPLITK_SUM if form == "split_sum" else ga.flags
        _check(dev._lib.mg_gemm(dev._ctx, C.byref(ga)), "gemm")
        dev.sync()
        out.append((c.download(np.uint32, (m, n)), y.download(np.uint16, (m, n))))
        c.destroy(), y.destroy()
    for c, y in out[:2]:
        assert np.array_equal(c, out[2][0]) and np.array_equal(y, out[2][1])
    if form != "grad":
        want = a @ b + bias + dict(accumulate=5, res=z).get(form, 0)
        assert np.array_equal(out[0][0].view(np.float32), want.astype(np.float32))
    for x in bufs.values():
        x.destroy()


@pytest.mark.parametrize("k", [40, 88, 96, 1000])
@pytest.mark.parametrize("layout", ["nn", "nt"])
def test_remainders_of_k_in_the_fused_form(dev, layout, k):
    """The fused form multiplies K % 32 first, the kernel with K-blocks of 64 that it stands in for K % 64: from 32 on
    not the same, so that sums of products that do not come out whole round otherwise.  Each is within what K adds in
    f32 allow, rounded or cut off, and where K % 64 is below 32 they are the same bits."""
    m, n, dtype = 2950, 3000, "bf16"
    rng = np.random.default_rng(k)
    a, b = (O.round_to(rng.standard_normal(x).astype(np.float32), dtype) for x in ((m, k), (n, k) if layout == "nt" else (k, n)))
    bufs = [dev.buffer(x.nbytes + 16, "device") for x in (a, b)]
    for buf, x in zip(bufs, (a, b)):
        buf.upload(x)
    c, y = dev.buffer(m * n * 4, "device"), dev.buffer(m * n * 2, "device")
    rows = (1408, m)   # 264 tiles of 128 x 128, and 576: two workgroups a CU at the most, and more
    assert -(-rows[0] // 128) * -(-n // 128) <= 2 * dev.compute_units < -(-rows[1] // 128) * -(-n // 128)
    got = []
    for r in rows:
        c.upload(np.full((m, n), np.nan, np.float32))
        ga = Matmul(dev, trans_b=layout == "nt", dtype=dtype, tile=3, split_k=1)._args(
            *bufs, c, r, n, k, 1, (0, 0, 0), bias=None, accumulate=False, lda=None, ldb=None, ldc=None, act="gelu", y16=y)
        _check(dev._lib.mg_gemm(dev._ctx, C.byref(ga)), "gemm")
        dev.sync()
        got.append(c.download(np.float32, (m, n))[:r])
    a64, b64 = (O.widen(x, dtype).astype(np.float64) for x in (a, b))
    b64 = b64.T if layout == "nt" else b64
    exact, bound = a64 @ b64, 2.0 ** -23 * k * (np.abs(a64) @ np.abs(b64))   # any order of K adds in f32
    for z in got:
        assert (np.abs(z - exact[:len(z)]) <= bound[:len(z)]).all()
    if k % 64 < 32:
        assert np.array_equal(got[1][:rows[0]], got[0])
    for x in (*bufs, c, y):
        x.destroy()
