"""The 128 x 128 tile with K-blocks of 32 in its form for three workgroups a CU, which products of more than two
workgroups for a CU run: integer operands, so that every sum is exact, against the same product in 64 x 64 tiles and a CPU product."""

import ctypes as C

import numpy as np
import pytest

from oracle import ref_gemm as O
from vkgrad_amd.kernels import Matmul, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["plain", "accumulate", "res", "gelu", "relu", "narrow", "grad", "split"])
@pytest.mark.parametrize("layout,m,n,k", [("nn", 3001, 2936, 72), ("nt", 2945, 3000, 96), ("tn", 3008, 2952, 33), ("nn", 4096, 2176, 64)])
def test_same_as_small_tiles(dev, layout, m, n, k, form):
    if layout == "tn" and form in ("gelu", "relu", "narrow", "grad"):
        pytest.skip("no fused 16-bit output in this layout")
    if form == "split":
        m, n, k = m // 2 // 8 * 8, n // 2 // 8 * 8, 32 * 8 + k
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
    kw = dict(plain={}, accumulate=dict(accumulate=True), res=dict(res=bufs["z"]), split={})
    out = []
    for tile in (14, 3, 4):   # (tile 3: with the fused outputs the same kernel)
        c, y = dev.buffer(m * n * 4, "device"), dev.buffer(m * n * 2, "device")
        c.upload(np.full((m, n), 5, np.float32))
        y.upload(np.zeros((m, n), np.uint16))
        extra = kw.get(form) or dict(gelu=dict(act="gelu", y16=y), relu=dict(act="relu", y16=y), narrow=dict(y16=y),
                                     grad=dict(act="gelu_grad", z=bufs["z"], y16=y)).get(form, {})
        extra = dict(bias=None if form == "grad" else bufs["bias"], accumulate=False, lda=ah.shape[1], ldb=bh.shape[1], ldc=n) | extra
        mm = Matmul(dev, trans_a=ta, trans_b=tb, dtype=dtype, tile=tile, split_k=3 if form == "split" and tile != 4 else 1)
        ga = mm._args(bufs["a"], bufs["b"], c, m, n, k, 1, (0, 0, 0), **extra)
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
