"""The any-alignment loads (dword addresses, odd pieces moved by 16 bits): every register-staged tile, both operands odd, one of
them, neither; bases in the middle of a dword; tiles at the edges, where pieces of columns run on into the next row; K around whole
blocks.  The elements around every row are NaN, the data small integers: results are exact or wrong."""

import ctypes as C

import numpy as np
import pytest

from oracle import ref_gemm as O

pytestmark = pytest.mark.gpu

LAYOUT_ID = {"NN": 0, "NT": 1, "TN": 2}
# m, n, k; a pitch is the number of columns plus a pad
SIZES = [(64, 64, 64), (65, 63, 129), (129, 257, 191), (300, 5, 192), (7, 130, 200), (257, 255, 321), (128, 128, 448)]
PADS = [(0, 0), (1, 0), (0, 1), (3, 9), (17, 16)]


@pytest.fixture(scope="module")
def dev():
    from vkgrad_amd.vk import Device
    d = Device(0)
    yield d
    d.destroy()


def _put(dev, x, pitch, shift):
    """x in rows of `pitch` elements, `shift` elements into a buffer, NaN around it: (buffer, address)."""
    flat = np.full(shift + x.shape[0] * pitch + 64, 0x7FC0, np.uint16)
    rows = flat[shift:shift + x.shape[0] * pitch].reshape(x.shape[0], pitch)
    rows[:, :x.shape[1]] = x.view(np.uint16)
    buf = dev.buffer(flat.nbytes, "device")
    buf.upload(flat)
    return buf, buf.ptr + 2 * shift


@pytest.mark.parametrize("layout", sorted(LAYOUT_ID))
@pytest.mark.parametrize("tile", range(9))
def test_odd_pieces(dev, layout, tile):
    from vkgrad_amd import _lib as L
    ta, tb = O.LAYOUTS[layout]
    for case, (m, n, k) in enumerate(SIZES):
        a, b = O.make_operands(m, n, k, ta, tb, "bf16", seed=case, integer=True)
        ref = O.ref_gemm(a, b, ta, tb, "bf16")
        for j, (pa, pb) in enumerate(PADS):
            shift_a, shift_b = (case + j) % 3, (2 * case + j) % 4
            lda, ldb = a.shape[1] + pa, b.shape[1] + pb
            (ba, at), (bb, bt), bc = _put(dev, a, lda, shift_a), _put(dev, b, ldb, shift_b), dev.buffer(m * n * 4, "device")
            for split in (1, 2):
                g = L.GemmArgs()
                g.struct_size, g.layout, g.dtype, g.tile, g.split_k = C.sizeof(L.GemmArgs), LAYOUT_ID[layout], 1, tile, split
                g.m, g.n, g.k, g.a, g.b, g.c, g.lda, g.ldb, g.ldc, g.nbatch = m, n, k, at, bt, bc.ptr, lda, ldb, n, 1
                bc.upload(np.full((m, n), np.nan, np.float32))
                assert dev._lib.mg_gemm(dev._ctx, C.byref(g)) == 0
                assert np.array_equal(bc.download(np.float32, (m, n)), ref), (m, n, k, lda, ldb, shift_a, shift_b, split)
            for x in (ba, bb, bc):
                x.destroy()


@pytest.mark.parametrize("layout,m,n,k,lda,ldb", [
    ("NN", 5, 70, 130, (1 << 21) + 1, 71), ("NN", 70, 33, 66, 67, 1 << 21), ("NT", 3, 4, 200, (1 << 21) - 1, (1 << 21) + 1),
    ("TN", 6, 65, 66, (1 << 21) + 3, 65), ("TN", 6, 65, 66, (1 << 21) - 1, 65)])
def test_pitches_on_both_sides_of_32_bit_offsets(dev, layout, m, n, k, lda, ldb):
    """Whole K-blocks are loaded at 32-bit offsets from their first dword; pitches of 2^21 elements and more go the careful way."""
    from vkgrad_amd import _lib as L
    ta, tb = O.LAYOUTS[layout]
    a, b = O.make_operands(m, n, k, ta, tb, "bf16", seed=m, integer=True)
    ref = O.ref_gemm(a, b, ta, tb, "bf16")
    (ba, at), (bb, bt), bc = _put(dev, a, lda, 1), _put(dev, b, ldb, 1), dev.buffer(m * n * 4, "device")
    for tile in (3, 4):
        g = L.GemmArgs()
        g.struct_size, g.layout, g.dtype, g.tile, g.split_k = C.sizeof(L.GemmArgs), LAYOUT_ID[layout], 1, tile, 1
        g.m, g.n, g.k, g.a, g.b, g.c, g.lda, g.ldb, g.ldc, g.nbatch = m, n, k, at, bt, bc.ptr, lda, ldb, n, 1
        bc.upload(np.full((m, n), np.nan, np.float32))
        assert dev._lib.mg_gemm(dev._ctx, C.byref(g)) == 0
        assert np.array_equal(bc.download(np.float32, (m, n)), ref), tile
    for x in (ba, bb, bc):
        x.destroy()
