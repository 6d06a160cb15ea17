"""The backward pass of a linear layer in one launch (mg_gemm_backward): dW, the column sums of dy and dX next to each
other.  Integer operands, so that every sum is exact in any order; edges of the tiles, remainders of K, every kind of
kernel, K slices of both products, and the launches in turn that the library takes where it estimates them to be
faster.  What it picks is checked without a device."""

import ctypes as C

import numpy as np
import pytest

from oracle import ref_gemm as O
from vkgrad_amd import _lib as L
from vkgrad_amd.kernels import Matmul, linear_backward
from vkgrad_amd.vk import Graph, VkError, _check

KINDS = [  # rows, fin, fout, tile, split_w, split_x
    (64, 64, 64, 4, 1, 1), (65, 72, 136, 4, 1, 2), (1100, 136, 264, 4, 6, 2),          # 64 x 64, direct loads
    (128, 128, 128, 11, 1, 1), (520, 264, 392, 11, 3, 2), (1031, 136, 128, 11, 5, 1),  # 128 x 128
    (1, 1, 1, 4, 1, 1), (131, 77, 45, 4, 2, 1), (1100, 33, 10, 4, 3, 1), (640, 65, 513, 4, 1, 3),  # any alignment
    (1665, 384, 1152, L.MG_BACKWARD_AUTO, 0, 0), (300, 999, 37, L.MG_BACKWARD_AUTO, 0, 0), (513, 64, 72, L.MG_BACKWARD_APART, 0, 0),
]


def _args(bufs, rows, fin, fout, tile, split_w, split_x, dtype, form, sums, accumulate):
    gw = Matmul(None, trans_a=True, dtype=dtype)._args(bufs["x"], bufs["dy"], bufs["dw"], fin, fout, rows, 1, (0, 0, 0), None,
                                                       accumulate, None, None, None)
    gx = None
    if form == "nn":      # W stored (fout, fin), a tied head
        gx = Matmul(None, dtype=dtype)._args(bufs["dy"], bufs["w"], bufs["dx"], rows, fin, fout, 1, (0, 0, 0), None, False, None, None, None)
    elif form != "none":
        extra = dict(act="relu_grad", z=bufs["z"], y16=bufs["y"]) if form == "act" else {}
        gx = Matmul(None, trans_b=True, dtype=dtype)._args(bufs["dy"], bufs["w"], bufs["dx"], rows, fin, fout, 1, (0, 0, 0), None, False,
                                                           None, None, None, **extra)
    b = L.BackwardArgs()
    b.struct_size, b.tile, b.split_w, b.split_x = C.sizeof(b), tile, split_w, split_x
    b.dw = C.pointer(gw)
    if gx is not None:
        b.dx = C.pointer(gx)
    if sums:
        g = bufs["g32"] if sums == "f32" else bufs["dy"]
        b.g, b.db, b.rows, b.cols, b.g_f32, b.accumulate = g.ptr, bufs["db"].ptr, rows, fout, int(sums == "f32"), int(accumulate)
    return b


@pytest.mark.gpu
@pytest.mark.parametrize("form,sums,accumulate", [("plain", "16", False), ("act", "f32", False), ("nn", "", False), ("none", "f32", True),
                                                  ("plain", "16", True)])
@pytest.mark.parametrize("rows,fin,fout,tile,split_w,split_x", KINDS)
def test_exact_on_integers(dev, rows, fin, fout, tile, split_w, split_x, form, sums, accumulate):
    dtype = "f16" if (rows + len(form)) % 2 else "bf16"
    rng = np.random.default_rng(rows + fin)
    x, w, dy = (rng.integers(-3, 4, s).astype(np.float32) for s in ((rows, fin), (fout, fin) if form == "nn" else (fin, fout), (rows, fout)))
    z, g32 = rng.standard_normal((rows, fin)).astype(np.float32), rng.integers(-9, 10, (rows, fout)).astype(np.float32)
    bufs = {}
    for name, a in (("x", O.round_to(x, dtype)), ("w", O.round_to(w, dtype)), ("dy", O.round_to(dy, dtype)), ("z", z), ("g32", g32),
                    ("dw", np.full((fin, fout), 5, np.float32)), ("dx", np.full((rows, fin), 5, np.float32)),
                    ("y", np.zeros((rows, fin), np.uint16)), ("db", np.full(fout, 3, np.float32))):
        bufs[name] = dev.buffer(a.nbytes + 16, "device")   # (a piece past a ragged edge lies inside)
        bufs[name].upload(a)
    b = _args(bufs, rows, fin, fout, tile, split_w, split_x, dtype, form, sums, accumulate)
    _check(dev._lib.mg_gemm_backward(dev._ctx, C.byref(b)), "backward")
    dev.sync()
    get = lambda name, t, shape: bufs[name].download(t, shape)
    assert np.array_equal(get("dw", np.float32, (fin, fout)), x.T @ dy + (5 if accumulate else 0))
    if form != "none":
        want = dy @ (w if form == "nn" else w.T)
        if form == "act":
            want = want * (z > 0)
            got16 = get("y", np.uint16, (rows, fin))
            assert np.array_equal(O.widen(got16.view(np.float16) if dtype == "f16" else got16, dtype), O.widen(O.round_to(want, dtype), dtype))
        assert np.array_equal(get("dx", np.float32, (rows, fin)), want)
    db = (g32 if sums == "f32" else dy).sum(0) + (3 if accumulate else 0) if sums else np.full(fout, 3)
    assert np.array_equal(get("db", np.float32, (fout,)), db)
    for buf in bufs.values():
        buf.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("tile,split_w,split_x,pad", [(4, 3, 2, 8), (11, 2, 2, 8), (21, 2, 2, 8), (4, 2, 1, 1), (4, 1, 3, 5)])
@pytest.mark.parametrize("form", ["bias", "accumulate", "res", "act"])
def test_padded_pitches_and_what_dx_adds(dev, tile, split_w, split_x, pad, form):
    """Every matrix with a pitch of its own, NaN between the rows of the operands; dX onto its bias, onto itself, onto a residual, or
    times the derivative with its column sums."""
    if tile == 21 and form == "act":
        form = "narrow"    # (those tiles have no derivative in one launch)
    rows, fin, fout = (528, 264, 392) if pad == 8 else (301, 77, 139)
    dtype = "f16" if (split_w + len(form)) % 2 else "bf16"
    rng = np.random.default_rng(tile + pad)
    data, host, bufs, pitch = {}, {}, {}, {}
    shapes = dict(x=(rows, fin), w=(fin, fout), dy=(rows, fout), g32=(rows, fout), dw=(fin, fout), dx=(rows, fin), res=(rows, fin), z=(rows, fin),
                  y=(rows, fin), bias=(1, fin), cs=(1, fin), db=(1, fout))
    for i, (name, (r, c)) in enumerate(shapes.items()):
        ld = pitch[name] = c if name in ("g32", "bias", "cs", "db") else c + pad * (1 + i % 3)
        p = np.full((r, ld), np.nan if name in ("x", "w", "dy", "res", "z") else 5, np.float32)
        data[name] = p[:, :c] = rng.integers(-3, 4, (r, c))
        host[name] = O.round_to(p, dtype) if name in ("x", "w", "dy") else np.full((r, ld), 7, np.uint16) if name == "y" else p
        bufs[name] = dev.buffer(host[name].nbytes + 16, "device")
        bufs[name].upload(host[name])
    B, P = bufs, pitch
    gw = Matmul(None, trans_a=True, dtype=dtype)._args(B["x"], B["dy"], B["dw"], fin, fout, rows, 1, (0, 0, 0), None, True, P["x"], P["dy"], P["dw"])
    extra = dict(bias=dict(bias=B["bias"]), accumulate=dict(accumulate=True), res=dict(res=B["res"], ldr=P["res"]),
                 act=dict(act="relu_grad", z=B["z"], ldz=P["z"], y16=B["y"], ldy=P["y"], colsum=B["cs"]), narrow=dict(y16=B["y"], ldy=P["y"]))[form]
    gx = Matmul(None, trans_b=True, dtype=dtype)._args(B["dy"], B["w"], B["dx"], rows, fin, fout, 1, (0, 0, 0), **{
        **dict(bias=None, accumulate=False, lda=P["dy"], ldb=P["w"], ldc=P["dx"]), **extra})
    b = L.BackwardArgs()
    b.struct_size, b.tile, b.split_w, b.split_x, b.dw, b.dx = C.sizeof(b), tile, split_w, split_x, C.pointer(gw), C.pointer(gx)
    b.g, b.db, b.rows, b.cols, b.g_f32 = B["g32"].ptr, B["db"].ptr, rows, fout, 1
    _check(dev._lib.mg_gemm_backward(dev._ctx, C.byref(b)), "backward")
    dev.sync()

    def get(name):   # and what lies between the rows is as it was
        got = bufs[name].download(host[name].dtype, host[name].shape)
        c = shapes[name][1]
        assert np.array_equal(got[:, c:], host[name][:, c:])
        return got[:, :c]
    assert np.array_equal(get("dw"), data["dw"] + data["x"].T @ data["dy"])
    assert np.array_equal(get("db"), data["g32"].sum(0, keepdims=True))
    want = data["dy"] @ data["w"].T
    want += dict(bias=data["bias"], accumulate=data["dx"], res=data["res"]).get(form, 0)
    if form == "act":
        want *= data["z"] > 0
        assert np.array_equal(get("cs"), data["cs"] + want.sum(0, keepdims=True))
    if form in ("act", "narrow"):
        y = get("y")
        assert np.array_equal(O.widen(y.view(np.float16) if dtype == "f16" else y, dtype), O.widen(O.round_to(want.astype(np.float32), dtype), dtype))
    assert np.array_equal(get("dx"), want)
    for buf in bufs.values():
        buf.destroy()


class _Mem:
    host_visible, size = False, 1 << 40

    def __init__(self, ptr):
        self.ptr = ptr


def test_what_is_picked():
    lib = L.load()

    def pick(rows, fin, fout, form="plain", tile=L.MG_BACKWARD_AUTO, **at):
        names = ("x", "w", "dy", "dw", "dx", "y", "z", "g32", "db")
        bufs = {n: _Mem(at.get(n, (i + 1) << 33)) for i, n in enumerate(names)}
        b = _args(bufs, rows, fin, fout, tile, 1, 1, "bf16", form, "16", False)
        out = [C.c_int() for _ in range(3)]
        assert lib.mg_backward_pick(C.byref(b), 256, *(C.byref(o) for o in out)) == L.MG_OK
        return tuple(o.value for o in out)

    assert pick(128, 64, 256) == (4, 1, 1)
    assert pick(4096, 1024, 1024)[0] == 11
    assert pick(16384, 1024, 50304)[0] == L.MG_BACKWARD_APART      # 256 x 256 tiles
    assert pick(128, 64, 256, tile=L.MG_BACKWARD_APART)[0] == L.MG_BACKWARD_APART
    assert pick(128, 77, 45) == (4, 1, 1) and pick(128, 77, 45, tile=11)[0] == L.MG_BACKWARD_APART   # no direct loads
    # what one product writes is read or written by another: in turn, as mg_gemm would
    for clash in (dict(dx=3 << 33), dict(dx=(1 << 33) + 64), dict(dw=(2 << 33) - 64), dict(db=4 << 33), dict(db=3 << 33)):
        assert pick(128, 64, 256, **clash)[0] == L.MG_BACKWARD_APART, clash


@pytest.mark.parametrize("which", ["dw", "dx"])
def test_refused_where_it_is_recorded(which):
    """A product that the library refuses (a misaligned result) never enters a graph, as with a product by itself."""
    class Dev:
        _lib, _ctx = L.load(), None

    g = Graph(Dev(), "g")
    bufs = {n: _Mem((i + 1) << 33) for i, n in enumerate(("x", "w", "dy", "dw", "dx"))}

    def record():
        linear_backward(Dev(), (Matmul(Dev(), trans_a=True), (bufs["x"], bufs["dy"], bufs["dw"], 64, 64, 32), {}),
                        (Matmul(Dev(), trans_b=True), (bufs["dy"], bufs["w"], bufs["dx"], 32, 64, 64), {}), graph=g)

    record()
    assert g.n_dispatch == 1
    bufs[which] = _Mem((7 << 33) + 2)
    with pytest.raises(VkError):
        record()
    assert g.n_dispatch == 1


def test_named_plans_bind():
    """A tile or K split that a product names is what it runs with, in one launch or by itself; MG_BACKWARD_REPLAN is for plans that
    were measured on a product by itself."""
    lib = L.load()

    def pick(rows, fin, fout, how=L.MG_BACKWARD_AUTO, w=(-1, 0), x=(-1, 0)):
        bufs = {n: _Mem((i + 1) << 33) for i, n in enumerate(("x", "w", "dy", "dw", "dx", "y", "z", "g32", "db"))}
        b = _args(bufs, rows, fin, fout, how, 0, 0, "bf16", "plain", "16", False)
        (b.dw.contents.tile, b.dw.contents.split_k), (b.dx.contents.tile, b.dx.contents.split_k) = w, x
        out = [C.c_int() for _ in range(3)]
        assert lib.mg_backward_pick(C.byref(b), 256, *(C.byref(o) for o in out)) == L.MG_OK
        return tuple(o.value for o in out)

    apart = (L.MG_BACKWARD_APART, 0, 0)
    for shape, w in (((8192, 768, 3072), (21, 5)), ((1665, 384, 1152), (11, 1)), ((128, 64, 256), (3, 2)), ((4096, 1024, 1024), (11, 3))):
        free, bound = pick(*shape), pick(*shape, w=w)
        assert free[0] >= 0 and free[:2] != w
        assert bound == apart or bound[:2] == w
        assert pick(*shape, how=L.MG_BACKWARD_REPLAN, w=w)[0] >= 0     # (compared with what the named plan takes)
    assert pick(128, 64, 256, w=(3, 2)) == apart                       # no one-launch kernel has that tile
    assert pick(1665, 384, 1152, w=(4, 2), x=(4, 1)) == (4, 2, 1)
    assert pick(1665, 384, 1152, w=(4, 1), x=(11, 1)) == apart
    assert pick(1665, 384, 1152, x=(-1, 2))[2] in (0, 2) and pick(1665, 384, 1152, w=(-1, 2))[1] in (0, 2)
    assert pick(8192, 768, 3072, x=(21, 2)) == apart


def test_whose_plans_bind(monkeypatch):
    """Plans from the shipped table give way to the one launch, plans that the caller or the tuner named do not."""
    from vkgrad_amd import kernels as K
    from vkgrad_amd.autograd import Ctx

    class Dev:
        _lib, _ctx, name, compute_units = L.load(), None, "fake", 256

    entry = {"tile_id": 11, "split_k": 3, "group_m": 4}
    key = K.tune_key("fake", 64, 64, 32, True, False)
    bufs = {n: _Mem((i + 1) << 33) for i, n in enumerate(("x", "w", "dy", "dw", "dx"))}

    def recorded(mw, mx):
        g = Graph(Dev(), "g")
        linear_backward(Dev(), (mw, (bufs["x"], bufs["dy"], bufs["dw"], 64, 64, 32), {}),
                        (mx, (bufs["dy"], bufs["w"], bufs["dx"], 32, 64, 64), {}), graph=g)
        return g._thunks[0].__defaults__[0].tile

    plain = Matmul(Dev(), trans_b=True)
    assert recorded(Matmul(Dev(), trans_a=True), plain) == L.MG_BACKWARD_AUTO
    assert recorded(Matmul(Dev(), trans_a=True, tile=11), plain) == L.MG_BACKWARD_AUTO
    for shipped, user, want in (({key: entry}, {}, L.MG_BACKWARD_REPLAN), ({}, {key: entry}, L.MG_BACKWARD_AUTO)):
        monkeypatch.setattr(K, "_shipped_table", lambda t=shipped: t)
        monkeypatch.setattr(K, "_load_cache", lambda path=None, t=user: t)
        ctx = Ctx.__new__(Ctx)
        ctx.dev, ctx.tune, ctx.dtype, ctx._mm = Dev(), False, "f16", {}
        mm = ctx.matmul(64, 64, 32, trans_a=True)
        assert mm.tile == 11 and recorded(mm, plain) == want
        assert recorded(mm, Matmul(Dev(), trans_b=True, split_k=2)) == L.MG_BACKWARD_AUTO


def test_how_slices_of_a_shipped_plan_meet(monkeypatch):
    """Slices that add with atomics keep a pass in turn where the caller asked for them, not where a shipped plan has them."""
    from vkgrad_amd import kernels as K
    from vkgrad_amd.autograd import Ctx

    class Dev:
        _lib, _ctx, name, compute_units = L.load(), None, "fake", 256

    key = K.tune_key("fake", 1024, 256, 16384, True, False)
    table = {key: {"tile_id": 14, "split_k": 15, "group_m": 4, "atomic_split": True}}
    monkeypatch.setattr(K, "_shipped_table", lambda: table)
    monkeypatch.setattr(K, "_load_cache", lambda path=None: {})
    ctx = Ctx.__new__(Ctx)
    ctx.dev, ctx.tune, ctx.dtype, ctx._mm = Dev(), False, "f16", {}
    shipped = ctx.matmul(1024, 256, 16384, trans_a=True)
    assert shipped.atomic_split and shipped.from_table
    bufs = {n: _Mem((i + 1) << 33) for i, n in enumerate(("x", "w", "dy", "dw", "z", "y"))}

    def pick(mw, mx=None):
        g = Graph(Dev(), "g")
        linear_backward(Dev(), (mw, (bufs["x"], bufs["dy"], bufs["dw"], 1024, 256, 16384), {}),
                        (mx or Matmul(Dev(), trans_b=True), (bufs["dy"], bufs["w"], None, 16384, 1024, 256),
                         dict(act="gelu_grad", z=bufs["z"], y16=bufs["y"])), graph=g)
        ba, out = g._thunks[0].__defaults__[0], [C.c_int() for _ in range(3)]
        assert Dev._lib.mg_backward_pick(C.byref(ba), 256, *(C.byref(o) for o in out)) == L.MG_OK
        return ba.dw.contents.flags & L.MG_FLAG_SPLITK_ATOMIC, out[0].value

    flag, tile = pick(shipped)
    assert flag == 0 and tile in (4, 11)
    named = Matmul(Dev(), trans_a=True, tile=14, split_k=15, atomic_split=True)
    assert pick(named) == (L.MG_FLAG_SPLITK_ATOMIC, L.MG_BACKWARD_APART)


def test_keywords_of_a_product_arrive():
    """Every keyword of Matmul's call reaches the product, with its buffer; others are refused."""
    class Dev:
        _lib, _ctx = L.load(), None

    bufs = {n: _Mem((i + 1) << 33) for i, n in enumerate(("x", "w", "dy", "dw", "dx", "res", "bias"))}

    def record(graph=True, **kw):
        g = Graph(Dev(), "g") if graph else None
        linear_backward(Dev(), (Matmul(Dev(), trans_a=True), (bufs["x"], bufs["dy"], bufs["dw"], 64, 64, 32), dict(ldc=72, accumulate=True)),
                        (Matmul(Dev(), trans_b=True), (bufs["dy"], bufs["w"], bufs["dx"], 32, 64, 64), kw), graph=g)
        return g

    g = record(res=bufs["res"], ldr=80, bias=bufs["bias"], lda=96, ldb=104, ldc=112)
    ba = g._thunks[0].__defaults__[0]
    dw, dx = ba.dw.contents, ba.dx.contents
    assert (dw.lda, dw.ldb, dw.ldc, dw.beta) == (64, 64, 72, 1)
    assert (dx.lda, dx.ldb, dx.ldc, dx.beta, dx.res, dx.ldr, dx.bias) == (96, 104, 112, 1, bufs["res"].ptr, 80, bufs["bias"].ptr)
    assert all(id(b) in g._buffers for b in bufs.values())
    assert record(side=True)._thunks[0].__defaults__[0].dx.contents.flags & L.MG_FLAG_SIDE_STREAM
    with pytest.raises(VkError):
        record(graph=False, side=True)
    with pytest.raises(TypeError):
        record(acumulate=True)
    with pytest.raises(VkError):
        record(tri="diagonal")
