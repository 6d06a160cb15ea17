"""GEMM objects, tile table, autotuner and the companion elementwise kernels.

Call surface of the reference's kernels.py (Matmul: /root/reference/kernels.py:232-315,
CONFIGS: 326-331, warmup: 353-381, autotune_matmul: 450-603, Elementwise and
make_kernels: 668-862) over libmigemm.so.  Differences a caller can see:

  * any positive M, N, K is legal (the reference refuses non-tile-multiples,
    kernels.py:271-276);
  * keyword-only extensions on a Matmul call: bias=, accumulate=, lda/ldb/ldc=;
    and on its constructor: dtype= ("f16" | "bf16"), tile=, split_k=;
  * eager calls are timed with HIP events on the device, not host wall clock.
"""

import ctypes as C
import json
import os
import time

import numpy as np

from . import _lib as L
from .vk import VkError, _check

TILE = 32  # MFMA accumulator tile edge (v_mfma_f32_32x32x16); the reference's is 16


def _tiles():
    lib = L.load()
    out = []
    for i in range(lib.mg_tile_count()):
        t = L.Tile()
        _check(lib.mg_tile_info(i, C.byref(t)), "tile table")
        out.append(dict(id=t.id, bm=t.bm, bn=t.bn, bk=t.bk, waves_m=t.waves_m, waves_n=t.waves_n,
                        threads=t.threads, lds_bytes=t.lds_bytes, stages=t.stages, fallback=t.fallback, persistent=t.persistent,
                        name=t.name.decode()))
    return out


# The tile table the tuner walks; one dict per block tile built into the library.
CONFIGS = _tiles()


def layout_of(trans_a, trans_b):
    if trans_a and trans_b:
        raise VkError("the (trans_a, trans_b) = (True, True) layout is not provided: no call site uses it")
    return L.MG_TN if trans_a else (L.MG_NT if trans_b else L.MG_NN)


def _nearest_tile(bm, bn):
    """Tile of the table closest to a requested bm x bn (log-distance)."""
    best = min(CONFIGS, key=lambda t: abs(np.log2(t["bm"] / bm)) + abs(np.log2(t["bn"] / bn)))
    return best["id"]


class Matmul:
    """One GEMM configuration: C[m,n] f32 = op(A) @ op(B), 16-bit inputs.

    Positional arguments follow the reference (sg, wm, wn described a
    sg*wm*16 x wn*16 block tile there); here they select the nearest tile of the
    library's table, tile= selects one by id, and with neither the built-in
    picker chooses per call.
    """

    def __init__(self, dev, sg=None, wm=None, wn=None, trans_a=False, trans_b=False,
                 capture_stats=False, lds=True, bk=64, batched=False, acc16=False,
                 group_m=0, *, tile=None, dtype="f16", split_k=0, atomic_split=False, xcd_rotate=None):
        if acc16:
            raise VkError("acc16 (f16 output) is not provided: no call site of the path uses it")
        if dtype not in L.DTYPES:
            raise VkError(f"unknown dtype {dtype!r}; use 'f16' or 'bf16'")
        self.dev = dev
        self.sg, self.wm, self.wn = sg, wm, wn
        self.trans_a, self.trans_b = bool(trans_a), bool(trans_b)
        self.layout = layout_of(trans_a, trans_b)
        self.lds, self.bk, self.batched = True, bk, bool(batched)
        self.acc16 = False
        self.group_m = int(group_m)
        self.dtype = dtype
        self.split_k = int(split_k)
        self.atomic_split = bool(atomic_split)   # K slices add into C with atomics, not via the workspace
        # walk of the XCDs over their shares of the tiles: True rotated, False in step, None the library's choice
        self.xcd_rotate = None if xcd_rotate is None else bool(xcd_rotate)
        if tile is None and sg is not None:
            tile = _nearest_tile(sg * (wm or 1) * 16, (wn or 1) * 16)
        if tile is not None and not 0 <= tile < len(CONFIGS):
            raise VkError(f"unknown tile id {tile}")
        self.tile = -1 if tile is None else int(tile)
        if self.tile >= 0:
            t = CONFIGS[self.tile]
            self.bm, self.bn, self.bk = t["bm"], t["bn"], t["bk"]
            base = t["name"]
        else:
            self.bm = self.bn = None
            base = "mm_auto"
        self.name = (f"{base}_{dtype}{'_ta' if trans_a else ''}{'_tb' if trans_b else ''}"
                     f"{'_bat' if batched else ''}{'_g' + str(group_m) if group_m else ''}"
                     f"{'_s' + str(split_k) if split_k > 1 else ''}{'_at' if atomic_split else ''}"
                     f"{'' if xcd_rotate is None else ('_rot' if xcd_rotate else '_ins')}")
        # the plan is the shipped table's, measured on the product by itself: `linear_backward` may take another
        self.from_table = False
        self._keep = []
        self._sent = {}   # enqueue's checked arguments

    def fits(self, m, n, k):
        """Every tile handles ragged shapes; only positivity is required."""
        return m > 0 and n > 0 and k > 0

    def _args(self, a, b, c, m, n, k, nbatch, strides, bias, accumulate, lda, ldb, ldc, side=False,
              act=None, y16=None, ldy=None, z=None, ldz=None, colsum=None, res=None, ldr=None, tri=None,
              p16=None, ldp=None, rowsub=None, scale=1.0):
        if self.batched:
            nb = int(nbatch)
            sa, sb, sc = (int(s) for s in strides)
        else:
            nb, sa, sb, sc = 1, 0, 0, 0
        ga = L.GemmArgs()
        ga.struct_size = C.sizeof(L.GemmArgs)
        ga.layout, ga.dtype = self.layout, L.DTYPES[self.dtype]
        ga.beta = 1 if accumulate else 0
        ga.m, ga.n, ga.k = int(m), int(n), int(k)
        ga.a, ga.b, ga.c = a.ptr, b.ptr, (c.ptr if c is not None else None)
        ga.lda = int(lda) if lda is not None else (m if self.trans_a else k)
        ga.ldb = int(ldb) if ldb is not None else (k if self.trans_b else n)
        ga.ldc = int(ldc) if ldc is not None else n
        ga.bias = bias.ptr if bias is not None else None
        ga.nbatch, ga.tile = nb, self.tile
        ga.sa, ga.sb, ga.sc = sa, sb, sc
        ga.split_k, ga.group_m = self.split_k, self.group_m
        # buffers must cover what the kernel touches
        esz = 2
        a_rows = k if self.trans_a else m
        b_rows = n if self.trans_b else k
        a_cols = m if self.trans_a else k
        b_cols = k if self.trans_b else n
        need_a = ((nb - 1) * sa + (a_rows - 1) * ga.lda + a_cols) * esz
        need_b = ((nb - 1) * sb + (b_rows - 1) * ga.ldb + b_cols) * esz
        need_c = ((nb - 1) * sc + (m - 1) * ga.ldc + n) * 4
        # the fast kernels may read (never use) the last row's padding up to the next
        # multiple of 8 columns; tell the library when a buffer does not contain it
        full_a = ((nb - 1) * sa + (a_rows - 1) * ga.lda + ((a_cols + 7) & ~7)) * esz
        full_b = ((nb - 1) * sb + (b_rows - 1) * ga.ldb + ((b_cols + 7) & ~7)) * esz
        ga.flags = L.MG_FLAG_TIGHT_BUFFERS if (full_a > a.size or full_b > b.size) else 0
        ga.flags |= L.MG_FLAG_SPLITK_ATOMIC if self.atomic_split else L.MG_FLAG_SPLITK_SUM
        if side:
            ga.flags |= L.MG_FLAG_SIDE_STREAM
        if self.xcd_rotate is not None:
            ga.flags |= L.MG_FLAG_XCD_ROTATE if self.xcd_rotate else L.MG_FLAG_XCD_IN_STEP
        if act not in L.ACTS:
            raise VkError(f"{self.name}: unknown activation {act!r}; use None, 'gelu', 'relu', "
                          f"'gelu_grad', 'relu_grad' or 'softmax_grad'")
        ga.act = L.ACTS[act]
        if ga.act == L.MG_ACT_SOFTMAX_GRAD:
            if p16 is None or rowsub is None:
                raise VkError(f"{self.name}: act='softmax_grad' needs p16= (the 16-bit softmax output) and rowsub=")
            if z is not None or colsum is not None:
                raise VkError(f"{self.name}: z= and colsum= belong to act='gelu_grad' or 'relu_grad'")
            ga.p16, ga.rowsub, ga.scale = p16.ptr, rowsub.ptr, float(scale)
            ga.ldp = int(ldp) if ldp is not None else n
            if m > 0 and n > 0:
                if p16.size < ((nb - 1) * sc + (m - 1) * ga.ldp + n) * 2:
                    raise VkError(f"{self.name}: p16 buffer of {p16.size} bytes is too small for {nb} x {m}x{n}")
                if rowsub.size < nb * m * 4:
                    raise VkError(f"{self.name}: rowsub buffer of {rowsub.size} bytes is shorter than {nb * m} floats")
        elif p16 is not None or rowsub is not None:
            raise VkError(f"{self.name}: p16= and rowsub= belong to act='softmax_grad'")
        elif ga.act >= L.MG_ACT_GELU_GRAD:
            if z is None:
                raise VkError(f"{self.name}: act={act!r} needs z= (the pre-activation, f32)")
            ga.z = z.ptr
            ga.ldz = int(ldz) if ldz is not None else n
            if m > 0 and n > 0 and z.size < ((m - 1) * ga.ldz + n) * 4:
                raise VkError(f"{self.name}: z buffer of {z.size} bytes is too small for {m}x{n} (pitch {ga.ldz})")
            if colsum is not None:
                if colsum.size < n * 4:
                    raise VkError(f"{self.name}: colsum buffer of {colsum.size} bytes is shorter than N={n} floats")
                ga.colsum = colsum.ptr
        elif z is not None or colsum is not None:
            raise VkError(f"{self.name}: z= and colsum= belong to act='gelu_grad' or 'relu_grad'")
        if y16 is not None:
            ga.y16 = y16.ptr
            ga.ldy = int(ldy) if ldy is not None else n
            if m > 0 and n > 0 and y16.size < ((nb - 1) * sc + (m - 1) * ga.ldy + n) * 2:
                raise VkError(f"{self.name}: y16 buffer of {y16.size} bytes is too small for {m}x{n} (pitch {ga.ldy})")
        elif ga.act:
            raise VkError(f"{self.name}: act= needs y16= (the activated 16-bit output)")
        if c is None and y16 is None:
            raise VkError(f"{self.name}: C may only be omitted when y16 is given")
        if tri not in L.TRI:
            raise VkError(f"{self.name}: unknown tri {tri!r}; use None, 'c_lower', 'a_lower' or 'a_upper'")
        ga.tri = L.TRI[tri]
        if res is not None:
            if c is None:
                raise VkError(f"{self.name}: res= needs C (C = res + result)")
            ga.beta = 1
            ga.res = res.ptr
            ga.ldr = int(ldr) if ldr is not None else n
            if m > 0 and n > 0 and res.size < ((m - 1) * ga.ldr + n) * 4:
                raise VkError(f"{self.name}: res buffer of {res.size} bytes is too small for {m}x{n} (pitch {ga.ldr})")
        if m > 0 and n > 0 and k > 0:
            if need_a > a.size or need_b > b.size or (c is not None and need_c > c.size):
                raise VkError(f"{self.name}: shape {m}x{n}x{k} (nbatch {nb}) needs {need_a}/{need_b}/{need_c} "
                              f"bytes but buffers hold {a.size}/{b.size}/{c.size if c is not None else 0}")
            if bias is not None and bias.size < n * 4:
                raise VkError(f"{self.name}: bias buffer of {bias.size} bytes is shorter than N={n} floats")
        return ga

    def __call__(self, a, b, c, m, n, k, repeat=1, graph=None, nbatch=1, strides=(0, 0, 0),
                 *, bias=None, accumulate=False, lda=None, ldb=None, ldc=None, side=False,
                 act=None, y16=None, ldy=None, z=None, ldz=None, colsum=None, res=None, ldr=None, tri=None,
                 p16=None, ldp=None, rowsub=None, scale=1.0):
        """side=True (recorded calls only) puts the GEMM on the device's side stream:
        it runs concurrently with the main stream between graph.fork() and graph.join().
        y16= (with act=None, 'gelu' or 'relu') makes the epilogue also write
        narrow(act(result)) in the input dtype, the separate bias_gelu pass of the
        reference (kernels.py:709-718) folded into the GEMM; c may then be None.
        act='gelu_grad' / 'relu_grad' with z= (f32 pre-activation of the layer below)
        folds bias_gelu_bwd (kernels.py:720-739) into a dX GEMM instead: y16 and c
        receive g = result * act'(z), and colsum= (N floats, cleared by the caller unless
        accumulating) has the column sums of g added to it (col_sum, kernels.py:753-761).
        res= (an (m, n) f32 matrix) makes it C = res + result (+ bias): the `residual`
        pass of the reference's transformer (tkernels.py:362-371) in the epilogue.
        act='softmax_grad' with p16= (the 16-bit softmax output P), rowsub= (one float per
        row: sum_j P_j dP_j) and scale= folds attn_softmax_bwd (tkernels.py:167-187) into the
        dP = dOut V^T GEMM: y16 = narrow(scale * P * (result - rowsub[row])); batches allowed
        (y16 and p16 advance strides[2] elements per batch, rowsub m floats).
        tri= declares the causal structure of an attention GEMM so that work on masked
        entries is skipped: 'c_lower' (only C[i, j <= i] is needed; the rest of C is left
        as it was), 'a_lower' / 'a_upper' (op(A)[i, k] is zero for k > i / k < i)."""
        lib, ctx = self.dev._lib, self.dev._ctx
        if side and graph is None:
            raise VkError(f"{self.name}: side=True needs graph= (eager calls wait for their result); "
                          f"use enqueue(..., side=True) between dev.side_fork() and dev.side_join()")
        ga = self._args(a, b, c, m, n, k, nbatch, strides, bias, accumulate, lda, ldb, ldc, side, act, y16, ldy, z, ldz, colsum, res, ldr, tri,
                        p16, ldp, rowsub, scale)
        if graph is not None:
            _check(lib.mg_gemm_check(C.byref(ga)), self.name)
            self._keep.append(ga)

            def launch(ga=ga):
                _check(lib.mg_gemm(ctx, C.byref(ga)), self.name)

            graph.record(launch, [x for x in (a, b, c, bias, y16, z, colsum, res, p16, rowsub) if x is not None], name=self.name,
                         bytes_hint=self.traffic_bytes(m, n, k, nbatch))
            nb_ = nbatch if self.batched else 1
            graph.mm_split.append((nb_ * 2 * (m * k + k * n), nb_ * m * n * 4))
            return 0.0
        dt = C.c_double()
        _check(lib.mg_gemm_time(ctx, C.byref(ga), int(repeat), C.byref(dt)), self.name)
        return dt.value

    def time_rotating(self, sets, m, n, k, repeat=1, nbatch=1, strides=(0, 0, 0), *, accumulate=False,
                      lda=None, ldb=None, ldc=None):
        """Seconds for `repeat` back-to-back launches that take their buffers from
        `sets` in turn; each set is (a, b, c) or (a, b, c, bias).  Enough sets to
        overflow the last-level cache make every launch read its operands from HBM."""
        arr = (L.GemmArgs * len(sets))()
        for i, st in enumerate(sets):
            bias = st[3] if len(st) > 3 else None
            arr[i] = self._args(st[0], st[1], st[2], m, n, k, nbatch, strides, bias, accumulate, lda, ldb, ldc)
        dt = C.c_double()
        _check(self.dev._lib.mg_gemm_time_rotating(self.dev._ctx, arr, len(sets), int(repeat), C.byref(dt)),
               self.name)
        return dt.value

    def enqueue(self, a, b, c, m, n, k, nbatch=1, strides=(0, 0, 0), *, bias=None,
                accumulate=False, lda=None, ldb=None, ldc=None, side=False, act=None, y16=None, ldy=None,
                z=None, ldz=None, colsum=None, res=None, ldr=None, tri=None):
        """Launch without waiting (the stream keeps order); for pipelined callers.  The checked
        arguments of the last few calls are kept, by everything they were checked against."""
        key = (a.ptr, a.size, b.ptr, b.size, c is not None and (c.ptr, c.size), m, n, k, nbatch, tuple(strides),
               bias is not None and (bias.ptr, bias.size), accumulate, lda, ldb, ldc, side, act,
               y16 is not None and (y16.ptr, y16.size), z is not None and (z.ptr, z.size),
               colsum is not None and (colsum.ptr, colsum.size), res is not None and (res.ptr, res.size),
               ldy, ldz, ldr, tri, self.tile, self.split_k, self.group_m, self.atomic_split, self.xcd_rotate)
        ref = self._sent.get(key)
        if ref is None:
            ga = self._args(a, b, c, m, n, k, nbatch, strides, bias, accumulate, lda, ldb, ldc, side, act, y16, ldy, z, ldz, colsum, res, ldr, tri)
            if len(self._sent) >= 64:
                self._sent.clear()
            ref = self._sent[key] = C.byref(ga)
        _check(self.dev._lib.mg_gemm(self.dev._ctx, ref), self.name)

    def plan(self, m, n, k, nbatch=1, lda=None, ldb=None, ldc=None):
        """(tile id, split_k, group_m) the library would use for this shape."""
        ga = L.GemmArgs()
        ga.struct_size = C.sizeof(L.GemmArgs)
        ga.layout, ga.dtype = self.layout, L.DTYPES[self.dtype]
        ga.m, ga.n, ga.k = int(m), int(n), int(k)
        ga.a = ga.b = ga.c = 16     # placeholders: the picker never dereferences
        ga.lda = int(lda) if lda is not None else (m if self.trans_a else k)
        ga.ldb = int(ldb) if ldb is not None else (k if self.trans_b else n)
        ga.ldc = int(ldc) if ldc is not None else n
        ga.nbatch, ga.tile = (int(nbatch) if self.batched else 1), self.tile
        ga.sc = m * ga.ldc
        ga.split_k, ga.group_m = self.split_k, self.group_m
        ga.flags = L.MG_FLAG_SPLITK_ATOMIC if self.atomic_split else L.MG_FLAG_SPLITK_SUM
        t, s, g = C.c_int(), C.c_int(), C.c_int()
        _check(L.load().mg_pick(C.byref(ga), getattr(self.dev, "compute_units", 256), C.byref(t), C.byref(s), C.byref(g)),
               self.name)
        return t.value, s.value, g.value

    def statistics(self, m, n, k, nbatch=1, lda=None, ldb=None, ldc=None):
        """Runtime-reported resource usage of the kernel this Matmul launches for a shape
        (Kernel.statistics, vk.py:690-736), with the reference's key names where they have a
        counterpart: numUsedVgprs, ldsUsageSizeInBytes, scratchMemUsageInBytes, plus
        workgroupThreads, workgroupsPerCU, wavesPerSimd and the tile id that would run."""
        ga = L.GemmArgs()
        ga.struct_size = C.sizeof(L.GemmArgs)
        ga.layout, ga.dtype = self.layout, L.DTYPES[self.dtype]
        ga.m, ga.n, ga.k = int(m), int(n), int(k)
        ga.a = ga.b = ga.c = 16     # placeholders: nothing is launched
        ga.lda = int(lda) if lda is not None else (m if self.trans_a else k)
        ga.ldb = int(ldb) if ldb is not None else (k if self.trans_b else n)
        ga.ldc = int(ldc) if ldc is not None else n
        ga.nbatch, ga.tile = (int(nbatch) if self.batched else 1), self.tile
        ga.sc = m * ga.ldc
        ga.split_k, ga.group_m = self.split_k, self.group_m
        ga.flags = L.MG_FLAG_SPLITK_ATOMIC if self.atomic_split else L.MG_FLAG_SPLITK_SUM
        st, tile = L.KernelStats(), C.c_int()
        _check(self.dev._lib.mg_kernel_stats_for(self.dev._ctx, C.byref(ga), C.byref(tile), C.byref(st)), self.name)
        return stats_dict(st, tile.value)

    def traffic_bytes(self, m, n, k, nbatch=1, bias=False, accumulate=False):
        """Algorithmic (compulsory) bytes: each operand once.  The reference's
        upper bound (kernels.py:299-309) counts per-tile re-reads instead; with
        LDS-staged 256-wide tiles and L2-aware rasterisation those mostly hit
        cache, so the compulsory figure is the one rooflines are priced on."""
        nb = nbatch if self.batched else 1
        return nb * (2 * (m * k + k * n) + 4 * m * n * (2 if accumulate else 1) + (4 * n if bias else 0))

    def flops(self, m, n, k):
        return 2 * m * n * k

    def destroy(self):
        self._keep.clear()
        self._sent.clear()


def linear_backward(dev, dw, dx=None, db=None, graph=None):
    """The backward pass of a linear layer: dW, the bias gradient and dX, which share no result, in one
    launch where the library estimates that to be faster (autograd.py:213-228 issues them in turn).
    dw, dx: (Matmul, positional arguments, keyword arguments) of its call; db: (matrix, sums,
    columns, rows, accumulate, f32) - the column sums of a dense matrix, f32 or 16 bits.  A tile or a K split
    that a Matmul was made with is what its product runs with, except from the shipped table (`from_table`)."""
    lib, ctx = dev._lib, dev._ctx
    args, buffers, traffic, splits = [], [], 0, []
    for mm, (a, b, c, m, n, k), kw in (p for p in (dw, dx) if p is not None):
        if kw.get("side") and graph is None:
            raise VkError(f"{mm.name}: side=True needs graph=")
        named = dict(bias=None, accumulate=False, lda=None, ldb=None, ldc=None)
        named.update(kw)   # (what a product does not take is refused by name)
        args.append(mm._args(a, b, c, m, n, k, 1, (0, 0, 0), **named))
        if graph is not None:   # refused where it is recorded, like a product by itself
            _check(lib.mg_gemm_check(C.byref(args[-1])), mm.name)
        buffers += [x for x in (a, b, c, *kw.values()) if hasattr(x, "ptr")]
        traffic += mm.traffic_bytes(m, n, k)
        splits.append((2 * (m * k + k * n), m * n * 4))
    ba = L.BackwardArgs()
    ba.struct_size, ba.tile = C.sizeof(L.BackwardArgs), L.MG_BACKWARD_AUTO
    named = [p[0] for p in (dw, dx) if p is not None and (p[0].tile >= 0 or p[0].split_k > 0)]
    if named and all(mm.from_table for mm in named):
        ba.tile = L.MG_BACKWARD_REPLAN
        # how slices meet is part of such a plan, not a wish to stay off the workspace, which would rule the one launch out
        # (16384 rows, 1024 -> 256 with the derivative: 70 us in turn, its dW in 15 slices that add with atomics, 46 in one launch;
        # none of the plans that ship splits K that way now)
        for ga, (mm, *_) in zip(args, (p for p in (dw, dx) if p is not None)):
            if mm.from_table and ga.flags & L.MG_FLAG_SPLITK_ATOMIC:
                ga.flags = ga.flags & ~L.MG_FLAG_SPLITK_ATOMIC | L.MG_FLAG_SPLITK_SUM
    ba.dw = C.pointer(args[0])   # (ctypes keeps what a pointer points to)
    if dx is not None:
        ba.dx = C.pointer(args[1])
    if db is not None:
        g, sums, cols, rows, accumulate, f32 = db
        if g.size < rows * cols * (4 if f32 else 2) or sums.size < cols * 4:
            raise VkError(f"linear_backward: column sums of {rows} x {cols} from {g.size} bytes into {sums.size}")
        ba.g, ba.db, ba.rows, ba.cols, ba.g_f32, ba.accumulate = g.ptr, sums.ptr, rows, cols, int(f32), int(accumulate)
        buffers += [g, sums]
        traffic += rows * cols * (4 if f32 else 2)

    if any(x.ptr is None for x in buffers):
        raise VkError("linear_backward: a buffer was destroyed")

    def launch(ba=ba):
        _check(lib.mg_gemm_backward(ctx, C.byref(ba)), "linear_backward")

    if graph is None:
        launch()
        _check(lib.mg_sync(ctx), "linear_backward")
        return
    graph.record(launch, buffers, name="linear_backward", bytes_hint=traffic)
    graph.mm_split += splits


# --------------------------------------------------------------------------
# autotuner
# --------------------------------------------------------------------------

def time_sequence(dev, calls):
    """Seconds each GEMM of a sequence costs inside it: every call behind the previous one on
    the device's stream, HIP events between them.  calls: (mm, a, b, c, m, n, k, kwargs) with
    kwargs from lda / ldb / ldc / bias / accumulate."""
    arr = (L.GemmArgs * len(calls))()
    for i, (mm, a, b, c, m, n, k, kw) in enumerate(calls):
        arr[i] = mm._args(a, b, c, m, n, k, 1, (0, 0, 0), kw.get("bias"), kw.get("accumulate", False),
                          kw.get("lda"), kw.get("ldb"), kw.get("ldc"))
    out = (C.c_double * len(calls))()
    _check(dev._lib.mg_gemm_time_each(dev._ctx, arr, len(calls), out), "time_sequence")
    return list(out)


def stats_dict(st, tile):
    return {"numUsedVgprs": st.vgprs, "ldsUsageSizeInBytes": st.static_lds_bytes + st.dynamic_lds_bytes,
            "scratchMemUsageInBytes": st.scratch_bytes, "workgroupThreads": st.threads,
            "workgroupsPerCU": st.wgs_per_cu, "wavesPerSimd": st.waves_per_simd, "tile_id": tile}


def tile_statistics(dev, tile, layout, dtype="f16", variant=0):
    """statistics() of one instantiation named directly (tile id, layout MG_NN.., dtype,
    variant 0 aligned / 1 any alignment or bias epilogue / 2 fused activation / 3 the same with direct
    loads, or for three workgroups a CU / 4 aligned, for three workgroups a CU); None when the
    library holds no such instantiation."""
    st = L.KernelStats()
    rc = dev._lib.mg_tile_kernel_stats(dev._ctx, int(tile), int(layout), L.DTYPES[dtype], int(variant), C.byref(st))
    if rc == L.MG_ERR_ARG:
        return None
    _check(rc, "tile_statistics")
    return stats_dict(st, int(tile))


def occupancy(dev, stats, workgroup_threads=None, min_waves=1):
    """Waves resident per SIMD for a compiled kernel, and why it is not worth timing (or
    None) - the reference's pruning signal (kernels.py:384-411).  There the reason is too
    few waves to hide DRAM latency on a 12-CU part; the kernels here are built for one or two
    wavefronts per SIMD with explicit prefetch, so the default bar is one wave, and the
    reason that does prune is a register spill: a kernel that uses scratch memory turns
    accumulator traffic into vector memory operations inside the K loop."""
    waves = stats.get("wavesPerSimd")
    if not stats.get("numUsedVgprs") or waves is None:
        return None, None          # unknown: benchmark it rather than guess
    if stats.get("scratchMemUsageInBytes", 0) > 0:
        return waves, f"spills {stats['scratchMemUsageInBytes']} bytes of scratch per lane (vgpr={stats['numUsedVgprs']})"
    if waves < min_waves:
        return waves, f"only {waves} waves/SIMD (vgpr={stats['numUsedVgprs']})"
    return waves, None


_HERE = os.path.dirname(os.path.abspath(__file__))
# Shipped table of tuned picks for MI355X, consulted read-only after the user cache.  Its keys name the architecture:
# what the runtime calls the device ("gfx950:sramecc+:xnack-", or a marketing name such as "AMD Radeon Graphics") differs
# from machine to machine for the same chip, and the library is built for no other.
_SHIPPED_CACHE = os.path.join(_HERE, "tuned_mi355x.json")
_SHIPPED_DEVICE = "gfx950:sramecc+:xnack-"
_TUNE_CACHE = os.environ.get("VKGRAD_AMD_TUNE_CACHE", os.path.join(_HERE, ".autotune.json"))


def _load_cache(path=None):
    path = path or _TUNE_CACHE
    if os.path.exists(path):
        try:
            with open(path) as f:
                return json.load(f)
        except (OSError, ValueError):
            return {}
    return {}


_shipped = (None, {})   # (path, its content): read-only, parsed once - a model asks for a plan per GEMM shape


def _shipped_table():
    global _shipped
    if _shipped[0] != _SHIPPED_CACHE:
        _shipped = (_SHIPPED_CACHE, _load_cache(_SHIPPED_CACHE))
    return _shipped[1]


def _save_cache(cache, path=None):
    path = path or _TUNE_CACHE
    tmp = path + f".{os.getpid()}.tmp"
    with open(tmp, "w") as f:
        json.dump(cache, f, indent=1, sort_keys=True)
    os.replace(tmp, path)


def _pitch_tag(m, n, k, trans_a, trans_b, lda, ldb, ldc):
    """Non-default row pitches as a key suffix (they decide which kernels are eligible)."""
    d = (m if trans_a else k, k if trans_b else n, n)
    got = tuple(int(x) if x is not None else dflt for x, dflt in zip((lda, ldb, ldc), d))
    return "" if got == d else f"|ld{got[0]},{got[1]},{got[2]}"


def tune_key(dev_name, m, n, k, trans_a, trans_b, dtype="f16", batched=False, nbatch=1,
             accumulate=False, lda=None, ldb=None, ldc=None, context=None):
    """Cache key; the reference's shape (kernels.py:459-460) plus dtype, beta and pitches, and the
    context a plan was tuned in when that is not "alone" (see tune_in_context)."""
    return (f"{dev_name}|{m}x{n}x{k}|ta{int(trans_a)}tb{int(trans_b)}|{dtype}"
            f"{'|acc' if accumulate else ''}{'|bat' + str(nbatch) if batched else ''}"
            f"{_pitch_tag(m, n, k, trans_a, trans_b, lda, ldb, ldc)}{'|in:' + context if context else ''}")


def lookup_tuned(dev_name, m, n, k, trans_a, trans_b, dtype="f16", batched=False, nbatch=1,
                 accumulate=False, lda=None, ldb=None, ldc=None, context=None):
    """Cached pick for a shape, user cache first, then the shipped table; with a context, the
    pick made in that context if there is one, else the one made alone."""
    for ctx in ((context, None) if context else (None,)):
        shipped = _shipped_table()
        for table, name in ((_load_cache(), dev_name), (shipped, dev_name), (shipped, _SHIPPED_DEVICE)):
            e = table.get(tune_key(name, m, n, k, trans_a, trans_b, dtype, batched, nbatch, accumulate, lda, ldb,
                                   ldc, ctx))
            if e is not None:
                return e
    return None


def is_shipped(e):
    """Whether lookup_tuned found the entry in the shipped table, not in the user's cache."""
    return any(e is x for x in _shipped_table().values())


def matmul_from_entry(dev, e, trans_a=False, trans_b=False, dtype="f16", batched=False):
    """The Matmul a cache entry (or a candidate of tune_in_context) describes; tile_id -1: the library's own choice."""
    tile = e["tile_id"]
    return Matmul(dev, trans_a=trans_a, trans_b=trans_b, batched=batched, dtype=dtype, tile=tile if tile >= 0 else None,
                  split_k=e.get("split_k", 0), group_m=e.get("group_m", 0),
                  atomic_split=e.get("atomic_split", False), xcd_rotate=e.get("xcd_rotate"))


def tuned_matmul(dev, m, n, k, trans_a=False, trans_b=False, dtype="f16", batched=False, nbatch=1,
                 accumulate=False, lda=None, ldb=None, ldc=None, context=None):
    """(Matmul, how) for one shape as the benchmarks run it: the cached pick (tile,
    K split, rasterisation band, split mode, walk) when a cache holds the shape, else a
    Matmul that leaves the choice to the library's picker.  how is 'tuned table' or
    'picker'.  The parity tests build their GEMMs through this same function, so what
    is timed is what is checked."""
    e = lookup_tuned(dev.name, m, n, k, trans_a, trans_b, dtype, batched, nbatch, accumulate, lda, ldb, ldc, context)
    if e is None:
        return Matmul(dev, trans_a=trans_a, trans_b=trans_b, batched=batched, dtype=dtype), "picker"
    return matmul_from_entry(dev, e, trans_a, trans_b, dtype, batched), "tuned table"


def plan_candidates(m, n, k, layout, cus=256, splits=(1, 2, 3, 4, 6, 8)):
    """Candidate plans for tune_in_context: one tile of every family and size (64 x 64
    register-staged, the direct-to-LDS 128 x 128 with 64- and 32-wide K-blocks, 128 x 256,
    256 x 128, the persistent 128 x 128, the ping-pong 256 x 256) with K splits from none up to
    where a slice has fewer than four K-blocks or the grid has more than twice the resident
    workgroups - beside another stream's kernels a GEMM is often better off with few, large
    workgroups than with the grid that fills the chip by itself - each split both through
    the workspace and with atomics."""
    fams = [t for t in CONFIGS if t["name"] in ("mm_64x64x64_w2x2", "mmd_128x128x64_w2x2_s2", "mmd_128x128x32_w2x2_s3",
                                                "mmd_128x256x32_w2x2_s3", "mmd_256x128x32_w2x2_s3",
                                                "mmp_128x128x64_w2x2_s2", "mmq_256x256x64_w2x4_s2")]
    out = []
    for t in fams:
        tiles = -(-m // t["bm"]) * -(-n // t["bn"])
        if tiles * t["bm"] * t["bn"] > 2.0 * m * n:
            continue                                    # more padding than matrix
        for sp in splits:
            if sp > 1 and (k // (4 * t["bk"]) < sp or tiles * sp > 4 * cus):
                continue
            for at in ((False, True) if sp > 1 else (False,)):
                out.append({"tile_id": t["id"], "split_k": sp, "atomic_split": at, "group_m": 0, "xcd_rotate": None,
                            "tile": [t["bm"], t["bn"]], "config": [t["bm"], t["bn"], t["bk"]], "lds": True})
    return out


def tune_in_context(slots, measure, passes=2, min_gain=0.003, refine=True, verbose=False):
    """Plans for GEMMs that run beside each other, chosen by what the whole sequence takes.

    The per-shape tuner times a GEMM alone; a GEMM that shares the chip with another stream's
    kernels wants a different plan (a weight-gradient GEMM beside the forward / dX chain of a
    training step: fewer, larger workgroups than the grid that is fastest alone).  slots maps
    a name to its candidate plans (dicts with tile_id, split_k, atomic_split, group_m,
    xcd_rotate), the first being the current one; measure(assignment) returns the seconds the
    sequence takes with {name: plan}.  Coordinate descent: for one slot after the other every
    candidate is measured with the others held, and kept when it beats the held plan by more
    than min_gain (relative; below that a difference is noise); `passes` sweeps or until a
    sweep changes nothing.  With refine, a last sweep tries the rasterisation band and the walk
    of the XCDs on each kept plan.  Returns (assignment, seconds, log); no counterpart in the
    reference, whose steps run on one queue (vk.py:848-851)."""
    cur = {name: dict(c[0]) for name, c in slots.items()}
    best = measure(cur)
    log = [("start", None, best)]

    def sweep(options_of):
        nonlocal best
        changed = False
        for name in slots:
            held, held_t = cur[name], best
            for cand in options_of(name):
                if cand == held:
                    continue
                cur[name] = cand
                t = measure(cur)
                if verbose:
                    print(f"    {name}: tile {cand['tile_id']} split {cand['split_k']}{' at' if cand['atomic_split'] else ''} "
                          f"g{cand['group_m']} walk {cand['xcd_rotate']}: {t * 1e3:.4f} ms (held {held_t * 1e3:.4f})", flush=True)
                if t < held_t * (1.0 - min_gain):
                    # confirm: a second measurement must agree before a plan is replaced
                    t2 = measure(cur)
                    if t2 < held_t * (1.0 - min_gain):
                        held, held_t = cand, max(t, t2)
            cur[name] = held
            if held_t < best:
                changed = True
                log.append((name, dict(held), held_t))
            best = held_t
        return changed

    for _ in range(passes):
        if not sweep(lambda name: [dict(c) for c in slots[name]]):
            break
    if refine:
        def variants(name):
            base = cur[name]
            walks = (True, False) if walk_matters(base["tile_id"]) else (base["xcd_rotate"],)
            return [dict(base, group_m=g, xcd_rotate=w) for g in (0, 1, 2, 4, 16) for w in walks]
        sweep(variants)
    return cur, best, log


_WARMED = set()


def warmup(dev, seconds=2.0, force=False):
    """Sustained GEMM load until clocks settle (kernels.py:353-381).  On MI355X
    the effect is a power-managed clock under MFMA load rather than an idle
    ramp, but timing anything before the chip is in its loaded state still
    biases a comparison."""
    if not force and id(dev) in _WARMED:
        return 0.0
    m = n = k = 2048
    a = dev.buffer(m * k * 2, "device")
    b = dev.buffer(k * n * 2, "device")
    c = dev.buffer(m * n * 4, "device")
    K = make_kernels(dev)
    K["fill_uniform16"]([a], m * k, 3)
    K["fill_uniform16"]([b], k * n, 4)
    mm = Matmul(dev)
    t0 = time.perf_counter()
    try:
        while time.perf_counter() - t0 < seconds:
            mm(a, b, c, m, n, k, repeat=20)
    finally:
        mm.destroy()
        for x in (a, b, c):
            x.destroy()
    _WARMED.add(id(dev))
    return time.perf_counter() - t0


_MEASURE_S = 0.02     # GPU time per measurement (kernels.py:424)
_SUBMIT_CAP_S = 0.2   # one timed batch stays under this (kernels.py:421)


def _repeat_for(t_one):
    """Launches per measurement so every candidate is timed over equal GPU
    time, not an equal number of launches (kernels.py:433-447)."""
    return max(1, int(min(_MEASURE_S, _SUBMIT_CAP_S) / max(t_one, 1e-7)))


LAST_LEVEL_CACHE_BYTES = 256 << 20


MAX_OPERAND_SETS = 32


def buffer_sets_for(read_bytes):
    """How many operand sets a timing loop rotates through so that no launch finds what it
    reads in the last-level cache: the sets between two uses of one set are read in between,
    and together they are twice the cache (3 to MAX_OPERAND_SETS sets; one when a single set
    already is).  Only what a GEMM reads counts: the results it writes pass through that
    cache without displacing operands (8192 x 50257 x 768 finds its 90 MB of operands there
    after the 1.65 GB of logits of the previous launch)."""
    if read_bytes >= 2 * LAST_LEVEL_CACHE_BYTES:
        return 1
    return max(3, min(MAX_OPERAND_SETS, -(-2 * LAST_LEVEL_CACHE_BYTES // max(1, read_bytes)) + 1))


def walk_matters(tile_id):
    """Whether a tile's kernel walks the tile order per XCD (MG_FLAG_XCD_ROTATE / _IN_STEP mean
    something to it): the one-tile-per-workgroup kernels do, the persistent, stream-K and
    skinny ones place their work themselves.  tile_id -1: whatever the library chooses may."""
    return tile_id < 0 or CONFIGS[tile_id]["name"].split("_")[0] in ("mm", "mmd", "mmq")


def skinny_stream_fits(m, k, layout):
    """The skinny-M streaming tile (name mv_*): NT layout, at most 8 rows of A and
    K <= 2048 in whole 8-element pieces."""
    return layout == L.MG_NT and m <= 8 and k <= 2048 and k % 8 == 0


def skinny_mfma_fits(m, k, layout):
    """The skinny-M tile on the matrix cores (name ms_*): NT layout, at most 64 rows of A,
    which must fit LDS whole beside the phase buffers of B (K <= 2176 for up to 32 rows,
    K <= 960 for up to 64), K in whole 8-element pieces."""
    kpad = -(-k // 64) * 64
    blocks = -(-m // 32)
    lds = (4 if blocks == 1 else 8) * 32 * (64 * 2 + 16) + blocks * 32 * (kpad * 2 + 16)
    return layout == L.MG_NT and m <= 64 and k % 8 == 0 and lds <= 160 * 1024


def candidate_space(m, n, k, cus=256, nbatch=1, layout=None):
    """(tile, split_k) pairs worth timing for a shape: every tile whose padding
    waste is tolerable, with K splits that bring an under-filled grid up to
    about one or two workgroups per CU."""
    def useful_of(t):
        gm, gn = -(-m // t["bm"]), -(-n // t["bn"])
        return (m * n) / (gm * t["bm"] * gn * t["bn"])

    tiled = [t for t in CONFIGS if not t["name"].startswith(("mv_", "ms_"))]
    # skinny problems waste most of every tile: keep the tiles that waste least
    floor = min(0.45, 0.45 * max(useful_of(t) for t in tiled))
    out = [(t["id"], 1) for t in CONFIGS if t["name"].startswith("mv_") and skinny_stream_fits(m, k, layout)]
    if nbatch == 1:
        out += [(t["id"], 1) for t in CONFIGS if t["name"].startswith("ms_") and skinny_mfma_fits(m, k, layout)]
    for t in tiled:
        gm, gn = -(-m // t["bm"]), -(-n // t["bn"])
        if useful_of(t) < floor and len(tiled) > 1:
            continue
        groups = gm * gn * nbatch
        kblocks = -(-k // t["bk"])
        splits = {1}
        if groups < cus and kblocks >= 4 and t.get("persistent") != 2:   # stream-K tiles cut K themselves
            for target in (cus, 2 * cus, 3 * cus):
                s = max(1, min(target // groups, kblocks // 2))
                # the neighbours too: atomic traffic grows with the split, so the
                # fastest one is often just below what fills the chip
                for c in (s - 1, s, s + 1, s // 2):
                    if 1 <= c <= kblocks // 2:
                        splits.add(c)
        for s in sorted(splits):
            out.append((t["id"], s))
    if not out:
        out = [(CONFIGS[0]["id"], 1)]
    return out


def autotune_matmul(dev, m, n, k, trans_a=False, trans_b=False, reps=3, verbose=False,
                    use_cache=True, batched=False, nbatch=1, *, dtype="f16", accumulate=False,
                    timer=None, lda=None, ldb=None, ldc=None):
    """Pick the fastest (tile, split_k, group_m) for one shape (kernels.py:450-603).

    Stage one times every candidate round-robin over equal GPU time and keeps
    the best-of-`reps`; stage two sweeps the rasterisation band on the winner
    only, re-measuring group_m's default alongside (kernels.py:539-584).
    `timer(mm, repeat) -> seconds` replaces the device for tests of the logic.
    Returns (Matmul, best) with best keys config, lds, tflops, ms, tile,
    evaluated, pruned, group_m, xcd_rotate, split_k, tile_id.

    What the library runs when no tile is named is a candidate too (tile_id -1; config and tile then say
    what that was): it alone packs operands with odd pitches.  It has to be 2 % faster than the best named
    plan, because a name stays what it is when the library learns to choose differently.
    """
    key = tune_key(dev.name, m, n, k, trans_a, trans_b, dtype, batched, nbatch, accumulate, lda, ldb, ldc)
    if use_cache:
        e = lookup_tuned(dev.name, m, n, k, trans_a, trans_b, dtype, batched, nbatch, accumulate, lda, ldb, ldc)
        if e is not None:
            return matmul_from_entry(dev, e, trans_a, trans_b, dtype, batched), e

    nb = nbatch if batched else 1
    pa = int(lda) if lda is not None else (m if trans_a else k)      # row pitches
    pb = int(ldb) if ldb is not None else (k if trans_b else n)
    pc = int(ldc) if ldc is not None else n
    ea, eb, ec = (k if trans_a else m) * pa, (n if trans_b else k) * pb, m * pc   # elements per matrix
    strides = (ea, eb, ec)
    call = dict(nbatch=nb, strides=strides) if batched else {}
    sets = None
    if timer is None:
        warmup(dev)
        read_bytes = nb * (2 * (ea + eb) + (4 * ec if accumulate else 0))
        K = make_kernels(dev, dtype)
        sets, outs = [], []
        for s in range(buffer_sets_for(read_bytes)):
            # results that are only written share three buffers: they do not displace operands
            if accumulate or s < 3:
                outs.append(dev.buffer(nb * ec * 4, "device"))
            st = (dev.buffer(nb * ea * 2, "device"), dev.buffer(nb * eb * 2, "device"), outs[s % len(outs)])
            sets.append(st)
            # random operands: zeros or garbage bit patterns misstate the timing (data
            # toggling sets MFMA power and with it the clock)
            K["fill_uniform16"]([st[0]], nb * ea, 1 + 2 * s)
            K["fill_uniform16"]([st[1]], nb * eb, 2 + 2 * s)

        def timer(mm, repeat):
            # operands rotate through sets that together overflow the last-level cache:
            # a layer of a training step finds its operands in HBM, not in cache
            return mm.time_rotating(sets, m, n, k, repeat=repeat, accumulate=accumulate,
                                    lda=lda, ldb=ldb, ldc=ldc, **call)

    try:
        # a K split is timed both ways: slices meeting in the workspace, and adding atomically
        cands = [Matmul(dev, trans_a=trans_a, trans_b=trans_b, batched=batched, tile=t, dtype=dtype,
                        split_k=s, group_m=0, atomic_split=at, xcd_rotate=True)
                 for t, s in candidate_space(m, n, k, getattr(dev, "compute_units", 256), nb,
                                             layout_of(trans_a, trans_b))
                 for at in ((False, True) if s > 1 else (False,))]
        if not cands:
            raise VkError(f"no matmul config fits {m}x{n}x{k}")
        own = Matmul(dev, trans_a=trans_a, trans_b=trans_b, batched=batched, dtype=dtype, xcd_rotate=True)
        cands.append(own)
        # resource usage of each candidate's kernel; a spilling one is not timed (kernels.py:478-503)
        info, pruned = {}, []
        if sets is not None:
            kept = []
            for x in cands:
                st = x.statistics(m, n, k, nb, lda, ldb, ldc)
                occ, reason = occupancy(dev, st)
                info[id(x)] = (st["numUsedVgprs"], occ)
                if reason:
                    pruned.append((x.tile, x.split_k, reason))
                    if verbose:
                        print(f"    tile {x.name} split_k={x.split_k:2d}  pruned: {reason}")
                else:
                    kept.append(x)
            cands = kept or cands

        def measure(mms):
            warm = {id(x): timer(x, 1) for x in mms}
            best_t = {id(x): float("inf") for x in mms}
            for _ in range(reps):
                for x in mms:   # round-robin: drift spreads evenly over candidates
                    r = max(_repeat_for(warm[id(x)]), len(sets) if sets else 1)
                    best_t[id(x)] = min(best_t[id(x)], timer(x, r) / r)
            return best_t

        best_t = measure(cands)
        results = []
        for x in cands:
            t = best_t[id(x)]
            tf = x.flops(m, n, k) * nb / t / 1e12
            c = CONFIGS[x.tile if x is not own else x.plan(m, n, k, nb, lda, ldb, ldc)[0]]
            results.append({"config": [c["bm"], c["bn"], c["bk"]], "lds": True, "tflops": tf, "ms": t * 1e3,
                            "tile": [c["bm"], c["bn"]], "tile_id": x.tile, "split_k": x.split_k,
                            "atomic_split": x.atomic_split, "vgpr": info.get(id(x), (None, None))[0],
                            "occupancy": info.get(id(x), (None, None))[1]})
            if verbose:
                v, o = info.get(id(x), (None, None))
                print(f"    tile {c['bm']:3d}x{c['bn']:3d} id={x.tile:2d} split_k={x.split_k:2d}{' at' if x.atomic_split else '   '}  "
                      f"{tf:8.2f} TFLOPS  {t * 1e6:9.1f} us  vgpr={v or '?'} waves={o or '?'}")
        results.sort(key=lambda r: -r["tflops"])
        named = next((r for r in results if r["tile_id"] >= 0), results[0])
        best = dict(results[0] if results[0]["tflops"] > 1.02 * named["tflops"] else named)

        # stage two: rasterisation band and the walk of the XCDs (in step or rotated) on the winner
        variants = [matmul_from_entry(dev, dict(best, group_m=g, xcd_rotate=rot), trans_a, trans_b, dtype, batched)
                    for g in (0, 1, 2, 4, 16) for rot in ((True, False) if walk_matters(best["tile_id"]) else (False,))]
        gt = measure(variants)
        scored = sorted(((v.flops(m, n, k) * nb / gt[id(v)] / 1e12, v.group_m, v.xcd_rotate) for v in variants),
                        reverse=True)
        if verbose:
            for tf, g, rot in scored:
                print(f"    group_m={g:2d}{' rotated' if rot else '        '} on winning tile   {tf:8.2f} TFLOPS")
        tf, g, rot = scored[0]
        best.update(tflops=tf, ms=2.0 * m * n * k * nb / tf / 1e9, group_m=g, xcd_rotate=rot)
        best["pruned"] = len(CONFIGS) * 1 - len({c.tile for c in cands if c is not own})
        best["spilling"] = [list(x) for x in pruned]
        best["evaluated"] = len(results)
        if use_cache:
            cache = _load_cache()
            cache[key] = best
            _save_cache(cache)
        return matmul_from_entry(dev, best, trans_a, trans_b, dtype, batched), best
    finally:
        for x in {id(b): b for st in sets or () for b in st}.values():
            x.destroy()


# --------------------------------------------------------------------------
# companion elementwise kernels
# --------------------------------------------------------------------------

class Elementwise:
    """One elementwise kernel with the reference's call shape
    (kernels.py:687-693): k(buffers, n, *args, graph=None)."""

    def __init__(self, dev, name, launch):
        self.dev, self.name, self._launch = dev, name, launch

    def __call__(self, buffers, n, *args, repeat=1, graph=None):
        lib, ctx = self.dev._lib, self.dev._ctx
        ptrs = [b.ptr for b in buffers]
        if any(p is None for p in ptrs):
            raise VkError(f"{self.name}: a buffer was destroyed")

        def launch():
            _check(self._launch(lib, ctx, ptrs, int(n), *args), self.name)

        if graph is not None:
            graph.record(launch, buffers, name=self.name)
            return 0.0
        t0 = time.perf_counter()
        for _ in range(repeat):
            launch()
        _check(lib.mg_sync(ctx), self.name)
        return time.perf_counter() - t0

    def destroy(self):
        pass


def make_kernels(dev, dtype="f16"):
    """The elementwise kernels the training loop needs (kernels.py:699-862), by
    the reference's names.  `dtype` is the 16-bit type of narrowed outputs.
    bias_relu / bias_relu_bwd are the ReLU counterparts of the GELU pair."""
    dt = L.DTYPES[dtype]
    K = {}

    def add(name, fn):
        K[name] = Elementwise(dev, name, fn)

    # buffers: acc, bias, z, y16 ; args: ncol
    add("bias_gelu", lambda lib, ctx, p, n, ncol:
        lib.mg_ew_bias_act(ctx, p[0], p[1], p[2], p[3], n, int(ncol), L.MG_ACT_GELU, dt))
    add("bias_relu", lambda lib, ctx, p, n, ncol:
        lib.mg_ew_bias_act(ctx, p[0], p[1], p[2], p[3], n, int(ncol), L.MG_ACT_RELU, dt))
    # buffers: dy, z, dz16, dz32
    add("bias_gelu_bwd", lambda lib, ctx, p, n:
        lib.mg_ew_act_bwd(ctx, p[0], p[1], p[2], p[3], n, L.MG_ACT_GELU, dt))
    add("bias_relu_bwd", lambda lib, ctx, p, n:
        lib.mg_ew_act_bwd(ctx, p[0], p[1], p[2], p[3], n, L.MG_ACT_RELU, dt))
    # buffers: dy, z, dz16
    add("bias_gelu_bwd16", lambda lib, ctx, p, n:
        lib.mg_ew_act_bwd(ctx, p[0], p[1], p[2], None, n, L.MG_ACT_GELU, dt))
    # buffers: acc, bias, z ; args: ncol
    add("bias", lambda lib, ctx, p, n, ncol:
        lib.mg_ew_bias_act(ctx, p[0], p[1], p[2], None, n, int(ncol), L.MG_ACT_NONE, dt))
    # buffers: g, sums ; n = ncol ; args: nrow
    add("col_sum", lambda lib, ctx, p, n, nrow: lib.mg_ew_col_sum(ctx, p[0], p[1], n, int(nrow), 0))
    add("col_sum_acc", lambda lib, ctx, p, n, nrow: lib.mg_ew_col_sum(ctx, p[0], p[1], n, int(nrow), 1))
    # buffers: z, y16 — activation + narrowing of a pre-activation that already holds its bias
    add("gelu16", lambda lib, ctx, p, n:
        lib.mg_ew_bias_act(ctx, p[0], None, None, p[1], n, 1, L.MG_ACT_GELU, dt))
    add("relu16", lambda lib, ctx, p, n:
        lib.mg_ew_bias_act(ctx, p[0], None, None, p[1], n, 1, L.MG_ACT_RELU, dt))
    # buffers: logits, labels, dl16, dl32, loss ; n = rows ; args: stride, ncls
    add("softmax_ce", lambda lib, ctx, p, n, stride, ncls:
        lib.mg_ew_softmax_ce(ctx, p[0], p[1], p[2], p[3], p[4], n, int(stride), int(ncls), dt))
    # buffers: w, g, m, v, w16, hp ; args: wd
    add("adamw", lambda lib, ctx, p, n, wd:
        lib.mg_ew_adamw(ctx, p[0], p[1], p[2], p[3], p[4], p[5], n, float(wd), dt))
    add("zero", lambda lib, ctx, p, n: lib.mg_ew_zero(ctx, p[0], n))
    # buffers: src, dst ; n = bytes — recordable device-side copy (stages CPU-written inputs into HBM)
    add("copy", lambda lib, ctx, p, n: lib.mg_ew_copy(ctx, p[1], p[0], n))
    add("cast16", lambda lib, ctx, p, n: lib.mg_ew_cast16(ctx, p[0], p[1], n, dt))
    # dataparallel.py:54-58 — buffers: dst, src
    add("grad_add", lambda lib, ctx, p, n: lib.mg_ew_grad_add(ctx, p[0], p[1], n))
    # buffers: dst (16-bit) ; args: seed — pseudo-random operands in [-1, 1) for warm-up and tuning
    add("fill_uniform16", lambda lib, ctx, p, n, seed: lib.mg_ew_fill_uniform16(ctx, p[0], n, int(seed), dt))
    return K
