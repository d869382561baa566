"""The strided element-wise kernels on the GPU: copies and casts, ADD / MUL,
REPEAT, CONCAT and SOFT_MAX at sizes with and without whole 4- and 8-element
chunks, on permuted and broadcast operands.  Every op but SOFT_MAX rounds
once, so the results must match numpy bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_fusion import Graph

pytestmark = pytest.mark.gpu

TYPES = {"f32": 0, "f16": 1, "bf16": 30}


def to_bits(wx, a, typ):
    a = np.ascontiguousarray(a, np.float32)
    return a if typ == "f32" else a.astype(np.float16) if typ == "f16" else wx.f32_to_bf16(a)


def value(wx, a, typ):
    """What `a` reads back as in typ."""
    b = to_bits(wx, a, typ)
    return b if typ == "f32" else b.astype(np.float32) if typ == "f16" else wx.bf16_to_f32(b)


class G(Graph):
    def leaf(self, wx, a, typ):
        t = self.t(TYPES[typ], *reversed(a.shape))
        self.todo = getattr(self, "todo", []) + [(t, to_bits(wx, a, typ))]
        return t

    def run(self, y, typ, shape):
        self.alloc()
        for t, a in self.todo:
            self.set(t, a)
        self.compute(y)
        return self.get(y, {"f32": np.float32, "f16": np.float16, "bf16": np.uint16}[typ], shape)


SHAPES = [(1, 1, 1, 1), (2, 3, 5, 7), (1, 24, 49, 128), (3, 1, 33, 12), (1, 2, 200, 520), (2, 2, 7, 3121),
          (1, 1, 1, 1 << 18 | 3), (1, 16, 160, 520)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("src,dst", [("f32", "bf16"), ("bf16", "f32"), ("bf16", "bf16"), ("f32", "f32"), ("f16", "f32")])
@pytest.mark.parametrize("perm", [(0, 1, 2, 3), (0, 2, 1, 3), (1, 2, 0, 3), (2, 0, 1, 3)])
def test_copies_and_casts(wx, be, rng, shape, src, dst, perm):
    print(f"copy {shape} {src}->{dst} perm {perm}", flush=True)
    a = rng.standard_normal(shape).astype(np.float32)
    g = G(wx, be)
    try:
        p = be.lib.wamx_permute(g.ctx, g.leaf(wx, a, src), *perm)
        y = be.lib.wamx_cast(g.ctx, p, TYPES[dst]) if src != dst else be.lib.wamx_cont(g.ctx, p)
        # ggml's permute sends dim i to perm[i]; numpy axis 3 - i is dim i.
        axes = [0] * 4
        for i, q in enumerate(perm):
            axes[3 - q] = 3 - i
        ref = to_bits(wx, np.transpose(value(wx, a, src), axes), dst)
        assert np.array_equal(g.run(y, dst, ref.shape), ref)
    finally:
        g.close()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("keep", [(1, 1, 1, 1), (0, 0, 0, 1), (0, 1, 0, 0), (0, 0, 0, 0), (1, 0, 1, 1)])
@pytest.mark.parametrize("ta,tb", [("f32", "f32"), ("bf16", "bf16"), ("f32", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("op", ["add", "mul"])
def test_broadcast_binary(wx, be, rng, shape, keep, ta, tb, op):
    """b has a's extent where keep is 1 and one element elsewhere."""
    print(f"{op} {shape} keep {keep} {ta} {tb}", flush=True)
    bs = tuple(n if k else 1 for n, k in zip(shape, keep))
    a, b = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(bs).astype(np.float32)
    g = G(wx, be)
    try:
        y = getattr(be.lib, "wamx_" + op)(g.ctx, g.leaf(wx, a, ta), g.leaf(wx, b, tb))
        assert y, wx.last_error()
        va, vb = value(wx, a, ta), value(wx, b, tb)
        ref = to_bits(wx, va + vb if op == "add" else va * vb, ta)
        assert np.array_equal(g.run(y, ta, shape), ref)
    finally:
        g.close()


@pytest.mark.parametrize("bs", [(1, 1, 5, 4), (2, 1, 1, 8), (1, 3, 5, 8)])
def test_modulo_broadcast(wx, be, rng, bs):
    """b repeats by modulo in a dim longer than one: the general kernel."""
    a, b = rng.standard_normal((2, 3, 10, 8)).astype(np.float32), rng.standard_normal(bs).astype(np.float32)
    g = G(wx, be)
    try:
        y = be.lib.wamx_add(g.ctx, g.leaf(wx, a, "f32"), g.leaf(wx, b, "f32"))
        ref = a + np.tile(b, [n // m for n, m in zip(a.shape, bs)])
        assert np.array_equal(g.run(y, "f32", a.shape), ref)
    finally:
        g.close()


@pytest.mark.parametrize("dim,sa,sb", [
    (0, (2, 3, 5, 1), (2, 3, 5, 511)), (0, (1, 2, 7, 1000), (1, 2, 7, 1)), (0, (1, 3, 2, 2043), (1, 3, 2, 13)),
    (0, (2, 3, 5, 1), (2, 3, 5, 48)), (0, (1, 24, 128, 49), (1, 24, 128, 3072)), (0, (1, 2, 3, 8), (1, 2, 3, 16)),
    (1, (1, 24, 1, 128), (1, 24, 48, 128)), (1, (1, 24, 49, 128), (1, 24, 3072, 128)), (2, (2, 3, 5, 7), (2, 4, 5, 7)),
    (3, (1, 3, 4, 8), (2, 3, 4, 8))])
@pytest.mark.parametrize("typ", ["f32", "bf16"])
def test_concat(wx, be, rng, dim, sa, sb, typ):
    print(f"concat dim {dim} {sa} {sb} {typ}", flush=True)
    a, b = rng.standard_normal(sa).astype(np.float32), rng.standard_normal(sb).astype(np.float32)
    g = G(wx, be)
    try:
        y = be.lib.wamx_concat(g.ctx, g.leaf(wx, a, typ), g.leaf(wx, b, typ), dim)
        ref = to_bits(wx, np.concatenate([value(wx, a, typ), value(wx, b, typ)], 3 - dim), typ)
        assert np.array_equal(g.run(y, typ, ref.shape), ref)
    finally:
        g.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 169, 512, 513, 2048, 2049, 3121, 4096, 4097])
@pytest.mark.parametrize("mask", [False, True])
def test_soft_max_rows(wx, be, rng, n, mask):
    """Each row length bracket of the kernel; expf and the sum's rounding are
    a few 2^-24 each."""
    print(f"soft_max rows of {n} mask={mask}", flush=True)
    x = (rng.standard_normal((1, 3, 5, n)) * 4).astype(np.float32)
    m = rng.standard_normal((1, 3, 5, n)).astype(np.float32)
    g = G(wx, be)
    try:
        y = be.lib.wamx_soft_max_ext(g.ctx, g.leaf(wx, x, "f32"), g.leaf(wx, m, "f32") if mask else None, 0.125, 0.0)
        assert y, wx.last_error()
        got = g.run(y, "f32", x.shape)
        w = x.astype(np.float64) * 0.125 + (m if mask else 0)
        e = np.exp(w - w.max(-1, keepdims=True))
        assert np.allclose(got, e / e.sum(-1, keepdims=True), rtol=32 * 2.0 ** -24, atol=0)
    finally:
        g.close()


@pytest.mark.parametrize("mask", [False, True])
def test_soft_max_rows_of_no_elements(wx, be, rng, mask):
    """Nothing to read or write: the graph runs, and the soft_max of the
    tensor beside it in memory is what it is without the empty one."""
    print(f"soft_max rows of 0 mask={mask}", flush=True)
    x = rng.standard_normal((1, 1, 5, 7)).astype(np.float32)
    got = []
    for empty in (False, True):
        g = G(wx, be)
        try:
            outs = [be.lib.wamx_soft_max_ext(g.ctx, g.leaf(wx, x, "f32"), None, 1.0, 0.0)]
            if empty:
                m = g.t(wx.TYPE_F32, 0, 5) if mask else None
                outs.insert(0, be.lib.wamx_soft_max_ext(g.ctx, g.t(wx.TYPE_F32, 0, 5), m, 0.125, 0.0))
                assert outs[0], wx.last_error()
            g.alloc()
            g.set(*g.todo[0])
            g.compute(*outs)
            got.append(g.get(outs[-1], np.float32, x.shape))
        finally:
            g.close()
    assert np.array_equal(*got)


@pytest.mark.parametrize("n", [1, 7, 520, 70001])
@pytest.mark.parametrize("src,dst", [("f32", "f32"), ("f32", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("side", ["src", "dst"])
def test_reshaping_copy_of_a_transposed_row(wx, be, rng, n, src, dst, side):
    """A row [n] seen as [1, n] through a transpose: dense, but the stride of
    its first dim (one element) is the whole row.  Copied to, or filled from,
    a tensor of another shape, in memory order."""
    print(f"reshaping copy {n} {src}->{dst} transposed {side}", flush=True)
    a = rng.standard_normal((1, 1, 1, n)).astype(np.float32)
    g = G(wx, be)
    try:
        x = g.leaf(wx, a, src)
        d = g.t(TYPES[dst], n)
        if side == "src":
            y = be.lib.wamx_cpy(g.ctx, be.lib.wamx_transpose(g.ctx, x), d)
        else:
            y = be.lib.wamx_cpy(g.ctx, x, be.lib.wamx_transpose(g.ctx, d))
        assert y, wx.last_error()
        g.alloc()
        g.set(*g.todo[0])
        g.compute(y)
        assert np.array_equal(g.get(d, {"f32": np.float32, "bf16": np.uint16}[dst], a.shape), to_bits(wx, value(wx, a, src), dst))
    finally:
        g.close()
