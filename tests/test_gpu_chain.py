"""Element-wise nodes after a product, applied by the product's own reduce: the
same bits in every node's output as the nodes computed apart (the product
fetched and fed to a graph of the element-wise nodes alone), for products that
split along K and products that do not, and with operands that keep the nodes
apart (an operand that is a view of the product, a row length that is not a
multiple of 4)."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_fusion import Graph

pytestmark = pytest.mark.gpu

CHAINS = {
    "bias": ["row"], "bias_residual": ["row", "add"], "bias_gate_residual": ["row", "mulrow", "add"],
    "residual": ["radd"], "gelu": ["gelu"], "mul": ["mul"], "bias_gelu_mul": ["row", "gelu", "mul"],
    "gated": ["row", "gated"], "bias_gelu_node": ["biasgelu"], "self": ["selfview"], "four": ["row", "add", "mul", "row"],
}
BF16_ONLY = {"gated", "bias_gelu_node"}
SHAPES = [(3072, 48, 3072), (3072, 1, 14336), (1000, 33, 1024), (14336, 16, 256), (258, 20, 1024), (3072, 64, 4104)]


def stage(wx, lib, g, kind, cur, leaf):
    if kind == "row":
        return lib.wamx_add(g.ctx, cur, leaf("row"))
    if kind == "add":
        return lib.wamx_add(g.ctx, cur, leaf("full"))
    if kind == "radd":
        return lib.wamx_add(g.ctx, leaf("full"), cur)
    if kind == "mulrow":
        return lib.wamx_mul(g.ctx, cur, leaf("row"))
    if kind == "mul":
        return lib.wamx_mul(g.ctx, cur, leaf("full"))
    if kind == "gelu":
        return lib.wamx_gelu(g.ctx, cur)
    if kind == "gated":
        return lib.wamx_gated_residual_bf16(g.ctx, leaf("full"), cur, leaf("gate"))
    if kind == "biasgelu":
        return lib.wamx_bias_gelu_bf16(g.ctx, cur, leaf("row"))
    # an operand that is the product itself, seen through a reshape
    t = cur.contents
    return lib.wamx_add(g.ctx, cur, lib.wamx_reshape_2d(g.ctx, cur, t.ne[0], t.ne[1]))


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("chain", list(CHAINS))
@pytest.mark.parametrize("typ", ["f32", "bf16"])
def test_chain_same_bits_as_nodes_apart(wx, be, M, N, K, chain, typ):
    if chain in BF16_ONLY and typ == "f32":
        pytest.skip("a bf16 node")
    print(f"chain {chain} {typ} {M}x{N}x{K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    lib, T = be.lib, wx.TYPE_F32 if typ == "f32" else wx.TYPE_BF16
    dt = np.float32 if typ == "f32" else np.uint16
    bits = lambda a: np.asarray(a, np.float32) if typ == "f32" else wx.f32_to_bf16(np.asarray(a, np.float32))  # noqa: E731
    w, x = rng.standard_normal((M, K)) * 0.02, rng.standard_normal((N, K))
    data = [{"row": rng.standard_normal(M), "full": rng.standard_normal((N, M)), "gate": rng.standard_normal(M)}
            for _ in CHAINS[chain]]

    def build(g, cur, sets):
        outs = []
        for kind, d in zip(CHAINS[chain], data):
            def leaf(what, d=d):
                t = g.t(wx.TYPE_F32 if what == "gate" else T, *reversed(d[what].shape))
                sets.append((t, d[what].astype(np.float32) if what == "gate" else bits(d[what])))
                return t
            cur = stage(wx, lib, g, kind, cur, leaf)
            assert cur, wx.last_error()
            outs.append(cur)
        return outs

    def run(g, outs, sets):
        g.alloc()
        for t, a in sets:
            g.set(t, a)
        g.compute(outs[-1])
        return [g.get(t, dt, (N, M)) for t in outs]

    g = Graph(wx, be)
    try:
        sets = []
        tw, tx = g.t(T, K, M), g.t(T, K, N)
        sets += [(tw, bits(w)), (tx, bits(x))]
        mm = lib.wamx_mul_mat_out_type(g.ctx, tw, tx, T)
        assert mm, wx.last_error()
        got = run(g, [mm] + build(g, mm, sets), sets)
    finally:
        g.close()
    g = Graph(wx, be)
    try:
        sets = []
        leaf = g.t(T, M, N)
        sets.append((leaf, got[0]))
        apart = run(g, build(g, leaf, sets), sets)
    finally:
        g.close()
    for a, b in zip(got[1:], apart):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    # and the product itself is the product
    ref = (x if typ == "f32" else wx.bf16_to_f32(bits(x)).astype(np.float64)) @ \
        (w if typ == "f32" else wx.bf16_to_f32(bits(w)).astype(np.float64)).T
    p = got[0] if typ == "f32" else wx.bf16_to_f32(got[0])
    assert np.abs(p - ref).max() <= 1e-2 * np.abs(ref).max()


@pytest.mark.parametrize("IC,OC,IW,IH,B", [(160, 160, 40, 33, 1), (640, 640, 12, 10, 2), (12, 30, 50, 20, 1)])
def test_conv_bias_same_bits_as_nodes_apart(wx, be, IC, OC, IW, IH, B):
    print(f"conv + bias {IC}->{OC} {IW}x{IH}x{B}", flush=True)
    rng = np.random.default_rng(IC)
    lib = be.lib
    k, x, b = (wx.f32_to_bf16(rng.standard_normal(s).astype(np.float32)) for s in ((OC, IC, 3, 3), (B, IC, IH, IW), (OC,)))
    def run(g, outs, sets):
        g.alloc()
        for t, a in sets:
            g.set(t, a)
        g.compute(outs[-1])
        return [g.get(t, np.uint16, (B, OC, IH, IW)) for t in outs]
    g = Graph(wx, be)
    try:
        tk, tx, tb = g.t(30, 3, 3, IC, OC), g.t(30, IW, IH, IC, B), g.t(30, 1, 1, OC, 1)
        y = lib.wamx_conv_2d_direct(g.ctx, tk, tx, 1, 1, 1, 1, 1, 1)
        conv, out = run(g, [y, lib.wamx_add(g.ctx, y, tb)], [(tk, k), (tx, x), (tb, b)])
    finally:
        g.close()
    g = Graph(wx, be)
    try:
        ty, tb = g.t(30, IW, IH, OC, B), g.t(30, 1, 1, OC, 1)
        apart, = run(g, [lib.wamx_add(g.ctx, ty, tb)], [(ty, conv), (tb, b)])
    finally:
        g.close()
    assert np.array_equal(out, apart)


@pytest.mark.parametrize("node,IC,OC,IW,IH", [(n, *s) for n in ("gelu", "bias_gelu") for s in
                                              ((32, 160, 40, 33), (640, 640, 12, 10), (32, 1, 40, 33))] +
                         [("gated", 32, 1, 40, 33)])  # 2-D tensors only
def test_conv_before_other_nodes_runs_apart(wx, be, node, IC, OC, IW, IH):
    """A convolution followed by GELU, bias + GELU (a bias per column of the
    image: more output channels than bias values) or, with one output channel,
    a gated residual: nodes that its epilogue does not know, in one K slice and
    in several.  The same bits as the node on the fetched convolution."""
    print(f"conv + {node} {IC}->{OC} {IW}x{IH}", flush=True)
    rng = np.random.default_rng(IC + OC)
    lib = be.lib
    k, x, row, full = (wx.f32_to_bf16(rng.standard_normal(s).astype(np.float32))
                       for s in ((OC, IC, 3, 3), (1, IC, IH, IW), (IW,), (IH, IW)))
    gate = rng.standard_normal(IW).astype(np.float32)

    def run(conv):
        """(convolution, node): the node after the convolution, or on `conv`."""
        g = Graph(wx, be)
        try:
            sets, outs = [], []
            def leaf(a, typ, *ne):
                t = g.t(typ, *ne)
                sets.append((t, a))
                return t
            if conv is None:
                cur = lib.wamx_conv_2d_direct(g.ctx, leaf(k, wx.TYPE_BF16, 3, 3, IC, OC),
                                              leaf(x, wx.TYPE_BF16, IW, IH, IC, 1), 1, 1, 1, 1, 1, 1)
                outs.append(cur)
            else:
                cur = leaf(conv, wx.TYPE_BF16, IW, IH, OC, 1)
            if node == "gelu":
                y = lib.wamx_gelu(g.ctx, cur)
            elif node == "bias_gelu":
                y = lib.wamx_bias_gelu_bf16(g.ctx, cur, leaf(row, wx.TYPE_BF16, IW))
            else:
                y = lib.wamx_gated_residual_bf16(g.ctx, leaf(full, wx.TYPE_BF16, IW, IH), cur,
                                                 leaf(gate, wx.TYPE_F32, IW))
            assert y, wx.last_error()
            outs.append(y)
            g.alloc()
            for t, a in sets:
                g.set(t, a)
            g.compute(y)
            return [g.get(t, np.uint16, (1, OC, IH, IW)) for t in outs]
        finally:
            g.close()

    conv, got = run(None)
    apart, = run(conv)
    assert np.array_equal(got, apart)
