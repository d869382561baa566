"""Products and the element-wise nodes after them, where their tensors share
memory: which nodes the product's launch takes along (an operand or the
product overwritten in place, an earlier output overwritten by a later one,
strided operands) and which stay apart (an operand or gate that overlaps an
earlier output, an output over the product's inputs or over another operand),
with tensors placed by the graph allocator and in two-lane graphs.  Values are
small integers, so f32 results are exact and bf16 ones are the rounding of
each node, whatever the order of summation; wamx_backend_fused_nodes says how
many nodes went along."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_fusion import Graph

pytestmark = pytest.mark.gpu


class Typ:
    def __init__(self, wx, name):
        self.wx, self.f32 = wx, name == "f32"
        self.id, self.size, self.dt = (wx.TYPE_F32, 4, np.float32) if self.f32 else (wx.TYPE_BF16, 2, np.uint16)

    def bits(self, a):
        a = np.asarray(a, np.float32)
        return a if self.f32 else self.wx.f32_to_bf16(a)

    def rnd(self, a):
        """What a node of this type that computes `a` reads back as."""
        a = np.asarray(a, np.float64).astype(np.float32)
        return (a if self.f32 else self.wx.bf16_to_f32(self.wx.f32_to_bf16(a))).astype(np.float64)


class Case(Graph):
    """Integer operands of a product M x N x K and the nodes after it."""

    def __init__(self, wx, be, typ, M, N, K):
        super().__init__(wx, be)
        self.T, self.M, self.N, self.K = Typ(wx, typ), M, N, K
        self.rng = np.random.default_rng(M + N + K)
        self.sets = []
        self.w, self.x, hw, hx = self.operands(M, N, K)
        self.p = self.lib.wamx_mul_mat_out_type(self.ctx, self.w, self.x, self.T.id)
        assert self.p, wx.last_error()
        self.P = self.T.rnd(hx @ hw.T)

    def operands(self, M, N, K):
        hw, hx = self.rng.integers(-1, 2, (M, K)), np.zeros((N, K), np.int64)
        for row in hx:  # 64 terms: |sums| <= 128, exact in bf16 too
            row[self.rng.choice(K, min(K, 64), replace=False)] = self.rng.integers(-2, 3, min(K, 64))
        return self.leaf(hw, K, M), self.leaf(hx, K, N), hw.astype(np.float64), hx.astype(np.float64)

    def leaf(self, a, *ne, typ=None):
        t = self.t(self.T.id if typ is None else typ, *ne)
        self.sets.append((t, a.astype(np.float32) if typ == self.wx.TYPE_F32 else self.T.bits(a)))
        return t

    def row(self):
        a = self.rng.integers(-9, 10, self.M).astype(np.float64)
        return self.leaf(a, self.M), a

    def full(self):
        a = self.rng.integers(-9, 10, (self.N, self.M)).astype(np.float64)
        return self.leaf(a, self.M, self.N), a

    def add(self, a, b):
        t = self.lib.wamx_add(self.ctx, a, b)
        assert t, self.wx.last_error()
        return t

    def mul(self, a, b):
        t = self.lib.wamx_mul(self.ctx, a, b)
        assert t, self.wx.last_error()
        return t

    def run(self, nodes, place=(), along=0):
        """Places `t` at `at` + offset bytes for each (t, at, offset), computes
        the nodes in order and checks how many went along with an earlier one."""
        self.alloc()
        for t, at, off in place:
            t.contents.data = at.contents.data + off
        for t, a in self.sets:
            self.set(t, a)
        before = self.lib.wamx_backend_fused_nodes(self.be.ptr)
        self.compute(*nodes)
        assert self.lib.wamx_backend_fused_nodes(self.be.ptr) - before == along

    def check(self, t, ref, what):
        assert np.array_equal(self.get(t, self.T.dt, ref.shape), self.T.bits(ref)), what


# f32: K slices and their reduce; bf16 also the one-launch kernel (1024 x 8).
SHAPES = [("f32", 1024, 33, 1024), ("bf16", 1024, 64, 1024), ("bf16", 1024, 8, 1024)]


@pytest.fixture(params=SHAPES, ids=lambda s: f"{s[0]}-{s[1]}x{s[2]}x{s[3]}")
def case(request, wx, be):
    c = Case(wx, be, *request.param)
    yield c
    c.close()


def test_residual_in_place(case):
    r, R = case.full()
    t = case.add(case.p, r)
    case.run([t], [(t, r, 0)], along=1)
    case.check(case.p, case.P, "product")
    case.check(t, case.T.rnd(case.P + R), "sum")


def test_bias_in_place_on_the_product(case):
    b, B = case.row()
    t = case.add(case.p, b)
    case.run([t], [(t, case.p, 0)], along=1)
    case.check(t, case.T.rnd(case.P + B), "sum")


def test_later_output_over_an_earlier_one(case):
    (b, B), (f, F), (h, H) = case.row(), case.full(), case.full()
    t1 = case.add(case.p, b)
    t2 = case.mul(t1, f)
    t3 = case.add(t2, h)
    case.run([t3], [(t2, case.p, 0), (t3, t1, 0)], along=3)
    v = case.T.rnd(case.T.rnd(case.P + B) * F)
    case.check(t2, v, "over the product")
    case.check(t3, case.T.rnd(v + H), "over the first sum")


def test_operand_of_two_nodes_overwritten_by_the_second(case):
    r, R = case.full()
    t1 = case.add(case.p, r)
    t2 = case.mul(t1, r)
    case.run([t2], [(t2, r, 0)], along=2)
    v = case.T.rnd(case.P + R)
    case.check(t1, v, "sum")
    case.check(t2, case.T.rnd(v * R), "product of the two")


@pytest.mark.parametrize("pad,along", [(4, 1), (3, 0)])
def test_strided_matrix_operand(case, pad, along):
    """Rows apart by a multiple of four elements go along, others do not."""
    a = case.rng.integers(-9, 10, (case.N, case.M + pad)).astype(np.float64)
    wide = case.leaf(a, case.M + pad, case.N)
    v = case.lib.wamx_view_2d(case.ctx, wide, case.M, case.N, wide.contents.nb[1], 0)
    t = case.add(case.p, v)
    case.run([t], along=along)
    case.check(t, case.T.rnd(case.P + a[:, :case.M]), "sum")


def test_operand_one_row_into_the_product_stays_apart(case):
    """The operand is the product seen one row on: it must read what the
    product wrote."""
    a = case.rng.integers(-9, 10, (case.N + 1, case.M)).astype(np.float64)
    room = case.leaf(a, case.M, case.N + 1)
    o = case.t(case.T.id, case.M, case.N)
    t = case.add(case.p, o)
    case.run([t], [(case.p, room, 0), (o, room, case.M * case.T.size)], along=0)
    case.check(t, case.T.rnd(case.P + np.vstack([case.P[1:], a[-1:]])), "sum")


@pytest.mark.parametrize("over", ["activations", "weight"])
def test_output_over_the_products_inputs_stays_apart(case, over):
    b, B = case.row()
    t = case.add(case.p, b)
    case.run([t], [(t, case.x if over == "activations" else case.w, 0)], along=0)
    case.check(case.p, case.P, "product")
    case.check(t, case.T.rnd(case.P + B), "sum")


def test_output_over_an_earlier_row_operand_stays_apart(case):
    """The second sum's output covers the first one's bias row."""
    (b, B), (f, F) = case.row(), case.full()
    t1 = case.add(case.p, b)
    t2 = case.add(t1, f)
    case.run([t2], [(b, t2, 64)], along=1)
    v = case.T.rnd(case.P + B)
    case.check(t1, v, "first sum")
    case.check(t2, case.T.rnd(v + F), "second sum")


@pytest.mark.parametrize("N", [64, 8])
def test_gate_that_is_a_row_of_the_product_stays_apart(wx, be, N):
    c = Case(wx, be, "bf16", 1024, N, 1024)
    try:
        r, R = c.full()
        gate = c.t(wx.TYPE_BF16, c.M)
        t = c.lib.wamx_gated_residual_bf16(c.ctx, r, c.p, gate)
        assert t, wx.last_error()
        c.run([t], [(gate, c.p, 0)], along=0)
        c.check(t, c.T.rnd(R + c.P * c.P[0]), "gated")
    finally:
        c.close()


@pytest.mark.parametrize("N", [64, 8])
@pytest.mark.parametrize("beside", [False, True])
def test_gate_inside_or_beside_a_later_output(wx, be, N, beside):
    """A gate that the node after the gated residual overwrites keeps that node
    apart; one that ends where the node's output begins does not."""
    c = Case(wx, be, "bf16", 1024, N, 1024)
    try:
        (r, R), (f, F) = c.full(), c.full()
        G = c.rng.integers(-3, 4, c.M).astype(np.float64)
        gate = c.leaf(G, c.M, typ=wx.TYPE_F32)
        t1 = c.lib.wamx_gated_residual_bf16(c.ctx, r, c.p, gate)
        t2 = c.add(t1, f)
        room = c.t(wx.TYPE_F32, c.M * (1 + c.N))
        c.run([t2], [(gate, room, 0), (t2, room, 4 * c.M if beside else 64)], along=2 if beside else 1)
        v = c.T.rnd(R + c.P * G)
        c.check(t1, v, "gated")
        c.check(t2, c.T.rnd(v + F), "sum")
    finally:
        c.close()


@pytest.mark.parametrize("IC,OC,IW,IH,B", [(32, 160, 160, 128, 1), (640, 640, 12, 10, 2), (320, 30, 13, 7, 1)])
@pytest.mark.parametrize("place", ["apart", "in place"])
def test_conv_bias_sum_in_place(wx, be, orc, IC, OC, IW, IH, B, place):
    """One K slice, several, and several with an odd number of pixels (the
    reduce's one-element form)."""
    print(f"conv + bias {place} {IC}->{OC} {IW}x{IH}x{B}", flush=True)
    rng = np.random.default_rng(IC + IW)
    k, x, b = (rng.integers(-2, 3, s).astype(np.float32) for s in ((OC, IC, 3, 3), (B, IC, IH, IW), (OC,)))
    bf = wx.f32_to_bf16
    g = Graph(wx, be)
    try:
        tk, tx, tb = g.t(30, 3, 3, IC, OC), g.t(30, IW, IH, IC, B), g.t(30, 1, 1, OC, 1)
        y = be.lib.wamx_conv_2d_direct(g.ctx, tk, tx, 1, 1, 1, 1, 1, 1)
        t = be.lib.wamx_add(g.ctx, y, tb)
        g.alloc()
        if place == "in place":
            t.contents.data = y.contents.data
        for q, a in ((tk, k), (tx, x), (tb, b)):
            g.set(q, bf(a))
        before = be.lib.wamx_backend_fused_nodes(be.ptr)
        g.compute(t)
        assert be.lib.wamx_backend_fused_nodes(be.ptr) - before == 1
        conv = wx.bf16_to_f32(bf(orc.conv_2d(k, x, 1, 1, 1, 1, 1, 1)))
        assert np.array_equal(g.get(t, np.uint16, conv.shape), bf(conv + b[:, None, None]))
        if place == "apart":
            assert np.array_equal(g.get(y, np.uint16, conv.shape), bf(conv))
    finally:
        g.close()


@pytest.mark.parametrize("typ,N", [("f32", 33), ("bf16", 8), ("bf16", 64)])
def test_chain_placed_by_the_graph_allocator(wx, be, typ, N):
    """x2 = x + x is scratch whose memory is free after the product: an output
    of the product's chain placed there would keep the nodes apart.  Two such
    layers, intermediates recycled between them."""
    M = 1024
    c = Case(wx, be, typ, M, N, M)  # leaves; its own product is not used
    lib, ga = be.lib, None
    ctx = lib.wamx_init(64)
    try:
        leaves = [(c.row(), c.full()) for _ in range(2)]
        hw, hx = (next(a for t, a in c.sets if t is s) for s in (c.w, c.x))
        hw, hx = ((a if typ == "f32" else wx.bf16_to_f32(a)).astype(np.float64) for a in (hw, hx))
        c.alloc()
        for t, a in c.sets:
            c.set(t, a)
        cur, ref = c.x, hx
        for (b, B), (f, F) in leaves:
            x2 = lib.wamx_add(ctx, cur, cur)
            p = lib.wamx_mul_mat_out_type(ctx, c.w, x2, c.T.id)
            cur = lib.wamx_add(ctx, lib.wamx_add(ctx, p, b), f)
            ref = c.T.rnd(c.T.rnd(c.T.rnd(c.T.rnd(2 * ref) @ hw.T) + B) + F)
        assert np.abs(ref).max() < 2 ** 24
        lib.wamx_set_output(cur)
        g = lib.wamx_new_graph(ctx, 64)
        lib.wamx_build_forward_expand(g, cur)
        ga = lib.wamx_gallocr_new(be.ptr)
        assert lib.wamx_gallocr_alloc_graph(ga, g), wx.last_error()
        for _ in range(2):
            before = lib.wamx_backend_fused_nodes(be.ptr)
            wx.check(lib.wamx_backend_graph_compute(be.ptr, g), "graph_compute")
            be.sync()
            assert lib.wamx_backend_fused_nodes(be.ptr) - before == 4
            c.check(cur, ref, "second layer")
    finally:
        if ga:
            lib.wamx_gallocr_free(ga)
        lib.wamx_free(ctx)
        c.close()


@pytest.mark.parametrize("capture", [True, False])
@pytest.mark.parametrize("form,along", [("reads_product", 2), ("writes_operand", 0), ("reads_sum", 2)])
def test_chain_in_a_two_lane_graph(wx, be, form, along, capture):
    """Lane 0: p = x w, t = p + r, u = t * f.  Lane 1, built between them,
    reads the product (or the sum) that the fused launch writes, or overwrites
    the operand r before the sum reads it, which keeps the nodes apart."""
    print(f"chain beside another lane: {form} capture={capture}", flush=True)
    c = Case(wx, be, "f32", 1024, 33, 1024)
    lib = be.lib
    try:
        (r, R), (f, F), (z, Z) = c.full(), c.full(), c.full()
        nodes = [c.p]
        if form == "writes_operand":
            lib.wamx_set_lane(c.ctx, 1)
            r2 = lib.wamx_cpy(c.ctx, z, r)
            nodes.append(r2)
            lib.wamx_set_lane(c.ctx, 0)
            t, R = c.add(c.p, r), Z
        else:
            t = c.add(c.p, r)
        u = c.mul(t, f)
        if form != "writes_operand":
            lib.wamx_set_lane(c.ctx, 1)
            q = c.mul(c.p if form == "reads_product" else t, z)
            nodes += [q] if form == "reads_product" else [t, q]
        nodes += [u]
        c.alloc()
        g = lib.wamx_new_graph(c.ctx, 64)
        for n in nodes:
            lib.wamx_build_forward_expand(g, n)
        if capture:
            lib.wamx_graph_assign_uid(g)
        for run in range(3):
            for s, a in c.sets:
                c.set(s, a)
            before = lib.wamx_backend_fused_nodes(be.ptr)
            wx.check(lib.wamx_backend_graph_compute(be.ptr, g), "graph_compute")
            be.sync()
            if run == 0 or not capture:
                assert lib.wamx_backend_fused_nodes(be.ptr) - before == along
            c.check(c.p, c.P, "product")
            c.check(t, c.P + R, "sum")
            c.check(u, (c.P + R) * F, "product of the sum")
            if form != "writes_operand":
                c.check(q, (c.P if form == "reads_product" else c.P + R) * Z, "other lane")
    finally:
        c.close()
