"""The work that a program has this backend do, as cases that can be timed.

Each case names a kind of call, its sizes and its data types.  The kinds are
the layers and requests of a GWP-0.5-shaped policy as the backend is used:

  linear     one projection of a few tokens (the state token, the 48 action
             tokens, a prompt), weights row-major or in the tiled layout
  mul_mat    one MUL_MAT of more tokens with f32 or bf16 activations
  ffn        the visual expert's FFN half: adaLN norm, up + GELU, down + gated
             residual, on the tokens of one canvas
  attention  Q (and K) norm + RoPE and the attention over resident keys, as a
             computed graph: the prefix pass (many queries) and the denoise
             step (48 queries over the cached prefix and their own keys)
  layer      one action-expert layer as an unfused ggml graph, which is what a
             ggml host submits: in the bf16 profile and in the f32 reference
             profile
  conv       one VAE encoder convolution with its bias
  t5         one prompt through the UMT5 text encoder
  chunk      one whole request of the model driver: upload, prompt projection,
             prefix pass, unrolled flow-matching denoise, actions back

Inputs come from the seed alone.  Tensors are torch's; the backend takes
their device pointers and runs on a blocking stream, which the null stream
that torch uses is ordered with.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "wam.cpp_amd"))

import wamx  # noqa: E402

EPS = 1e-6
BF16, F32, I32 = wamx.TYPE_BF16, wamx.TYPE_F32, wamx.TYPE_I32
EPI = {"none": wamx.EPI_NONE, "bias": wamx.EPI_BIAS, "gelu": wamx.EPI_BIAS_GELU, "gated": wamx.EPI_BIAS_GATED,
       "residual": wamx.EPI_BIAS_RESIDUAL}
# Widths of the policy: hidden 3072 = 24 heads of 128, FFN 14336.
D, HEADS, DH, FFN = 3072, 24, 128, 14336


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The state token's QKV-sized product: one token, all latency and weight bytes.
        dict(name="linear_1_token", kind="linear", m=3072, n=1, k=3072, tiled=False, x="bf16", epi="bias"),
        # FFN-up of the 48-token action expert, weights in the tiled buffer type (the denoise step's largest product).
        dict(name="linear_48_tiled", kind="linear", m=14336, n=48, k=3072, tiled=True, x="bf16", epi="gelu"),
        # The benchmark's single MUL_MAT: f32 activations, f32 result.
        dict(name="mul_mat_256_f32", kind="mul_mat", m=3072, n=256, k=3072, x="f32", y="f32"),
        # The visual FFN at the published canvas (384 x 320 pixels: 120 visual tokens).
        dict(name="ffn_120", kind="ffn", n=120),
        # The benchmark's FFN block.
        dict(name="ffn_2048", kind="ffn", n=2048),
        # Prefix self-attention of 3 x 1024 visual tokens and the state token.
        dict(name="attention_prefix", kind="attention", tq=3072, na=3073, nb=0, own_k=True),
        # One denoise step's attention: 48 action queries over the cached prefix and their own keys.
        dict(name="attention_denoise", kind="attention", tq=48, na=3073, nb=48, own_k=False),
        # An action layer as a ggml host submits it, bf16 profile, over a 3073-key prefix and a 512-token prompt.
        dict(name="layer_bf16", kind="layer", profile="bf16", t=48, prefix=3073, prompt=512),
        # The same in the f32 reference profile, at the published geometry (120 visual tokens, 64 prompt tokens).
        dict(name="layer_f32", kind="layer", profile="f32", t=48, prefix=121, prompt=64),
        # The VAE encoder's first-level residual convolution for a 384 x 320 image.
        dict(name="conv_vae", kind="conv", ic=160, oc=160, w=192, h=160, ks=3, s=1, p=1),
        # A full 64-token prompt through the XXL-sized encoder.
        dict(name="t5_xxl", kind="t5", layers=24, hidden=4096, ffn=10240, heads=64, tokens=64),
        # A whole request at the published canvas with the default depth, widths and prompt length.
        dict(name="chunk", kind="chunk", layers=30, grid_h=10, grid_w=12, prompt=512, steps=10, batch=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "mul_mat", "ffn", "attention", "layer", "conv", "t5", "chunk"])
    if kind == "linear":
        tiled = rng.random() < 0.5
        # The policy's widths, and others as a smaller action expert has them.
        m = rng.choice([1024, 1536, 2304, 3072, 4096, 9216, 14336, 16 * rng.randint(24, 500)])
        k = rng.choice([1024, 2048, 3072, 4096, 14336, 32 * rng.randint(12, 200)])
        return dict(kind=kind, m=m, n=_log(rng, 1, 64), k=k, tiled=tiled, x=rng.choice(["bf16", "bf16", "f32"]),
                    epi=rng.choice(["none", "bias", "gelu", "gated", "residual"]))
    if kind == "mul_mat":
        m = rng.choice([1024, 3072, 4096, 9216, 14336, rng.randint(300, 9000)])
        k = rng.choice([1024, 3072, 4096, 14336, 8 * rng.randint(40, 900)])
        return dict(kind=kind, m=m, n=_log(rng, 65, 2048), k=k, x=rng.choice(["f32", "bf16"]),
                    y=rng.choice(["f32", "bf16"]))
    if kind == "ffn":
        return dict(kind=kind, n=_log(rng, 65, 3072))
    if kind == "attention":
        if rng.random() < 0.5:  # prefix: every token's queries over all keys
            na = _log(rng, 81, 3073)
            return dict(kind=kind, tq=na - 1, na=na, nb=0, own_k=True)
        return dict(kind=kind, tq=rng.choice([16, 24, 32, 48, 48, 64]), na=_log(rng, 64, 4097),
                    nb=rng.choice([0, 16, 48]), own_k=False)
    if kind == "layer":
        return dict(kind=kind, profile=rng.choice(["bf16", "f32"]), t=rng.choice([16, 33, 48, 48, 64]),
                    prefix=1 + _log(rng, 64, 3072), prompt=rng.choice([16, 64, 77, 128, 512]))
    if kind == "conv":
        ks, s, p = rng.choice([(3, 1, 1), (3, 1, 1), (3, 2, 0), (1, 1, 0)])
        level = rng.choice([(160, 1), (160, 2), (320, 2), (320, 4), (640, 4), (640, 8)])
        ic = rng.choice([level[0], level[0], max(12, level[0] // 2)])
        return dict(kind=kind, ic=ic, oc=level[0], w=rng.randint(120, 192) // level[1] + (s == 2),
                    h=rng.randint(96, 160) // level[1] + (s == 2), ks=ks, s=s, p=p)
    if kind == "t5":
        heads = rng.randint(16, 64)
        return dict(kind=kind, layers=rng.randint(2, 24), hidden=64 * heads, ffn=32 * rng.randint(80, 320), heads=heads,
                    tokens=_log(rng, 6, 64))
    return dict(kind="chunk", layers=rng.randint(2, 8), grid_h=rng.randint(6, 16), grid_w=rng.randint(8, 24),
                prompt=rng.choice([72, 77, 128, 200]), steps=rng.choice([4, 10]), batch=rng.choice([1, 1, 1, 2, 4]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
_BE = None


def _backend():
    """The process's backend (a program opens one per GPU)."""
    global _BE
    if _BE is None:
        _BE = wamx.Backend(0)
    return _BE


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    if std != 1.0:
        x.mul_(std)
    if mean:
        x.add_(mean)
    return x.to(dtype)


def _weight(g, m, k, dtype=torch.bfloat16):
    return _normal(g, (m, k), 0.02, dtype=dtype)


class _Device:
    """Device memory of `state` as an array interface, which keeps `state` alive."""

    def __init__(self, state, ptr, n, typestr):
        self.state = state
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


class Graph:
    """One computed graph: leaves and outputs are torch tensors, intermediates the graph allocator's."""

    def __init__(self, tensors=256):
        self.be = _backend()
        self.lib = self.be.lib
        self.ctx = self.lib.wamx_init(tensors)
        self.galloc = None
        self.kept = []

    def __getattr__(self, name):  # g.mul_mat(a, b) is wamx_mul_mat(ctx, a, b)
        fn = getattr(self.lib, "wamx_" + name)

        def call(*args):
            t = fn(self.ctx, *args)
            if not t:
                raise RuntimeError(f"wamx_{name}: {wamx.last_error()}")
            return t

        return call

    def leaf(self, x, *ne):
        """A graph tensor over torch tensor x (ne: ggml order, default x's shape reversed)."""
        ne = list(ne) or list(reversed(x.shape))
        typ = {torch.bfloat16: BF16, torch.float32: F32, torch.int32: I32}[x.dtype]
        t = self.lib.wamx_new_tensor_4d(self.ctx, typ, *(ne + [1] * (4 - len(ne))))
        t.contents.data = x.data_ptr()
        self.lib.wamx_set_input(t)
        self.kept.append(x)
        return t

    def out(self, t, x):
        """Places node t in torch tensor x."""
        t.contents.data = x.data_ptr()
        self.lib.wamx_set_output(t)
        self.kept.append(x)
        return t

    def finish(self, *outputs):
        self.graph = self.lib.wamx_new_graph(self.ctx, 256)
        for t in outputs:
            self.lib.wamx_build_forward_expand(self.graph, t)
        self.lib.wamx_graph_assign_uid(self.graph)
        self.galloc = self.lib.wamx_gallocr_new(self.be.ptr)
        if not self.lib.wamx_gallocr_alloc_graph(self.galloc, self.graph):
            raise RuntimeError("graph allocation failed: " + wamx.last_error())

    def compute(self):
        wamx.check(self.lib.wamx_backend_graph_compute(self.be.ptr, self.graph), "graph_compute")

    def __del__(self):
        if getattr(self, "galloc", None):
            self.lib.wamx_gallocr_free(self.galloc)
        if getattr(self, "ctx", None):
            self.lib.wamx_free(self.ctx)


def _pad8(n):
    return (n + 7) // 8 * 8


def _linear_inputs(c, seed):
    g = _gen(seed)
    s = {"w": _weight(g, c["m"], c["k"]), "x": _normal(g, (c["n"], c["k"]), dtype=getattr(torch, {"bf16": "bfloat16", "f32": "float32"}[c["x"]]))}
    s["bias"] = _normal(g, (c["m"],), 0.02)
    s["res"] = _normal(g, (c["n"], c["m"]))
    s["gate"] = _normal(g, (c["m"],), 0.5, dtype=torch.float32)
    return s


def _prepare_linear(c, seed):
    s = _linear_inputs(c, seed)
    be = _backend()
    s["y"] = torch.empty((c["n"], c["m"]), device="cuda", dtype=torch.bfloat16)
    w = s["w"].data_ptr()
    if c["tiled"]:
        # The weight lives in a tensor of the tiled buffer type, set once.
        lib = be.lib
        rows, held = lib.wamx_init(4), lib.wamx_init(4)
        src = lib.wamx_new_tensor_2d(rows, BF16, c["k"], c["m"])
        src.contents.data = w
        dst = lib.wamx_new_tensor_2d(held, BF16, c["k"], c["m"])
        buf = lib.wamx_backend_alloc_ctx_tensors_from_buft(held, lib.wamx_backend_tiled_buffer_type(0))
        torch.cuda.synchronize()
        wamx.check(lib.wamx_backend_tensor_copy(src, dst), "tiled weight")
        lib.wamx_free(rows)
        s["tiled_weight"] = _Held(lib, held, buf)
        w = dst.contents.data
        del s["w"]
    epi = EPI[c["epi"]]
    ptr = lambda k, on: s[k].data_ptr() if on else None  # noqa: E731
    fn = be.lib.wamx_op_linear_tiled if c["tiled"] else be.lib.wamx_op_linear
    args = (be.ptr, w, s["x"].data_ptr(), BF16 if c["x"] == "bf16" else F32, ptr("bias", c["epi"] != "none"), epi,
            ptr("res", c["epi"] in ("gated", "residual")), ptr("gate", c["epi"] == "gated"), s["y"].data_ptr(), c["m"],
            c["n"], c["k"])
    s["call"] = lambda: wamx.check(fn(*args), "linear")
    s["outputs"] = s["y"]
    return s


class _Held:
    """A context and its buffer, freed with the state."""

    def __init__(self, lib, ctx, buf):
        self.lib, self.ctx, self.buf = lib, ctx, buf

    def __del__(self):
        self.lib.wamx_buffer_free(self.buf)
        self.lib.wamx_free(self.ctx)


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _exact_linear(c, seed):
    s = _linear_inputs(c, seed)
    x = s["x"].to(torch.bfloat16).double()  # the op's products take bf16 activations
    y = x @ s["w"].double().T
    if c["epi"] == "none":
        return y
    y = y + s["bias"].double()
    if c["epi"] == "gelu":
        return _gelu64(y)
    if c["epi"] == "gated":
        return s["res"].double() + y * s["gate"].double()
    return s["res"].double() + y if c["epi"] == "residual" else y


def _prepare_mul_mat(c, seed):
    g = _gen(seed)
    be = _backend()
    s = {"w": _weight(g, c["m"], c["k"]), "x": _normal(g, (c["n"], c["k"]), dtype=torch.float32 if c["x"] == "f32" else torch.bfloat16)}
    s["y"] = torch.empty((c["n"], c["m"]), device="cuda", dtype=torch.float32 if c["y"] == "f32" else torch.bfloat16)
    args = (be.ptr, s["w"].data_ptr(), c["k"], s["x"].data_ptr(), F32 if c["x"] == "f32" else BF16, c["k"],
            s["y"].data_ptr(), F32 if c["y"] == "f32" else BF16, c["m"], c["m"], c["n"], c["k"])
    s["call"] = lambda: wamx.check(be.lib.wamx_op_mul_mat(*args), "mul_mat")
    s["outputs"] = s["y"]
    return s


def _exact_mul_mat(c, seed):
    g = _gen(seed)
    w = _weight(g, c["m"], c["k"])
    x = _normal(g, (c["n"], c["k"]), dtype=torch.float32).to(torch.bfloat16)
    return x.double() @ w.double().T


def _ffn_inputs(c, seed):
    g = _gen(seed)
    n = c["n"]
    return {"x": _normal(g, (n, D)), "shift": _normal(g, (D,), 0.1, dtype=torch.float32),
            "scale": _normal(g, (D,), 0.1, dtype=torch.float32), "gate": _normal(g, (D,), 0.1, dtype=torch.float32),
            "wu": _weight(g, FFN, D), "bu": _normal(g, (FFN,), 0.02), "wd": _weight(g, D, FFN),
            "bd": _normal(g, (D,), 0.02)}


def _prepare_ffn(c, seed):
    s = _ffn_inputs(c, seed)
    n, lib, be = c["n"], _backend().lib, _backend().ptr
    s["h"], s["u"], s["y"] = (torch.empty((n, k), device="cuda", dtype=torch.bfloat16) for k in (D, FFN, D))
    p = {k: v.data_ptr() for k, v in s.items()}

    def call():
        wamx.check(lib.wamx_op_norm_modulation_bf16(be, p["x"], D, p["scale"], p["shift"], 0, p["h"], n, D, EPS))
        wamx.check(lib.wamx_op_linear(be, p["wu"], p["h"], BF16, p["bu"], EPI["gelu"], None, None, p["u"], FFN, n, D))
        wamx.check(lib.wamx_op_linear(be, p["wd"], p["u"], BF16, p["bd"], EPI["gated"], p["x"], p["gate"], p["y"], D, n,
                                      FFN))

    s["call"] = call
    s["outputs"] = [s["h"], s["u"], s["y"]]
    return s


def _ln64(x):
    mu = x.mean(-1, keepdim=True)
    return (x - mu) / torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + EPS)


def _exact_ffn(c, seed):
    s = {k: v.double() for k, v in _ffn_inputs(c, seed).items()}
    h = _ln64(s["x"]) * (1 + s["scale"]) + s["shift"]
    u = _gelu64(h @ s["wu"].T + s["bu"])
    return [h, u, s["x"] + (u @ s["wd"].T + s["bd"]) * s["gate"]]


def _attention_inputs(c, seed):
    g = _gen(seed)
    tq, na, nb = c["tq"], c["na"], c["nb"]
    s = {"xq": _normal(g, (tq, D)), "wq": _normal(g, (D,), 0.02, 1.0), "ka": _normal(g, (HEADS, na, DH)),
         "va": _normal(g, (HEADS, DH, na))}
    if c["own_k"]:  # K of the tokens after the state's is normalised and rotated here too
        s["xk"], s["wk"] = _normal(g, (tq, D)), _normal(g, (D,), 0.02, 1.0)
    if nb:
        s["kb"], s["vb"] = _normal(g, (HEADS, nb, DH)), _normal(g, (HEADS, DH, nb))
    # The prefix rotates by the (t, h, w) grid position, the action tokens by 1..T.
    i = torch.arange(tq, device="cuda", dtype=torch.int32)
    side = max(1, int(math.sqrt(tq)))
    s["pos"] = [torch.zeros_like(i), i // side, i % side] if c["own_k"] else [i + 1]
    return s


def _prepare_attention(c, seed):
    s = _attention_inputs(c, seed)
    tq, na, nb = c["tq"], c["na"], c["nb"]
    g = Graph()

    def vt(v, n):  # V^T rows padded to a multiple of 8 keys
        rows = torch.zeros((HEADS, DH, _pad8(n)), device="cuda", dtype=torch.bfloat16)
        rows[:, :, :n] = v
        t = g.leaf(rows)
        return g.view_3d(t, n, DH, HEADS, 2 * _pad8(n), 2 * _pad8(n) * DH, 0)

    s["q"] = torch.empty((HEADS, tq, DH), device="cuda", dtype=torch.bfloat16)
    s["y"] = torch.empty((tq, D), device="cuda", dtype=torch.bfloat16)
    mode = 1 if c["own_k"] else 0
    pos = [g.leaf(p) for p in s["pos"]] + [None] * (3 - len(s["pos"]))
    q = g.qk_norm_rope(g.leaf(s["xq"]), g.leaf(s["wq"]), g.leaf(s["q"]), 0, mode, *pos, EPS, 10000.0)
    ka = g.leaf(s["ka"])
    if c["own_k"]:
        ka = g.qk_norm_rope(g.leaf(s["xk"]), g.leaf(s["wk"]), ka, 1, mode, *pos, EPS, 10000.0)
    va = vt(s["va"], na)
    kb, vb = (g.leaf(s["kb"]), vt(s["vb"], nb)) if nb else (None, None)
    y = g.out(g.joint_attn(q, ka, va, kb, vb, 1 if nb else 0, 1 / math.sqrt(DH)), s["y"])
    g.finish(y)
    s["call"] = g.compute
    s["graph"] = g
    s["outputs"] = [s["q"], s["ka"], s["y"]] if c["own_k"] else [s["q"], s["y"]]
    return s


def _rope64(x, pos):
    """x [T, H, dh] rotated in (even, odd) pairs: one position over dh, or three over {44, 42, 42}."""
    out = torch.empty_like(x)
    at = 0
    for n, p in zip([x.shape[2]] if len(pos) == 1 else (44, 42, 42), pos):
        i = torch.arange(n // 2, device=x.device, dtype=torch.float64)
        th = (p.double()[:, None] * 10000.0 ** (-2 * i / n))[:, None, :]
        a, b = x[..., at:at + n:2], x[..., at + 1:at + n:2]
        out[..., at:at + n:2] = a * th.cos() - b * th.sin()
        out[..., at + 1:at + n:2] = a * th.sin() + b * th.cos()
        at += n
    return out


def _rms64(x, w):
    return x / torch.sqrt((x ** 2).mean(-1, keepdim=True) + EPS) * w


def _attend64(q, k, vt):
    """q [H, T, dh], k [H, n, dh], vt [H, dh, n] -> [T, H * dh]."""
    out = []
    for h in range(q.shape[0]):
        p = torch.softmax(q[h] @ k[h].T / math.sqrt(q.shape[2]), -1)
        out.append(p @ vt[h].T)
    return torch.cat(out, 1)


def _exact_attention(c, seed):
    s = {k: v if k == "pos" else v.double() for k, v in _attention_inputs(c, seed).items()}
    head = lambda x, w: _rope64(_rms64(x, w).reshape(c["tq"], HEADS, DH), s["pos"]).transpose(0, 1)  # noqa: E731
    q = head(s["xq"], s["wq"])
    k, v = s["ka"], s["va"]
    if c["own_k"]:
        k = torch.cat([k[:, :1], head(s["xk"], s["wk"])], 1)
        return [q, k, _attend64(q, k, v)]
    if c["nb"]:
        k, v = torch.cat([k, s["kb"]], 1), torch.cat([v, s["vb"]], 2)
    return [q, _attend64(q, k, v)]


_LAYER = {"attn1.norm_q": None, "attn1.norm_k": None, "attn1.to_out.0": (D, D), "norm2": None, "attn2.to_q": (D, D),
          "attn2.norm_q": None, "attn2.to_out.0": (D, D), "ffn.net.0.proj": (FFN, D), "ffn.net.2": (D, FFN)}


def _layer_inputs(c, seed):
    g = _gen(seed)
    typ = torch.bfloat16 if c["profile"] == "bf16" else torch.float32
    t, p, nl = c["t"], c["prefix"], c["prompt"]
    w = {}
    qkv = {"attn1.to_qkv": (3 * D, D)} if c["profile"] == "bf16" else {f"attn1.to_{i}": (D, D) for i in "qkv"}
    for name, shape in {**qkv, **_LAYER}.items():
        if shape:
            w[name + ".weight"] = _weight(g, *shape, dtype=typ)
            w[name + ".bias"] = _normal(g, (shape[0],), 0.02, dtype=typ)
        else:
            w[name + ".weight"] = _normal(g, (D,), 0.02, 1.0, dtype=typ)
            if name == "norm2":
                w[name + ".bias"] = _normal(g, (D,), 0.02, dtype=typ)
    s = {"h": _normal(g, (t, D), dtype=typ), "mod": _normal(g, (6, D), 0.5, dtype=typ),
         "table": _normal(g, (6, D), 0.1, dtype=typ), "pk": _normal(g, (HEADS, p, DH), dtype=typ),
         "pv": _normal(g, (HEADS, DH, p), dtype=typ), "lk": _normal(g, (HEADS, nl, DH), dtype=typ),
         "lv": _normal(g, (HEADS, DH, nl), dtype=typ)}
    s["pos"] = torch.arange(1, t + 1, device="cuda", dtype=torch.int32)
    return w, s


def _prepare_layer(c, seed):
    """The nodes a ggml host builds for one action-expert layer over the cached prefix and prompt."""
    w, s = _layer_inputs(c, seed)
    bf = c["profile"] == "bf16"
    es, t, p = 2 if bf else 4, c["t"], c["prefix"]
    g = Graph(512)
    lib = g.lib
    wt = {k: g.leaf(v) for k, v in w.items()}
    lf = {k: g.leaf(v) for k, v in s.items()}

    def linear(name, x):
        if bf:
            if x.contents.type != BF16:
                x = g.cast(x, BF16)
            return g.add(g.mul_mat_out_type(wt[name + ".weight"], x, BF16), wt[name + ".bias"])
        return g.add(g.mul_mat(wt[name + ".weight"], x), wt[name + ".bias"])

    def rms(x, name):
        n = wt[name + ".weight"]
        return g.rms_norm_bf16_f32(x, n, EPS) if bf else g.mul(g.rms_norm(x, EPS), g.cast(n, F32))

    def layer_norm(x, name):
        n, b = wt[name + ".weight"], wt[name + ".bias"]
        return g.layer_norm_bf16(x, n, b, EPS) if bf else g.add(g.mul(g.norm(x, EPS), g.cast(n, F32)), g.cast(b, F32))

    def modulated(x, scale, shift):
        if bf:
            return g.norm_modulation_bf16(x, scale, shift, EPS)
        n = g.norm(x, EPS)
        return g.add(g.add(n, g.mul(n, scale)), shift)

    def gated(h, x, gate):
        return g.gated_residual_bf16(h, x, gate) if bf else g.add(h, g.mul(x, gate))

    def heads(x):  # [d, T] -> [dh, T, H]
        return g.cont(g.permute(x, 0, 2, 1, 3))

    def attend(k, v, q):
        scores = g.mul_mat(k, q)
        lib.wamx_mul_mat_set_prec(scores, 10)
        probs = g.soft_max_ext(scores, None, 1 / math.sqrt(DH), 0.0)
        return g.reshape_2d(g.cont(g.permute(g.mul_mat(v, probs), 0, 2, 1, 3)), D, t)

    def rope(x):
        x = g.rope_ext(x, lf["pos"], None, DH, 0, 0, 10000.0, 1.0, 0.0, 1.0, 32.0, 1.0)
        return g.cast(x, BF16) if bf else x

    comb = g.add(g.cast(lf["mod"], F32), g.cast(lf["table"], F32)) if bf else g.add(lf["mod"], lf["table"])
    shift, scale, gate, cshift, cscale, cgate = (g.view_2d(comb, D, 1, 4 * 6 * D, i * 4 * D) for i in range(6))
    n = modulated(lf["h"], scale, shift)
    if bf:
        qkv = linear("attn1.to_qkv", n)
        q, k, v = (g.cont(g.view_2d(qkv, D, t, 3 * D * es, i * D * es)) for i in range(3))
    else:
        q, k, v = (linear(f"attn1.to_{i}", n) for i in "qkv")
    q, k = (rope(g.reshape_3d(rms(x, "attn1.norm_" + i), DH, HEADS, t)) for x, i in ((q, "q"), (k, "k")))
    v = g.reshape_3d(v, DH, HEADS, t)
    kb, vb = p * DH * es, p * es  # bytes of a head of K, of a row of V^T
    jk = g.concat(g.concat(g.view_3d(lf["pk"], DH, 1, HEADS, DH * es, kb, 0), heads(k), 1),
                  g.view_3d(lf["pk"], DH, p - 1, HEADS, DH * es, kb, DH * es), 1)
    jv = g.concat(g.concat(g.view_3d(lf["pv"], 1, DH, HEADS, vb, vb * DH, 0), g.cont(g.permute(v, 1, 2, 0, 3)), 0),
                  g.view_3d(lf["pv"], p - 1, DH, HEADS, vb, vb * DH, es), 0)
    h = gated(lf["h"], linear("attn1.to_out.0", attend(jk, jv, heads(q))), gate)
    cq = g.reshape_3d(rms(linear("attn2.to_q", layer_norm(h, "norm2")), "attn2.norm_q"), DH, HEADS, t)
    if bf:
        cq = g.cast(cq, BF16)
    h = g.add(h, linear("attn2.to_out.0", attend(lf["lk"], lf["lv"], heads(cq))))
    n3 = modulated(h, cscale, cshift)
    if bf:
        u = g.bias_gelu_bf16(g.mul_mat_out_type(wt["ffn.net.0.proj.weight"], n3, BF16), wt["ffn.net.0.proj.bias"])
    else:
        u = g.gelu(linear("ffn.net.0.proj", n3))
    y = torch.empty((t, D), device="cuda", dtype=s["h"].dtype)
    g.finish(g.out(gated(h, linear("ffn.net.2", u), cgate), y))
    return {"graph": g, "call": g.compute, "outputs": y}


def _exact_layer(c, seed):
    w, s = _layer_inputs(c, seed)
    w = {k: v.double() for k, v in w.items()}
    pos = s.pop("pos")
    s = {k: v.double() for k, v in s.items()}
    t = c["t"]
    lin = lambda name, x: x @ w[name + ".weight"].T + w[name + ".bias"]  # noqa: E731
    m = s["mod"] + s["table"]
    n = _ln64(s["h"]) * (1 + m[1]) + m[0]
    q, k, v = lin("attn1.to_qkv", n).split(D, 1) if c["profile"] == "bf16" else (lin(f"attn1.to_{i}", n) for i in "qkv")
    head = lambda x, name: _rms64(x, w[name + ".weight"]).reshape(t, HEADS, DH)  # noqa: E731
    q = _rope64(head(q, "attn1.norm_q"), [pos]).transpose(0, 1)
    k = _rope64(head(k, "attn1.norm_k"), [pos]).transpose(0, 1)
    v = v.reshape(t, HEADS, DH).permute(1, 2, 0)
    a = _attend64(q, torch.cat([k, s["pk"]], 1), torch.cat([v, s["pv"]], 2))
    h = s["h"] + lin("attn1.to_out.0", a) * m[2]
    n2 = _ln64(h) * w["norm2.weight"] + w["norm2.bias"]
    cq = head(lin("attn2.to_q", n2), "attn2.norm_q").transpose(0, 1)
    h = h + lin("attn2.to_out.0", _attend64(cq, s["lk"], s["lv"]))
    u = _gelu64(lin("ffn.net.0.proj", _ln64(h) * (1 + m[4]) + m[3]))
    return h + lin("ffn.net.2", u) * m[5]


def _conv_inputs(c, seed):
    g = _gen(seed)
    k = c["ic"] * c["ks"] ** 2
    return {"w": _normal(g, (c["oc"], c["ic"], c["ks"], c["ks"]), 1 / math.sqrt(k)),
            "x": _normal(g, (1, c["ic"], c["h"], c["w"])), "b": _normal(g, (c["oc"],), 0.1)}


def _conv_out(c):
    return tuple((c[k] + 2 * c["p"] - c["ks"]) // c["s"] + 1 for k in ("w", "h"))


def _prepare_conv(c, seed):
    s = _conv_inputs(c, seed)
    ow, oh = _conv_out(c)
    g = Graph()
    s["y"] = torch.empty((1, c["oc"], oh, ow), device="cuda", dtype=torch.bfloat16)
    y = g.conv_2d_direct(g.leaf(s["w"]), g.leaf(s["x"]), c["s"], c["s"], c["p"], c["p"], 1, 1)
    g.finish(g.out(g.add(y, g.leaf(s["b"], 1, 1, c["oc"], 1)), s["y"]))
    s["graph"], s["call"], s["outputs"] = g, g.compute, s["y"]
    return s


def _exact_conv(c, seed):
    s = {k: v.double() for k, v in _conv_inputs(c, seed).items()}
    col = torch.nn.functional.unfold(s["x"], c["ks"], padding=c["p"], stride=c["s"])[0]
    ow, oh = _conv_out(c)
    return (s["w"].reshape(c["oc"], -1) @ col + s["b"][:, None]).reshape(1, c["oc"], oh, ow)


def _t5_vocab():
    return 4096


def _t5_weights(c, seed):
    """Name -> (rows, columns, std, mean), in the order they are drawn."""
    d, f = c["hidden"], c["ffn"]
    out = {"t5.shared.weight": (_t5_vocab(), d, 1.0, 0.0)}
    for i in range(c["layers"]):
        p = f"t5.encoder.block.{i}.layer."
        for j in "qkvo":  # scores are not scaled, so q's weights are smaller by the root of the head width
            out[p + f"0.SelfAttention.{j}.weight"] = (d, d, (1 / 8 if j == "q" else 1) / math.sqrt(d), 0.0)
        out[p + "0.SelfAttention.relative_attention_bias.weight"] = (32, c["heads"], 1.0, 0.0)
        out[p + "0.layer_norm.weight"] = (1, d, 0.05, 1.0)
        out[p + "1.DenseReluDense.wi_0.weight"] = (f, d, 1 / math.sqrt(d), 0.0)
        out[p + "1.DenseReluDense.wi_1.weight"] = (f, d, 1 / math.sqrt(d), 0.0)
        out[p + "1.DenseReluDense.wo.weight"] = (d, f, 1 / math.sqrt(f), 0.0)
        out[p + "1.layer_norm.weight"] = (1, d, 0.05, 1.0)
    out["t5.encoder.final_layer_norm.weight"] = (1, d, 0.05, 1.0)
    return out


class T5:
    def __init__(self, c):
        self.lib = _backend().lib
        cfg = wamx.T5Config(vocab=_t5_vocab(), hidden=c["hidden"], ffn_dim=c["ffn"], heads=c["heads"],
                            head_dim=c["hidden"] // c["heads"], layers=c["layers"], max_tokens=64, eps=EPS)
        self.ptr = self.lib.wamx_t5_create(_backend().ptr, C.byref(cfg))
        if not self.ptr:
            raise RuntimeError("out of memory: " + wamx.last_error())

    def __del__(self):
        if getattr(self, "ptr", None):
            self.lib.wamx_t5_free(self.ptr)


def _t5_tokens(c, seed):
    return np.random.default_rng(seed).integers(0, _t5_vocab(), c["tokens"]).astype(np.int32)


def _prepare_t5(c, seed):
    g = _gen(seed)
    t = T5(c)
    lib = t.lib
    for name, (m, k, std, mean) in _t5_weights(c, seed).items():
        w = lib.wamx_t5_weight(t.ptr, name.encode()).contents
        torch.as_tensor(_Device(t, w.data, m * k, "<i2"), device="cuda").view(torch.bfloat16).copy_(
            _normal(g, (m * k,), std, mean))
    # New prompts each time: a program whose prompts repeat would not encode them again.
    wamx.check(lib.wamx_t5_set_prompt_cache(t.ptr, 0))
    tokens = _t5_tokens(c, seed)
    s = {"t5": t, "tokens": tokens}

    def call():
        out = np.empty((64, c["hidden"]), np.float32)
        wamx.check(lib.wamx_t5_encode(t.ptr, tokens.ctypes.data, None, tokens.size, out.ctypes.data), "t5_encode")
        s["outputs"] = out

    s["call"] = call
    return s


def _bucket(rel, buckets=32, most=128):
    half = buckets // 2
    at = half if rel > 0 else 0
    rel = abs(rel)
    if rel < half // 2:
        return at + rel
    e = half // 2
    return at + min(half - 1, e + int(math.log(rel / e) / math.log(most / e) * (half - e)))


def _exact_t5(c, seed):
    g = _gen(seed)
    w = {}
    n, heads = c["tokens"], c["heads"]
    tok = torch.from_numpy(_t5_tokens(c, seed).astype(np.int64)).cuda()
    at = torch.tensor([[_bucket(j - i) for j in range(n)] for i in range(n)], device="cuda")
    h = None
    for name, (m, k, std, mean) in _t5_weights(c, seed).items():
        key = name.rsplit(".layer.", 1)[-1]
        w[key] = _normal(g, (m * k,), std, mean).double().reshape(m, k)
        if key == "t5.shared.weight":
            h = w[key][tok]
        elif key == "1.layer_norm.weight":  # the block's last
            x = _rms64(h, w["0.layer_norm.weight"])
            q, k_, v = ((x @ w[f"0.SelfAttention.{j}.weight"].T).reshape(n, heads, -1).transpose(0, 1) for j in "qkv")
            bias = w["0.SelfAttention.relative_attention_bias.weight"][at].permute(2, 0, 1)
            a = torch.softmax(q @ k_.transpose(1, 2) + bias, -1) @ v
            h = h + a.transpose(0, 1).reshape(n, -1) @ w["0.SelfAttention.o.weight"].T
            x = _rms64(h, w["1.layer_norm.weight"])
            f = _gelu64(x @ w["1.DenseReluDense.wi_0.weight"].T) * (x @ w["1.DenseReluDense.wi_1.weight"].T)
            h = h + f @ w["1.DenseReluDense.wo.weight"].T
            w = {}
    out = torch.zeros((64, c["hidden"]), device="cuda", dtype=torch.float64)
    out[:n] = _rms64(h, w["t5.encoder.final_layer_norm.weight"])
    return out.cpu().numpy()


def _chunk_config(c):
    cfg = _backend().lib.wamx_gwp_default_config()
    cfg.n_layers, cfg.grid_h, cfg.grid_w = c["layers"], c["grid_h"], c["grid_w"]
    cfg.n_lang, cfg.num_steps, cfg.batch = c["prompt"], c["steps"], c["batch"]
    return cfg


class Model:
    def __init__(self, c, seed):
        self.lib = _backend().lib
        self.cfg = _chunk_config(c)
        self.ptr = self.lib.wamx_gwp_create(_backend().ptr, C.byref(self.cfg))
        if not self.ptr:
            raise RuntimeError("out of memory: " + wamx.last_error())
        wamx.check(self.lib.wamx_gwp_init_synthetic(self.ptr, 0x5EED0000 + seed, 0.02), "init_synthetic")

    def __del__(self):
        if getattr(self, "ptr", None):
            self.lib.wamx_gwp_free(self.ptr)


def _prepare_chunk(c, seed):
    m = Model(c, seed)
    cfg, lib = m.cfg, m.lib
    rng = np.random.default_rng(seed)
    b = c["batch"]
    normal = lambda *shape: rng.standard_normal(shape, dtype=np.float32)  # noqa: E731
    state, latent = normal(b, cfg.action_dim), normal(b, cfg.z_dim, 2 * cfg.grid_h, 2 * cfg.grid_w)
    prompt, noise = normal(b, cfg.n_lang, cfg.t5_hidden), normal(b, cfg.action_chunk, cfg.action_dim)
    s = {"model": m}

    def call():
        wamx.check(lib.wamx_gwp_set_inputs(m.ptr, state.ctypes.data, latent.ctypes.data, prompt.ctypes.data,
                                           noise.ctypes.data), "set_inputs")
        wamx.check(lib.wamx_gwp_predict(m.ptr, None), "predict")
        out = [np.empty((b, cfg.action_chunk, cfg.action_dim), np.float32) for _ in range(3)]
        wamx.check(lib.wamx_gwp_get_action(m.ptr, out[0].ctypes.data), "get_action")
        for i, step in ((1, 0), (2, cfg.num_steps - 1)):
            wamx.check(lib.wamx_gwp_get_velocity(m.ptr, step, out[i].ctypes.data), "get_velocity")
        s["outputs"] = out

    s["call"] = call
    return s


_PREPARE = {"linear": _prepare_linear, "mul_mat": _prepare_mul_mat, "ffn": _prepare_ffn, "attention": _prepare_attention,
            "layer": _prepare_layer, "conv": _prepare_conv, "t5": _prepare_t5, "chunk": _prepare_chunk}
_EXACT = {"linear": _exact_linear, "mul_mat": _exact_mul_mat, "ffn": _exact_ffn, "attention": _exact_attention,
          "layer": _exact_layer, "conv": _exact_conv, "t5": _exact_t5}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    state["call"]()
    return state["outputs"]


def exact(case, seed):
    # A whole request has its weights from the backend's own generator, and its 10 denoise steps over 10 G
    # weights take more than 20 seconds in 64 bits.
    fn = _EXACT.get(case["kind"])
    return fn(case, seed) if fn else None


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _product(m, n, k, wb=2, xb=2, yb=2):
    return m * k * wb + n * k * xb + n * m * yb, 2 * m * n * k


def _chunk_work(c):
    cfg = _chunk_config(c)
    d, f, L, b = cfg.hidden, cfg.ffn_dim, cfg.n_layers, cfg.batch
    nimg, nl, t, steps = cfg.grid_h * cfg.grid_w, cfg.n_lang, cfg.action_chunk, cfg.num_steps
    attn1, cross, ffn = 4 * d * d, 2 * d * d, 2 * d * f        # self-attention, cross Q and O, FFN
    visual = attn1 + cross + 2 * d * d + ffn                   # with its text K and V
    action = attn1 + cross + ffn
    text = 2 * (cfg.t5_hidden * d + d * d)
    weights = L * (visual + action + 2 * d * d) + text + 2 * (256 * d + 7 * d * d)
    kv = 2 * d * (nimg + 1 + nl) * L * 2                       # K and V caches of a chunk
    bytes_ = 2 * weights + 2 * b * kv + steps * (2 * L * action + b * kv)
    flops = 2 * L * b * (nimg * (attn1 + cross + ffn) + nl * 4 * d * d + action) + 2 * b * nl * text
    flops += 4 * d * L * b * nimg * (nimg + 1 + nl)
    flops += steps * b * t * L * (2 * action + 4 * d * (nimg + 1 + t + nl))
    return bytes_, flops


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        b, f = _product(c["m"], c["n"], c["k"], xb=4 if c["x"] == "f32" else 2)
        b += {"none": 0, "bias": 2 * c["m"], "gelu": 2 * c["m"], "gated": 6 * c["m"] + 2 * c["n"] * c["m"],
              "residual": 2 * c["m"] + 2 * c["n"] * c["m"]}[c["epi"]]
    elif kind == "mul_mat":
        b, f = _product(c["m"], c["n"], c["k"], xb=4 if c["x"] == "f32" else 2, yb=4 if c["y"] == "f32" else 2)
    elif kind == "ffn":
        n = c["n"]
        b, f = 2 * 2 * D * FFN + 2 * n * (D + D + FFN + D), 4 * n * D * FFN
    elif kind == "attention":
        keys = c["na"] + c["nb"]
        b = 2 * D * (2 * keys + 3 * c["tq"] + (c["tq"] if c["own_k"] else 0))
        f = 4 * c["tq"] * keys * D
    elif kind == "layer":
        es, t, keys = (2 if c["profile"] == "bf16" else 4), c["t"], c["prefix"] + c["prompt"]
        weights = 6 * D * D + 2 * D * FFN
        b = es * (weights + 2 * D * keys + 2 * t * D)
        f = 2 * t * weights + 4 * t * D * (keys + t)
    elif kind == "conv":
        ow, oh = _conv_out(c)
        k = c["ic"] * c["ks"] ** 2
        b = 2 * (c["oc"] * k + c["ic"] * c["w"] * c["h"] + c["oc"] * ow * oh)
        f = 2 * c["oc"] * k * ow * oh
    elif kind == "t5":
        n, d = c["tokens"], c["hidden"]
        weights = c["layers"] * (4 * d * d + 3 * d * c["ffn"])
        b, f = 2 * weights + 4 * n * d, 2 * n * weights + 4 * c["layers"] * n * n * d
    else:
        b, f = _chunk_work(c)
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind == "mul_mat" and case["y"] == "f32":
        return {"rel": 1e-5}   # exact products of bf16 values, 32-bit sums
    if kind == "layer" and case["profile"] == "f32":
        return {"rel": 1e-5}   # 32-bit throughout
    if kind in ("t5", "chunk"):
        return {"rel": 0.03}   # bf16 roundings of every layer travel through the rest
    return {"rel": 1e-2}       # bf16 results
