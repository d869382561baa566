"""MUL_MAT with f32 weights (the f32 reference profile), and with bf16 weights
in batches or with unaligned rows at few tokens, on the GPU: one kernel, at the
edges of its tiles, K steps and K slices.  Integer operands whose sums stay
below 2^24 have one f32 result in any order of summation, so the products must
match exactly."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_fusion import Graph

pytestmark = pytest.mark.gpu


def mul_mat(wx, be, w, x, ld=None, xtype="f32", wtype="f32"):
    """w [B][M][K] (leading dimension ld >= K), x [B2][N][K] -> [B2][N][M]."""
    B, M, K = w.shape
    B2, N, _ = x.shape
    ld = ld or K
    g = Graph(wx, be)
    try:
        wt = g.t(wx.TYPE_F32 if wtype == "f32" else wx.TYPE_BF16, ld, M, B)
        xt = g.t(wx.TYPE_F32 if xtype == "f32" else wx.TYPE_BF16, ld, N, B2)
        es = 4 if xtype == "f32" else 2
        ws = 4 if wtype == "f32" else 2
        wv = be.lib.wamx_view_3d(g.ctx, wt, K, M, B, ws * ld, ws * ld * M, 0)
        xv = be.lib.wamx_view_3d(g.ctx, xt, K, N, B2, es * ld, es * ld * N, 0)
        y = be.lib.wamx_mul_mat(g.ctx, wv, xv)
        assert y, wx.last_error()
        g.alloc()
        # Columns past K are NaN: they must not be read into a product.
        wp = np.full((B, M, ld), np.nan, np.float32)
        xp = np.full((B2, N, ld), np.nan, np.float32)
        wp[:, :, :K], xp[:, :, :K] = w, x
        g.set(wt, wp if wtype == "f32" else wx.f32_to_bf16(wp))
        g.set(xt, xp if xtype == "f32" else wx.f32_to_bf16(xp))
        g.compute(y)
        return g.get(y, np.float32, (B2, N, M))
    finally:
        g.close()


# Token tiles of 1-4 and 8 sixteens with remainders; feature blocks of 64 and
# 128 with remainders; K below a 16-byte chunk, below, at and past a 128-byte
# step, in slices (the last one shorter), ending inside a chunk; batches with w
# broadcast, and in slices; rows whose stride is not a multiple of 16 bytes.
@pytest.mark.parametrize("M,N,K,B,r,ld", [
    (3072, 48, 3072, 1, 1, 3072), (14336, 33, 512, 1, 1, 512), (200, 1, 4100, 1, 1, 4100), (65, 17, 36, 1, 1, 40),
    (1, 1, 1, 1, 1, 1), (169, 48, 128, 24, 1, 128), (128, 48, 169, 24, 1, 169), (64, 64, 64, 4, 3, 64),
    (130, 65, 4, 2, 1, 4), (3072, 121, 3072, 1, 1, 3072), (300, 160, 90, 1, 1, 93), (1000, 300, 1440, 1, 1, 1440),
    (129, 128, 31, 1, 1, 33), (128, 48, 3121, 24, 1, 3121), (3121, 48, 128, 4, 6, 128), (40, 5, 7, 3, 1, 9),
    (64, 16, 3, 2, 1, 3), (70, 64, 1001, 1, 2, 1003), (128, 20, 263, 5, 1, 264)])
@pytest.mark.parametrize("xtype", ["f32", "bf16"])
@pytest.mark.parametrize("wtype", ["f32", "bf16"])
def test_mul_mat_integers_exact(wx, be, rng, M, N, K, B, r, ld, xtype, wtype):
    print(f"mul_mat M={M} N={N} K={K} B={B}x{r} ld={ld} w={wtype} x={xtype}", flush=True)
    w = rng.integers(-8, 9, (B, M, K)).astype(np.float32)
    x = rng.integers(-8, 9, (B * r, N, K)).astype(np.float32)
    got = mul_mat(wx, be, w, x, ld, xtype, wtype)
    ref = x.astype(np.float64) @ np.repeat(w, r, 0).transpose(0, 2, 1).astype(np.float64)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("M,N,K", [(3072, 48, 3072), (3072, 48, 14336), (256, 200, 1440)])
def test_f32_mul_mat_error(wx, be, rng, M, N, K):
    """Against 64-bit sums: K products summed in f32 in any order are off by
    at most K 2^-24 sum|a b|; errors of either sign make the observed one grow
    as sqrt(K), so an eighth of that bound is generous."""
    print(f"f32 mul_mat error M={M} N={N} K={K}", flush=True)
    w = rng.standard_normal((1, M, K)).astype(np.float32)
    x = rng.standard_normal((1, N, K)).astype(np.float32)
    got = mul_mat(wx, be, w, x)[0].astype(np.float64)
    wd, xd = w[0].astype(np.float64), x[0].astype(np.float64)
    bound = np.abs(xd) @ np.abs(wd).T * (K / 8 * 2.0 ** -24)
    assert (np.abs(got - xd @ wd.T) <= bound).all()
