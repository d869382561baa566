"""wamx_op_linear_noalloc against wamx_op_linear, through the C ABI: the
same product on the same device arrays gives the same bits, on calls in a row
(each smaller than the one before, so it runs on what that one left in the
shared scratch array), on the K-split paths (few tokens; K-sliced 128 x 128,
192 x 192 and 256 x 256 tiles), and a product of which a plain K split would
need more than half of the scratch array is refused before anything runs."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(wx, be, orc, M, N, K, epi, seed):
    w = orc.fill_normal(M * K, seed, 0.0, 0.02, orc.BF16)
    x = orc.fill_normal(N * K, seed + 1, 0.0, 1.0, orc.BF16)
    b = orc.fill_normal(M, seed + 2, 0.0, 0.02, orc.BF16)
    r = orc.fill_normal(N * M, seed + 3, 0.0, 1.0, orc.BF16)
    g = orc.fill_normal(M, seed + 4, 0.0, 0.5)
    dw, dx, db, dr, dg = (be.array(a) for a in (w, x, b, r, g))
    y_ref, y_na = be.empty(N * M * 2), be.empty(N * M * 2)
    res = dr.ptr if epi in (wx.EPI_BIAS_GATED, wx.EPI_BIAS_RESIDUAL) else None
    gate = dg.ptr if epi == wx.EPI_BIAS_GATED else None
    lib = be.lib
    wx.check(lib.wamx_op_linear(be.ptr, dw.ptr, dx.ptr, wx.TYPE_BF16, db.ptr, epi, res, gate, y_ref.ptr, M, N, K),
             "linear")
    be.sync()
    stream = lib.wamx_backend_stream(be.ptr)
    wx.check(lib.wamx_op_linear_noalloc(stream, dw.ptr, dx.ptr, wx.TYPE_BF16, db.ptr, epi, res, gate, y_na.ptr, M, N,
                                        K), "linear_noalloc")
    be.sync()
    a = y_ref.download(np.uint16, (N, M))
    c = y_na.download(np.uint16, (N, M))
    assert np.array_equal(a, c), f"{N}x{M}x{K}"
    return dw, dx, db, y_na


def test_linear_noalloc_matches_linear(wx, be, orc):
    print("linear_noalloc: 384 x 3072 x 14336, 384 x 3072 x 3072, 48 x 14336 x 3072, 16 x 3072 x 14336, "
          "8 x 256 x 512", flush=True)
    lib = be.lib
    # batch-8 denoise FFN-down and 3072^2 projection: 8 slices of 192 x 192
    # tiles and 6 of 128 x 128, partials in the scratch array
    for M, K, seed in ((3072, 14336, 400), (3072, 3072, 500)):
        _case(wx, be, orc, M, 384, K, wx.EPI_BIAS_GATED, seed)
    _case(wx, be, orc, 14336, 48, 3072, wx.EPI_BIAS_GELU, 100)       # FFN-up of the 48-token step
    _case(wx, be, orc, 3072, 16, 14336, wx.EPI_BIAS_GATED, 200)      # smaller: FFN-down shape on 16 tokens
    dw, dx, db, y = _case(wx, be, orc, 256, 8, 512, wx.EPI_BIAS_RESIDUAL, 300)
    # 64 tokens x 65536 x 14336, split plainly, would need far more partials
    # than the limit: refused, nothing launched
    st = lib.wamx_op_linear_noalloc(lib.wamx_backend_stream(be.ptr), dw.ptr, dx.ptr, wx.TYPE_BF16, db.ptr,
                                    wx.EPI_BIAS, None, None, y.ptr, 65536, 64, 14336)
    assert st != 0 and "split-K scratch" in wx.last_error()
    be.sync()


# Planes past the first half of the scratch array (48 MiB each): 8 and 2 slices
# of 256 x 256 tiles; then 4 of 192 x 192, on what those left there.
def test_linear_noalloc_large_tiles(wx, be, orc):
    print("linear_noalloc: 512 x 3072 x 14336, 2048 x 3072 x 14336, 192 x 9216 x 3072", flush=True)
    _case(wx, be, orc, 3072, 512, 14336, wx.EPI_BIAS_GATED, 600)
    _case(wx, be, orc, 3072, 2048, 14336, wx.EPI_BIAS_RESIDUAL, 700)
    _case(wx, be, orc, 9216, 192, 3072, wx.EPI_BIAS, 800)
