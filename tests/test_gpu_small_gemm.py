"""The GEMMs on 32 x 32 fp32 tiles (csrc/gemm_small.h), which small shapes take:
edges of tiles, of steps of 8 and batches of 32 k, K pieces, and the ends of
their range, in the three layouts; accumulating and with the residual; the
maxima they leave; the grouped weight gradients; and the fused epilogues bit
for bit against the separate passes.

Bound: sums of 32 terms in chunks, then of the K / 32 chunks and at most 16
waves and pieces: about 32 + K / 32 roundings of 2^-24 in random directions.
"""
import ctypes

import numpy as np
import pytest

from util import rel_l2

SHAPES = [(1, 1, 1), (1, 7, 33), (31, 8, 32), (33, 31, 65), (64, 64, 64), (65, 100, 130), (256, 64, 128), (30, 1536, 40),
          (16, 8192, 16), (100, 1000, 300), (2048, 33, 64), (500, 515, 700), (64, 4096, 1024), (8192, 20, 48)]


def up(fh, a):
    return fh.DeviceArray.from_numpy(np.ascontiguousarray(a, np.float32))


def _bound(K):
    return 2.0 ** -24 * np.sqrt(32 + K / 32)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_small_gemms_vs_fp64(fh, M, K, N):
    rs = np.random.default_rng(M * 7 + K)
    X, W, G = (rs.standard_normal(s, dtype=np.float32) for s in ((M, K), (N, K), (M, N)))
    Xd, Wd, Gd = (a.astype(np.float64) for a in (X, W, G))
    dX, dW, dG = up(fh, X), up(fh, W), up(fh, G)
    Y, gX, gW = fh.DeviceArray((M, N)), fh.DeviceArray((M, K)), fh.DeviceArray((N, K))
    xx, xw, xg = (up(fh, np.full(256, np.nan)) for _ in range(3))
    fh.call("matmulT_fwd_p", Y, dX, dW, M, K, N, xx, xw, 0)
    y = Y.numpy()
    assert rel_l2(y, Xd @ Wd.T) < _bound(K)
    fh.call("matmulT_bwd_p", gX, 0, gW, 0, dG, dX, dW, M, K, N, xg, xx, xw, 6)
    gx, gw = gX.numpy(), gW.numpy()
    assert rel_l2(gx, Gd @ Wd) < _bound(N)
    assert rel_l2(gw, Gd.T @ Xd) < _bound(M)
    for xp, a in ((xx, X), (xw, W), (xg, G)):
        assert xp.numpy().max() == np.abs(a).max()
    fh.call("matmulT_bwd", gX, 1, gW, 1, dG, dX, dW, M, K, N)
    # K pieces are added to the incoming gradient one by one: a rounding each, at most 16
    assert rel_l2(gX.numpy(), 2.0 * gx) < 2.0 ** -24 * 4
    assert rel_l2(gW.numpy(), 2.0 * gw) < 2.0 ** -24 * 4
    fh.call("matmulT_fwd_resid", Y, dG, dX, dW, M, K, N)
    np.testing.assert_array_equal(Y.numpy(), G + y)


# the input gradient in two pieces
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(128, 128, 700), (70, 130, 600)])
def test_small_input_gradient_halves(fh, M, K, N):
    assert fh.lib.fg_matmulT_bwd_x_pieces(M, K, N) == 2
    rs = np.random.default_rng(5)
    G, W = up(fh, rs.standard_normal((M, N))), up(fh, rs.standard_normal((N, K)))
    H, gX = fh.DeviceArray((2, M, K)), fh.DeviceArray((M, K))
    fh.call("matmulT_bwd_x_halves", H, G, W, M, K, N)
    fh.call("matmulT_bwd_x", gX, G, W, M, K, N, 0)
    h = H.numpy()
    np.testing.assert_array_equal(gX.numpy(), h[0] + h[1])


# more jobs than a table holds, one output named twice, accumulating ones among them
@pytest.mark.gpu
def test_small_weight_gradients_grouped(fh):
    rs = np.random.default_rng(9)
    shapes = [(64, 16 + 3 * i, 8 + 5 * i) for i in range(17)] + [(100, 33, 20)]
    jobs, want, keep = [], [], []
    for i, (M, K, N) in enumerate(shapes):
        G, X, C = rs.standard_normal((M, N)), rs.standard_normal((M, K)), rs.standard_normal((N, K))
        G, X, C = (a.astype(np.float32) for a in (G, X, C))
        d = [up(fh, a) for a in (C, G, X)]
        keep.append(d)
        jobs.append(fh.WgradJob(d[0].ptr, d[1].ptr, d[2].ptr, M, K, N, i % 2, None, None))
        want.append(G.astype(np.float64).T @ X + (C if i % 2 else 0.0))
    M, K, N = shapes[-1]
    G, X = (rs.standard_normal(s).astype(np.float32) for s in ((M, N), (M, K)))
    d = [up(fh, a) for a in (G, X)]
    jobs.append(fh.WgradJob(keep[-1][0].ptr, d[0].ptr, d[1].ptr, M, K, N, 1, None, None))
    want[-1] = want[-1] + G.astype(np.float64).T @ X
    fh.check(fh.lib.fg_matmulT_bwd_w_grouped((fh.WgradJob * len(jobs))(*jobs), len(jobs)), "grouped")
    for (M, K, N), d, w in zip(shapes, keep, want):
        assert rel_l2(d[0].numpy(), w) < 2 * _bound(M)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,H", [(33, 64, 48), (256, 64, 128), (70, 30, 31), (300, 256, 100)])
def test_small_fused_epilogues_are_the_separate_passes(fh, M, K, H):
    rs = np.random.default_rng(M)
    X, W = up(fh, rs.standard_normal((M, K))), up(fh, rs.standard_normal((2 * H, K)))
    GU, O, GU2, O2 = (fh.DeviceArray(s) for s in ((M, 2 * H), (M, H)) * 2)
    xx, xw = fh.DeviceArray((256,)), fh.DeviceArray((256,))
    fh.call("matmulT_fwd_swiglu_p", O, GU, X, W, M, K, H, xx, xw, 0)
    fh.call("matmulT_fwd", GU2, X, W, M, K, 2 * H)
    fh.call("swiglu_gu_fwd", O2, GU2, M, H)
    np.testing.assert_array_equal(GU.numpy(), GU2.numpy())
    np.testing.assert_array_equal(O.numpy(), O2.numpy())
    assert xw.numpy().max() == np.abs(W.numpy()).max() and xx.numpy().max() == np.abs(X.numpy()).max()
    # RoPE of two query heads and a key head of 6, the rest of the columns as they are
    nH, nKV, dH, T = 2, 1, 6, 40
    N = (nH + 2 * nKV) * dH + 5
    Wq = up(fh, rs.standard_normal((N, K)))
    ang = rs.uniform(0, 6, (T, dH // 2))
    cos, sin = (fh.DeviceArray.from_numpy(f(ang)) for f in (np.cos, np.sin))
    Y, Y2 = fh.DeviceArray((M, N)), fh.DeviceArray((M, N))
    fh.call("matmulT_fwd_rope", Y, X, Wq, M, K, N, cos, sin, T, nH, nKV, dH, 0, T)
    fh.call("matmulT_fwd", Y2, X, Wq, M, K, N)
    y = Y2.numpy()
    c, s = (np.tile(a, (M // T + 1, nH + nKV))[:M] for a in (np.cos(ang), np.sin(ang)))
    q = y[:, :(nH + nKV) * dH].astype(np.float64)
    a, b = q[:, 0::2], q[:, 1::2]
    want = y.copy()
    want[:, 0:(nH + nKV) * dH:2], want[:, 1:(nH + nKV) * dH:2] = a * c - b * s, a * s + b * c
    np.testing.assert_array_equal(Y.numpy(), want)


# the fused SwiGLU form at a longer K (pairs of tiles that fit a round of CUs), and
# few tiles over a long K, which run as the GEMM and the pass
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,H", [(512, 200, 400), (1030, 477, 60), (416, 1440, 32), (17, 1396, 887)])
def test_small_swiglu_projection_at_longer_k(fh, M, K, H):
    test_small_fused_epilogues_are_the_separate_passes(fh, M, K, H)
