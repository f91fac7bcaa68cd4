"""The GEMMs on operands split ahead of time (csrc/gemm_pieces.h), which large
shapes take: ragged rows, columns and k against fp64 on sampled rows and
columns, in the three layouts, with the residual and accumulating; the K
split; the grouped weight gradients over jobs of different lengths; and the
fused SwiGLU epilogue bit for bit against the separate pass.

Bound: the two-piece split leaves 3 * 2^-22 (7e-7) of a product and the fp32
sums of random-sign terms about 2^-24 sqrt(K / 2) <= 5e-6 of the result's norm
only at K ~ 10^4, less for the chunked order: 2e-6 up to K = 8000, 4e-6 above.
"""
import ctypes

import numpy as np
import pytest

from util import rel_l2


def up(fh, a):
    return fh.DeviceArray.from_numpy(np.ascontiguousarray(a, np.float32))


def _sample(rs, n, k=48):
    """k indexes of [0, n), the edges among them."""
    return np.unique(np.concatenate([[0, 1, n - 2, n - 1], rs.integers(0, n, k)]))


def _check(got, ref, K):
    assert rel_l2(got, ref) < (2e-6 if K <= 8000 else 4e-6)


# forward tiles of 256 rows ragged in M, N and K; of 128 rows; split over K
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(8187, 2003, 4090), (4045, 1228, 8091), (3031, 11946, 7906)])
def test_matmulT_on_pieces_vs_fp64(fh, M, K, N):
    rs = np.random.default_rng(M)
    X = rs.standard_normal((M, K), dtype=np.float32)
    W = rs.standard_normal((N, K), dtype=np.float32) * np.float32(0.05)
    R = rs.standard_normal((M, N), dtype=np.float32)
    dX, dW, dR, dY = up(fh, X), up(fh, W), up(fh, R), fh.DeviceArray((M, N))
    i, j = _sample(rs, M), _sample(rs, N)
    fh.call("matmulT_fwd", dY, dX, dW, M, K, N)
    Y = dY.numpy()
    Xd, Wd = X.astype(np.float64), W.astype(np.float64)
    _check(Y[i], Xd[i] @ Wd.T, K)
    _check(Y[:, j], Xd @ Wd[j].T, K)
    fh.call("matmulT_fwd_resid", dY, dR, dX, dW, M, K, N)
    np.testing.assert_array_equal(dY.numpy(), R + Y)
    # gradients, written and accumulated (R is the incoming gradient)
    gX, gW = fh.DeviceArray((M, K)), fh.DeviceArray((N, K))
    fh.call("matmulT_bwd", gX, 0, gW, 0, dR, dX, dW, M, K, N)
    x0, w0 = gX.numpy(), gW.numpy()
    Rd = R.astype(np.float64)
    _check(x0[i], Rd[i] @ Wd, N)
    _check(w0[j], Rd[:, j].T @ Xd, M)
    fh.call("matmulT_bwd", gX, 1, gW, 1, dR, dX, dW, M, K, N)
    _check(gX.numpy()[i], 2 * x0[i].astype(np.float64), 1)
    _check(gW.numpy()[j], 2 * w0[j].astype(np.float64), 1)


@pytest.mark.gpu
def test_grouped_weight_gradients_on_pieces(fh):
    """Jobs of different token counts (one shorter than a K piece of the
    others) and ragged outputs in one launch, fresh and accumulating."""
    rs = np.random.default_rng(5)
    shapes = [(8190, 4093, 4100), (8190, 1021, 4100), (70, 300, 500), (4096, 4096, 4096)]  # M (tokens), K, N
    host, rows = [], []
    for M, K, N in shapes:
        g, x = rs.standard_normal((M, N), dtype=np.float32), rs.standard_normal((M, K), dtype=np.float32)
        w0 = rs.standard_normal((N, K), dtype=np.float32)
        host.append((g, x, w0, up(fh, g), up(fh, x), up(fh, w0)))
    for beta in (1, 0):
        jobs = (fh.WgradJob * len(shapes))(*[
            fh.WgradJob(h[5].ptr, h[3].ptr, h[4].ptr, M, K, N, beta, None, None)
            for h, (M, K, N) in zip(host, shapes)])
        fh.check(fh.lib.fg_matmulT_bwd_w_grouped(ctypes.cast(jobs, ctypes.c_void_p), len(shapes)), "grouped")
        for (g, x, w0, _, _, dw), (M, K, N) in zip(host, shapes):
            j = _sample(rs, N)
            ref = g[:, j].astype(np.float64).T @ x.astype(np.float64) + beta * w0[j].astype(np.float64)
            _check(dw.numpy()[j], ref, M)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,H", [(4096, 2048, 4096), (8064, 1030, 4096)])
def test_swiglu_epilogue_on_pieces_is_the_separate_pass(fh, M, K, H):
    rs = np.random.default_rng(H)
    dX, dW = up(fh, rs.standard_normal((M, K))), up(fh, rs.standard_normal((2 * H, K)) * 0.02)
    gu, o, gu2, o2 = (fh.DeviceArray(s) for s in ((M, 2 * H), (M, H), (M, 2 * H), (M, H)))
    fh.call("matmulT_fwd_swiglu", o, gu, dX, dW, M, K, H)
    fh.call("matmulT_fwd", gu2, dX, dW, M, K, 2 * H)
    fh.call("swiglu_gu_fwd", o2, gu2, M, H)
    np.testing.assert_array_equal(gu.numpy(), gu2.numpy())
    np.testing.assert_array_equal(o.numpy(), o2.numpy())


# shapes of a middle size take this form where their tiles or vectors are not
# whole: odd rows of each operand, and K pieces in all three layouts
@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(777, 1555, 666), (1501, 1499, 1502), (2048, 1026, 1537), (4095, 515, 771)])
def test_uneven_shapes_vs_fp64(fh, M, K, N):
    test_matmulT_on_pieces_vs_fp64(fh, M, K, N)


# operands that start between 16-byte boundaries
@pytest.mark.gpu
def test_unaligned_operands_on_pieces(fh):
    M, K, N = 1536, 1024, 1536
    rs = np.random.default_rng(3)
    X, W = rs.standard_normal(M * K + 1, dtype=np.float32), rs.standard_normal(N * K + 3, dtype=np.float32)
    dX, dW, Y = up(fh, X), up(fh, W), fh.DeviceArray((M, N))
    fh.call("matmulT_fwd", Y, dX.ptr + 4, dW.ptr + 12, M, K, N)
    _check(Y.numpy(), X[1:].reshape(M, K).astype(np.float64) @ W[3:].reshape(N, K).astype(np.float64).T, K)


# jobs whose partial sums end between 16-byte boundaries, before others: odd
# outputs over an odd number of K pieces
@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(8192, 1535, 1535), (8192, 1536, 512)],
                                    [(8192, 1103, 1101), (8192, 511, 1001), (8192, 512, 512)]])
def test_grouped_partial_sums_of_odd_outputs(fh, shapes):
    rs = np.random.default_rng(8)
    host = [(rs.standard_normal((M, N), dtype=np.float32), rs.standard_normal((M, K), dtype=np.float32)) for M, K, N in shapes]
    dev = [(up(fh, g), up(fh, x), fh.DeviceArray((N, K))) for (g, x), (M, K, N) in zip(host, shapes)]
    jobs = (fh.WgradJob * len(shapes))(*[fh.WgradJob(w.ptr, g.ptr, x.ptr, M, K, N, 0, None, None)
                                         for (g, x, w), (M, K, N) in zip(dev, shapes)])
    fh.check(fh.lib.fg_matmulT_bwd_w_grouped(ctypes.cast(jobs, ctypes.c_void_p), len(shapes)), "grouped")
    for (g, x), (_, _, w), (M, K, N) in zip(host, dev, shapes):
        j = _sample(rs, N)
        _check(w.numpy()[j], g[:, j].astype(np.float64).T @ x.astype(np.float64), M)


# lists whose jobs are told apart: uneven ones go to pieces, even ones stay with
# the kernels that split while staging; a list on pieces as a whole; more jobs
# than a window; a job on an earlier job's output after it
@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [
    [(4096, 2048, 4001), (4096, 1024, 8192), (4096, 1024, 8192), (4096, 1024, 8192), (4096, 1024, 8192)],
    [(8192, 1024, 4096), (8192, 1025, 1001), (8192, 1024, 4096), (8192, 1025, 1001), (8192, 1025, 1001)],
    [(4096, 4096, 4096), (4096, 768, 16385), (4096, 4096, 4096)],
    [(1024, 512, 512)] * 50 + [(1024, 300, 1001)] * 6,
])
def test_grouped_lists_told_apart(fh, shapes):
    rs = np.random.default_rng(len(shapes))
    host, dev = {}, {}
    for M, K, N in set(shapes):
        host[M, K, N] = rs.standard_normal((M, N), dtype=np.float32), rs.standard_normal((M, K), dtype=np.float32)
        dev[M, K, N] = [up(fh, a) for a in host[M, K, N]]
    w = [up(fh, np.full((N, K), 0.5, np.float32)) for M, K, N in shapes]
    order = list(range(len(shapes))) + [0, len(shapes) - 1]  # the last two accumulate onto written outputs
    jobs = (fh.WgradJob * len(order))(*[
        fh.WgradJob(w[i].ptr, dev[shapes[i]][0].ptr, dev[shapes[i]][1].ptr, *shapes[i], int(p >= len(shapes) or p % 2), None, None)
        for p, i in enumerate(order)])
    fh.check(fh.lib.fg_matmulT_bwd_w_grouped(ctypes.cast(jobs, ctypes.c_void_p), len(order)), "grouped")
    for i, (M, K, N) in enumerate(shapes):
        g, x = host[M, K, N]
        j = _sample(rs, N, 12)
        ref = g[:, j].astype(np.float64).T @ x.astype(np.float64)
        _check(w[i].numpy()[j], ref * order.count(i) + 0.5 * (i % 2), M)
