"""Attention at head sizes below 32 (a workgroup's waves share a row's keys) at
the edges of rows, waves and classes, against fp64.

Bound: a score is a sum of dH products, an output of up to T weights, each
rounding 2^-24 of terms of one size; exp turns a score's absolute error (|s|
<= 20 here: 20 * 2^-24 = 1.2e-6) into a relative one of its weight.  4e-6 of
the result's norm holds both.

Gradients that share a buffer (attention of a tensor with itself) are added in
the order dQ, dK, dV: one fp32 addition each after those of the separate run.
"""
import numpy as np
import pytest

from util import rel_l2


def attention64(q, k, v, go):
    """o, lse, dq, dk, dv of one sample's causal attention; q [T, nH, dH], k, v [T, nKV, dH]."""
    T, nH, dH = q.shape
    nKV = k.shape[1]
    group = max(1, nH // nKV)
    o, lse, dq = np.zeros_like(q), np.zeros((nH, T)), np.zeros_like(q)
    dk, dv = np.zeros_like(k), np.zeros_like(v)
    future = np.triu(np.ones((T, T), bool), 1)
    for h in range(nH):
        z = h // group
        s = q[:, h] @ k[:, z].T / np.sqrt(dH)
        s[future] = -np.inf
        m = s.max(1, keepdims=True)
        e = np.exp(s - m)
        lse[h] = m[:, 0] + np.log(e.sum(1))
        p = e / e.sum(1, keepdims=True)
        o[:, h] = p @ v[:, z]
        dv[:, z] += p.T @ go[:, h]
        dp = go[:, h] @ v[:, z].T
        ds = p * (dp - (p * dp).sum(1, keepdims=True)) / np.sqrt(dH)
        dq[:, h] = ds @ k[:, z]
        dk[:, z] += ds.T @ q[:, h]
    return o, lse, dq, dk, dv


def check(fh, B, T, nH, nKV, dH, beta, tol=4e-6):
    rs = np.random.default_rng(T * 31 + dH)
    q, go = (rs.standard_normal((B, T, nH, dH)).astype(np.float32) for _ in range(2))
    k, v = (rs.standard_normal((B, T, nKV, dH)).astype(np.float32) for _ in range(2))
    d = [fh.DeviceArray.from_numpy(a) for a in (q, k, v, go)]
    o, lse = fh.DeviceArray(q.shape), fh.DeviceArray((B, nH, T))
    fh.call("attn_fwd", o, lse, d[0], d[1], d[2], B, T, nH, nKV, dH)
    g = [fh.DeviceArray.from_numpy(np.ones(a.shape, np.float32)) for a in (q, k, v)]
    fh.call("attn_bwd", g[0], beta, g[1], beta, g[2], beta, d[3], d[0], d[1], d[2], o, lse, B, T, nH, nKV, dH)
    want = [np.stack(a) for a in zip(*[attention64(*(a[b].astype(np.float64) for a in (q, k, v, go))) for b in range(B)])]
    got = [o.numpy(), lse.numpy()] + [a.numpy() - np.float32(beta) for a in g]
    for a, w in zip(got, want):
        if w.any():
            assert rel_l2(a, w) < tol
        else:
            assert not a.any()


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,nH,nKV,dH", [(1, 1, 1, 1, 1), (2, 7, 4, 2, 8), (1, 8, 2, 2, 13), (3, 63, 4, 1, 16),
                                           (1, 64, 2, 1, 24), (2, 65, 6, 3, 16), (1, 130, 2, 2, 31), (1, 333, 4, 2, 9),
                                           (1, 70, 2, 4, 16)])
@pytest.mark.parametrize("beta", [0, 1])
def test_attention_below_32_vs_fp64(fh, B, T, nH, nKV, dH, beta):
    check(fh, B, T, nH, nKV, dH, beta)


# few heads over long rows: chains in pieces, a last row block of one row, GQA, more and fewer blocks than a piece
@pytest.mark.gpu
@pytest.mark.parametrize("B,T,nH,nKV,dH", [(1, 513, 1, 1, 32), (1, 897, 4, 2, 64), (2, 777, 3, 1, 96), (1, 1100, 2, 2, 128),
                                           (1, 640, 6, 2, 80), (1, 400, 2, 1, 64)])
@pytest.mark.parametrize("beta", [0, 1])
def test_attention_in_pieces_vs_fp64(fh, B, T, nH, nKV, dH, beta):
    check(fh, B, T, nH, nKV, dH, beta)


# padded, scalar, MFMA (whole and in pieces) and GEMM heads
@pytest.mark.gpu
@pytest.mark.parametrize("T,dH", [(130, 80), (700, 48), (70, 16), (65, 64), (600, 64), (40, 32), (33, 160)])
@pytest.mark.parametrize("shared", ["kv", "qkv", "qk"])
def test_gradients_that_share_a_buffer(fh, T, dH, shared):
    B, nH = 2, 3
    rs = np.random.default_rng(T + dH)
    q, k, v, go = (fh.DeviceArray.from_numpy(rs.standard_normal((B, T, nH, dH)).astype(np.float32)) for _ in range(4))
    shape = (B, T, nH, dH)
    o, lse = fh.DeviceArray(shape), fh.DeviceArray((B, nH, T))
    fh.call("attn_fwd", o, lse, q, k, v, B, T, nH, nH, dH)
    own = [fh.DeviceArray(shape) for _ in range(3)]
    fh.call("attn_bwd", own[0], 0, own[1], 0, own[2], 0, go, q, k, v, o, lse, B, T, nH, nH, dH)
    for first in (0, 1):  # the shared gradient fresh, or there already
        g = [fh.DeviceArray.from_numpy(np.ones(shape, np.float32)) for _ in range(3)]
        want = [np.full(shape, float(first)) for _ in range(3)]
        use = {"q": 0, "k": 1, "v": 2}
        at, beta, seen = [0, 1, 2], [first] * 3, False
        for c in shared:
            at[use[c]] = use[shared[0]]
            beta[use[c]] = 1 if seen else first
            seen = True
        fh.call("attn_bwd", g[at[0]], beta[0], g[at[1]], beta[1], g[at[2]], beta[2], go, q, k, v, o, lse, B, T, nH, nH, dH)
        for i in range(3):
            want[at[i]] += own[i].numpy().astype(np.float64)
        for i in set(at):
            assert rel_l2(g[i].numpy(), want[i]) < 3 * 2.0 ** -24
