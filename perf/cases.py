"""The work that programs have this framework do, as timed cases.

Training: one transformer layer forward and backward, recorded and replayed as
one graph the way train() replays its steps; a single matmulT and a single
causal attention with their gradients; the final norm, LM head and loss; one
Adam step over a model's parameters; and the token side of a step (windows,
embedding, embedding gradient).  Inference: one decode step of a model over
f32 or quantized matrices, replayed as one graph, and one quantized linear
layer.  Everything goes through the C ABI of include/forge_hip.h, as the
JavaScript host's calls do.

Tensors are torch's (any device memory will do for the library); the library
queues its work on a stream of its own.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "forge-llm_amd"))
import forge_hip as fh  # noqa: E402

XP = 256  # FG_XP_PARTS: floats per buffer of operand maxima
EPS = 1e-5
F32, F16, Q8_0, Q4_K, Q5_K, Q6_K = 0, 1, 8, 12, 13, 14
BLOCK = {F32: (1, 4), F16: (1, 2), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}
MFMA_HEADS = (32, 64, 96, 128)  # head sizes whose attention reads the fused q, k, v projection


def listed():
    return [
        # the training demo's layer (dim 64, 8 windows of 32 tokens): the smallest step, launches and latency
        {"name": "layer-demo", "kind": "layer", "B": 8, "T": 32, "nH": 4, "nKV": 2, "dH": 16, "hidden": 128, "theta": 1e4},
        # a layer of the 125M model at the benchmark's batch: the ordinary training step
        {"name": "layer-125m", "kind": "layer", "B": 8, "T": 1024, "nH": 12, "nKV": 12, "dH": 64, "hidden": 2048, "theta": 1e4},
        # a Llama-3-8B layer over one 4096-token window: the largest
        {"name": "layer-8b", "kind": "layer", "B": 1, "T": 4096, "nH": 32, "nKV": 8, "dH": 128, "hidden": 14336, "theta": 5e5},
        # one projection with its gradients, the shape of the isolated op benchmark
        {"name": "matmul-2k", "kind": "matmul", "M": 2048, "K": 1024, "N": 4096},
        # attention and its gradient with a head size and a length that fill no tile
        {"name": "attention-ragged", "kind": "attention", "B": 3, "T": 777, "nH": 12, "nKV": 6, "dH": 80},
        # final norm, LM head, loss and their gradients of the 125M model
        {"name": "head-125m", "kind": "head", "rows": 8192, "dim": 768, "V": 32000},
        # one optimizer step over the 125M model's parameters
        {"name": "adam-125m", "kind": "adam", "dim": 768, "hidden": 2048, "layers": 12, "V": 32000},
        # windows, embedding and embedding gradient of one step of the 125M model
        {"name": "tokens-125m", "kind": "tokens", "B": 8, "T": 1024, "V": 32000, "dim": 768},
        # a token of the small decode benchmark's model (f32, tied head)
        {"name": "decode-small", "kind": "decode", "dim": 256, "hidden": 512, "layers": 4, "nH": 8, "nKV": 4, "V": 4096,
         "maxSeq": 512, "pos": 200, "mat": F32, "down": F32, "emb": F32, "cls": -1, "theta": 1e4},
        # a token of the 125M model in f32
        {"name": "decode-125m", "kind": "decode", "dim": 768, "hidden": 2048, "layers": 12, "nH": 12, "nKV": 12, "V": 32000,
         "maxSeq": 1024, "pos": 500, "mat": F32, "down": F32, "emb": F32, "cls": F32, "theta": 1e4},
        # a token through Llama-3-8B layers in K-quants, with its head, deep in its context
        {"name": "decode-8b-q4k", "kind": "decode", "dim": 4096, "hidden": 14336, "layers": 8, "nH": 32, "nKV": 8, "V": 128256,
         "maxSeq": 4096, "pos": 2047, "mat": Q4_K, "down": Q6_K, "emb": Q4_K, "cls": Q6_K, "theta": 5e5},
        # one quantized linear layer on its own (QuantLinear.forward)
        {"name": "qlinear-q8", "kind": "qlinear", "type": Q8_0, "N": 4096, "K": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "matmul", "attention", "head", "adam", "tokens", "decode", "decode", "qlinear"])
    if kind in ("layer", "attention"):
        while True:
            dH = rng.choice([16, 32, 48, 64, 64, 80, 96, 128, 128] + ([192, 256] if kind == "attention" else []))
            nKV = rng.choice([1, 2, 3, 4, 6, 8, 12])
            nH = nKV * rng.choice([1, 1, 2, 4])
            T = _log(rng, 24, 1024 if dH < 32 else 4096)
            B = _log(rng, 1, 16)
            if nH * dH > 4096 or not 64 <= B * T <= 8192:
                continue
            c = {"kind": kind, "B": B, "T": T, "nH": nH, "nKV": nKV, "dH": dH}
            if kind == "layer":
                c.update(hidden=max(32, int(nH * dH * rng.uniform(1.5, 3.6))), theta=rng.choice([1e4, 5e5]))
            return c
    if kind == "matmul":
        while True:
            M, K, N = _log(rng, 16, 8192), _log(rng, 16, 8192), _log(rng, 16, 32000)
            if M * K * N <= 2e11:
                return {"kind": kind, "M": M, "K": K, "N": N}
    if kind == "head":
        while True:
            c = {"kind": kind, "rows": _log(rng, 64, 8192), "dim": 16 * _log(rng, 4, 256), "V": _log(rng, 31, 128256)}
            if c["rows"] * c["dim"] * c["V"] <= 2.1e11 and c["rows"] * c["V"] <= 3e8:
                return c
    if kind == "adam":
        dim = 16 * _log(rng, 4, 48)
        return {"kind": kind, "dim": dim, "hidden": int(dim * rng.uniform(1.5, 3.6)), "layers": _log(rng, 2, 12), "V": _log(rng, 31, 32000)}
    if kind == "tokens":
        while True:
            c = {"kind": kind, "B": _log(rng, 1, 16), "T": _log(rng, 24, 2048), "V": _log(rng, 31, 32000), "dim": 16 * _log(rng, 4, 64)}
            if c["B"] * c["T"] <= 16384:
                return c
    if kind == "decode":
        while True:
            dH = rng.choice([32, 48, 64, 64, 96, 128])
            nKV = rng.choice([1, 2, 4, 8, 12])
            nH = nKV * rng.choice([1, 2, 4])
            mat = rng.choice([F32, F32, F16, Q8_0, Q4_K, Q5_K, Q6_K])
            if nH * dH > 4096 or (nH * dH) % BLOCK[mat][0]:
                continue
            hidden = int(nH * dH * rng.uniform(1.5, 3.5))
            hidden = max(1, hidden // BLOCK[mat][0]) * BLOCK[mat][0]
            maxSeq = rng.choice([256, 512, 1024, 2048, 4096])
            return {"kind": kind, "dim": nH * dH, "hidden": hidden, "layers": rng.randint(1, 8), "nH": nH, "nKV": nKV,
                    "V": _log(rng, 300, 65536), "maxSeq": maxSeq, "pos": rng.randint(0, maxSeq - 1), "mat": mat, "down": mat,
                    "emb": mat, "cls": rng.choice([-1, mat]), "theta": rng.choice([1e4, 5e5])}
    t = rng.choice([F32, F16, Q8_0, Q4_K, Q5_K, Q6_K])
    return {"kind": "qlinear", "type": t, "N": _log(rng, 64, 32000), "K": max(256, BLOCK[t][0] * (_log(rng, 64, 14336) // BLOCK[t][0]))}


# ── inputs ────────────────────────────────────────────────────────────────
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _rope(npos, dH, theta, dtype):
    p = np.arange(npos, dtype=np.float64)[:, None]
    a = p * (1.0 / np.power(theta, np.arange(0, dH, 2, dtype=np.float64) / dH))[None, :]
    return (torch.from_numpy(np.ascontiguousarray(np.cos(a))).to("cuda", dtype),
            torch.from_numpy(np.ascontiguousarray(np.sin(a))).to("cuda", dtype))


def _call(name, *args):
    fh.call(name, *[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args])


_ready = False


def _init():
    global _ready
    if not _ready:
        torch.cuda.init()
        fh.init(0)
        _ready = True


class _Graph:
    """A recorded pass (fg_graph_*), given back when its state goes."""

    def __init__(self, record):
        torch.cuda.synchronize()
        record()  # op by op once, as train() and Transformer.forward do before they record
        fh.check(fh.lib.fg_graph_begin(), "fg_graph_begin")
        record()
        p = ctypes.c_void_p()
        fh.check(fh.lib.fg_graph_end(ctypes.byref(p)), "fg_graph_end")
        self.ptr = p.value

    def launch(self):
        fh.check(fh.lib.fg_graph_launch(self.ptr), "fg_graph_launch")

    def __del__(self):
        fh.lib.fg_graph_destroy(self.ptr)


def _jobs(cls, rows):
    return (cls * len(rows))(*[cls(*[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in r]) for r in rows])


# ── a training layer ──────────────────────────────────────────────────────
def _layer_sizes(c):
    qD, kD = c["nH"] * c["dH"], c["nKV"] * c["dH"]
    return c["B"] * c["T"], qD, kD, qD + 2 * kD, c["hidden"]


def _layer_inputs(c, seed):
    M, D, _, Q, H = _layer_sizes(c)
    g = _gen(seed)
    return {"x": _randn(g, M, D), "gy": _randn(g, M, D, std=1e-3), "ln1": _randn(g, D, std=0.1, mean=1.0),
            "ln2": _randn(g, D, std=0.1, mean=1.0), "wqkv": _randn(g, Q, D, std=0.02), "wo": _randn(g, D, D, std=0.01),
            "wgu": _randn(g, 2 * H, D, std=0.02), "wdown": _randn(g, D, H, std=0.01)}


def _pieces(M, K, N):
    return fh.lib.fg_matmulT_bwd_x_pieces(M, K, N)


class _Norm:
    """rmsNorm with its gradient: the weight's left as partial rows for the grouped column sums, where it has that form."""

    def __init__(self, w, M, D):
        self.w, self.M, self.D = w, M, D
        self.y, self.inv, self.gx, self.gw = _empty(M, D), _empty(M), _empty(M, D), _empty(D)
        self.parts = fh.lib.fg_rmsnorm_bwd_parts(M, D)
        self.part = _empty(self.parts, D) if self.parts > 0 else None

    def fwd(self, x):
        _call("rmsnorm_fwd", self.y, self.inv, x, self.w, self.M, self.D, EPS)

    def bwd(self, gx_in, g, halves, x):
        if self.part is not None:
            _call("rmsnorm_bwd_partial", self.gx, gx_in, self.part, g, int(halves), x, self.w, self.inv, self.M, self.D)
        elif halves:
            _call("rmsnorm_bwd_from_halves", self.gx, gx_in, self.gw, 0, g, x, self.w, self.inv, self.M, self.D)
        else:
            _call("rmsnorm_bwd_from", self.gx, gx_in, self.gw, 0, g, x, self.w, self.inv, self.M, self.D)

    def job(self):
        return (self.gw, self.part, self.parts, self.D, 0)


class _InputGrad:
    """The gradient of a projection's normed input: in two halves where the split leaves them."""

    def __init__(self, M, K, N):
        self.M, self.K, self.N = M, K, N
        self.halves = _pieces(M, K, N) == 2
        self.g = _empty((2 if self.halves else 1) * M * K)

    def bwd(self, gy, w, xp_gy, xp_w, have):
        if self.halves:
            _call("matmulT_bwd_x_halves_p", self.g, gy, w, self.M, self.K, self.N, xp_gy, xp_w, have)
        else:
            _call("matmulT_bwd_x_p", self.g, gy, w, self.M, self.K, self.N, 0, xp_gy, xp_w, have)


def _layer(c, seed):
    i = _layer_inputs(c, seed)
    B, T, nH, nKV, dH = c["B"], c["T"], c["nH"], c["nKV"], c["dH"]
    M, D, kD, Q, H = _layer_sizes(c)
    cos, sin = _rope(T, dH, c["theta"], torch.float64)
    fused = dH in MFMA_HEADS
    n1, n2 = _Norm(i["ln1"], M, D), _Norm(i["ln2"], M, D)
    qkv, att, lse = _empty(M, Q), _empty(M, D), _empty(B * nH * T)
    x1, gu, act, y = _empty(M, D), _empty(M, 2 * H), _empty(M, H), _empty(M, D)
    gact, ggu, gatt, gqkv = _empty(M, H), _empty(M, 2 * H), _empty(M, D), _empty(M, Q)
    g2, g1 = _InputGrad(M, D, 2 * H), _InputGrad(M, D, Q)
    gw = {k: torch.empty_like(i[k]) for k in ("wqkv", "wo", "wgu", "wdown")}
    if not fused:
        q, k, v = _empty(M, D), _empty(M, kD), _empty(M, kD)
        gq, gk, gv = _empty(M, D), _empty(M, kD), _empty(M, kD)
    (x_qkv, w_qkv, x_wo, w_wo, x_gu, w_gu, x_down, w_down, g_down, g_gu, g_wo, g_qkv) = (_empty(XP) for _ in range(12))
    xp_att = _empty(3 * XP)
    wjobs = _jobs(fh.WgradJob, [(gw["wdown"], i["gy"], act, M, H, D, 0, g_down, x_down),
                                (gw["wgu"], ggu, n2.y, M, D, 2 * H, 0, g_gu, x_gu),
                                (gw["wo"], n2.gx, att, M, D, D, 0, g_wo, x_wo),
                                (gw["wqkv"], gqkv, n1.y, M, D, Q, 0, g_qkv, x_qkv)])
    cjobs = _jobs(fh.ColsumJob, [n.job() for n in (n2, n1) if n.part is not None])

    def step():
        n1.fwd(i["x"])
        if fused:
            _call("matmulT_fwd_rope_p", qkv, n1.y, i["wqkv"], M, D, Q, cos, sin, T, nH, nKV, dH, 0, T, x_qkv, w_qkv, 0)
            _call("attn_fwd_qkv_p", att, lse, qkv, B, T, nH, nKV, dH, xp_att)
        else:
            _call("matmulT_fwd_p", qkv, n1.y, i["wqkv"], M, D, Q, x_qkv, w_qkv, 0)
            _call("qkv_rope_fwd", q, k, v, qkv, cos, sin, T, M, nH, nKV, dH, 0, T)
            _call("attn_fwd", att, lse, q, k, v, B, T, nH, nKV, dH)
        _call("matmulT_fwd_resid_p", x1, i["x"], att, i["wo"], M, D, D, x_wo, w_wo, 0)
        n2.fwd(x1)
        _call("matmulT_fwd_swiglu_p", act, gu, n2.y, i["wgu"], M, D, H, x_gu, w_gu, 0)
        _call("matmulT_fwd_resid_p", y, x1, act, i["wdown"], M, H, D, x_down, w_down, 0)
        _call("matmulT_bwd_x_p", gact, i["gy"], i["wdown"], M, H, D, 0, g_down, w_down, 2)
        _call("swiglu_gu_bwd_p", ggu, 0, gact, gu, M, H, g_gu)
        g2.bwd(ggu, i["wgu"], g_gu, w_gu, 3)
        n2.bwd(i["gy"], g2.g, g2.halves, x1)
        _call("matmulT_bwd_x_p", gatt, n2.gx, i["wo"], M, D, D, 0, g_wo, w_wo, 2)
        if fused:
            _call("attn_bwd_qkv_p", gqkv, gatt, qkv, att, lse, B, T, nH, nKV, dH, cos, sin, T, 0, T, xp_att)
        else:
            _call("attn_bwd", gq, 0, gk, 0, gv, 0, gatt, q, k, v, att, lse, B, T, nH, nKV, dH)
            _call("qkv_rope_bwd", gqkv, gq, gk, gv, cos, sin, T, M, nH, nKV, dH, 0, T, 0)
        g1.bwd(gqkv, i["wqkv"], g_qkv, w_qkv, 2)
        n1.bwd(n2.gx, g1.g, g1.halves, i["x"])
        fh.check(fh.lib.fg_matmulT_bwd_w_grouped(wjobs, 4), "fg_matmulT_bwd_w_grouped")
        if len(cjobs):
            fh.check(fh.lib.fg_colsum_grouped(cjobs, len(cjobs)), "fg_colsum_grouped")

    out = {"y": y, "gx": n1.gx, "gln1": n1.gw, "gln2": n2.gw, **{"g" + k: v for k, v in gw.items()}}
    return {"graph": _Graph(step), "out": out, "keep": (i, cos, sin, locals())}


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w


def _rot64(x, cos, sin, B):
    # x [B*T, heads, dH]; interleaved pairs
    n = x.shape[0] // B
    c, s = (t[:n].repeat(B, 1)[:, None, :] for t in (cos, sin))
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _attn64(q, k, v, B, T):
    # q [B*T, nH, dH], k, v [B*T, nKV, dH] → [B*T, nH*dH]
    nH, nKV, dH = q.shape[1], k.shape[1], q.shape[2]
    mask = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    rows = []
    for b in range(B):
        heads = []
        for h in range(nH):
            z = h // max(1, nH // nKV)
            s = (q[b * T:(b + 1) * T, h] @ k[b * T:(b + 1) * T, z].t().contiguous()) / math.sqrt(dH)
            p = torch.softmax(s.masked_fill(mask, -math.inf), 1)
            heads.append(p @ v[b * T:(b + 1) * T, z].contiguous())
        rows.append(torch.cat(heads, 1))
    return torch.cat(rows, 0)


def _layer64(c, seed):
    i = {k: t.double().requires_grad_(k != "gy") for k, t in _layer_inputs(c, seed).items()}
    B, T, nH, nKV, dH = c["B"], c["T"], c["nH"], c["nKV"], c["dH"]
    M, D, kD, _, H = _layer_sizes(c)
    cos, sin = _rope(T, dH, c["theta"], torch.float64)
    qkv = _rms64(i["x"], i["ln1"]) @ i["wqkv"].t()
    q = _rot64(qkv[:, :D].reshape(M, nH, dH), cos, sin, B)
    k = _rot64(qkv[:, D:D + kD].reshape(M, nKV, dH), cos, sin, B)
    x1 = i["x"] + _attn64(q, k, qkv[:, D + kD:].reshape(M, nKV, dH), B, T) @ i["wo"].t()
    gu = _rms64(x1, i["ln2"]) @ i["wgu"].t()
    y = x1 + (torch.nn.functional.silu(gu[:, :H]) * gu[:, H:]) @ i["wdown"].t()
    y.backward(i["gy"])
    return {"y": y.detach(), "gx": i["x"].grad, **{"g" + n: i[n].grad for n in ("ln1", "ln2", "wqkv", "wo", "wgu", "wdown")}}


# ── one matmulT, one attention ────────────────────────────────────────────
def _matmul_inputs(c, seed):
    g = _gen(seed)
    return _randn(g, c["M"], c["K"]), _randn(g, c["N"], c["K"], std=0.02), _randn(g, c["M"], c["N"], std=1e-3)


def _matmul(c, seed):
    M, K, N = c["M"], c["K"], c["N"]
    x, w, gy = _matmul_inputs(c, seed)
    return {"x": x, "w": w, "gy": gy, "dims": (M, K, N), "xp": [_empty(XP) for _ in range(3)],
            "out": {"y": _empty(M, N), "gx": _empty(M, K), "gw": _empty(N, K)}}


def _matmul_run(s):
    o, (xx, xw, xg) = s["out"], s["xp"]
    _call("matmulT_fwd_p", o["y"], s["x"], s["w"], *s["dims"], xx, xw, 0)
    _call("matmulT_bwd_p", o["gx"], 0, o["gw"], 0, s["gy"], s["x"], s["w"], *s["dims"], xg, xx, xw, 6)


def _attn_inputs(c, seed):
    g = _gen(seed)
    M, qD, kD = c["B"] * c["T"], c["nH"] * c["dH"], c["nKV"] * c["dH"]
    return _randn(g, M, qD), _randn(g, M, kD), _randn(g, M, kD), _randn(g, M, qD, std=1e-3)


def _attn(c, seed):
    q, k, v, go = _attn_inputs(c, seed)
    return {"in": (q, k, v, go), "dims": [c[n] for n in ("B", "T", "nH", "nKV", "dH")],
            "out": {"o": torch.empty_like(q), "lse": _empty(c["B"] * c["nH"] * c["T"]), "gq": torch.empty_like(q),
                    "gk": torch.empty_like(k), "gv": torch.empty_like(v)}}


def _attn_run(s):
    o, (q, k, v, go) = s["out"], s["in"]
    _call("attn_fwd", o["o"], o["lse"], q, k, v, *s["dims"])
    _call("attn_bwd", o["gq"], 0, o["gk"], 0, o["gv"], 0, go, q, k, v, o["o"], o["lse"], *s["dims"])


# ── final norm, LM head, loss ─────────────────────────────────────────────
def _head_inputs(c, seed):
    g = _gen(seed)
    t = torch.randint(0, c["V"], (c["rows"],), generator=g, device="cuda", dtype=torch.int32)
    return _randn(g, c["rows"], c["dim"]), _randn(g, c["dim"], std=0.1, mean=1.0), _randn(g, c["V"], c["dim"], std=0.02), t


def _head(c, seed):
    M, D, V = c["rows"], c["dim"], c["V"]
    x, ln, w, t = _head_inputs(c, seed)
    n, gx = _Norm(ln, M, D), _InputGrad(M, D, V)
    logits, glogits, loss, lse, gw = _empty(M, V), _empty(M, V), _empty(1), _empty(M), torch.empty_like(w)
    xx, xw, xg = (_empty(XP) for _ in range(3))
    job = _jobs(fh.WgradJob, [(gw, glogits, n.y, M, D, V, 0, xg, xx)])
    col = _jobs(fh.ColsumJob, [n.job()]) if n.part is not None else None

    def step():
        n.fwd(x)
        _call("matmulT_fwd_p", logits, n.y, w, M, D, V, xx, xw, 0)
        _call("ce_fwd_bwd_p", loss, lse, glogits, logits, t, M, V, xg)
        gx.bwd(glogits, w, xg, xw, 3)
        n.bwd(None, gx.g, gx.halves, x)
        fh.check(fh.lib.fg_matmulT_bwd_w_grouped(job, 1), "fg_matmulT_bwd_w_grouped")
        if col is not None:
            fh.check(fh.lib.fg_colsum_grouped(col, 1), "fg_colsum_grouped")

    return {"step": step, "out": {"loss": loss, "logits": logits, "gx": n.gx, "gln": n.gw, "gw": gw}, "keep": (x, ln, w, t)}


def _head64(c, seed):
    x, ln, w, t = _head_inputs(c, seed)
    x, ln, w = (a.double().requires_grad_() for a in (x, ln, w))
    logits = _rms64(x, ln) @ w.t()
    loss = torch.nn.functional.cross_entropy(logits, t.long())
    loss.backward()
    return {"loss": loss.detach().reshape(1), "logits": logits.detach(), "gx": x.grad, "gln": ln.grad, "gw": w.grad}


# ── optimizer ─────────────────────────────────────────────────────────────
ADAM = {"lr": 3e-4, "b1": 0.9, "b2": 0.999, "eps": 1e-8, "wd": 0.01, "clip": 1.0, "bc1": 1 - 0.9 ** 100, "bc2": 1 - 0.999 ** 100}


def _adam_sizes(c):
    D, H, V = c["dim"], c["hidden"], c["V"]
    return [V * D, D, V * D] + [D, 3 * D * D, D * D, D, 2 * H * D, H * D] * c["layers"]


def _adam_inputs(c, seed):
    n = sum(_adam_sizes(c))
    g = _gen(seed)
    return _randn(g, n, std=0.02), _randn(g, n, std=1e-3), _randn(g, n, std=1e-4), _randn(g, n, std=1e-3).square_()


class _Adam:
    def __init__(self, tensors):
        self.keep = tensors
        p = ctypes.c_void_p()
        fh.check(fh.lib.fg_adam_plan_create(tensors, len(tensors), ctypes.byref(p)), "fg_adam_plan_create")
        self.ptr = p.value

    def __del__(self):
        fh.lib.fg_adam_plan_destroy(self.ptr)


def _adam(c, seed):
    p, g, m, v = _adam_inputs(c, seed)
    rows, at = [], 0
    for n in _adam_sizes(c):
        rows.append(tuple(t.data_ptr() + 4 * at for t in (p, g, m, v)) + (n,))
        at += n
    stats = _empty(2, dtype=torch.float64)
    return {"plan": _Adam(_jobs(fh.AdamTensor, rows)), "keep": g, "out": {"p": p, "m": m, "v": v, "stats": stats}}


def _adam_run(s):
    a = ADAM
    _call("adam_step_plan", s["plan"].ptr, a["lr"], a["b1"], a["b2"], a["eps"], a["wd"], a["clip"], a["bc1"], a["bc2"],
          s["out"]["stats"])


def _adam64(c, seed):
    a = ADAM
    p, g, m, v = (t.double() for t in _adam_inputs(c, seed))
    norm = torch.sqrt((g * g).sum())
    scale = torch.where(norm > a["clip"], a["clip"] / norm, torch.ones_like(norm))
    g = g * scale + a["wd"] * p
    m = a["b1"] * m + (1 - a["b1"]) * g
    v = a["b2"] * v + (1 - a["b2"]) * g * g
    p = p - a["lr"] * (m / a["bc1"]) / (torch.sqrt(v / a["bc2"]) + a["eps"])
    return {"p": p, "m": m, "v": v, "stats": torch.stack([norm, scale])}


# ── the token side of a step ──────────────────────────────────────────────
def _tokens_inputs(c, seed):
    g = _gen(seed)
    M, V, D = c["B"] * c["T"], c["V"], c["dim"]
    # ids as text has them: their frequency falls with their rank
    u = torch.rand(1 << 20, generator=g, device="cuda", dtype=torch.float64)
    rank = torch.exp(u * math.log(V + 1)).sub_(1).floor_().clamp_(0, V - 1).to(torch.int64)
    data = torch.randperm(V, generator=g, device="cuda")[rank].to(torch.int32)
    starts = torch.randint(0, (1 << 20) - c["T"] - 1, (c["B"],), generator=g, device="cuda", dtype=torch.int32)
    return data, starts, _randn(g, V, D, std=0.02), _randn(g, M, D, std=1e-3)


def _tokens(c, seed):
    data, starts, w, gx = _tokens_inputs(c, seed)
    M = c["B"] * c["T"]
    n = ctypes.c_int64()
    fh.check(fh.lib.fg_embed_keys_len(M, ctypes.byref(n)), "fg_embed_keys_len")
    return {"in": (data, starts, w, gx), "dims": (c["B"], c["T"], c["V"], c["dim"]), "keys": _empty(n.value, dtype=torch.int64),
            "out": {"ids": _empty(M, dtype=torch.int32), "targets": _empty(M, dtype=torch.int32), "x": _empty(M, c["dim"]),
                    "gw": torch.empty_like(w)}}


def _tokens_run(s):
    o, (data, starts, w, gx), (B, T, V, D), keys = s["out"], s["in"], s["dims"], s["keys"]
    _call("batch_gather", o["ids"], o["targets"], data, data.numel(), starts, B, T, V)
    _call("embed_fwd", o["x"], w, o["ids"], B * T, V, D)
    _call("embed_sort_keys", keys, keys.numel(), o["ids"], B * T, V)
    _call("zero", o["gw"], 4 * V * D)
    _call("embed_bwd_sorted", o["gw"], gx, keys, B * T, V, D, 0)


def _tokens64(c, seed):
    data, starts, w, gx = _tokens_inputs(c, seed)
    at = (starts.long()[:, None] + torch.arange(c["T"], device="cuda")[None, :]).reshape(-1)
    ids = data[at].long()
    gw = torch.zeros(w.shape, dtype=torch.float64, device="cuda").index_add_(0, ids, gx.double())
    return {"ids": None, "targets": None, "x": w[ids].double(), "gw": gw}


# ── quantized matrices ────────────────────────────────────────────────────
def _matrix(g, t, N, K, std):
    """Rows of a ggml type, about std in spread: the blocks' integers uniform, their scales to match."""
    if t == F32:
        return _randn(g, N, K, std=std)
    if t == F16:
        return _randn(g, N, K, std=std).half()
    el, nb = BLOCK[t]
    blocks = N * (K // el)
    q = torch.randint(0, 256, (blocks, nb), generator=g, device="cuda", dtype=torch.uint8)

    def half(x):
        u = torch.rand(blocks, 1, generator=g, device="cuda").mul_(0.5).add_(0.75)
        return (u * x).half().view(torch.uint8)

    if t == Q8_0:
        q[:, 0:2] = half(std / 74)
    elif t == Q6_K:  # (q - 32) times an int8 scale: 18.5 times 74
        q[:, 208:210] = half(std / (18.5 * 74))
    else:  # d·sc·q - dmin·m, sc and m 6 bits: dmin·m takes the mean of d·sc·q away
        top = 15 if t == Q4_K else 31
        d = std / (32 * top / 3.4641 * 1.6)
        q[:, 0:2] = half(d)
        q[:, 2:4] = half(d * top / 2)
    return q


def _values(q, t, N, K):
    """What _matrix's bytes stand for, in 64 bits."""
    if t in (F32, F16):
        return q.double()
    if t == Q8_0:
        return (q[:, 2:].contiguous().view(torch.int8).double() * q[:, 0:2].contiguous().view(torch.float16).double()).reshape(N, K)
    if t == Q6_K:
        ql, qh = q[:, 0:128].reshape(-1, 2, 64).int(), q[:, 128:192].reshape(-1, 2, 32).int()
        lo, hi = ql[:, :, :32], ql[:, :, 32:]
        v = torch.stack([(lo & 15) | ((qh & 3) << 4), (hi & 15) | (((qh >> 2) & 3) << 4),
                         (lo >> 4) | (((qh >> 4) & 3) << 4), (hi >> 4) | (((qh >> 6) & 3) << 4)], 2).reshape(-1, 256) - 32
        sc = q[:, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 1)
        return (q[:, 208:210].contiguous().view(torch.float16).double() * sc * v).reshape(N, K)
    d, dm = (q[:, a:a + 2].contiguous().view(torch.float16).double() for a in (0, 2))
    s = q[:, 4:16].int()
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    qs = q[:, -128:].int().reshape(-1, 4, 32)
    v = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if t == Q5_K:
        qh = q[:, 16:48].int()
        v = v + 16 * torch.stack([(qh >> b) & 1 for b in range(8)], 1)
    return ((d * sc)[:, :, None] * v - (dm * mn)[:, :, None]).reshape(N, K)


def _qlinear(c, seed):
    g = _gen(seed)
    w = _matrix(g, c["type"], c["N"], c["K"], 0.02)
    return {"w": w, "x": _randn(g, c["K"]), "dims": (c["type"], c["N"], c["K"]), "out": {"y": _empty(c["N"])}}


def _qlinear_run(s):
    t, N, K = s["dims"]
    _call("qmatvec", t, s["out"]["y"], s["w"], s["x"], N, K)


def _qlinear64(c, seed):
    s = _qlinear(c, seed)
    return {"y": _values(s["w"], c["type"], c["N"], c["K"]) @ s["x"].double()}


# ── decode ────────────────────────────────────────────────────────────────
def _decode_inputs(c, seed):
    g = _gen(seed)
    D, H, V, L = c["dim"], c["hidden"], c["V"], c["layers"]
    dH = D // c["nH"]
    kD = c["nKV"] * dH
    w = {"emb": _matrix(g, c["emb"], V, D, 0.5), "ln_f": _randn(g, D, std=0.1, mean=1.0), "layers": []}
    w["cls"] = w["emb"] if c["cls"] < 0 else _matrix(g, c["cls"], V, D, 0.02)
    for _ in range(L):
        w["layers"].append({"ln1": _randn(g, D, std=0.1, mean=1.0), "wqkv": _matrix(g, c["mat"], D + 2 * kD, D, 0.02),
                            "wo": _matrix(g, c["mat"], D, D, 0.01), "ln2": _randn(g, D, std=0.1, mean=1.0),
                            "gate": _matrix(g, c["mat"], H, D, 0.02), "up": _matrix(g, c["mat"], H, D, 0.02),
                            "down": _matrix(g, c["down"], D, H, 0.01)})
    kc, vc = (torch.zeros(L, c["maxSeq"], kD, device="cuda") for _ in range(2))
    for t in (kc, vc):  # the tokens before this one
        t[:, :c["pos"]] = _randn(g, L, c["pos"], kD, std=0.5)
    token = int(torch.randint(0, V, (1,), generator=g, device="cuda"))
    return w, kc, vc, token


def _decode(c, seed):
    w, kc, vc, token = _decode_inputs(c, seed)
    D, H, V, L, nH, nKV = c["dim"], c["hidden"], c["V"], c["layers"], c["nH"], c["nKV"]
    dH = D // nH
    cos, sin = _rope(c["maxSeq"], dH, c["theta"], torch.float32)
    n = ctypes.c_int64()
    fh.check(fh.lib.fg_decode_part_len(nH, dH, c["maxSeq"], ctypes.byref(n)), "fg_decode_part_len")
    x, q, h, part, logits = _empty(D), _empty(nH * dH), _empty(H), _empty(n.value, dtype=torch.float64), _empty(V)
    layers = (fh.DecodeLayer * L)(*[
        fh.DecodeLayer(*[a[k].data_ptr() for k in ("ln1", "wqkv", "wo", "ln2", "gate", "up", "down")],
                       c["mat"], c["mat"], c["mat"], c["mat"], c["down"]) for a in w["layers"]])
    model = fh.DecodeModel(D, H, L, nH, nKV, V, c["maxSeq"], c["emb"], c["emb"] if c["cls"] < 0 else c["cls"], EPS,
                           w["emb"].data_ptr(), w["ln_f"].data_ptr(), w["cls"].data_ptr(),
                           ctypes.cast(layers, ctypes.c_void_p), cos.data_ptr(), sin.data_ptr(), x.data_ptr(), q.data_ptr(),
                           h.data_ptr(), part.data_ptr())
    host = np.array([token, c["pos"]], np.int32)
    state = torch.from_numpy(host).cuda()

    def step():
        fh.check(fh.lib.fg_decode_step(ctypes.byref(model), kc.data_ptr(), vc.data_ptr(), state.data_ptr(), logits.data_ptr()),
                 "fg_decode_step")

    return {"graph": _Graph(step), "state": state, "host": host, "out": {"logits": logits, "k": kc, "v": vc},
            "keep": (w, cos, sin, x, q, h, part, layers, model)}


def _decode_run(s):
    # what Transformer.forward does for each token: the token and its position up, then the recorded step
    fh.check(fh.lib.fg_h2d(s["state"].data_ptr(), s["host"].ctypes.data, 8), "fg_h2d")
    s["graph"].launch()


def _decode64(c, seed):
    w, kc, vc, token = _decode_inputs(c, seed)
    D, H, V, nH, nKV, pos = c["dim"], c["hidden"], c["V"], c["nH"], c["nKV"], c["pos"]
    dH = D // nH
    kD = nKV * dH
    cos, sin = (t.double()[pos:pos + 1] for t in _rope(c["maxSeq"], dH, c["theta"], torch.float32))
    el = BLOCK[c["emb"]][0]
    row = w["emb"][token * (D // el):(token + 1) * (D // el)] if el > 1 else w["emb"][token:token + 1]
    x = _values(row, c["emb"], 1, D)[0]
    kc, vc = kc.double(), vc.double()
    for n, a in enumerate(w["layers"]):
        qkv = _values(a["wqkv"], c["mat"], D + 2 * kD, D) @ _rms64(x[None], a["ln1"].double())[0]
        q = _rot64(qkv[:D].reshape(1, nH, dH), cos, sin, 1)[0]
        kc[n, pos] = _rot64(qkv[D:D + kD].reshape(1, nKV, dH), cos, sin, 1).reshape(-1)
        vc[n, pos] = qkv[D + kD:]
        k, v = (t[n, :pos + 1].reshape(pos + 1, nKV, dH).repeat_interleave(nH // nKV, 1) for t in (kc, vc))
        p = torch.softmax((k * q[None]).sum(2) / math.sqrt(dH), 0)
        x = x + _values(a["wo"], c["mat"], D, D) @ (p[:, :, None] * v).sum(0).reshape(-1)
        xn = _rms64(x[None], a["ln2"].double())[0]
        g, u = (_values(a[k2], c["mat"], H, D) @ xn for k2 in ("gate", "up"))
        x = x + _values(a["down"], c["down"], D, H) @ (torch.nn.functional.silu(g) * u)
    t = c["emb"] if c["cls"] < 0 else c["cls"]
    logits, xn = [], _rms64(x[None], w["ln_f"].double())[0]
    per = D // BLOCK[t][0] if BLOCK[t][0] > 1 else 1
    for r in range(0, V, 16384):  # the head's rows in parts: it is the largest matrix
        n = min(16384, V - r)
        logits.append(_values(w["cls"][r * per:(r + n) * per], t, n, D) @ xn)
    return {"logits": torch.cat(logits), "k": kc, "v": vc}


# ── the interface ─────────────────────────────────────────────────────────
_PREPARE = {"layer": _layer, "matmul": _matmul, "attention": _attn, "head": _head, "adam": _adam, "tokens": _tokens,
            "decode": _decode, "qlinear": _qlinear}
_RUN = {"layer": lambda s: s["graph"].launch(), "matmul": _matmul_run, "attention": _attn_run, "head": lambda s: s["step"](),
        "adam": _adam_run, "tokens": _tokens_run, "decode": _decode_run, "qlinear": _qlinear_run}


def prepare(case, seed):
    _init()
    s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    return s


def run(state):
    _RUN[state["kind"]](state)
    return state["out"]


def _matrix_bytes(t, N, K):
    return N * (K // BLOCK[t][0]) * BLOCK[t][1]


def work(case):
    c, k = case, case["kind"]
    if k == "layer":
        M, D, _, Q, H = _layer_sizes(c)
        P = Q * D + D * D + 3 * H * D
        pairs = c["T"] * (c["T"] + 1) / 2 * c["B"] * c["nH"]
        return {"bytes": 4.0 * (4 * M * D + 2 * P), "flops": 6.0 * M * P + 12.0 * c["dH"] * pairs}
    if k == "matmul":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 8.0 * (M * K + N * K + M * N), "flops": 6.0 * M * K * N}
    if k == "attention":
        n = c["B"] * c["T"] * c["dH"]
        pairs = c["T"] * (c["T"] + 1) / 2 * c["B"] * c["nH"]
        return {"bytes": 4.0 * n * (4 * c["nH"] + 4 * c["nKV"]), "flops": 12.0 * c["dH"] * pairs}
    if k == "head":
        M, D, V = c["rows"], c["dim"], c["V"]
        return {"bytes": 4.0 * (2 * M * D + 2 * V * D + M * V), "flops": 6.0 * M * D * V}
    if k == "adam":
        n = sum(_adam_sizes(c))
        return {"bytes": 28.0 * n, "flops": 16.0 * n}
    if k == "tokens":
        M = c["B"] * c["T"]
        return {"bytes": 4.0 * (3 * M * c["dim"] + c["V"] * c["dim"] + 3 * M), "flops": 1.0 * M * c["dim"]}
    if k == "qlinear":
        return {"bytes": _matrix_bytes(c["type"], c["N"], c["K"]) + 4.0 * (c["N"] + c["K"]), "flops": 2.0 * c["N"] * c["K"]}
    D, H, L = c["dim"], c["hidden"], c["layers"]
    kD = c["nKV"] * (D // c["nH"])
    t = c["emb"] if c["cls"] < 0 else c["cls"]
    b = L * (_matrix_bytes(c["mat"], 2 * D + 2 * kD + 2 * H, D) + _matrix_bytes(c["down"], D, H) + 8.0 * kD * (c["pos"] + 1))
    f = 2.0 * L * (D * (2 * D + 2 * kD) + 3 * D * H + 2 * D * (c["pos"] + 1)) + 2.0 * D * c["V"]
    return {"bytes": b + _matrix_bytes(t, c["V"], D) + 4.0 * c["V"], "flops": f}


def tolerance(case):
    # about four times the errors against 64 bits that the largest sizes show: fp32 products from split pieces,
    # fp32 sums (over up to 32000 terms, attention's over a long window above all) and fp32 stores between the ops
    return {"rel": {"layer": 3e-5, "matmul": 2e-6, "attention": 2e-5, "head": 5e-6, "adam": 2e-7, "tokens": 1e-6,
                    "decode": 5e-6, "qlinear": 1e-6}[case["kind"]]}


_EXACT = {"layer": _layer64, "head": _head64, "adam": _adam64, "tokens": _tokens64, "decode": _decode64, "qlinear": _qlinear64}


def exact(case, seed):
    if case["kind"] == "matmul":
        x, w, gy = (t.double() for t in _matmul_inputs(case, seed))
        return {"y": x @ w.t(), "gx": gy @ w, "gw": gy.t() @ x}
    if case["kind"] == "attention":
        B, T, nH, nKV, dH = (case[n] for n in ("B", "T", "nH", "nKV", "dH"))
        q, k, v, go = (t.double() for t in _attn_inputs(case, seed))
        for t in (q, k, v):
            t.requires_grad_()
        o = _attn64(q.reshape(-1, nH, dH), k.reshape(-1, nKV, dH), v.reshape(-1, nKV, dH), B, T)
        o.backward(go)
        return {"o": o.detach(), "lse": None, "gq": q.grad, "gk": k.grad, "gv": v.grad}
    return _EXACT[case["kind"]](case, seed)
