"""Performance cases of the layer path: what a program that uses this library
has it do, through the public entry points of ``mimir_hip``.

Every case is a dict of plain values; ``prepare`` makes its inputs on the GPU
from a seed, ``run`` is one pass, ``exact`` the same pass in 64-bit torch.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mimir-framework_amd"))
import mimir_hip as M  # noqa: E402

DEV = "cuda:0"
F64 = torch.float64
_CTX = []


def ctx():
    """The one context that a single-threaded program keeps."""
    if not _CTX:
        _CTX.append(M.Context(0))
    return _CTX[0]


class Rand:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, scale=1.0, mean=0.0):
        t = torch.randn(shape, generator=self.g, device=DEV)
        if scale != 1.0:
            t *= scale
        if mean:
            t += mean
        return t

    def ids(self, n, vocab, zipf):
        """Token ids: uniform, or with frequencies falling as 1 / rank, the
        ranks spread over the vocabulary."""
        if not zipf:
            return torch.randint(vocab, (n,), generator=self.g, device=DEV, dtype=torch.int32)
        u = torch.rand(n, generator=self.g, device=DEV, dtype=F64)
        ranks = ((vocab + 1.0) ** u).long() - 1
        perm = torch.randperm(vocab, generator=self.g, device=DEV)
        return perm[ranks.clamp_(0, vocab - 1)].to(torch.int32)


def like(t):
    return torch.empty_like(t)


def done(state):
    # The library works on a stream of its own: the inputs have to be there.
    torch.cuda.synchronize()
    return state


# --- residual add + RMSNorm --------------------------------------------------

def add_rmsnorm_prepare(c, r):
    n, w = c["rows"], c["cols"]
    s = {"x": r.normal(n, w), "res": r.normal(n, w), "w": r.normal(w, scale=0.02, mean=1.0)}
    s["y"], s["h"] = like(s["x"]), like(s["x"])
    return s


def add_rmsnorm_run(c, s):
    ctx().add_rmsnorm(s["x"].data_ptr(), s["res"].data_ptr(), s["h"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(),
                      c["rows"], c["cols"], 1e-6)
    return {"y": s["y"], "h": s["h"]}


def add_rmsnorm_exact(c, s):
    h = (s["x"] + s["res"]).to(F64)  # the sum is stored in 32 bits and read back
    return {"y": h / torch.sqrt((h * h).mean(1, keepdim=True) + 1e-6) * s["w"].to(F64), "h": h}


def add_rmsnorm_work(c):
    n = c["rows"] * c["cols"]
    return {"bytes": 4 * (4 * n + c["cols"]), "flops": 5 * n}


# --- row softmax of causal scores --------------------------------------------

def softmax_prepare(c, r):
    n, q, k = c["rows"], c["q"], c["cols"]
    x = r.normal(n // q, q, k, scale=3.0)
    x.masked_fill_(torch.ones(q, k, device=DEV, dtype=torch.bool).triu_(1 + max(0, k - q)), -math.inf)
    x = x.reshape(n // q * q, k)
    return {"x": x, "y": like(x)}


def softmax_run(c, s):
    ctx().softmax(s["x"].data_ptr(), s["y"].data_ptr(), s["x"].shape[0], c["cols"], M.SOFTMAX_DIV_EPS)
    return s["y"]


def softmax_exact(c, s):
    out = torch.empty(s["x"].shape, device=DEV, dtype=F64)
    for at in range(0, out.shape[0], 65536):
        x = s["x"][at:at + 65536].to(F64)
        x = torch.exp(x - x.amax(1, keepdim=True))
        out[at:at + 65536] = x / (x.sum(1, keepdim=True) + 1e-9)
    return out


def softmax_work(c):
    n = c["rows"] // c["q"] * c["q"] * c["cols"]
    return {"bytes": 8 * n, "flops": 5 * n}


# --- token gather, then RoPE on q and k --------------------------------------

def embed_rope_prepare(c, r):
    t, d = c["batch"] * c["seq"], c["heads"] * c["head_dim"]
    cos, sin = M.rope_table(c["seq"], c["head_dim"], 10000.0)
    s = {"table": r.normal(c["vocab"], d, scale=0.02), "ids": r.ids(t, c["vocab"], c["zipf"]),
         "q": r.normal(t, d), "k": r.normal(t, c["k_heads"] * c["head_dim"]),
         "cos": torch.from_numpy(cos).to(DEV), "sin": torch.from_numpy(sin).to(DEV)}
    s["y"], s["qo"], s["ko"] = torch.empty(t, d, device=DEV), like(s["q"]), like(s["k"])
    return s


def embed_rope_run(c, s):
    d = c["heads"] * c["head_dim"]
    ctx().embedding(s["ids"].data_ptr(), s["ids"].numel(), s["table"].data_ptr(), c["vocab"] * d, c["vocab"], d, -1,
                    s["y"].data_ptr())
    ctx().rope(s["q"].data_ptr(), s["qo"].data_ptr(), c["heads"], s["k"].data_ptr(), s["ko"].data_ptr(), c["k_heads"],
               c["batch"], c["seq"], c["head_dim"], 0, s["cos"].data_ptr(), s["sin"].data_ptr(), c["seq"])
    # The gathered rows are copies, bit for bit: returned as whole numbers.
    return {"rows": s["y"].view(torch.int32), "q": s["qo"], "k": s["ko"]}


def embed_rope_exact(c, s):
    def rot(x, heads):
        x = x.to(F64).reshape(c["batch"], c["seq"], heads, 2, c["head_dim"] // 2)
        cos, sin = (t.to(F64)[None, :, None, :] for t in (s["cos"], s["sin"]))
        a, b = x[..., 0, :], x[..., 1, :]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], 3).reshape(c["batch"] * c["seq"], -1)
    return {"rows": None, "q": rot(s["q"], c["heads"]), "k": rot(s["k"], c["k_heads"])}


def embed_rope_work(c):
    t, d, kd = c["batch"] * c["seq"], c["heads"] * c["head_dim"], c["k_heads"] * c["head_dim"]
    return {"bytes": 4 * t * (1 + 2 * d + 2 * d + 2 * kd) + 4 * c["seq"] * c["head_dim"], "flops": 3 * t * (d + kd)}


# --- the elementwise chain of a decoder MLP, forward -------------------------

def mlp_prepare(c, r):
    n, h, m = c["rows"], c["hidden"], c["inner"]
    s = {"x": r.normal(n, h), "res": r.normal(n, h), "g": r.normal(h, scale=0.02, mean=1.0), "b": r.normal(h, scale=0.02),
         "gate": r.normal(n, m), "up": r.normal(n, m)}
    for name, src in (("ln", "x"), ("gelu", "up"), ("glu", "gate"), ("sum", "x")):
        s[name] = like(s[src])
    return s


def mlp_run(c, s):
    n, nh, nm = c["rows"], s["x"].numel(), s["gate"].numel()
    ctx().layernorm(s["x"].data_ptr(), s["g"].data_ptr(), s["b"].data_ptr(), s["ln"].data_ptr(), n, c["hidden"], 1e-5)
    ctx().gelu(s["up"].data_ptr(), s["gelu"].data_ptr(), nm)
    ctx().silu_mul(s["gate"].data_ptr(), s["up"].data_ptr(), s["glu"].data_ptr(), nm)
    ctx().add(s["ln"].data_ptr(), nh, s["res"].data_ptr(), nh, s["sum"].data_ptr())
    return {k: s[k] for k in ("ln", "gelu", "glu", "sum")}


def gelu64(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def norm64(x, eps):
    x = x.to(F64)
    x = x - x.mean(1, keepdim=True)
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + eps)


def mlp_exact(c, s):
    ln = norm64(s["x"], 1e-5) * s["g"].to(F64) + s["b"].to(F64)
    gate, up = s["gate"].to(F64), s["up"].to(F64)
    return {"ln": ln, "gelu": gelu64(up), "glu": gate * torch.sigmoid(gate) * up, "sum": ln + s["res"].to(F64)}


def mlp_work(c):
    nh, nm = c["rows"] * c["hidden"], c["rows"] * c["inner"]
    return {"bytes": 4 * (5 * nh + 5 * nm + 2 * c["hidden"]), "flops": 9 * nh + 18 * nm}


# --- rows of any width: LayerNorm both ways, log-softmax ----------------------

def rows_prepare(c, r):
    n, w = c["rows"], c["cols"]
    s = {"x": r.normal(n, w), "dy": r.normal(n, w), "g": r.normal(w, scale=0.02, mean=1.0), "b": r.normal(w, scale=0.02)}
    for name in ("ln", "dx", "ls"):
        s[name] = like(s["x"])
    s["dw"] = torch.empty(2, w, device=DEV)
    return s


def rows_run(c, s):
    n, w = c["rows"], c["cols"]
    ctx().layernorm(s["x"].data_ptr(), s["g"].data_ptr(), s["b"].data_ptr(), s["ln"].data_ptr(), n, w, 1e-5)
    ctx().softmax(s["ln"].data_ptr(), s["ls"].data_ptr(), n, w, M.SOFTMAX_LOG)
    ctx().fill(s["dw"].data_ptr(), 0.0, 2 * w)  # gradients of the weights are added to
    ctx().layernorm_bwd(s["x"].data_ptr(), s["dy"].data_ptr(), s["g"].data_ptr(), s["dx"].data_ptr(), s["dw"].data_ptr(),
                        s["dw"].data_ptr() + 4 * w, n, w, 1e-5)
    return {k: s[k] for k in ("ln", "ls", "dx", "dw")}


def norm_bwd64(x, dy, g, eps):
    x, dy = x.to(F64), dy.to(F64)
    rstd = 1 / torch.sqrt(x.var(1, unbiased=False, keepdim=True) + eps)
    xh = (x - x.mean(1, keepdim=True)) * rstd
    gy = dy * g.to(F64)
    dx = rstd * (gy - gy.mean(1, keepdim=True) - xh * (gy * xh).mean(1, keepdim=True))
    return dx, torch.stack([(dy * xh).sum(0), dy.sum(0)])


def rows_exact(c, s):
    ln = norm64(s["x"], 1e-5) * s["g"].to(F64) + s["b"].to(F64)
    dx, dw = norm_bwd64(s["x"], s["dy"], s["g"], 1e-5)
    return {"ln": ln, "ls": torch.log_softmax(ln, 1), "dx": dx, "dw": dw}


def rows_work(c):
    n = c["rows"] * c["cols"]
    return {"bytes": 4 * (7 * n + 5 * c["cols"]), "flops": 30 * n}


# --- the backward of an elementwise residual block ---------------------------

def block_bwd_prepare(c, r):
    n, w = c["rows"], c["cols"]
    s = {"h": r.normal(n, w), "gate": r.normal(n, w), "dy": r.normal(n, w), "gamma": r.normal(w, scale=0.02, mean=1.0)}
    # What the forward Add -> LayerNorm -> GELU -> Multiply -> SiLU kept.
    s["n"] = torch.nn.functional.layer_norm(s["h"], (w,), s["gamma"])
    s["g"] = torch.nn.functional.gelu(s["n"], approximate="tanh")
    s["m"] = s["g"] * s["gate"]
    for name in ("dm", "dg", "dgate", "dn", "dh", "da", "db"):
        s[name] = like(s["h"])
    s["dw"] = torch.empty(2, w, device=DEV)
    return s


def block_bwd_run(c, s):
    p = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    n, w = c["rows"], c["cols"]
    x = ctx()
    x.fill(p["dw"], 0.0, 2 * w)
    x.silu_bwd(p["m"], p["dy"], p["dm"], n * w)
    x.mul_bwd(p["g"], p["gate"], p["dm"], p["dg"], p["dgate"], n * w)
    x.gelu_bwd(p["n"], p["dg"], p["dn"], n * w)
    x.layernorm_bwd(p["h"], p["dn"], p["gamma"], p["dh"], p["dw"], p["dw"] + 4 * w, n, w, 1e-5)
    x.add_bwd(p["dh"], n * w, n * w, p["da"], p["db"])
    return {k: s[k] for k in ("dgate", "dw", "da", "db")}


def block_bwd_exact(c, s):
    dy, m = s["dy"].to(F64), s["m"].to(F64)
    sg = torch.sigmoid(m)
    dm = dy * (sg + m * sg * (1 - sg))
    del m, sg
    dgate = dm * s["g"].to(F64)
    n = s["n"].to(F64).requires_grad_()
    dn, = torch.autograd.grad(gelu64(n), n, dm * s["gate"].to(F64))
    dx, dw = norm_bwd64(s["h"], dn, s["gamma"], 1e-5)
    return {"dgate": dgate, "dw": dw, "da": dx, "db": dx}


def block_bwd_work(c):
    n = c["rows"] * c["cols"]
    return {"bytes": 4 * (17 * n + 5 * c["cols"]), "flops": 50 * n}


# --- the embedding's gradient -------------------------------------------------

def embed_bwd_prepare(c, r):
    return {"ids": r.ids(c["tokens"], c["vocab"], c["zipf"]), "dy": r.normal(c["tokens"], c["dim"], scale=0.01),
            "grad": torch.empty(c["vocab"], c["dim"], device=DEV)}


def embed_bwd_run(c, s):
    n = c["vocab"] * c["dim"]
    ctx().fill(s["grad"].data_ptr(), 0.0, n)
    ctx().embedding_bwd(s["ids"].data_ptr(), c["tokens"], s["dy"].data_ptr(), s["grad"].data_ptr(), n, c["vocab"],
                        c["dim"], -1)
    return s["grad"]


def embed_bwd_exact(c, s):
    out = torch.zeros(c["vocab"], c["dim"], device=DEV, dtype=F64)
    return out.index_add_(0, s["ids"].long(), s["dy"].to(F64))


def embed_bwd_work(c):
    return {"bytes": 4 * (c["tokens"] * (1 + c["dim"]) + c["vocab"] * c["dim"]), "flops": c["tokens"] * c["dim"]}


# --- the attention core, forward and backward ---------------------------------

def attn_prepare(c, r):
    b, lq, lk, w = c["batch"], c["q_len"], c["kv_len"], c["heads"] * c["head_dim"]
    if lq == lk:  # the projection's output, [rows, 3 width]
        qkv = r.normal(b * lq, 3 * w)
        s = {"q": qkv[:, :w], "k": qkv[:, w:2 * w], "v": qkv[:, 2 * w:]}
    else:
        kv = r.normal(b * lk, 2 * w)
        s = {"q": r.normal(b * lq, w), "k": kv[:, :w], "v": kv[:, w:]}
    if c["kind"] == "attn_bwd":
        s["do"] = r.normal(b * lq, w)
        s["dq"], s["dkv"] = torch.empty(b * lq, w, device=DEV), torch.empty(b * lk, 2 * w, device=DEV)
    else:
        s["out"] = torch.empty(b * lq, w, device=DEV)
    return s


def attn_run(c, s):
    b, lq, lk, h, d = c["batch"], c["q_len"], c["kv_len"], c["heads"], c["head_dim"]
    w, ld_q, ld_kv = h * d, s["q"].stride(0), s["k"].stride(0)
    q, k, v = s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr()
    if c["kind"] == "attn_bwd":
        ctx().attention_bwd(q, k, v, s["do"].data_ptr(), s["dq"].data_ptr(), s["dkv"].data_ptr(),
                            s["dkv"].data_ptr() + 4 * w, b, lq, lk, h, d, c["causal"], ld_q=ld_q, ld_kv=ld_kv, ld_dkv=2 * w)
        return {"dq": s["dq"], "dkv": s["dkv"]}
    ctx().attention(q, k, v, s["out"].data_ptr(), b, lq, lk, h, d, c["causal"], ld_q=ld_q, ld_kv=ld_kv)
    return s["out"]


def attn_one64(q, k, v, causal):
    """One sequence, [heads, rows, head_dim] in 64 bits: (out, probabilities)."""
    sc = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[2])
    if causal:
        hide = torch.ones(sc.shape[1:], device=DEV, dtype=torch.bool).triu_(1)
        sc.masked_fill_(hide, -math.inf)
    p = torch.softmax(sc, 2)
    return torch.matmul(p, v), p


def attn_exact(c, s):
    b, lq, lk, h, d = c["batch"], c["q_len"], c["kv_len"], c["heads"], c["head_dim"]
    w = h * d

    def heads(t, i, n):  # [n, heads, d] rows of sequence i -> [heads, n, d]
        return t[i * n:(i + 1) * n].to(F64).reshape(n, h, d).transpose(0, 1).contiguous()

    def rows(t):
        return t.transpose(0, 1).reshape(-1, w)

    if c["kind"] == "attn":
        out = torch.empty(b * lq, w, device=DEV, dtype=F64)
        for i in range(b):
            o, _ = attn_one64(heads(s["q"], i, lq), heads(s["k"], i, lk), heads(s["v"], i, lk), c["causal"])
            out[i * lq:(i + 1) * lq] = rows(o)
        return out
    dq, dkv = torch.empty(b * lq, w, device=DEV, dtype=F64), torch.empty(b * lk, 2 * w, device=DEV, dtype=F64)
    for i in range(b):
        q, k, v, do = heads(s["q"], i, lq), heads(s["k"], i, lk), heads(s["v"], i, lk), heads(s["do"], i, lq)
        _, p = attn_one64(q, k, v, c["causal"])
        dkv[i * lk:(i + 1) * lk, w:] = rows(torch.matmul(p.transpose(1, 2).contiguous(), do))
        ds = torch.matmul(do, v.transpose(1, 2).contiguous())
        ds = p * (ds - (p * ds).sum(2, keepdim=True)) / math.sqrt(d)
        dq[i * lq:(i + 1) * lq] = rows(torch.matmul(ds, k))
        dkv[i * lk:(i + 1) * lk, :w] = rows(torch.matmul(ds.transpose(1, 2).contiguous(), q))
    return {"dq": dq, "dkv": dkv}


def pairs(q_len, kv_len, causal):
    return sum(min(i + 1, kv_len) for i in range(q_len)) if causal else q_len * kv_len


def attn_work(c):
    b, lq, lk, w = c["batch"], c["q_len"], c["kv_len"], c["heads"] * c["head_dim"]
    n = b * pairs(lq, lk, c["causal"]) * w
    seen = min(lq, lk) if c["causal"] else lk  # keys that some query reads
    if c["kind"] == "attn":
        return {"bytes": 4 * b * w * (2 * lq + 2 * seen), "flops": 4 * n}
    return {"bytes": 4 * b * w * (3 * lq + 2 * seen + 2 * lk), "flops": 10 * n}


# --- a whole attention layer with its projections, both ways ------------------

def layer_prepare(c, r):
    lq, lk, e = c["q_len"], c["kv_len"], c["heads"] * c["head_dim"]
    s = {"x": r.normal(lq, e), "w": r.normal(4 * e * e, scale=e ** -0.5), "dy": r.normal(lq, e)}
    s["y"], s["dx"], s["dw"] = like(s["x"]), like(s["x"]), like(s["w"])
    if c["cross"]:
        s["kv"] = r.normal(lk, e)
        s["dkv"] = like(s["kv"])
    return s


def layer_run(c, s):
    lq, lk, h, e = c["q_len"], c["kv_len"], c["heads"], c["heads"] * c["head_dim"]
    p = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    x, n = ctx(), 4 * e * e
    if c["cross"]:
        x.cross_attention(p["x"], lq, p["kv"], lk, e, h, c["causal"], p["w"], n, p["y"])
    else:
        x.self_attention(p["x"], lq, e, h, c["causal"], p["w"], n, p["y"])
    if not c["train"]:
        return s["y"]
    x.fill(p["dw"], 0.0, n)  # gradients of the weights are added to
    if c["cross"]:
        x.cross_attention_bwd(p["x"], lq, p["kv"], lk, p["dy"], e, h, c["causal"], p["w"], n, p["dw"], p["dx"], p["dkv"])
        return {k: s[k] for k in ("y", "dx", "dkv", "dw")}
    x.self_attention_bwd(p["x"], p["dy"], lq, e, h, c["causal"], p["w"], n, p["dw"], p["dx"])
    return {k: s[k] for k in ("y", "dx", "dw")}


def attention64(q, k, v, h, causal):
    def split(t):
        return t.reshape(t.shape[0], h, -1).transpose(0, 1).contiguous()
    o, _ = attn_one64(split(q), split(k), split(v), causal)
    return o.transpose(0, 1).reshape(q.shape[0], -1)


def layer_exact(c, s):
    h, e = c["heads"], c["heads"] * c["head_dim"]
    x, w = s["x"].to(F64).requires_grad_(c["train"]), s["w"].to(F64).requires_grad_(c["train"])
    src = [x, w]
    wo = w[3 * e * e:].reshape(e, e)
    if c["cross"]:
        kv = s["kv"].to(F64).requires_grad_(c["train"])
        src.append(kv)
        q, k, v = (x @ w[:e * e].reshape(e, e), *(kv @ w[e * e:3 * e * e].reshape(e, 2 * e)).chunk(2, 1))
    else:
        q, k, v = (x @ w[:3 * e * e].reshape(e, 3 * e)).chunk(3, 1)
    y = attention64(q, k, v, h, c["causal"]) @ wo
    if not c["train"]:
        return y
    g = torch.autograd.grad(y, src, s["dy"].to(F64))
    out = {"y": y.detach(), "dx": g[0], "dw": g[1]}
    if c["cross"]:
        out["dkv"] = g[2]
    return out


def layer_work(c):
    lq, lk, e = c["q_len"], c["kv_len"], c["heads"] * c["head_dim"]
    rows = 4 * lq if not c["cross"] else 2 * lq + 2 * lk  # rows times e^2 of the projections
    n, way = pairs(lq, lk, c["causal"]) * e, 1 + 2 * c["train"]
    moved = 2 * lq + (lk if c["cross"] else 0)  # rows in and out
    if c["train"]:
        moved += 2 * lq + (lk if c["cross"] else 0)
    return {"bytes": 4 * (moved * e + way * 4 * e * e),
            "flops": way * 2 * rows * e * e + (14 if c["train"] else 4) * n}


# --- a small stack through the runtime: one whole call ------------------------

class Stack:
    """A graph of pre-norm half blocks (LayerNorm -> SelfAttention -> Add ->
    LayerNorm -> GELU) with its weights on the device, its store, and the host
    inputs of one call."""

    def __init__(self, c, seed):
        r = np.random.default_rng(seed)
        e, seq, n = c["heads"] * c["head_dim"], c["seq"], c["blocks"]
        self.layers, cur = [], "inp"
        for b in range(n):
            g = np.concatenate([1 + 0.05 * r.standard_normal(e), 0.05 * r.standard_normal(e)]).astype(np.float32)
            w = (r.standard_normal(4 * e * e) / np.sqrt(e)).astype(np.float32)
            out = "x" if b == n - 1 else f"h{b}"
            self.layers += [
                dict(name=f"ln{b}", type="LayerNorm", inputs=[cur], output=f"n{b}", in_features=e, weights=g),
                dict(name=f"attn{b}", type="SelfAttention", inputs=[f"n{b}"], output=f"a{b}", seq_len=seq, embed_dim=e,
                     num_heads=c["heads"], causal=True, weights=w),
                dict(name=f"res{b}", type="Add", inputs=[f"a{b}", cur], output=f"r{b}"),
                dict(name=f"ln2_{b}", type="LayerNorm", inputs=[f"r{b}"], output=f"m{b}", in_features=e, weights=g),
                dict(name=f"act{b}", type="GELU", inputs=[f"m{b}"], output=out)]
            cur = out
        self.inp = r.standard_normal(seq * e).astype(np.float32)
        self.graph, self.store, self.captured = M.DeviceGraph(ctx(), self.layers), M.Store(ctx()), None
        self.store.set_fusion(True)
        if c["captured"]:
            self.captured = self.store.capture(self.graph, {"inp": self.inp}, {})

    def run(self):
        if self.captured is None:
            return self.store.forward_named(self.graph, {"inp": self.inp}, {})
        self.captured.set_input("inp", self.inp)
        self.captured.launch()
        return self.captured.get("x")

    def __del__(self):
        for part in (self.captured, self.store, self.graph):
            if part is not None:
                part.close()


def stack_prepare(c, seed):
    return {"stack": Stack(c, seed)}


def stack_run(c, s):
    return s["stack"].run()


def stack_exact(c, s):
    e, h = c["heads"] * c["head_dim"], c["heads"]

    def norm(x, w):
        return norm64(x, 1e-5) * w[:e] + w[e:]
    x = torch.from_numpy(s["stack"].inp).to(DEV).to(F64).reshape(c["seq"], e)
    for b in range(c["blocks"]):
        g, w = (torch.from_numpy(s["stack"].layers[5 * b + i]["weights"]).to(DEV).to(F64) for i in (0, 1))
        q, k, v = (norm(x, g) @ w[:3 * e * e].reshape(e, 3 * e)).chunk(3, 1)
        x = x + attention64(q, k, v, h, True) @ w[3 * e * e:].reshape(e, e)
        x = gelu64(norm(x, g))
    return x.reshape(-1).cpu().numpy()


def stack_work(c):
    e, n, seq = c["heads"] * c["head_dim"], c["blocks"], c["seq"]
    return {"bytes": 4 * (2 * seq * e + n * (4 * e * e + 2 * e)),
            "flops": n * (8 * seq * e * e + 4 * pairs(seq, seq, True) * e + 40 * seq * e)}


# --- the cases ----------------------------------------------------------------

def listed():
    return [
        # A small model served one call at a time from host data: launches and latency.
        {"name": "stack_small", "kind": "stack", "blocks": 4, "seq": 128, "heads": 4, "head_dim": 64, "captured": False},
        # The library's headline workload: residual add + RMSNorm over 4096 tokens.
        {"name": "add_rmsnorm", "kind": "add_rmsnorm", "rows": 4096, "cols": 4096},
        # Softmax of a causal score tensor, 8 x 32 heads x 1024 x 1024: the most bytes.
        {"name": "softmax_causal", "kind": "softmax", "rows": 262144, "q": 1024, "cols": 1024},
        # The input side of a decoder: token rows, then RoPE on q and k, 16 x 2048 tokens.
        {"name": "embed_rope", "kind": "embed_rope", "batch": 16, "seq": 2048, "vocab": 32000, "heads": 32, "k_heads": 32,
         "head_dim": 128, "zipf": False},
        # The elementwise part of a decoder MLP over 8192 tokens.
        {"name": "mlp_chain", "kind": "mlp", "rows": 8192, "hidden": 4096, "inner": 11008},
        # Rows of an odd width (1001 classes): LayerNorm both ways and log-softmax.
        {"name": "rows_odd", "kind": "rows", "rows": 8191, "cols": 1001},
        # The backward of an elementwise residual block in a training step.
        {"name": "block_bwd", "kind": "block_bwd", "rows": 8192, "cols": 4096},
        # The embedding's gradient for token ids as frequent as in text.
        {"name": "embed_bwd", "kind": "embed_bwd", "tokens": 32768, "vocab": 32000, "dim": 4096, "zipf": True},
        # The attention core over whole prompts, causal, from a fused QKV buffer.
        {"name": "attn_prefill", "kind": "attn", "batch": 8, "q_len": 1024, "kv_len": 1024, "heads": 32, "head_dim": 128,
         "causal": True},
        # One new query for each of 16 sequences over their cached keys and values.
        {"name": "attn_decode", "kind": "attn", "batch": 16, "q_len": 1, "kv_len": 4000, "heads": 32, "head_dim": 128,
         "causal": False},
        # The core's gradient in training, at the prefill's shape.
        {"name": "attn_bwd", "kind": "attn_bwd", "batch": 8, "q_len": 1024, "kv_len": 1024, "heads": 32, "head_dim": 128,
         "causal": True},
        # A whole self-attention layer with its projections, forward and backward.
        {"name": "attn_layer", "kind": "layer", "q_len": 2048, "kv_len": 2048, "heads": 16, "head_dim": 64, "causal": True,
         "cross": False, "train": True},
    ]


def span(rng, lo, hi):
    """A size between lo and hi, even over the logarithm; odd ones among them."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and n >= 64:
        n = n // 64 * 64
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["stack", "add_rmsnorm", "softmax", "embed_rope", "mlp", "rows", "block_bwd", "embed_bwd", "attn", "attn",
                       "attn_bwd", "layer"])
    c = {"kind": kind}
    if kind == "stack":
        c.update(blocks=rng.randint(1, 6), seq=span(rng, 16, 256), heads=rng.choice([2, 4, 8]), head_dim=rng.choice([32, 64]),
                 captured=rng.random() < 0.5)
    elif kind == "add_rmsnorm":
        cols = span(rng, 256, 8192)
        c.update(rows=span(rng, 64, (1 << 26) // cols), cols=cols)
    elif kind == "softmax":
        q = rng.choice([128, 200, 512, 1000, 2048])
        cols = q if rng.random() < 0.5 else span(rng, 64, 8192)
        c.update(rows=q * rng.randint(1, max(1, (1 << 27) // (q * cols))), q=q, cols=cols)
    elif kind == "embed_rope":
        heads, head_dim = rng.choice([4, 8, 16, 32]), rng.choice([64, 80, 128])
        c.update(batch=rng.randint(1, 8), seq=span(rng, 16, 2048), vocab=span(rng, 1000, 32000), heads=heads,
                 k_heads=max(1, heads // rng.choice([1, 4])), head_dim=head_dim, zipf=rng.random() < 0.5)
    elif kind == "mlp":
        hidden = span(rng, 256, 4096)
        c.update(rows=span(rng, 32, 8192), hidden=hidden, inner=hidden * rng.choice([2, 3, 4]) - rng.choice([0, 0, 2]))
    elif kind == "rows":
        cols = span(rng, 100, 20000)
        c.update(rows=span(rng, 32, (1 << 25) // cols), cols=cols)
    elif kind == "block_bwd":
        cols = span(rng, 256, 8192)
        c.update(rows=span(rng, 64, (1 << 25) // cols), cols=cols)
    elif kind == "embed_bwd":
        c.update(tokens=span(rng, 64, 32768), vocab=span(rng, 1000, 32000), dim=rng.choice([256, 500, 768, 1024, 2048, 4096]),
                 zipf=rng.random() < 0.7)
    elif kind in ("attn", "attn_bwd"):
        heads, d = rng.choice([4, 8, 12, 16, 32]), rng.choice([32, 64, 64, 80, 96, 128, 128])
        how = rng.choice(["self", "self", "cross"] + (["decode", "decode"] if kind == "attn" else []))
        lq = 1 if how == "decode" else span(rng, 32, 2048)
        lk = lq if how == "self" else span(rng, 64, 8192 if how == "decode" else 2048)
        most = (1 << 21) // (lk * heads) if how == "decode" else (1 << 27) // (lq * lk * heads)
        c.update(batch=rng.randint(1, max(1, min(32, most))), q_len=lq, kv_len=lk, heads=heads, head_dim=d,
                 causal=how == "self" and rng.random() < 0.8)
    else:
        cross = rng.random() < 0.3
        lq = span(rng, 64, 2048)
        c.update(q_len=lq, kv_len=span(rng, 64, 2048) if cross else lq, heads=rng.choice([4, 8, 16]),
                 head_dim=rng.choice([32, 64, 80, 128]), causal=not cross, cross=cross, train=rng.random() < 0.6)
    return c


def _of(c, what):
    kind = "attn" if c["kind"] == "attn_bwd" else c["kind"]
    return globals()[f"{kind}_{what}"]


def prepare(case, seed):
    source = seed if case["kind"] == "stack" else Rand(seed)
    return done(dict(_of(case, "prepare")(case, source), case=case))


def run(state):
    return _of(state["case"], "run")(state["case"], state)


def exact(case, seed):
    return _of(case, "exact")(case, prepare(case, seed))


def work(case):
    return _of(case, "work")(case)


# About four times the error against `exact` over the ranges, which is what
# another order of 32-bit sums differs by.
TOLERANCE = {"add_rmsnorm": 5e-7, "softmax": 1e-6, "embed_rope": 5e-7, "mlp": 1e-6, "rows": 2e-6, "block_bwd": 2e-6,
             "embed_bwd": 1e-6, "attn": 5e-6, "attn_bwd": 5e-6, "layer": 1e-5, "stack": 5e-6}


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}
