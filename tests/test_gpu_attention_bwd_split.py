"""The attention backward on split bf16 operands: the edges of its key blocks
(128), query blocks (256), tiles (32) and splits, and values without a split,
against float64."""
import numpy as np
import pytest

import oracle as O
from _attention import assert_bwd_close, attention_bwd64, layer_case, self_attention_bwd64
from test_gpu_attention_bwd import _dev, _tuned_context, check_core, gpu_core_bwd, rand_core

pytestmark = pytest.mark.gpu

# One tile and less, one key block and one key more, more than one query block,
# few heads with long rows (both sides split) and heads that fill the GPU.
SHAPES = [(1, 1, 33, 1, 4), (1, 32, 32, 2, 32), (2, 31, 129, 1, 36), (1, 257, 128, 2, 64), (1, 129, 257, 1, 72),
          (1, 288, 288, 1, 96), (1, 1025, 200, 1, 32), (1, 200, 1030, 1, 128), (70, 33, 140, 8, 16), (1, 65, 65, 3, 7)]


@pytest.mark.parametrize("b,lq,lk,heads,hd", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
def test_split_backward(ctx, b, lq, lk, heads, hd, causal):
    q, k, v, dout = rand_core(lq + lk + hd, b, lq, lk, heads * hd)
    got = gpu_core_bwd(ctx, q, k, v, dout, heads, causal)
    for i in range(0, b, max(1, b // 2)):
        check_core([g[i:i + 1] for g in got], q[i:i + 1], k[i:i + 1], v[i:i + 1], dout[i:i + 1], heads, causal,
                   f"split backward {b} {lq} {lk} {heads} {hd} {causal} [{i}]", oracle=False)


def test_split_backward_groups():
    """(sequence, head) pairs in groups with a smaller last one."""
    c = _tuned_context("attnbwd_heads=3")
    try:
        q, k, v, dout = rand_core(8, 2, 300, 300, 4 * 32)
        check_core(gpu_core_bwd(c, q, k, v, dout, 4, True), q, k, v, dout, 4, True, "groups of 3", oracle=False)
    finally:
        c.close()


# 1000 x 1000: keys and queries dealt to several workgroups.
@pytest.mark.parametrize("n", [200, 1000])
def test_split_backward_special_values(ctx, n):
    """A NaN key reaches the gradients of the queries that see it and no
    other; a query value that rounds to infinity in bf16 multiplies zeros."""
    hd = 32
    q, k, v, dout = rand_core(4, 1, n, n, hd)
    k[0, :, 3] = 0.0
    q[0, 7, 3] = 3.4e38
    (dq, dk, dv), tol = attention_bwd64(q[0], k[0], v[0], dout[0], 1, True, O.attention_scale(hd))
    got = gpu_core_bwd(ctx, q, k, v, dout, 1, True)
    keep = [d for d in range(hd) if d != 3]
    for name, g, want, t, cols in (("dq", got[0][0], dq, tol[0], list(range(hd))), ("dk", got[1][0], dk, tol[1], keep),
                                   ("dv", got[2][0], dv, tol[2], list(range(hd)))):
        assert np.isfinite(g[:, cols]).all(), name
        t = np.where(np.isfinite(t[:, cols]), np.minimum(t[:, cols], 1e-3), 1e-3)
        np.testing.assert_array_less(np.abs(g[:, cols] - want[:, cols]), t + 1e-5, err_msg=name)
    q, k, v, dout = rand_core(5, 1, n, n, hd)
    (dq, _, _), tol = attention_bwd64(q[0], k[0], v[0], dout[0], 1, True, O.attention_scale(hd))
    k[0, n - 1, 5] = np.nan
    got = gpu_core_bwd(ctx, q, k, v, dout, 1, True)[0][0]
    assert np.isnan(got[n - 1]).all()
    assert_bwd_close(got[:n - 1], dq[:n - 1], tol[0][:n - 1], "queries that do not see the NaN key")


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("lk", [1, 40])
def test_split_backward_one_visible_key(ctx, bad, lk):
    """A query that sees a single key has dS = p (dP - dP): 0, but NaN where its
    dP is not finite, as the formula has it.  lk == 1: every query; lk == 40,
    causal: the first one."""
    n, hd, at = 40, 32, 0
    causal = lk > 1
    q, k, v, dout = rand_core(11, 1, n, lk, hd)
    if lk == 1:
        at = 17
    clean = dout.copy()
    clean[0, at] = 0.0
    (dq, dk, dv), tol = attention_bwd64(q[0], k[0], v[0], clean[0], 1, causal, O.attention_scale(hd))
    dout[0, at, 3] = bad
    got = [g[0] for g in gpu_core_bwd(ctx, q, k, v, dout, 1, causal)]
    assert np.isnan(got[0][at]).all() and np.isnan(got[1][0]).all(), "dq of the query, dk of its key"
    assert not np.isfinite(got[2][0, 3]), "dv of its key"
    rest = np.arange(n) != at
    if causal:  # no other gradient sees that query
        assert_bwd_close(got[0][rest], dq[rest], tol[0][rest], "dq")
        assert_bwd_close(got[1][1:], dk[1:], tol[1][1:], "dk")
        assert_bwd_close(got[2][1:], dv[1:], tol[2][1:], "dv")
    else:
        assert (got[0][rest] == 0.0).all()
    v[0, 0, 5] = bad  # the only visible value row of that query
    got = gpu_core_bwd(ctx, q, k, v, clean if causal else dout, 1, causal)[0][0]
    assert np.isnan(got[at]).all()


@pytest.mark.parametrize("n,hd,causal", [(200, 32, False), (512, 64, True), (333, 80, False), (1100, 128, True)])
def test_split_backward_saturated_rows(ctx, n, hd, causal):
    """Rows where one key has all but 1e-8 of the weight (scores of about +-40): dP
    of that key and delta cancel, so both must have the same rounding.  There l
    = 1 and delta = dP (1 + u) + at most 1e-8 of another dP, so dS, whose exact
    value is below 2e-8 max |dP|, is within 2 u max |dP| of it, and dq within that
    times scale max |k|."""
    q, k, v, dout = rand_core(n + hd, 1, n, n, hd)
    amp = np.float32(np.sqrt(40.0 / np.sqrt(hd)) * hd ** 0.25)
    q *= amp
    k *= amp
    scale = float(np.float32(O.attention_scale(hd)))
    q64, k64, v64, do64 = (a[0].astype(np.float64) for a in (q, k, v, dout))
    (dq, _, dv), _ = attention_bwd64(q64, k64, v64, do64, 1, causal, scale)
    s = scale * (q64 @ k64.T)
    if causal:
        s[np.triu(np.ones(s.shape, bool), 1)] = -np.inf
    p = np.exp(s - s.max(1, keepdims=True))
    rows = np.flatnonzero(p.sum(1) - 1 < 1e-8)
    assert rows.size > n // 10
    got = gpu_core_bwd(ctx, q, k, v, dout, 1, causal)
    g = np.abs(do64 @ v64.T).max(1)
    tol = 2 * O.U32 * scale * np.outer(g, np.abs(k64).max(0))
    err = np.abs(got[0][0] - dq)
    print(f"saturated n={n} hd={hd}: worst error {(err / tol)[rows].max():.3g} of the bound, {err[rows].max():.3g}", flush=True)
    assert (err <= tol)[rows].all()


@pytest.mark.parametrize("scale", [0.125, -0.125])
@pytest.mark.parametrize("causal", [False, True])
def test_split_backward_large_scores(ctx, causal, scale):
    """Integer q and k, so q . k is exact, with scores of about 256 that differ by a
    few units: the weights' error is that of exp at the difference (up to 16 in
    base-2 units where a weight matters: 16 x 2 u x ln 2, and 4 u for exp, the sum
    and its reciprocal), not of the scores."""
    r = np.random.default_rng(2)
    n, hd = 200, 64
    q, k = (r.integers(-2, 3, (1, n, hd)).astype(np.float32) for _ in range(2))
    q[..., 0], k[..., 0] = 64.0, np.copysign(32.0, scale)
    v, dout = (r.standard_normal((1, n, hd)).astype(np.float32) for _ in range(2))
    got = gpu_core_bwd(ctx, q, k, v, dout, 1, causal, scale=scale)
    want, _ = attention_bwd64(q[0], k[0], v[0], dout[0], 1, causal, scale)
    s = scale * (q[0].astype(np.float64) @ k[0].astype(np.float64).T)
    if causal:
        s[np.triu(np.ones(s.shape, bool), 1)] = -np.inf
    p = np.exp(s - s.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    rel = (32 * np.log(2) + 4) * O.U32
    tol = (rel + 1e-6) * (p.T @ np.abs(dout[0])) + 1e-9  # 1e-6: the sum over 200 queries, sqrt(n) u and its splits
    err = np.abs(got[2][0] - want[2])
    print(f"large scores: dv {(err / tol).max():.3g} of the bound", flush=True)
    assert (err <= tol).all()
    for g, w, name in zip(got[:2], want[:2], ("dq", "dk")):
        e = np.linalg.norm(g[0] - w) / np.linalg.norm(w)
        print(f"  {name} {e:.3g}", flush=True)
        assert e <= 2 * rel, name


def layer_bwd(ctx, x, w, dy, heads, causal):
    seq, e = x.shape
    bufs = [_dev(ctx, a) for a in (x, dy, w, np.zeros(w.size, np.float32), np.zeros_like(x))]
    xb, dyb, wb, gwb, gxb = bufs
    try:
        ctx.self_attention_bwd(xb, dyb, seq, e, heads, causal, wb, w.size, gwb, gxb)
        return gxb.numpy().reshape(seq, e), gwb.numpy()
    finally:
        for b in bufs:
            b.free()


# Heads up to 64 take the output from the statistics' kernel, unsplit and with the
# keys dealt to several workgroups (256 tokens and more); wider ones from the
# forward.  Head sizes that are and are not 16-byte multiples.
@pytest.mark.parametrize("seq,e,heads", [(33, 64, 1), (130, 96, 3), (300, 128, 2), (700, 96, 3), (290, 60, 3), (300, 42, 2),
                                         (270, 192, 2)])
@pytest.mark.parametrize("causal", [False, True])
def test_layer_output_beside_the_statistics(ctx, seq, e, heads, causal):
    x, w = layer_case(seq, e, seq + e, amp=1.5)
    dy = np.random.default_rng(e).standard_normal((seq, e)).astype(np.float32)
    wqkv, wout = w[:3 * e * e].reshape(e, 3 * e), w[3 * e * e:].reshape(e, e)
    (dx, dwqkv, dwout), (tx, twqkv, twout) = self_attention_bwd64(x, wqkv, wout, dy, heads, causal)
    gx, gw = layer_bwd(ctx, x, w, dy, heads, causal)
    assert_bwd_close(gx, dx, tx, "dx")
    assert_bwd_close(gw[:3 * e * e], dwqkv, twqkv, "dWqkv")
    assert_bwd_close(gw[3 * e * e:], dwout, twout, "dWout")


@pytest.mark.parametrize("seq", [100, 300])
def test_layer_output_without_a_split(ctx, seq):
    """A value that rounds to infinity in bf16 reaches its dimension of the output,
    which dWout = att^T dy shows."""
    e, hd = 64, 32
    x, w = layer_case(seq, e, 3)
    wqkv, wout = w[:3 * e * e].reshape(e, 3 * e), w[3 * e * e:].reshape(e, e)
    x[:, 7] = 0.0
    x[5, 7] = 3.4e38
    wqkv[7] = 0.0
    wqkv[7, 2 * e + 3] = 1.0  # v[5, 3] = 3.4e38
    wout[3] = 0.0             # and no gradient through it
    dy = (1e-3 * np.random.default_rng(1).standard_normal((seq, e))).astype(np.float32)
    qkv = x.astype(np.float64) @ wqkv.astype(np.float64)
    att = np.zeros((seq, e))
    for h in range(2):
        q, k, v = (qkv[:, i * e + h * hd:i * e + (h + 1) * hd] for i in range(3))
        s = q @ k.T * O.attention_scale(hd)
        p = np.exp(s - s.max(1, keepdims=True))
        att[:, h * hd:(h + 1) * hd] = p / p.sum(1, keepdims=True) @ v
    want = att.T @ dy.astype(np.float64)
    mag = np.abs(att).T @ np.abs(dy).astype(np.float64)
    got = layer_bwd(ctx, x, w, dy, 2, False)[1][3 * e * e:].reshape(e, e)
    assert (np.abs(got - want) <= 2e-5 * mag + 1e-9).all()
