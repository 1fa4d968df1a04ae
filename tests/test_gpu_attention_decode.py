"""The attention core for a few queries against many keys (a decoding step):
the vector kernel and its splits over workgroups against float64, at the edges
of its groups of keys, its vector widths and its split sizes."""
import numpy as np
import pytest

import oracle as O
from _attention import assert_attention_close, attention64
from test_gpu_attention import gpu_attention, rand_qkv
from test_gpu_attention_bwd import _tuned_context

pytestmark = pytest.mark.gpu


# 64 keys per step of a workgroup (16 lanes per key; 128 for heads up to 32),
# one split per 256 keys where few heads share the GPU; 1, 2 and 4 queries per
# workgroup; heads of 1 to 4 vectors per lane, odd ones in scalar loads.
@pytest.mark.parametrize("b,lq,lk,heads,hd", [
    (1, 1, 1, 1, 4), (2, 1, 15, 3, 32), (1, 1, 64, 2, 64), (3, 1, 65, 2, 64), (1, 1, 256, 2, 128), (1, 1, 257, 1, 128),
    (2, 2, 1000, 3, 80), (1, 3, 513, 2, 96), (1, 4, 127, 2, 32), (1, 5, 300, 1, 100), (2, 8, 2049, 2, 64),
    (1, 1, 5000, 1, 7), (1, 2, 130, 3, 33), (40, 1, 70, 16, 36), (1, 6, 64, 2, 125)])
def test_decode(ctx, b, lq, lk, heads, hd):
    q, k, v = rand_qkv(lq + lk + hd, b, lq, lk, heads * hd)
    got = gpu_attention(ctx, q, k, v, heads, False)
    for i in range(b):
        out, mag, cond = attention64(q[i], k[i], v[i], heads, False, O.attention_scale(hd))
        assert_attention_close(got[i], out, mag, cond, f"decode {b} {lq} {lk} {heads} {hd} [{i}]")


@pytest.mark.parametrize("splits", [1, 5, 64])
def test_decode_splits(splits):
    """Keys over a set number of workgroups, among them fewer keys than 64 each."""
    c = _tuned_context(f"decode={splits}")
    try:
        for lq, lk, hd in ((1, 1000, 64), (3, 130, 100), (8, 61, 33)):
            q, k, v = rand_qkv(lk, 2, lq, lk, 2 * hd)
            got = gpu_attention(c, q, k, v, 2, False)
            for i in range(2):
                out, mag, cond = attention64(q[i], k[i], v[i], 2, False, O.attention_scale(hd))
                assert_attention_close(got[i], out, mag, cond, f"decode splits {splits} {lq} {lk} {hd} [{i}]")
    finally:
        c.close()


@pytest.mark.parametrize("lk", [40, 700])
def test_decode_special_values(ctx, lk):
    """A key of -inf scores weighs nothing, an infinite value row reaches only
    its own dimension, NaN only the queries and dimensions that see it: as
    the float64 softmax has it."""
    q, k, v = rand_qkv(5, 1, 2, lk, 64)
    q[0, :, 3] = np.abs(q[0, :, 3]) + 0.5
    k[0, 7, 3] = -np.inf
    v[0, lk - 1, 5] = np.inf
    v[0, 2, 9] = np.nan
    got = gpu_attention(ctx, q, k, v, 1, False)[0]
    s = (q[0].astype(np.float64) @ k[0].astype(np.float64).T) * O.attention_scale(64)
    p = np.exp(s - s.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    keep = [d for d in range(64) if d not in (5, 9)]
    v64 = v[0].astype(np.float64)
    np.testing.assert_allclose(got[:, keep], p @ v64[:, keep], rtol=0, atol=1e-5)
    assert np.isposinf(got[:, 5]).all() and np.isnan(got[:, 9]).all()


# 2^32 work-items bound a grid: 9 million sequences have fewer with four waves
# per workgroup than with eight, or with a workgroup per few queries.  With one
# key the output is its value, up to the 1e-9 beside the sum.
@pytest.mark.parametrize("lq", [5, 9])
def test_more_sequences_than_the_wider_grids_hold(ctx, lq):
    n = 9_000_000
    q = np.ones((n * lq, 1), np.float32)
    kv = np.random.default_rng(3).standard_normal((n, 2)).astype(np.float32)
    print(f"attention of {n} sequences, {lq} queries, one key", flush=True)
    dq, dkv, out = ctx.to_device(q), ctx.to_device(kv), ctx.empty(q.shape)
    try:
        ctx.attention(dq, dkv, dkv.ptr + 4, out, n, lq, 1, 1, 1, ld_kv=2)
        got = out.numpy()
    finally:
        for d in (dq, dkv, out):
            d.free()
    np.testing.assert_allclose(got.reshape(n, lq), np.repeat(kv[:, 1:], lq, 1), rtol=2e-7, atol=0)
