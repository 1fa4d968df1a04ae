"""The matrix-core attention core with fp32 operands split into bf16 terms:
both workgroup sizes at the edges of their query blocks and key tiles, every
padded head size, and values that have no split (infinities, NaN, the largest
floats), against float64."""
import ctypes
import time

import numpy as np
import pytest

import mimir_hip as M
import oracle as O
from _attention import assert_attention_close, attention64
from test_gpu_attention import gpu_attention, rand_qkv
from test_gpu_attention_bwd import _tuned_context

pytestmark = pytest.mark.gpu

# 128-query workgroups up to 256 of them, 256-query ones above (and for up to
# 64 queries); 32-key tiles; heads padded to 32, 64, 96 and 128.
SHAPES = [(1, 65, 31, 2, 32), (1, 128, 32, 1, 64), (2, 129, 33, 2, 36), (1, 257, 257, 2, 96), (1, 300, 64, 1, 100),
          (1, 97, 160, 2, 70), (1, 70, 70, 3, 5), (40, 130, 70, 8, 32), (33, 257, 66, 8, 16), (1, 9, 95, 2, 128),
          (1, 64, 65, 1, 128)]


@pytest.mark.parametrize("b,lq,lk,heads,hd", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
def test_split_core(ctx, b, lq, lk, heads, hd, causal):
    q, k, v = rand_qkv(lq + lk + hd, b, lq, lk, heads * hd)
    got = gpu_attention(ctx, q, k, v, heads, causal)
    for i in range(0, b, max(1, b // 3)):
        out, mag, cond = attention64(q[i], k[i], v[i], heads, causal, O.attention_scale(hd))
        assert_attention_close(got[i], out, mag, cond, f"split core {b} {lq} {lk} {heads} {hd} {causal} [{i}]")


@pytest.mark.parametrize("lq,lk", [(70, 100), (300, 300)])
@pytest.mark.parametrize("causal", [False, True])
def test_split_core_special_values(ctx, lq, lk, causal):
    """What fp32 arithmetic gives: -inf scores weigh nothing, an infinite
    value reaches its dimension of the queries that see it, a NaN key every
    query that sees it, and masked keys nothing at all."""
    check_special_values(ctx, lq, lk, causal, 7, 40, 41, 60)


def check_special_values(ctx, lq, lk, causal, low, inf_row, big_row, nan_key):
    q, k, v = rand_qkv(3, 1, lq, lk, 64)
    q[0, :, 3] = np.abs(q[0, :, 3]) + 0.5
    k[0, low, 3] = -np.inf
    v[0, inf_row, 5] = np.inf
    v[0, big_row, 6] = 3.4e38  # rounds to infinity in bf16
    k[0, nan_key, 8] = np.nan
    got = gpu_attention(ctx, q, k, v, 1, causal)[0]
    s = (q[0].astype(np.float64) @ k[0].astype(np.float64).T) * O.attention_scale(64)
    hide = np.triu(np.ones(s.shape, bool), 1) if causal else np.zeros(s.shape, bool)
    s[hide] = -np.inf
    p = np.exp(s - np.nanmax(s, 1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    seen = ~hide
    bad = seen[:, nan_key]
    assert np.isnan(got[bad]).all(), "a NaN key"
    fine = ~bad
    v64 = np.where(np.isfinite(v[0]), v[0], 0.0).astype(np.float64)
    keep = [d for d in range(64) if d not in (5, 6)]
    want = np.where(np.isnan(p), 0.0, p) @ v64
    np.testing.assert_allclose(got[fine][:, keep], want[fine][:, keep], rtol=0, atol=1e-5)
    inf = fine & seen[:, inf_row]
    assert np.isposinf(got[inf, 5]).all(), "an infinite value"
    big = fine & seen[:, big_row]
    np.testing.assert_allclose(got[big, 6], want[big, 6], rtol=1e-4)
    clean = fine & ~seen[:, inf_row]
    np.testing.assert_allclose(got[clean][:, 5:7], want[clean][:, 5:7], rtol=0, atol=1e-5)


# The keys dealt to several workgroups (one head, 737 keys and more): values in the
# first, a middle and the last share; lq well below lk leaves causal shares without
# a tile.
@pytest.mark.parametrize("lq,lk", [(1000, 1000), (40, 1500), (300, 1100)])
@pytest.mark.parametrize("rows", [(7, 20, 21, 30), (7, 250, 280, 299), (990, 400, 401, 999)])
@pytest.mark.parametrize("causal", [False, True])
def test_split_core_special_values_over_key_splits(ctx, lq, lk, causal, rows):
    check_special_values(ctx, lq, lk, causal, *rows)


# Keys over several workgroups: what splits_for chooses (737 keys and more, few
# workgroups), and counts and workgroup sizes set by MIMIR_TUNE, among them more
# splits than a causal block has tiles.
@pytest.mark.parametrize("tune", ["", "attnsplits=3", "attnsplits=7,attnwaves=4", "attnsplits=40,attnwaves=8"])
@pytest.mark.parametrize("b,lq,lk,heads,hd", [(1, 1000, 1000, 1, 128), (1, 40, 1500, 2, 80), (2, 130, 900, 1, 5),
                                               (1, 300, 737, 3, 64)])
@pytest.mark.parametrize("causal", [False, True])
def test_split_core_over_key_splits(tune, b, lq, lk, heads, hd, causal):
    q, k, v = rand_qkv(lq + lk + hd, b, lq, lk, heads * hd)
    c = _tuned_context(tune)
    try:
        got = gpu_attention(c, q, k, v, heads, causal)
    finally:
        c.close()
    for i in range(b):
        out, mag, cond = attention64(q[i], k[i], v[i], heads, causal, O.attention_scale(hd))
        assert_attention_close(got[i], out, mag, cond, f"key splits {tune} {b} {lq} {lk} {heads} {hd} {causal} [{i}]")


@pytest.mark.parametrize("waves", [4, 8])
def test_split_core_workgroup_sizes(waves):
    c = _tuned_context(f"attnwaves={waves}")
    try:
        for lq, lk, hd, causal in ((40, 70, 32, False), (260, 260, 96, True), (513, 100, 64, True)):
            q, k, v = rand_qkv(lq + hd, 1, lq, lk, 2 * hd)
            out, mag, cond = attention64(q[0], k[0], v[0], 2, causal, O.attention_scale(hd))
            assert_attention_close(gpu_attention(c, q, k, v, 2, causal)[0], out, mag, cond, f"{waves} waves {lq} {lk} {hd}")
    finally:
        c.close()


def call_us(ctx, run, reps):
    """Microseconds per call, the smallest of three runs."""
    run()
    ctx.sync()
    best = float("inf")
    for _ in range(3):
        t = time.perf_counter()
        for _ in range(reps):
            run()
        ctx.sync()
        best = min(best, (time.perf_counter() - t) / reps * 1e6)
    return best


def test_a_nan_costs_no_more_than_a_few_calls(ctx):
    """One NaN key that every query sees makes every block of the output, and of
    the gradients, be computed again. Measured: 4.4 and 9.2 times a call without
    one; row by row the forward took 23 times, more where sequences are longer."""
    n, heads, hd = 1024, 16, 64
    w = heads * hd
    q, k, v = rand_qkv(9, 1, n, n, w)
    bufs = [ctx.to_device(a) for a in (q, k, v, v)] + [ctx.empty(q.shape) for _ in range(4)]
    dq, dk, dv, do, out, gq, gk, gv = bufs
    runs = (("forward", lambda: ctx.attention(dq, dk, dv, out, 1, n, n, heads, hd, causal=True)),
            ("backward", lambda: ctx.attention_bwd(dq, dk, dv, do, gq, gk, gv, 1, n, n, heads, hd, True)))
    try:
        clean = {name: call_us(ctx, run, 20) for name, run in runs}
        k[0, 0, ::hd] = np.nan
        ctx.upload(dk, k)
        for name, run in runs:
            us = call_us(ctx, run, 3)
            print(f"{name}: {clean[name]:.0f} us, with a NaN key {us:.0f} us", flush=True)
            assert us < 20 * clean[name], name
        assert np.isnan(out.numpy()).all()
    finally:
        for b in bufs:
            b.free()


def _hip():
    for name in ("libamdhip64.so", "/opt/rocm/lib/libamdhip64.so"):
        try:
            return ctypes.CDLL(name)
        except OSError:
            continue
    pytest.skip("libamdhip64 not loadable")


def test_a_context_takes_no_workspace_before_it_needs_it():
    hip = _hip()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    with M.Context(0):  # what the process and the GPU keep exists now
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        before = free.value
        with M.Context(0):
            assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            assert before - free.value < 16 << 20


@pytest.mark.parametrize("lq", [1, 300])
def test_first_split_call_under_capture(lq):
    """The first call that deals its keys to several workgroups, made while the
    stream is captured: replayed three times, the eager call's bits each time."""
    hip = _hip()
    lk, heads, hd = 1500, 2, 64
    q, k, v = rand_qkv(3, 1, lq, lk, heads * hd)
    graph, execution = ctypes.c_void_p(), ctypes.c_void_p()
    with M.Context(0) as c:
        bufs = [c.to_device(a) for a in (q, k, v)] + [c.empty(q.shape), c.empty(q.shape)]
        dq, dk, dv, out, eager = bufs
        c.sync()
        stream = ctypes.c_void_p(c.lib.mimir_ctx_stream(c.handle))
        try:
            assert hip.hipStreamBeginCapture(stream, 0) == 0  # the strictest mode
            c.attention(dq, dk, dv, out, 1, lq, lk, heads, hd)
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
            assert hip.hipGraphInstantiate(ctypes.byref(execution), graph, None, None, ctypes.c_size_t(0)) == 0
            c.attention(dq, dk, dv, eager, 1, lq, lk, heads, hd)
            want = eager.numpy()
            for _ in range(3):
                c.fill(out.ptr, np.nan, out.size)
                assert hip.hipGraphLaunch(execution, stream) == 0
                np.testing.assert_array_equal(out.numpy(), want)
                c.attention(dq, dk, dv, eager, 1, lq, lk, heads, hd)
        finally:
            if execution:
                hip.hipGraphExecDestroy(execution)
            if graph:
                hip.hipGraphDestroy(graph)
            for b in bufs:
                b.free()
    assert_attention_close(want.reshape(lq, -1), *attention64(q[0], k[0], v[0], heads, False, O.attention_scale(hd)), "captured")
