"""The attention layers' matrix products (gemm_split.hip) through the layers, which
use every layout (input x weights, gradients x transposed weights, transposed
inputs x gradients, added onto what is there): each kernel at odd and at
vector-aligned sizes, the edges of its tiles and of its steps of 32, and
operands that have no bf16 split, against float64."""
import numpy as np
import pytest

from _attention import assert_bwd_close, attention_layer64, layer_case, self_attention_bwd64
from test_gpu_attention_bwd import _dev, _tuned_context

pytestmark = pytest.mark.gpu


# e: odd, below and above one step, a multiple of 4 but not of 32, past a
# tile of 128; seq: one row, odd, past a tile.
@pytest.mark.parametrize("seq,e,heads", [(1, 4, 1), (33, 20, 4), (67, 35, 5), (130, 96, 3), (129, 132, 2), (260, 136, 2)])
@pytest.mark.parametrize("tile", [128, 16, 4])
def test_products(tile, seq, e, heads):
    c = _tuned_context(f"gemm={tile}")
    x, w = layer_case(seq, e, seq + e, amp=1.5)
    dy = np.random.default_rng(seq).standard_normal((seq, e)).astype(np.float32)
    wqkv, wout = w[:3 * e * e].reshape(e, 3 * e), w[3 * e * e:].reshape(e, e)
    bufs = []
    try:
        bufs = [_dev(c, a) for a in (x, dy, w, np.ones(w.size, np.float32), np.empty_like(x))]
        xb, dyb, wb, gwb, yb = bufs
        c.self_attention(xb, seq, e, heads, True, wb, w.size, yb)
        want, tol = attention_layer64(x, wqkv, wout, heads, True)
        got = yb.numpy().reshape(seq, e)
        assert (np.abs(got - want.reshape(seq, e)) <= np.asarray(tol).reshape(seq, e)).all(), "forward"
        (dx, dwqkv, dwout), (tx, twqkv, twout) = self_attention_bwd64(x, wqkv, wout, dy, heads, True)
        c.self_attention_bwd(xb, dyb, seq, e, heads, True, wb, w.size, gwb, yb)
        gw = gwb.numpy()
        assert_bwd_close(yb.numpy().reshape(seq, e), dx, tx, "dx")
        assert_bwd_close(gw[:3 * e * e] - 1, dwqkv, twqkv + 2e-7, "dWqkv", 2e-5)
        assert_bwd_close(gw[3 * e * e:] - 1, dwout, twout + 2e-7, "dWout", 2e-5)
    finally:
        for b in bufs:
            b.free()
        c.close()


@pytest.mark.parametrize("tile", [128, 16, 4])
def test_products_special_values(tile):
    """One token, so the layer is x Wv Wout: a value that rounds to infinity
    in bf16 against a zero row of Wv leaves the result alone, an infinity
    reaches what fp32 products give, NaN everything."""
    e = 40
    c = _tuned_context(f"gemm={tile}")
    r = np.random.default_rng(3)
    w = r.standard_normal(4 * e * e).astype(np.float32)
    wqkv, wout = w[:3 * e * e].reshape(e, 3 * e), w[3 * e * e:].reshape(e, e)
    wqkv[5] = 0.0
    wout[:, 7] = np.abs(wout[:, 7])
    x = r.standard_normal((1, e)).astype(np.float32)
    x[0, 5] = 3.4e38
    bufs = []
    try:
        bufs = [_dev(c, a) for a in (x, w, np.empty_like(x))]
        xb, wb, yb = bufs
        c.self_attention(xb, 1, e, 1, False, wb, w.size, yb)
        want = x.astype(np.float64) @ wqkv[:, 2 * e:].astype(np.float64) @ wout.astype(np.float64)
        np.testing.assert_allclose(yb.numpy().reshape(1, e), want, rtol=1e-4, atol=1e-4)
        x[0, 5] = np.inf  # inf * 0 = NaN in fp32 too
        c.upload(xb, x)
        c.self_attention(xb, 1, e, 1, False, wb, w.size, yb)
        assert np.isnan(yb.numpy()).all()
    finally:
        for b in bufs:
            b.free()
        c.close()


def test_products_of_one_term_are_rounded_once(ctx):
    """One token of width 1: the layer is x wv wout, two products of one term, each
    the float32 product."""
    r = np.random.default_rng(7)
    x, w = r.standard_normal(200).astype(np.float32), r.standard_normal((200, 4)).astype(np.float32)
    bufs = [_dev(ctx, x), _dev(ctx, w), _dev(ctx, np.zeros_like(x))]
    xb, wb, yb = bufs
    try:
        for i in range(x.size):
            ctx.self_attention(xb.offset(i, (1,)), 1, 1, 1, True, wb.offset(4 * i, (4,)), 4, yb.offset(i, (1,)))
        np.testing.assert_array_equal(yb.numpy().ravel(), x * w[:, 2] * w[:, 3])
    finally:
        for b in bufs:
            b.free()
