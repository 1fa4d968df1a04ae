"""Rows whose 16-byte vectors do not line up (a width that is not a multiple
of 4, or a pointer off 16 bytes): LayerNorm both ways, RMSNorm, add + RMSNorm
and the softmaxes at the edges of the row kernels' widths, against float64.

Tolerance: a float32 sum of n terms in any order is within n u of its summed
magnitudes; over these widths and N(0,1) rows that stays below 1e-5 of the
result's scale, the path's own bound."""
import numpy as np
import pytest

import mimir_hip as M

pytestmark = pytest.mark.gpu

# The last vector of one to three floats in the first, middle and last slot of
# each launch shape, and the first width of the next.
WIDTHS = [1, 2, 3, 5, 63, 66, 67, 254, 257, 511, 513, 1001, 1023, 1025, 2047, 2050, 4095, 4097, 8191, 8194, 16383]


def close(got, want, scale=1.0, tol=1e-5):
    np.testing.assert_array_less(np.abs(got.astype(np.float64) - want), tol * (np.abs(want) + scale) + 1e-30)


class Buffers:
    """Device copies `shift` floats past a 16-byte boundary."""

    def __init__(self, ctx, shift):
        self.ctx, self.shift, self.made = ctx, shift, []

    def put(self, a):
        d = self.ctx.empty((a.size + self.shift + 4,))
        self.made.append(d)
        v = d.offset(self.shift, a.shape)
        self.ctx.upload(v, np.ascontiguousarray(a, np.float32))
        return v

    def get(self, v):
        out = np.empty(v.shape, np.float32)
        self.ctx.download(out, v)
        return out

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for d in self.made:
            d.free()


def ln64(x, eps):
    d = x - x.mean(1, keepdims=True)
    rstd = 1 / np.sqrt((d * d).mean(1, keepdims=True) + eps)
    return d * rstd, rstd


CASES = [(rows, cols, 0) for cols in WIDTHS for rows in (1, 5)] + [(131, 1001, 0), (2500, 67, 0), (7, 64, 1), (6, 1024, 3),
                                                                  (3, 4096, 2), (600, 260, 1), (2048, 515, 0), (2049, 515, 0),
                                                                  (2048, 1535, 0), (2049, 1535, 0), (2049, 1537, 0),
                                                                  (2560, 1001, 0), (2561, 1001, 0), (2561, 1535, 0),
                                                                  (3072, 1027, 0), (3073, 1535, 0)]


@pytest.mark.parametrize("rows,cols,shift", CASES)
def test_rows_any(ctx, rows, cols, shift):
    r = np.random.default_rng(rows + cols)
    x, res, dy = (r.standard_normal((rows, cols)).astype(np.float32) for _ in range(3))
    g = (1 + 0.1 * r.standard_normal(cols)).astype(np.float32)
    be = (0.1 * r.standard_normal(cols)).astype(np.float32)
    x64, dy64, g64 = x.astype(np.float64), dy.astype(np.float64), g.astype(np.float64)
    eps = 1e-5
    with Buffers(ctx, shift) as b:
        dx_, dg_, db_, y = b.put(x), b.put(g), b.put(be), b.put(np.zeros_like(x))
        ctx.layernorm(dx_, dg_, db_, y, rows, cols, eps)
        xh, rstd = ln64(x64, eps)
        close(b.get(y), xh * g64 + be)
        ctx.layernorm(dx_, None, None, y, rows, cols, eps)
        close(b.get(y), xh)
        # RMSNorm with a weight shorter than the row, then in place.
        w_len = max(1, cols - 2)
        rms = x64 / np.sqrt((x64 * x64).mean(1, keepdims=True) + eps)
        ctx.rmsnorm(dx_, dg_, w_len, y, rows, cols, eps)
        close(b.get(y), np.concatenate([rms[:, :w_len] * g64[:w_len], rms[:, w_len:]], 1))
        # add + RMSNorm, the residual updated in place: the sum is exact in float32.
        rd = b.put(res)
        ctx.add_rmsnorm(dx_, rd, rd, dg_, y, rows, cols, eps)
        h = x + res
        assert np.array_equal(b.get(rd), h)
        h64 = h.astype(np.float64)
        close(b.get(y), h64 / np.sqrt((h64 * h64).mean(1, keepdims=True) + eps) * g64)
        # Softmaxes, the first in place, with a masked tail.
        s = x.copy()
        s[:, cols // 2 + 1:] = -np.inf
        sd = b.put(s)
        ctx.softmax(sd, sd, rows, cols, M.SOFTMAX_DIV_EPS)
        e = np.exp(s.astype(np.float64) - s.max(1, keepdims=True))
        p = e / e.sum(1, keepdims=True)
        close(b.get(sd), p, 1e-6 * np.ones_like(p))
        ctx.softmax(dx_, y, rows, cols, M.SOFTMAX_LOG)
        m = x64.max(1, keepdims=True)
        close(b.get(y), x64 - m - np.log(np.exp(x64 - m).sum(1, keepdims=True)))
        # LayerNorm backward: dx over dy, dgamma and dbeta added to, then dx added to.
        dyd, gg = b.put(dy), b.put(np.ones((2, cols), np.float32))
        gb = gg.offset(cols, (cols,))
        ctx.layernorm_bwd(dx_, dyd, dg_, dyd, gg, gb, rows, cols, eps)
        gy = dy64 * g64
        want = rstd * (gy - gy.mean(1, keepdims=True) - xh * (gy * xh).mean(1, keepdims=True))
        scale = rstd * np.abs(gy).max(1, keepdims=True) * 4
        close(b.get(dyd), want, scale)
        grads = b.get(gg)
        close(grads[0], 1 + (dy64 * xh).sum(0), 1 + np.abs(dy64 * xh).sum(0))
        close(grads[1], 1 + dy64.sum(0), 1 + np.abs(dy64).sum(0))
        acc = b.put(res)
        ctx.layernorm_bwd(dx_, b.put(dy), dg_, acc, None, None, rows, cols, eps, accumulate=True)
        close(b.get(acc), res + want, scale + np.abs(res))
