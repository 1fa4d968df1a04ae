"""The embedding backward's row sums at the edges of their column groups, of
their batches of eight rows and of the launch (more runs than workgroups),
through the counting sort's run list and by sorted position.  Runs below 32
tokens are added in token order, so they equal a float32 sum in that order bit
for bit; `dim` 516 x 4 and up take the 1024-thread form."""
import numpy as np
import pytest

from test_gpu_backward import _embedding_bwd_gpu
from test_gpu_attention_bwd import _tuned_context

pytestmark = pytest.mark.gpu


def _runs(counts, r):
    ids = np.repeat(np.arange(len(counts), dtype=np.int32), counts)
    return r.permutation(ids)


@pytest.mark.parametrize("tune", ["", "embruns=0"])
@pytest.mark.parametrize("dim,ids", [
    (4, 40000), (252, 300), (260, 300), (1028, 200), (2052, 9000), (4092, 60), (4100, 60)])
def test_short_runs(tune, dim, ids):
    r = np.random.default_rng(dim)
    counts = np.ones(ids, np.int64)
    counts[: 62] = np.tile(np.arange(31) + 1, 2)[: min(62, ids)]  # 1 .. 31 tokens
    tokens = _runs(counts, r)
    dy = r.standard_normal((tokens.size, dim)).astype(np.float32)
    grad = r.standard_normal((ids, dim)).astype(np.float32)
    want = grad.copy()
    order = np.argsort(tokens, kind="stable")
    first = np.concatenate([[0], np.cumsum(counts)[:-1]])
    for k in range(31):  # the k-th token of every run that has one
        rows = np.flatnonzero(counts > k)
        want[rows] += dy[order[first[rows] + k]]
    c = _tuned_context(tune)
    try:
        got = _embedding_bwd_gpu(c, tokens, dy, grad.reshape(-1), ids, dim, -1).reshape(ids, dim)
    finally:
        c.close()
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("dim", [12, 1020, 2060, 4104])
def test_long_runs(dim):
    """Runs of 32 to 200 tokens: regrouped, within the rounding of a float32
    sum of their length (n u per unit of the sum of magnitudes)."""
    r = np.random.default_rng(dim)
    counts = np.array([32, 33, 1, 63, 64, 65, 7, 200, 95, 96, 31])
    tokens = _runs(counts, r)
    dy = r.standard_normal((tokens.size, dim)).astype(np.float32)
    grad = r.standard_normal((counts.size, dim)).astype(np.float32)
    want = grad.astype(np.float64)
    mag = np.abs(want)
    np.add.at(want, tokens, dy.astype(np.float64))
    np.add.at(mag, tokens, np.abs(dy).astype(np.float64))
    c = _tuned_context("")
    try:
        got = _embedding_bwd_gpu(c, tokens, dy, grad.reshape(-1), counts.size, dim, -1).reshape(counts.size, dim)
    finally:
        c.close()
    assert (np.abs(got - want) <= (counts[:, None] + 1) * 2.0 ** -24 * mag).all()
