"""mimir_fill_f32 at every alignment and remainder, past a workgroup and past
the size kept in the caches: the range is filled, its neighbours are not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 1023, 1024, 1030, (1 << 25) + 3])
@pytest.mark.parametrize("start", [0, 1, 2, 3])
def test_fill(ctx, start, n):
    before = np.arange(n + 16, dtype=np.float32)
    buf = ctx.to_device(before)
    try:
        ctx.fill(buf.ptr + 4 * (4 + start), -0.0, n)
        got = buf.numpy()
    finally:
        buf.free()
    want = before.copy()
    want[4 + start:4 + start + n] = -0.0
    np.testing.assert_array_equal(got.view(np.int32), want.view(np.int32))
