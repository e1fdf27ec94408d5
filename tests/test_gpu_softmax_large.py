"""Row softmax over more than 256 MiB, whose rows are walked from the last: every row, also where the last workgroup is not full, in place and not."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("rows,cols", [(520001, 130), (134219, 501), (67110, 1001), (16411, 4093), (12003, 5600)])
def test_large(hip, rows, cols, in_place):
    say("large softmax", rows, cols, in_place)
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, cols), dtype=np.float32)
    x *= np.arange(1, rows + 1, dtype=np.float32)[:, None] / np.float32(rows / 8)
    dx = hip.array(x)
    out = dx if in_place else hip.array(np.full((rows + 1, cols), np.nan, np.float32))
    hip.check(hip.L.axhip_softmax_rows(dx.ptr, out.ptr, rows, cols))
    got = out.numpy()
    if not in_place:
        assert np.isnan(got[rows]).all()                                  # a row past the output: never written
    for r0 in range(0, rows, 1 << 14):
        e = np.exp(x[r0:r0 + (1 << 14)].astype(np.float64) - x[r0:r0 + (1 << 14)].max(axis=1, keepdims=True))
        want = e / e.sum(axis=1, keepdims=True)
        # |x| up to 40: a rounding of the difference (2^-24 of 64), exp's and the sum's few units
        assert (np.abs(got[r0:min(rows, r0 + (1 << 14))] - want) <= 6e-6 * want + 1e-37).all()
