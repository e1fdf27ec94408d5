"""Fused attention with few query tiles: both sides of the line for walks of ten key tiles and more, and for one tile a wave of the geometry 96."""
import numpy as np
import pytest

from test_gpu_parity import SDPA_TOL, run_sdpa, say
from test_gpu_sdpa_terms import attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,S,dk,causal,few", [(31, 1400, 64, 1, True), (32, 1400, 64, 1, False), (18, 1300, 32, 0, True), (19, 1300, 32, 0, False),
                                                (21, 1300, 128, 1, True), (22, 1300, 128, 1, False), (12, 1300, 80, 0, True), (13, 1300, 80, 0, False),
                                                (128, 128, 96, 0, True), (129, 128, 96, 0, False), (128, 97, 80, 1, True)])
def test_where_it_runs(hip, BH, S, dk, causal, few):
    """256 CUs."""
    say("sdpa few, long", BH, S, dk, causal)
    rng = np.random.default_rng(BH + S + dk)
    q, k, v = (rng.uniform(-0.5, 0.5, (BH, S, dk)).astype(np.float32) for _ in range(3))
    o, l = run_sdpa(hip, q, k, v, 0.3, causal)
    assert ("few" in hip.last_kernel()) == few, hip.last_kernel()
    some = [0, BH - 1]
    want, lse = attention(q[some], k[some], v[some], np.float32(0.3), causal)
    assert np.abs(o[some] - want).max() <= SDPA_TOL and np.abs(l[some] - lse).max() <= 1e-5 * max(1.0, np.abs(lse).max())
