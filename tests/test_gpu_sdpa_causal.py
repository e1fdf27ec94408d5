"""Causal attention as single query tiles, longest first, and as pairs of tiles: head counts that no eight divides, on four and on eight waves in every geometry,
against 64 bits; heads of the first, a middle and the last index."""
import numpy as np
import pytest

from test_gpu_parity import SDPA_TOL, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,S,dk", [(145, 192, 32), (381, 509, 32), (95, 322, 64), (127, 500, 64), (32, 2048, 64), (509, 129, 48), (99, 381, 96), (129, 280, 80),
                                     (43, 1000, 80), (97, 1000, 80), (64, 1024, 128), (178, 192, 128), (119, 300, 128), (151, 668, 128), (301, 100, 96)])
def test_causal_tiles(hip, BH, S, dk):
    say("causal tiles", BH, S, dk)
    rng = np.random.default_rng(BH + S + dk)
    q, k, v = (rng.normal(0, 1, (BH, S, dk)).astype(np.float32) for _ in range(3))
    dq, dk_, dv, do, dl = hip.array(q), hip.array(k), hip.array(v), hip.array(np.full((BH, S, dk), np.nan, np.float32)), hip.array(np.full((BH, S), np.nan, np.float32))
    scale = 1 / np.sqrt(dk)
    hip.check(hip.L.axhip_sdpa_fwd(dq.ptr, dk_.ptr, dv.ptr, do.ptr, dl.ptr, BH, S, dk, scale, 1))
    assert hip.last_kernel().startswith("sdpa_fused_dk")
    o, lse = do.numpy(), dl.numpy()
    assert np.isfinite(o).all() and np.isfinite(lse).all()
    hidden = np.triu(np.ones((S, S), bool), 1)
    for h in (0, BH // 2, BH - 1):
        s = np.where(hidden, -np.inf, scale * (q[h].astype(np.float64) @ k[h].astype(np.float64).T))
        m = s.max(1, keepdims=True)
        p = np.exp(s - m)
        want = (p / p.sum(1, keepdims=True)) @ v[h].astype(np.float64)
        assert np.abs(o[h] - want).max() <= SDPA_TOL
        assert np.abs(lse[h] - (m + np.log(p.sum(1, keepdims=True)))[:, 0]).max() <= SDPA_TOL
