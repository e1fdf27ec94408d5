"""Attention whose head size the fused kernel does not take, against fp64: a chunk of a single head, whose two products leave the shared
workspace (it holds their score matrix) alone although their K alone would be worth cutting into ranges."""
import numpy as np
import pytest

from test_gpu_parity import SDPA_TOL, run_sdpa, say
from test_gpu_sdpa_terms import attention

pytestmark = pytest.mark.gpu


# one head; 256 MiB of scores hold 268 heads of 500 keys, 66 of 1001: the last of these comes alone
@pytest.mark.parametrize("BH,S,dk", [(1, 300, 6), (1, 500, 130), (1, 501, 256), (1, 1001, 160), (1, 97, 33), (269, 500, 130), (67, 1001, 161)])
@pytest.mark.parametrize("causal", [0, 1])
def test_single_head_chunks(hip, BH, S, dk, causal):
    say("unfused attention", BH, S, dk, causal)
    rng = np.random.default_rng(S + dk)
    q, k, v = (rng.uniform(-0.5, 0.5, (BH, S, dk)).astype(np.float32) for _ in range(3))
    o, l = run_sdpa(hip, q, k, v, 0.25, causal)
    assert hip.last_kernel() == "sdpa_unfused"
    some = sorted({0, BH // 2, BH - 1})
    want, lse = attention(q[some], k[some], v[some], 0.25, causal)
    assert np.abs(o[some] - want).max() <= SDPA_TOL
    assert np.abs(l[some] - lse).max() <= 1e-5 * max(1.0, np.abs(lse).max())
