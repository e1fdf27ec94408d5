"""Fused attention with few query tiles, where four waves share 32 queries and take their keys in turn: which calls it takes, and the
same heads on both forms, among them ones that neither can hold in bf16 terms."""
import numpy as np
import pytest

from test_gpu_parity import SDPA_TOL, run_sdpa, say
from test_gpu_sdpa_terms import attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,S,dk,causal,few", [(256, 32, 64, 0, False), (128, 64, 64, 0, True), (129, 64, 64, 1, False),
                                                (128, 128, 64, 0, True), (129, 128, 32, 0, False), (64, 97, 96, 1, True), (65, 128, 128, 0, False),
                                                (36, 512, 64, 0, True), (37, 512, 80, 0, False), (57, 512, 64, 1, True), (58, 512, 64, 1, False),
                                                (32, 512, 128, 1, True), (33, 512, 128, 1, False), (36, 224, 96, 0, True), (37, 224, 96, 0, False),
                                                (51, 300, 128, 0, True), (52, 300, 128, 0, False), (53, 256, 64, 1, True), (54, 256, 64, 1, False),
                                                (85, 150, 80, 1, True), (86, 150, 80, 1, False), (64, 256, 64, 0, True), (65, 256, 64, 0, False),
                                                (25, 993, 96, 1, False), (36, 512, 32, 1, True)])
def test_where_it_runs(hip, BH, S, dk, causal, few):
    """Both sides of each limit of the rule (256 CUs)."""
    say("sdpa few", BH, S, dk, causal)
    rng = np.random.default_rng(BH + S + dk)
    q, k, v = (rng.uniform(-0.5, 0.5, (BH, S, dk)).astype(np.float32) for _ in range(3))
    o, l = run_sdpa(hip, q, k, v, 0.3, causal)
    assert ("few" in hip.last_kernel()) == few, hip.last_kernel()
    some = [0, BH // 2, BH - 1]
    want, lse = attention(q[some], k[some], v[some], np.float32(0.3), causal)
    assert np.abs(o[some] - want).max() <= SDPA_TOL and np.abs(l[some] - lse).max() <= 1e-5 * max(1.0, np.abs(lse).max())


@pytest.mark.parametrize("dk", [20, 64, 80, 128])
@pytest.mark.parametrize("S", [33, 96, 161, 230])
@pytest.mark.parametrize("causal", [0, 1])
def test_both_forms_on_the_same_heads(hip, S, dk, causal):
    """Six heads alone and fifty times over: the same numbers to twice the tolerance of each, infinities and NaNs in the same places."""
    say("sdpa few and many", S, dk, causal)
    rng = np.random.default_rng(S + dk)
    q, k, v = (rng.uniform(-0.5, 0.5, (6, S, dk)).astype(np.float32) for _ in range(3))
    v[0, 0, 3] = np.inf
    k[1, S // 2, 1] = np.nan
    q[2, S - 1, 0] = np.nan
    k[3, :S // 2, 1], q[3, :, 1] = -np.inf, 0.5                           # causal: rows that see nothing else
    v[4] *= np.float32(2.0 ** 110)
    o, l = run_sdpa(hip, q, k, v, 0.3, causal)
    assert "few" in hip.last_kernel()
    om, lm = run_sdpa(hip, *(np.tile(x, (50, 1, 1)) for x in (q, k, v)), 0.3, causal)
    assert "few" not in hip.last_kernel()
    om, lm = om.reshape((50, 6, S, dk)), lm.reshape((50, 6, S))
    for n in (0, 49):
        assert np.array_equal(np.isfinite(o), np.isfinite(om[n])) and np.array_equal(np.isnan(o), np.isnan(om[n])) and np.array_equal(np.isnan(l), np.isnan(lm[n]))
        size = np.where(np.arange(6) == 4, 2.0 ** 110, 1.0)[:, None, None]
        fine = np.isfinite(o)
        assert (np.abs(o.astype(np.float64) - om[n]) / size)[fine].max() <= 2 * SDPA_TOL
        assert np.nanmax(np.abs(l - lm[n])) <= 2e-5 * max(1.0, np.nanmax(np.abs(l)))


@pytest.mark.parametrize("BH,S,dk", [(6, 64, 20), (6, 128, 64), (3, 161, 80), (3, 512, 128)])
@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("power", [70, 72, 73, 74, 75, 76, 78, 80])
def test_values_of_one_sign_past_the_terms(hip, BH, S, dk, causal, power):
    """Waves whose own sums the terms hold while those of all four are above what they hold; scores near each other, so that all of them count."""
    say("sdpa few, values of one sign", BH, S, dk, causal, power)
    rng = np.random.default_rng(S + dk + power)
    q, k = (rng.uniform(-0.5, 0.5, (BH, S, dk)).astype(np.float32) for _ in range(2))
    v = rng.uniform(0.5, 1, (BH, S, dk)).astype(np.float32)
    v[0, :, 0] = 1
    o, l = run_sdpa(hip, q, k, v * np.float32(2.0 ** power), 0.05, causal)
    assert "few" in hip.last_kernel()
    want, lse = attention(q, k, v, np.float32(0.05), causal)
    assert np.abs(o.astype(np.float64) / 2.0 ** power - want).max() <= SDPA_TOL
    assert np.abs(l - lse).max() <= 1e-5 * max(1.0, np.abs(lse).max())
