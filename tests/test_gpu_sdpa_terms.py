"""Fused attention in bf16 terms against fp64: edges of key blocks, query tiles and head sizes, and the inputs that the terms cannot
hold, which the kernel computes with fp32 instructions instead."""
import numpy as np
import pytest

from test_gpu_parity import SDPA_TOL, run_sdpa, say

pytestmark = pytest.mark.gpu


def attention(q, k, v, scale, causal):
    """O and L in fp64; a key that the mask hides counts as absent, whatever it holds."""
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    with np.errstate(invalid="ignore", over="ignore"):
        s = scale * (q @ k.transpose(0, 2, 1))
        if causal:
            s = np.where(np.triu(np.ones(s.shape[1:], bool), 1), -np.inf, s)
        m = s.max(-1, keepdims=True)
        p = np.exp(s - m)
        total = p.sum(-1, keepdims=True)
        return (p / total) @ v, (m + np.log(total))[..., 0]


@pytest.mark.parametrize("dk", [4, 32, 36, 64, 68, 80, 96, 100, 128])
@pytest.mark.parametrize("S", [1, 31, 33, 64, 65, 97, 128, 161, 224, 321])
def test_tile_edges(hip, S, dk):
    rng = np.random.default_rng(1000 * S + dk)
    for BH, causal in ((3, 0), (9, 1), (260, 0), (260, 1)):               # the last two: more heads than CUs, on four and on eight waves
        say("sdpa terms", BH, S, dk, causal)
        q, k, v = (rng.uniform(-0.5, 0.5, (BH, S, dk)).astype(np.float32) for _ in range(3))
        o, l = run_sdpa(hip, q, k, v, 0.3, causal)
        assert hip.last_kernel().startswith("sdpa_fused")
        some = sorted({0, 1, 7, BH // 2, BH - 1} & set(range(BH)))
        o, l, q, k, v = (x[some] for x in (o, l, q, k, v))
        want, lse = attention(q, k, v, np.float32(0.3), causal)
        assert np.abs(o - want).max() <= SDPA_TOL and np.abs(l - lse).max() <= 1e-5 * max(1.0, np.abs(lse).max())


@pytest.mark.parametrize("dk", [32, 64, 80, 128])
@pytest.mark.parametrize("sq,sk,sv", [(1, 1, -115), (1, 1, 100), (1, 1, 120), (-100, 100, 0), (110, -110, 0), (0, 0, -100)])
def test_keeps_the_range(hip, dk, sq, sk, sv):
    """Magnitudes (powers of two) whose small terms leave the normal range, and large ones (not so large that the 150 terms of a sum
    before its division leave it in fp32): accuracy as in the middle of it."""
    say("sdpa range", dk, sq, sk, sv)
    rng = np.random.default_rng(dk)
    q, k, v = (np.ldexp(rng.uniform(-0.5, 0.5, (3, 150, dk)), e).astype(np.float32) for e in (sq, sk, sv))
    for causal in (0, 1):
        o, l = run_sdpa(hip, q, k, v, 0.125, causal)
        want, lse = attention(q, k, v, 0.125, causal)
        # SDPA_TOL is for values of V below one half; fp32 has no more than its smallest step to give
        assert (np.abs(o - want) <= np.ldexp(SDPA_TOL, sv) + 64 * 2.0 ** -149).all()
        assert np.abs(l - lse).max() <= 1e-5 * max(1.0, np.abs(lse).max())


@pytest.mark.parametrize("dk", [32, 64, 80, 128])
def test_small_probabilities_keep_their_bits(hip, dk):
    """Row 0 of K takes all the weight and has zeros in V, so the result is one probability near 2^-d: accurate to the rounding of the
    score difference (|d| * 2^-23 in base 2, and as much again for the two scores' own sums)."""
    S = 70
    q, k, v = np.zeros((12, S, dk), np.float32), np.zeros((12, S, dk), np.float32), np.zeros((12, S, dk), np.float32)
    depth = np.arange(12) * 10.0 + 12
    q[:, :, 0] = 1.0
    k[:, 1:, 0] = (-depth * np.log(2.0))[:, None]
    v[:, 1:] = 1.0 + np.arange(dk) / 64
    say("sdpa depth", dk)
    o, _ = run_sdpa(hip, q, k, v, 1.0, 0)
    want, _ = attention(q, k, v, 1.0, 0)
    err = (np.abs(o - want) / want).max(axis=(1, 2))
    assert (err <= 4 * depth * 2.0 ** -23 + 70 * 2.0 ** -24).all(), err


@pytest.mark.parametrize("dk", [32, 64, 80, 128])
@pytest.mark.parametrize("causal", [0, 1])
def test_non_finite(hip, dk, causal):
    """Infinities and NaNs reach the rows that see them and no others; a value next to the largest float comes out whole."""
    say("sdpa non-finite", dk, causal)
    rng = np.random.default_rng(dk + causal)
    S = 200
    q, k, v = (rng.uniform(-0.5, 0.5, (6, S, dk)).astype(np.float32) for _ in range(3))
    top = np.finfo(np.float32).max
    v[0, 0, 3] = np.inf
    k[1, 150, 1] = np.nan
    q[2, 77, 0] = np.nan
    v[3, 0] = top
    v[3, 1:] = 0
    q[5, 10, 2], k[5, :, 2] = np.inf, 0.25                                # every score of query 10 infinite
    o, l = run_sdpa(hip, q, k, v, 0.2, causal)
    assert np.isposinf(o[0, :, 3]).all()
    bad = np.zeros((6, S), bool)
    bad[1, 150 if causal else 0:] = True
    bad[2, 77] = bad[5, 10] = True
    assert np.isnan(o[bad]).all() and np.isnan(l[bad]).all()
    fine = ~bad
    v[0, 0, 3] = 0
    want, lse = attention(np.nan_to_num(q, nan=0.0, posinf=0.0), np.nan_to_num(k), v, np.float32(0.2), causal)
    o[0, :, 3] = want[0, :, 3]
    size = np.where(np.arange(6) == 3, float(top), 1.0)[:, None]
    if causal:
        assert o[3, 0, 0] == top
    assert (np.abs(o - want).max(-1)[fine] <= (2 * SDPA_TOL * size * np.ones((6, S)))[fine]).all()
    assert (np.abs(l - lse)[fine] <= 1e-5 * np.maximum(1.0, np.abs(lse[fine]))).all()


@pytest.mark.parametrize("dk", [32, 64, 80, 128])
@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("S,hidden", [(200, 32), (200, 33), (200, 64), (200, 130), (520, 500)])
def test_first_keys_hidden(hip, dk, causal, S, hidden):
    """The first keys of every row score minus infinity: their weight is zero, and the rows that see others come out as without them;
    rows that see no others are NaN, as the quotient of two zeros is."""
    say("sdpa first keys hidden", dk, causal, S, hidden)
    rng = np.random.default_rng(dk + hidden)
    for BH in (3, 260):
        q, k, v = (rng.uniform(-0.5, 0.5, (BH, S, dk)).astype(np.float32) for _ in range(3))
        q[:, :, 1] = 0.5
        k[:, :hidden, 1] = -np.inf
        o, l = run_sdpa(hip, q, k, v, 0.3, causal)
        some = [0, BH - 1]
        want, lse = attention(q[some], k[some], v[some], np.float32(0.3), causal)
        assert np.array_equal(np.isnan(o[some]), np.isnan(want)) and np.array_equal(np.isnan(l[some]), np.isnan(lse))
        assert np.isnan(lse).any() == bool(causal)
        assert np.nanmax(np.abs(o[some] - want)) <= SDPA_TOL and np.nanmax(np.abs(l[some] - lse)) <= 1e-5 * max(1.0, np.nanmax(np.abs(lse)))


@pytest.mark.parametrize("dk", [32, 64, 80, 128])
def test_small_values_among_others(hip, dk):
    """Values down to fp32's smallest beside ordinary ones are no reason for the fp32 pass: every result comes out as with zeros in their
    place, but for the few whose rounding is a tie."""
    say("sdpa small values", dk)
    rng = np.random.default_rng(dk)
    x = [rng.uniform(-0.5, 0.5, (9, 300, dk)).astype(np.float32) for _ in range(3)]
    for y in x:
        y[rng.random(y.shape) < 0.02] = 0
    clean = run_sdpa(hip, *x, 0.3, 0)
    for y in x:
        y[y == 0] = np.ldexp(1.0, rng.integers(-149, -100, (y == 0).sum())).astype(np.float32)
    for got, want in zip(run_sdpa(hip, *x, 0.3, 0), clean):
        assert (got != want).mean() < 0.01


@pytest.mark.parametrize("dk", [32, 64, 80, 128])
@pytest.mark.parametrize("exponent", [0, -126, 90])
def test_single_products(hip, dk, exponent):
    """One key: O is V but for the left-out terms (2^-24), one rounding to 2^-24 of the sum of the terms, one of the quotient and the
    division of 1 (2^-24 each), and the others' own roundings (2^-8 of that, seven at most).  L is one product of Q and K times the scale:
    the roundings of q * scale * log2(e) (two), of the sum of terms, the left-out terms and the two on the way back."""
    say("sdpa single products", dk, exponent)
    rng = np.random.default_rng(dk)
    q, k = np.zeros((500, 1, dk), np.float32), np.zeros((500, 1, dk), np.float32)
    at = rng.integers(0, dk, (500, 1, 1))
    np.put_along_axis(q, at, rng.uniform(1, 2, (500, 1, 1)).astype(np.float32), 2)
    np.put_along_axis(k, at, rng.uniform(1, 2, (500, 1, 1)).astype(np.float32), 2)
    v = np.ldexp(rng.uniform(1, 2, (500, 1, dk)), exponent).astype(np.float32)
    o, l = run_sdpa(hip, q, k, v, 0.7, 0)
    assert (np.abs(o - v.astype(np.float64)) <= 2.0 ** -24 * (4 + 7 / 128) * v).all()
    want = np.float32(0.7) * (q.astype(np.float64) * k).sum(-1)
    assert (np.abs(l - want) <= 2.0 ** -24 * 8 * want).all(), float((np.abs(l - want) / want).max() * 2 ** 24)
