"""Causal attention as single query tiles, in groups of 32 heads and longest first, and as pairs of tiles: head counts that no eight divides, on four and on eight waves
in every geometry, against 64 bits; heads of the first, a middle and the last index.  Pairs with a middle tile that stands alone too, and on inputs that the terms cannot hold."""
import numpy as np
import pytest

from test_gpu_parity import SDPA_TOL, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,S,dk,form", [(145, 192, 32, ""), (381, 509, 32, ""), (95, 322, 64, "_w8"), (127, 500, 64, "_pairs"), (32, 2048, 64, "_pairs"), (509, 129, 48, "_pairs"),
                                          (99, 381, 96, "_w8"), (129, 280, 80, ""), (43, 1000, 80, ""), (97, 1000, 80, "_w8"), (64, 1024, 128, "_pairs"), (178, 192, 128, "_w8"),
                                          (119, 300, 128, "_w8"), (151, 668, 128, "_w8"), (301, 100, 96, ""), (167, 700, 112, "_w8"), (203, 700, 48, "")])
def test_causal_tiles(hip, BH, S, dk, form):
    say("causal tiles", BH, S, dk)
    rng = np.random.default_rng(BH + S + dk)
    q, k, v = (rng.normal(0, 1, (BH, S, dk)).astype(np.float32) for _ in range(3))
    dq, dk_, dv, do, dl = hip.array(q), hip.array(k), hip.array(v), hip.array(np.full((BH, S, dk), np.nan, np.float32)), hip.array(np.full((BH, S), np.nan, np.float32))
    scale = 1 / np.sqrt(dk)
    hip.check(hip.L.axhip_sdpa_fwd(dq.ptr, dk_.ptr, dv.ptr, do.ptr, dl.ptr, BH, S, dk, scale, 1))
    assert hip.last_kernel() == f"sdpa_fused_dk{(dk + 31) // 32 * 32}_causal{form}"
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


@pytest.mark.parametrize("BH,S,dk,form", [(32, 1793, 64, "_pairs"), (32, 1900, 36, "_pairs"), (33, 3840, 64, "_pairs"), (64, 1021, 128, "_pairs"), (64, 1000, 100, "_pairs"),
                                          (12, 7200, 96, "_w8_pairs"), (12, 7300, 80, "_w8_pairs"), (8, 7200, 96, "_pairs"), (8, 7300, 68, "_pairs")])
def test_pairs(hip, BH, S, dk, form):
    """Odd and even counts of tiles.  Every head but the first and the last has something that reaches one tile of a pair or both: values past the terms, which send a tile through
    the second pass, first keys that weigh nothing, a key and a query that are NaN, an infinite value that all rows see; rows at the edges of all tiles."""
    say("causal pairs", BH, S, dk)
    rng = np.random.default_rng(BH + S + dk)
    q, k, v = (rng.uniform(-0.5, 0.5, (BH, S, dk)).astype(np.float32) for _ in range(3))
    v[1] *= np.float32(2.0 ** 110)
    k[2, :S // 2, 1], q[2, :, 1] = -np.inf, 0.5
    k[3, S // 3, 1] = np.nan
    q[4, [3, S - 1], 0] = np.nan
    v[5, 0, 3] = np.inf
    v[6, 2 * S // 3:] *= np.float32(2.0 ** 110)
    o, lse = np.full((BH, S, dk), np.nan, np.float32), np.full((BH, S), np.nan, np.float32)
    dq, dk_, dv, do, dl = (hip.array(x) for x in (q, k, v, o, lse))
    hip.check(hip.L.axhip_sdpa_fwd(dq.ptr, dk_.ptr, dv.ptr, do.ptr, dl.ptr, BH, S, dk, 0.3, 1))
    assert hip.last_kernel() == f"sdpa_fused_dk{(dk + 31) // 32 * 32}_causal{form}"
    o, lse = do.numpy(), dl.numpy()
    rows = np.array(sorted({x for t in range(0, S, 128) for x in (t, t + 31, t + 127) if x < S} | {3, S // 4 - 1, S // 4, S // 3 - 1, S // 3, S // 2 - 1, S // 2, 2 * S // 3, S - 1}))
    hidden = np.arange(S)[None, :] > rows[:, None]
    for h in (*range(7), BH - 1):
        with np.errstate(invalid="ignore", over="ignore"):
            s = np.where(hidden, -np.inf, np.float64(np.float32(0.3)) * (q[h, rows].astype(np.float64) @ k[h].astype(np.float64).T))
            m = s.max(1, keepdims=True)
            p = np.exp(s - m)
            vh = v[h].astype(np.float64)
            want, total = np.empty((len(rows), dk)), p.sum(1, keepdims=True)
            for i in range(len(rows)):                       # a key that the mask hides counts as absent, whatever its value holds
                want[i] = p[i, :rows[i] + 1] @ vh[:rows[i] + 1] / total[i]
            l_want = (m + np.log(total))[:, 0]
        got, l_got = o[h, rows], lse[h, rows]
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(np.isnan(l_got), np.isnan(l_want)), h
        fine = np.isfinite(want)
        size = np.maximum(1.0, np.abs(want[fine]).max() * 2) if h in (1, 6) else 1.0
        assert np.abs(got[fine] - want[fine]).max() <= 2 * SDPA_TOL * size, h
        assert np.nanmax(np.abs(l_got - l_want)) <= 1e-5 * max(1.0, np.nanmax(np.abs(l_want))), h


@pytest.mark.parametrize("causal", [0, 1])
def test_more_tiles_than_a_grid_holds(hip, causal):
    """2^24 workgroups of 256 threads are one launch too many threads: the heads go in two pieces.  One key a head: O is V but for the left-out terms, three roundings and the
    others' own (2^-24 each and 2^-8 of that), L the scaled product of Q and K."""
    BH = 2 ** 24 + 1021
    say("causal tiles in pieces", causal)
    rng = np.random.default_rng(BH)
    q, k, v = (rng.random((BH, 1, 4), np.float32) + 1 for _ in range(3))
    dq, dk_, dv, do, dl = hip.array(q), hip.array(k), hip.array(v), hip.array(np.full((BH, 1, 4), np.nan, np.float32)), hip.array(np.full((BH, 1), np.nan, np.float32))
    hip.check(hip.L.axhip_sdpa_fwd(dq.ptr, dk_.ptr, dv.ptr, do.ptr, dl.ptr, BH, 1, 4, 0.5, causal))
    assert (np.abs(do.numpy() - v) <= 2.0 ** -24 * (4 + 7 / 128) * v).all()
    want = 0.5 * (q * k).sum(-1)
    assert (np.abs(dl.numpy() - want) <= 1e-6 * want).all()
