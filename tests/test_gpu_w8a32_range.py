"""W8A32 on the register-staged tiles against fp64, at the ends of fp32's range: rows off the 16-byte grid, a K off the 32 grid, few hundred
rows against a long K, with one range of K and with several."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say

pytestmark = pytest.mark.gpu

# one tile height each, ranges of K, a last slab that hangs over
SHAPES = [(17, 129, 65), (60, 300, 321), (100, 515, 2047), (250, 1000, 2048), (834, 1100, 67)]


def product(hip, a, w, s):
    got = hip.qgemm_w8a32(hip.array(a), hip.array(w), hip.array(s)).numpy()
    assert hip.last_kernel().endswith("_staged") or hip.last_kernel() == "qgemm_w8a32_mfma_splitk", hip.last_kernel()
    return got


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("exponent", [-140, -126, -122, -118, -112, 100, 110])
def test_keeps_the_range(hip, M, N, K, exponent):
    """Small and large activations: relative accuracy as in the middle of the range, up to fp32's own smallest step (a multiple of it enters
    every sum exactly)."""
    say("w8a32 range", M, N, K, exponent)
    rng = np.random.default_rng(K + 200 + exponent)
    a = np.ldexp(rng.uniform(-1, 1, (M, K)), exponent).astype(np.float32)
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    got = product(hip, a, w, np.ones(N, np.float32))
    want = a.astype(np.float64) @ w.astype(np.float64).T
    size = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert (np.abs(got - want) <= BOUND_FP32 * size).all(), float((np.abs(got - want) / size).max())


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_non_finite(hip, oracle, M, N, K):
    """Infinities, NaNs and products past the largest float: as the reference's fp32 sum gives them; the other rows are untouched."""
    say("w8a32 non-finite", M, N, K)
    rng = np.random.default_rng(K)
    a = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    w[::3, 7] = 0
    a[1, 7], a[2, K - 1], a[3, 30], a[4, 0] = np.inf, -np.inf, np.nan, np.float32(3.0e38)
    a[5, K - 2] = np.array([0x7f800001], np.uint32).view(np.float32)[0]
    a[6], a[6, 9] = 0, np.float32(2.0 ** 110)
    s = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    got = product(hip, a, w, s)
    with np.errstate(all="ignore"):
        ref = oracle.qgemm_w8a32(a, w, s)
        want = (a.astype(np.float64) @ w.astype(np.float64).T) * s
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    assert np.array_equal(np.sign(got[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))
    rows = np.setdiff1d(np.arange(M), [1, 2, 3, 4, 5])
    size = (np.abs(a[rows]).astype(np.float64) @ np.abs(w).astype(np.float64).T) * s
    assert (np.abs(got[rows] - want[rows]) <= BOUND_FP32 * size ).all()
    assert (np.abs(got[6] - want[6]) <= 2.0 ** -22 * np.abs(want[6])).all()
