"""fp32 products in bf16 terms against fp64: tile edges and remainders of K on and off the 16-byte grid, every storage order, ranges
of K, batches; and the inputs that the terms cannot hold, which the kernel computes with fp32 instructions instead."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say

pytestmark = pytest.mark.gpu


def product(hip, a, b, order):
    sa, sb = np.ascontiguousarray(a.T if order[0] == "t" else a), np.ascontiguousarray(b.T if order[1] == "t" else b)
    M, K, N = a.shape[0], a.shape[1], b.shape[1]
    c = hip.array(np.full((M, N), np.nan, np.float32))
    da, db = hip.array(sa), hip.array(sb)
    hip.check(hip.L.axhip_sgemm(int(order[0] == "t"), int(order[1] == "t"), M, N, K, 1.0, da.ptr, sa.shape[1], db.ptr, sb.shape[1], 0.0, c.ptr,
                                N, None, 0))
    kernel = hip.last_kernel()
    assert kernel.endswith("x3_staged") or kernel == "sgemm_splitk_x3", kernel
    return c.numpy()


# the fp32 error bound K u sum |a||b| (u = 2^-24) holds with room for sums of random signs, see test_gpu_staged; the left-out terms
# add at most 2^-24 of each product
@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K", [(17, 33, 64), (65, 129, 65), (129, 65, 95), (161, 516, 256), (1152, 1152, 1152), (1153, 772, 2052), (644, 4096, 1024),
                                   (2049, 1028, 260), (200, 128, 4096), (1000, 1004, 1001)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_split_fp32(hip, M, N, K, order):
    say("split", M, N, K, order)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    got = product(hip, a, b, order)
    want = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - want) <= BOUND_FP32 * size).all(), float((np.abs(got - want) / size).max())


@pytest.mark.parametrize("Bn,M,N,K,transb", [(9, 333, 333, 64, 1), (5, 257, 260, 1030, 0), (16, 512, 512, 256, 0)])
def test_split_batched(hip, Bn, M, N, K, transb):
    say("split batched", Bn, M, N, K, transb)
    rng = np.random.default_rng(Bn + M + K)
    a = rng.uniform(-1, 1, (Bn, M, K)).astype(np.float32)
    b = rng.uniform(-1, 1, (Bn, N, K) if transb else (Bn, K, N)).astype(np.float32)
    got = hip.sgemm_batched(hip.array(a), hip.array(b), transb=bool(transb), alpha=0.25).numpy()
    assert "x3_staged" in hip.last_kernel()
    bt = b.astype(np.float64).transpose(0, 2, 1) if transb else b.astype(np.float64)
    want = 0.25 * (a.astype(np.float64) @ bt)
    size = 0.25 * (np.abs(a).astype(np.float64) @ np.abs(bt))
    assert (np.abs(got - want) <= BOUND_FP32 * size).all()


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K,tile", [(70, 90, 101, "64x64"), (501, 2053, 129, "128x64"), (513, 3583, 129, "64x128"), (1537, 1541, 129, "128x128")])
def test_every_tile(hip, M, N, K, tile):
    """The shapes of this file reach every tile: one row or column past whole tiles, a slab and one value more."""
    say("split tile", M, N, K)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    got = product(hip, a, b, "nn")
    assert hip.last_kernel() == f"sgemm_nn_{tile}x3_staged"
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= BOUND_FP32 * size).all()


SHAPES = [(70, 90, 101), (200, 132, 1029), (1152, 1152, 1152)]      # one tile, ranges of K, whole tiles


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("scale_a,scale_b", [(2.0 ** -115, 1.0), (2.0 ** -100, 2.0 ** 90), (2.0 ** -60, 2.0 ** -50), (2.0 ** 120, 2.0 ** -20), (1.0, 2.0 ** -118)])
def test_split_keeps_the_range(hip, M, N, K, scale_a, scale_b):
    """Magnitudes whose small terms leave the normal range, and large ones: relative accuracy as in the middle of it."""
    say("split range", M, N, K, scale_a, scale_b)
    rng = np.random.default_rng(K)
    a = (rng.uniform(-1, 1, (M, K)) * scale_a).astype(np.float32)
    b = (rng.uniform(-1, 1, (K, N)) * scale_b).astype(np.float32)
    a[3] = 0
    got = product(hip, a, b, "nn")
    want = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - want) <= BOUND_FP32 * size + K * 2.0 ** -149).all()


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_split_non_finite(hip, M, N, K):
    """Infinities, NaNs and values that round past the largest bf16 give what fp32 arithmetic gives; the other rows are untouched."""
    say("split non-finite", M, N, K)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    top = np.finfo(np.float32).max
    a[1, 7] = np.inf
    a[2, 7], a[2, 30] = np.inf, -np.inf
    a[4, 50] = np.nan
    a[5] = 0
    a[5, K - 1] = top
    b[K - 1, 2] = 1.0
    b[7, ::3] = 0
    got = product(hip, a, b, "nn")
    with np.errstate(invalid="ignore", over="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.array_equal(np.sign(got[1]), np.sign(ref[1]), equal_nan=True)
    assert got[5, 2] == top
    rows = np.setdiff1d(np.arange(M), [1, 2, 4])
    size = np.abs(a[rows]).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got[rows] - ref[rows]) <= BOUND_FP32 * size).all()


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("scale_a,scale_b", [(2.0 ** -60, 2.0 ** -60), (2.0 ** -55, 2.0 ** -68), (2.0 ** -20, 2.0 ** -110), (2.0 ** -127, 2.0 ** 10), (2.0 ** 50, 2.0 ** 40)])
def test_split_small_results(hip, M, N, K, scale_a, scale_b):
    """Ordinary or small operands whose products lie next to the smallest normal value (and above 2^80): relative accuracy as in the
    middle of the range, up to fp32's own smallest step (one for the sum, one for each of the sums of ranges and wave sets)."""
    say("split small results", M, N, K, scale_a, scale_b)
    rng = np.random.default_rng(K)
    a = (rng.uniform(-1, 1, (M, K)) * scale_a).astype(np.float32)
    b = (rng.uniform(-1, 1, (K, N)) * scale_b).astype(np.float32)
    got = product(hip, a, b, "nn")
    want = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - want) <= BOUND_FP32 * size + 32 * 2.0 ** -149).all(), float(((np.abs(got - want) - 32 * 2.0 ** -149) / size).max())


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_split_small_values_among_others(hip, M, N, K):
    """Values down to fp32's smallest beside ordinary ones, as GELU and softmax leave them, are no reason for the fp32 pass: every sum
    comes out as with zeros in their place, but for the few whose rounding is a tie.  (The fp32 instructions add in another order: they
    would change about half of the sums.)"""
    say("split small values", M, N, K)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    for x in (a, b):
        x[rng.random(x.shape) < 0.02] = 0
    clean = product(hip, a, b, "nn")
    for x in (a, b):
        x[x == 0] = np.ldexp(1.0, rng.integers(-149, -100, (x == 0).sum())).astype(np.float32)
    got = product(hip, a, b, "nn")
    assert (got != clean).mean() < 0.01


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K", SHAPES + [(65, 517, 257), (501, 2053, 129), (513, 3583, 129)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_split_single_products(hip, M, N, K, order):
    """Sums with one product that is not zero, of operands with all 24 bits: the left-out terms are at most 2^-24 of it; the large term is
    added to the others by a vector instruction (2^-24) or, on 128x128 tiles, by the matrix core, whose additions are taken as truncating
    (2^-23); the others' own seven are 2^-8 of that.  Any of the six products of terms left out would show as 2^-18 or more."""
    say("split single products", M, N, K, order)
    rng = np.random.default_rng(K)
    a, b = np.zeros((M, K), np.float32), np.zeros((K, N), np.float32)
    a[np.arange(M), rng.integers(0, K, M)] = rng.uniform(1, 2, M) * rng.choice([-1, 1], M)
    b[rng.integers(0, K, N), np.arange(N)] = rng.uniform(1, 2, N)
    for x, y in ((a, rng.uniform(1, 2, (K, N)).astype(np.float32)), (rng.uniform(1, 2, (M, K)).astype(np.float32), b)):
        got, want = product(hip, x, y, order), x.astype(np.float64) @ y.astype(np.float64)
        err = np.abs(got - want) / np.abs(want) * 2.0 ** 24
        assert (err <= 3 + 7 / 64).all(), float(err.max())
