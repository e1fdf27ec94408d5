"""fp32 products with few tiles and a long K in one launch of ranges of it: the limits of every form, tiles that hang over, a K that ends inside a step, calls in
a row on the same counters, and the inputs that bf16 terms cannot hold."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say
from test_gpu_planes import product

pytestmark = pytest.mark.gpu

#            M, N, K, whether ranges are taken (or in which orders)
SHAPES = [(17, 1, 761, True), (17, 1, 760, False), (100, 10, 960, True), (33, 33, 961, True), (100, 10, 1300, True), (100, 10, 1301, True), (100, 10, 4096, True),
          (64, 512, 4607, True), (100, 10, 4609, False), (65, 330, 761, True), (200, 255, 1024, True), (64, 1000, 1025, True), (64, 1024, 2600, True),
          (64, 1024, 2601, False), (320, 320, 961, True), (320, 320, 1280, True), (320, 320, 1281, "nn tn"), (320, 320, 1600, "nn tn"), (96, 1056, 1601, "tn"),
          (96, 1056, 1950, "tn"), (320, 320, 2601, False), (330, 330, 1700, False)]


@pytest.mark.parametrize("M,N,K,taken", SHAPES)
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_ranges(hip, M, N, K, taken, order):
    say("ranges", M, N, K, order)
    rng = np.random.default_rng(M + N + K)
    a, b, c = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    bias = rng.normal(0, 1, N).astype(np.float32)
    exact, size = a.astype(np.float64) @ b.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    for pads, off in (((3, 1, 5), 1), ((0, 0, 0), 0)):
        got = product(hip, a, b, order, c=c, alpha=0.5, beta=2.0, bias=bias, act=1, pads=pads, off=off)
        assert (hip.last_kernel() == f"sgemm_{order}_ranges32x3") == (taken is True or taken and order in taken), hip.last_kernel()
        want = np.maximum(0.5 * exact + 2.0 * c + bias, 0)
        assert (np.abs(got - want) <= BOUND_FP32 * (0.5 * size + 2.0 * np.abs(c) + np.abs(bias))).all()
        assert np.array_equal(product(hip, a, b, order, c=c, alpha=0.5, beta=2.0, bias=bias, act=1, pads=pads, off=off), got)


def test_calls_in_a_row(hip):
    """The counters are at zero after every call: products of different tile counts one after the other, unsynchronised, as a step of training makes them."""
    say("ranges in a row")
    rng = np.random.default_rng(8)
    work = []
    for M, N, K in [(100, 10, 4096), (64, 1024, 1500), (17, 1, 777), (320, 320, 1200), (100, 10, 1024)] * 4:
        a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
        work.append((a, b, hip.array(a), hip.array(b), hip.array(np.full((M, N), np.nan, np.float32))))
    for a, b, da, db, dc in work:
        M, K, N = a.shape[0], a.shape[1], b.shape[1]
        hip.check(hip.L.axhip_sgemm(0, 0, M, N, K, 1.0, da.ptr, K, db.ptr, N, 0.0, dc.ptr, N, None, 0))
        assert "ranges" in hip.last_kernel()
    for a, b, da, db, dc in work:
        size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
        assert (np.abs(dc.numpy() - a.astype(np.float64) @ b.astype(np.float64)) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("M,N,K", [(100, 10, 4095), (65, 330, 800), (320, 300, 1001)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_ranges_non_finite(hip, M, N, K, order):
    """In the first, a middle and the last range, and sums of one sign next to the largest float, whose parts fit the terms and whose sum does not."""
    say("ranges non-finite", M, N, K, order)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    a[1, 7], a[2, K // 2], a[2, K - 1], a[4, K - 1] = np.inf, np.inf, -np.inf, np.nan
    b[7, ::3] = 0
    a[6] *= np.float32(2.0 ** 120)
    a[8] = np.abs(a[8]) * np.float32(2.0 ** 70)
    got = product(hip, a, b, order)
    assert "ranges" in hip.last_kernel()
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.array_equal(np.sign(got[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))
    rows = np.setdiff1d(np.arange(M), [1, 2, 4])
    size = np.abs(a[rows]).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got[rows] - ref[rows]) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("M,N,K", [(100, 10, 4096), (64, 300, 1000), (300, 320, 1300)])
def test_ranges_large_sums(hip, M, N, K):
    """Operands whose products add up to just below the largest float: every range is finite in itself, and so is the sum."""
    say("ranges, large sums", M, N, K)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(1, 2, (M, K)).astype(np.float32) * np.float32(2.0 ** 60), rng.uniform(1, 2, (K, N)).astype(np.float32) * np.float32(2.0 ** 53)
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert want.max() < np.finfo(np.float32).max
    got = product(hip, a, b, "nn")
    assert "ranges" in hip.last_kernel() and (np.abs(got - want) <= BOUND_FP32 * want).all()


@pytest.mark.parametrize("M,N,K", [(100, 12, 4096), (64, 300, 1024), (300, 320, 1264), (50, 10, 777)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_ranges_single_products(hip, M, N, K, order):
    """Sums with one product that is not zero, of operands with all 24 bits, in any of the ranges: the left-out terms are at most 2^-24 of it, the matrix core's own
    addition truncates (2^-23), the others' are 2^-8 of that.  Any of the six products of terms left out would show as 2^-18 or more."""
    say("ranges single products", M, N, K, order)
    rng = np.random.default_rng(K)
    a = np.zeros((M, K), np.float32)
    a[np.arange(M), rng.integers(0, K, M)] = rng.uniform(1, 2, M) * rng.choice([-1, 1], M)
    b = rng.uniform(1, 2, (K, N)).astype(np.float32)
    got, want = product(hip, a, b, order), a.astype(np.float64) @ b.astype(np.float64)
    assert hip.last_kernel() == f"sgemm_{order}_ranges32x3"
    err = np.abs(got - want) / np.abs(want) * 2.0 ** 24
    assert (err <= 3 + 7 / 64).all(), float(err.max())
