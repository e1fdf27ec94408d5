"""fp32 products with few tiles, in one launch of 32x32 tiles whose waves share K (or, past the longest K of that, a range of it): edges of tiles, steps and strips in every storage order
and form, and the inputs that bf16 terms cannot hold."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say

pytestmark = pytest.mark.gpu


def padded(x, pad):                                           # the columns past the matrix hold NaN: read or written, they show
    out = np.full((x.shape[0], x.shape[1] + pad), np.nan, np.float32)
    out[:, :x.shape[1]] = x
    return out


def product(hip, a, b, order, alpha=1.0, beta=0.0, c=None, bias=None, act=0, pads=(3, 1, 5)):
    sa, sb = padded(a.T if order[0] == "t" else a, pads[0]), padded(b.T if order[1] == "t" else b, pads[1])
    M, N, K = a.shape[0], b.shape[1], a.shape[1]
    da, db, dc = hip.array(sa), hip.array(sb), hip.array(padded(np.zeros((M, N), np.float32) if c is None else c, pads[2]))
    dbias = None if bias is None else hip.array(bias)
    hip.check(hip.L.axhip_sgemm(int(order[0] == "t"), int(order[1] == "t"), M, N, K, alpha, da.ptr, sa.shape[1], db.ptr, sb.shape[1], beta, dc.ptr,
                                N + pads[2], None if bias is None else dbias.ptr, act))
    assert ("_ranges32x3" if in_ranges(M, N, K) else "_strips32") in hip.last_kernel(), hip.last_kernel()
    full = dc.numpy()
    assert np.isnan(full[:, N:]).all()
    return full[:, :N]


def tiles(M, N):
    return ((M + 31) // 32) * ((N + 31) // 32)


def in_ranges(M, N, K):
    """A longer K on few tiles: ranges of it in workgroups of their own (test_gpu_strips_ranges.py)."""
    return K > 760 and tiles(M, N) <= 64 or K > 960 and tiles(M, N) <= 100


def most(order, M, N):
    """The largest K that the strips take off the 16-byte grid (256 CUs)."""
    if tiles(M, N) > 256:
        return 0 if order == "nt" else 640 if tiles(M, N) <= 341 else 800
    if tiles(M, N) >= 128:
        return 1088 if order == "nt" else 1024 if M < 96 else 1536
    return 760 if tiles(M, N) <= 64 else 864 if order == "nt" else 960 if tiles(M, N) <= 100 else 1024


FORMS = [(order, M, N, K) for order in ("nn", "nt", "tn") for M, N in [(17, 1), (31, 33), (32, 32), (65, 95), (100, 10), (260, 1000), (250, 2020)]
         for K in (1, 2, 15, 16, 17, 31, 32, 47, 63, 121, 128, 129, 143, 144, 145, 176, 177, 255, 256, 257, 500, 640, 641, 760, 799) if K < 64 or K <= most(order, M, N)]


# K u sum |a||b| holds with room; with terms the left-out ones add at most 2^-24 of each product
@pytest.mark.parametrize("order,M,N,K", FORMS)
def test_every_form(hip, M, N, K, order):
    say("strips", M, N, K, order)
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    bias, c = rng.normal(0, 1, N).astype(np.float32), rng.uniform(-1, 1, (M, N)).astype(np.float32)
    exact, size = a.astype(np.float64) @ b.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    got = product(hip, a, b, order, 0.5, 2.0, c, bias, 1)
    want, size = np.maximum(0.5 * exact + 2.0 * c + bias, 0), 0.5 * size + 2.0 * np.abs(c) + np.abs(bias)
    assert (np.abs(got - want) <= BOUND_FP32 * size).all(), float((np.abs(got - want) / size).max())
    assert np.array_equal(product(hip, a, b, order, 0.5, 2.0, c, bias, 1), got)


@pytest.mark.parametrize("order,M,N,K", [(o, M, N, K) for o in ("nn", "nt", "tn") for M, N, K in [(64, 64, 128), (256, 768, 256), (128, 1024, 784),
    (1024, 96, 640), (192, 2048, 512), (20, 36, 32), (36, 1000, 44), (100, 2048, 60), (64, 64, 64), (96, 260, 100), (192, 2048, 112), (68, 100, 116), (160, 96, 132),
    (32, 1024, 340), (128, 672, 328), (160, 20, 572)] if K < 113 or K <= most(o, M, N)])
def test_on_the_grid(hip, M, N, K, order):
    """Rows on the 16-byte grid, K off and on the 32 grid; error no larger than fp32 instructions leave (2^-24 a product and sqrt(K) roundings)."""
    say("strips on the grid", M, N, K, order)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.normal(0, 1, (M, K)).astype(np.float32), rng.normal(0, 1, (K, N)).astype(np.float32)
    got = product(hip, a, b, order, pads=(0, 0, 0))
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.linalg.norm(got - want) <= 2.0 ** -24 * (1 + np.sqrt(K) / 4) * np.linalg.norm(want)


@pytest.mark.parametrize("order,M,N,K", [("nn", 100, 10, 1024), ("tn", 97, 31, 1000), ("nn", 97, 250, 1023), ("nt", 250, 100, 863), ("tn", 96, 257, 1024),
                                         ("nn", 100, 10, 760), ("tn", 97, 31, 757), ("nn", 97, 250, 759), ("nt", 250, 100, 760), ("nt", 250, 257, 863), ("nn", 250, 257, 960),
                                         ("tn", 250, 257, 959), ("tn", 330, 300, 1024), ("nt", 500, 255, 1088), ("nn", 256, 1000, 1536), ("tn", 510, 500, 1535)])
def test_longer_k(hip, order, M, N, K):
    say("strips of a longer K", M, N, K, order)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.normal(0, 1, (M, K)).astype(np.float32), rng.normal(0, 1, (K, N)).astype(np.float32)
    got = product(hip, a, b, order, 0.5, pads=(0, 0, 0)) * 2
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.linalg.norm(got - want) <= 2.0 ** -24 * (1 + np.sqrt(K) / 4) * np.linalg.norm(want)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - want) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
@pytest.mark.parametrize("K", [20, 60, 300])
def test_non_finite(hip, K, order):
    """Infinities and NaNs reach the rows and columns that hold them and no others; magnitudes up to the largest float come out."""
    say("strips non-finite", K, order)
    rng = np.random.default_rng(K)
    M, N = 70, 100
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    a[3, K - 1], a[40, 0], b[K // 2, 90], a[66, 5] = np.inf, np.nan, -np.inf, np.float32(3e38)
    b[5, :] = np.float32(2.0 ** -20)
    b[K - 1, 7] = 0
    got = product(hip, a, b, order)
    with np.errstate(invalid="ignore", over="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    fine = np.isfinite(want)
    a[3, K - 1] = a[40, 0] = b[K // 2, 90] = 0
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got[fine] - want[fine]) <= BOUND_FP32 * size[fine]).all()


@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
@pytest.mark.parametrize("K", [1, 2, 10, 15, 16, 17, 20, 31, 130, 300])
def test_infinities_at_the_end_of_k(hip, K, order):
    """The last k is what a step of 16 that hangs over K is filled with: an infinity there, in either operand, counts once."""
    say("strips, infinities in the last k", K, order)
    rng = np.random.default_rng(K)
    M, N = 70, 100
    a, b = rng.uniform(0.5, 1, (M, K)).astype(np.float32), rng.uniform(0.5, 1, (K, N)).astype(np.float32)
    b[K - 1, 90], b[K - 1, 3], b[0, 64], a[41, K - 1], a[66, 0] = -np.inf, np.inf, np.inf, np.inf, -np.inf
    a[9, K - 1] = 0
    got = product(hip, a, b, order)
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    fine = np.isfinite(want)
    assert fine.mean() > 0.9 and np.array_equal(got[~fine], want[~fine].astype(np.float32), equal_nan=True)
    assert (np.abs(got[fine] - want[fine]) <= BOUND_FP32 * want[fine]).all()


@pytest.mark.parametrize("scale_a,scale_b", [(2.0 ** -115, 1.0), (2.0 ** -60, 2.0 ** -60), (2.0 ** 100, 2.0 ** -40), (2.0 ** 120, 2.0 ** -20)])
def test_keeps_the_range(hip, scale_a, scale_b):
    say("strips range", scale_a, scale_b)
    rng = np.random.default_rng(9)
    a, b = (rng.uniform(-1, 1, (50, 200)) * scale_a).astype(np.float32), (rng.uniform(-1, 1, (200, 40)) * scale_b).astype(np.float32)
    got = product(hip, a, b, "nn")
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= BOUND_FP32 * size).all()


# (order, M, N, K): forms of four, eight and sixteen waves
@pytest.mark.parametrize("order,M,N,K", [("nn", 64, 64, 256), ("nt", 64, 64, 256), ("tn", 64, 64, 256), ("tn", 65, 97, 600), ("nn", 200, 100, 760), ("nn", 200, 100, 800),
                                         ("nn", 192, 2048, 512), ("tn", 192, 2048, 512)])
@pytest.mark.parametrize("power", [69, 71, 73, 75, 77, 79])
def test_sums_of_one_sign_past_the_terms(hip, order, M, N, K, power):
    """Strips whose own sums the terms hold (below 2^80) while their total is above it."""
    say("strips, sums of one sign", M, N, K, order, power)
    rng = np.random.default_rng(M + K + power)
    a, b = (rng.uniform(0.5, 1, (M, K)) * 2.0 ** 37).astype(np.float32), (rng.uniform(0.5, 1, (K, N)) * 2.0 ** (power - 37)).astype(np.float32)
    got, want = product(hip, a, b, order, pads=(0, 0, 0)), a.astype(np.float64) @ b.astype(np.float64)
    assert (np.abs(got - want) <= BOUND_FP32 * want).all()


def test_outer_products_are_rounded_once(hip):
    """K = 1 on fp32 instructions: the product itself."""
    say("strips outer")
    rng = np.random.default_rng(4)
    u, v = rng.normal(0, 1, (90, 1)).astype(np.float32), rng.normal(0, 1, (1, 300)).astype(np.float32)
    for order in ("nn", "nt", "tn"):
        assert np.array_equal(product(hip, u, v, order), u * v)


@pytest.mark.parametrize("order,M,N", [("nn", 50, 10), ("nn", 101, 99), ("nn", 250, 257), ("nt", 250, 257), ("tn", 330, 300), ("nn", 130, 1002), ("nn", 70, 1602), ("nn", 330, 990), ("tn", 351, 991), ("nt", 101, 99), ("nt", 130, 1002), ("tn", 101, 99),
                                       ("tn", 130, 1002), ("nn", 200, 2002)])
def test_where_k_ends(hip, order, M, N):
    """The last K that the strips take and the next one, which takes another route."""
    K = most(order, M, N)
    rng = np.random.default_rng(K)
    for k in (K, K + 1):
        say("strips, limit of K", order, M, N, k)
        a, b = rng.uniform(-1, 1, (M, k)).astype(np.float32), rng.uniform(-1, 1, (k, N)).astype(np.float32)
        da, db = hip.array(a.T if order[0] == "t" else a), hip.array(b.T if order[1] == "t" else b)
        got = hip.sgemm(da, db, transa=order[0] == "t", transb=order[1] == "t").numpy()
        assert ("_strips32" in hip.last_kernel()) == (k == K), hip.last_kernel()
        assert (np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= BOUND_FP32 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))).all()


@pytest.mark.parametrize("order,M,N,K", [(o, 255, 1021, K) for o in ("nn", "nt", "tn") for K in (121, 128, 150, 176, 177)] +
                         [(o, 321, 865, K) for o in ("nn", "tn") for K in (401, 600)])
def test_error_is_that_of_the_staged_tiles_or_less(hip, monkeypatch, order, M, N, K):
    """No larger than what the staged tiles in terms leave on the same operands, which the strips stand before; 1 % for the luck of the draw: over a quarter of a
    million sums whose errors are independent a norm is known to some 0.15 %."""
    say("strips, error", order, M, N, K)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    strips = np.linalg.norm(product(hip, a, b, order) - want)
    monkeypatch.setenv("AX_HIP_F32_NO_STRIPS", "1")
    assert hip.L.axhip_tuning_reload() == 1
    try:
        da, db = hip.array(a.T if order[0] == "t" else a), hip.array(b.T if order[1] == "t" else b)
        staged = np.linalg.norm(hip.sgemm(da, db, transa=order[0] == "t", transb=order[1] == "t").numpy() - want)
        assert hip.last_kernel().endswith("x3_staged") or hip.last_kernel() == "sgemm_splitk_x3"
    finally:
        monkeypatch.delenv("AX_HIP_F32_NO_STRIPS")
        assert hip.L.axhip_tuning_reload() == 0
    assert strips <= 1.01 * staged, (strips, staged)
