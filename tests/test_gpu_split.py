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
    assert "x3_staged" in kernel or kernel == "sgemm_splitk", kernel
    return c.numpy()


# the fp32 error bound K u sum |a||b| (u = 2^-24) holds with room for sums of random signs, see test_gpu_staged; the left-out terms
# add at most 2^-24 of each product
@pytest.mark.parametrize("M,N,K", [(17, 33, 64), (65, 129, 65), (129, 65, 95), (161, 516, 256), (1152, 1152, 1152), (1153, 772, 2052), (644, 4096, 1024),
                                   (2049, 1028, 260), (200, 128, 4096), (1000, 1004, 1001)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_split_fp32(hip, M, N, K, order):
    say("split", M, N, K, order)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    if (M % 4 or N % 4 or K % 4) == 0 and order == "tn" and M % 64:
        M = M // 4 * 4
        a = a[:M]
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


SHAPES = [(70, 90, 101), (200, 132, 1029), (1152, 1152, 1152)]      # one tile, ranges of K, whole tiles


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
