"""Batches of A B^T with a short K in bf16 terms against fp64: edges of row blocks and of the 256 columns, padded rows, every K; and the
inputs that the terms cannot hold, which the kernel computes with fp32 instructions instead."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say

pytestmark = pytest.mark.gpu


def product(hip, a, b, alpha, pad=0):
    """alpha * a b^T on operands and a result whose rows are `pad` floats longer than the matrices."""
    Bn, M, K = a.shape
    N = b.shape[1]
    fa, fb = np.full((Bn, M, K + pad), 1e30, np.float32), np.full((Bn, N, K + pad), -1e30, np.float32)
    fa[:, :, :K], fb[:, :, :K] = a, b
    da, db, c = hip.array(fa), hip.array(fb), hip.array(np.full((Bn, M, N + pad), 7.0, np.float32))
    hip.check(hip.L.axhip_sgemm_strided_batched(0, 1, M, N, K, alpha, da.ptr, K + pad, M * (K + pad), db.ptr, K + pad, N * (K + pad), 0.0, c.ptr,
                                                N + pad, M * (N + pad), Bn))
    assert hip.last_kernel() == "sgemm_nt_cols256x3"
    got = c.numpy()
    assert (got[:, :, N:] == 7.0).all()
    return got[:, :, :N]


def check(got, a, b, alpha, floor=0.0):
    bt = b.astype(np.float64).transpose(0, 2, 1)
    want, size = alpha * (a.astype(np.float64) @ bt), abs(alpha) * (np.abs(a).astype(np.float64) @ np.abs(bt))
    assert (np.abs(got - want) <= BOUND_FP32 * size + floor).all()


@pytest.mark.parametrize("Bn,M,N,K,pad", [(512, 256, 256, 64, 0), (260, 129, 141, 64, 0), (257, 128, 256 - 31, 32, 4), (131, 191, 333, 96, 0), (130, 193, 321, 128, 8),
                                          (90, 321, 515, 64, 12), (256, 160, 130, 96, 0), (280, 288, 512, 128, 4), (140, 161, 511, 32, 0)])
def test_edges(hip, Bn, M, N, K, pad):
    say("nt terms", Bn, M, N, K, pad)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (Bn, M, K)).astype(np.float32), rng.uniform(-1, 1, (Bn, N, K)).astype(np.float32)
    check(product(hip, a, b, 0.25, pad), a, b, 0.25)


@pytest.mark.parametrize("K", [32, 64, 96, 128])
@pytest.mark.parametrize("scale_a,scale_b", [(2.0 ** -115, 1.0), (2.0 ** -100, 2.0 ** 90), (2.0 ** -60, 2.0 ** -50), (2.0 ** 120, 2.0 ** -20), (1.0, 2.0 ** -118)])
def test_keeps_the_range(hip, K, scale_a, scale_b):
    """Magnitudes whose small terms leave the normal range, and large ones: relative accuracy as in the middle of it."""
    say("nt terms range", K, scale_a, scale_b)
    rng = np.random.default_rng(K)
    a, b = (rng.uniform(-1, 1, (260, 140, K)) * scale_a).astype(np.float32), (rng.uniform(-1, 1, (260, 170, K)) * scale_b).astype(np.float32)
    a[:, 3] = 0
    check(product(hip, a, b, 1.0), a, b, 1.0, K * 2.0 ** -149)


@pytest.mark.parametrize("K", [32, 64, 96, 128])
def test_non_finite(hip, K):
    """Infinities, NaNs and values that round past the largest bf16 give what fp32 arithmetic gives; the rest is untouched."""
    say("nt terms non-finite", K)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (260, 140, K)).astype(np.float32), rng.uniform(-1, 1, (260, 170, K)).astype(np.float32)
    top = np.finfo(np.float32).max
    a[1, 7, 3] = np.inf
    b[1, :, 3] = 0.5
    b[2, 149, K - 1] = np.nan
    a[3, 139], a[3, 139, 5], b[3, 2, 5] = 0, top, 1.0
    got = product(hip, a, b, 1.0)
    assert np.isposinf(got[1, 7]).all() and np.isnan(got[2, :, 149]).all() and got[3, 139, 2] == top
    got[1, 7], a[1, 7] = 0, 0
    got[2, :, 149], b[2, 149] = 0, 0
    check(got, a, b, 1.0)


@pytest.mark.parametrize("K", [32, 64, 96, 128])
@pytest.mark.parametrize("scale_a,scale_b", [(2.0 ** -60, 2.0 ** -60), (2.0 ** -20, 2.0 ** -110), (2.0 ** -127, 2.0 ** 10), (2.0 ** 50, 2.0 ** 40)])
def test_small_results(hip, K, scale_a, scale_b):
    """Products next to the smallest normal value (and above 2^80): relative accuracy as in the middle of the range, up to fp32's own
    smallest step."""
    say("nt terms small results", K, scale_a, scale_b)
    rng = np.random.default_rng(K)
    a, b = (rng.uniform(-1, 1, (260, 140, K)) * scale_a).astype(np.float32), (rng.uniform(-1, 1, (260, 170, K)) * scale_b).astype(np.float32)
    check(product(hip, a, b, 1.0), a, b, 1.0, 4 * 2.0 ** -149)


@pytest.mark.parametrize("K", [32, 64, 96, 128])
def test_small_values_among_others(hip, K):
    """Values down to fp32's smallest beside ordinary ones are no reason for the fp32 pass: every sum comes out as with zeros in their
    place, but for the few whose rounding is a tie."""
    say("nt terms small values", K)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (260, 140, K)).astype(np.float32), rng.uniform(-1, 1, (260, 170, K)).astype(np.float32)
    for x in (a, b):
        x[rng.random(x.shape) < 0.02] = 0
    clean = product(hip, a, b, 1.0)
    for x in (a, b):
        x[x == 0] = np.ldexp(1.0, rng.integers(-149, -100, (x == 0).sum())).astype(np.float32)
    assert (product(hip, a, b, 1.0) != clean).mean() < 0.01


@pytest.mark.parametrize("K", [32, 64, 96, 128])
def test_single_products(hip, K):
    """Sums with one product that is not zero, of operands with all 24 bits: the left-out terms are at most 2^-24 of it, the sum of the
    large term and of the others is rounded once to 2^-24, the others' own five roundings are 2^-8 of that.  Any of the six products of
    terms left out would show as 2^-18 or more in some of them."""
    say("nt terms single products", K)
    rng = np.random.default_rng(K)
    a, b = np.zeros((260, 140, K), np.float32), rng.uniform(1, 2, (260, 170, K)).astype(np.float32)
    np.put_along_axis(a, rng.integers(0, K, (260, 140, 1)), rng.uniform(1, 2, (260, 140, 1)).astype(np.float32), 2)
    got, want = product(hip, a, b, 1.0), a.astype(np.float64) @ b.astype(np.float64).transpose(0, 2, 1)
    err = np.abs(got - want) / want * 2.0 ** 24
    assert (err <= 2 + 5 / 128).all(), float(err.max())
