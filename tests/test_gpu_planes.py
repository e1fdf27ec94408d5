"""Products whose operands are cut into planes of bf16 terms first, against fp64: both tiles, whole and hanging over by a row, a column and a k, one k past a
block and one short of it, every storage order, padded pitches and unaligned operands; and the inputs that the terms cannot hold."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say

pytestmark = pytest.mark.gpu

LARGE, SMALL = "planes256x128x3", "planes128x64x3"


def padded(x, pad, off=0):
    """x in rows of a longer pitch, `off` elements into its array; the rest holds NaN: read or written, it shows."""
    full = np.full(off + x.shape[0] * (x.shape[1] + pad), np.nan, np.float32)
    full[off:].reshape(x.shape[0], -1)[:, :x.shape[1]] = x
    return full


def product(hip, a, b, order, c=None, alpha=1.0, beta=0.0, bias=None, act=0, pads=(0, 0, 0), off=0):
    M, K, N = a.shape[0], a.shape[1], b.shape[1]
    sa, sb = a.T if order[0] == "t" else a, b.T if order[1] == "t" else b
    da, db = hip.array(padded(sa, pads[0], off)), hip.array(padded(sb, pads[1], off))
    dc = hip.array(padded(np.full((M, N), np.nan, np.float32) if c is None else c, pads[2], off))
    dbias = hip.array(bias) if bias is not None else None
    hip.check(hip.L.axhip_sgemm(int(order[0] == "t"), int(order[1] == "t"), M, N, K, alpha, da.ptr + 4 * off, sa.shape[1] + pads[0], db.ptr + 4 * off,
                                sb.shape[1] + pads[1], beta, dc.ptr + 4 * off, N + pads[2], dbias.ptr if dbias else None, act))
    full = dc.numpy()
    assert np.isnan(full[:off]).all() and np.isnan(full[off:].reshape(M, -1)[:, N:]).all()
    return full[off:].reshape(M, -1)[:, :N]


# the fp32 error bound K u sum |a||b| (u = 2^-24) holds with room for sums of random signs; the left-out terms add at most 2^-24 of each product
@pytest.mark.parametrize("M,N,K,tile", [(2048, 4096, 512, LARGE), (1793, 3969, 545, LARGE), (2111, 3001, 607, LARGE), (2000, 3072, 512, SMALL),
                                        (1665, 3009, 545, SMALL), (1537, 3265, 513, SMALL)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_planes(hip, M, N, K, tile, order):
    say("planes", M, N, K, order)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    got = product(hip, a, b, order)
    assert hip.last_kernel() == f"sgemm_{order}_{tile}"
    want, size = a.astype(np.float64) @ b.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - want) <= BOUND_FP32 * size).all(), float((np.abs(got - want) / size).max())


@pytest.mark.parametrize("M,N,K,tile", [(1793, 3969, 545, LARGE), (1665, 3009, 545, SMALL)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_planes_write_back(hip, M, N, K, tile, order):
    """alpha, beta, bias and activation; pitches off the 16-byte grid, operands and result off it too."""
    say("planes write-back", M, N, K, order)
    rng = np.random.default_rng(M * 3 + N + K)
    a, b, c = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((M, K), (K, N), (M, N)))
    bias = rng.normal(0, 1, N).astype(np.float32)
    got = product(hip, a, b, order, c=c, alpha=0.5, beta=2.0, bias=bias, act=1, pads=(3, 1, 5), off=1)
    assert hip.last_kernel() == f"sgemm_{order}_{tile}"
    want = np.maximum(0.5 * (a.astype(np.float64) @ b.astype(np.float64)) + 2.0 * c + bias, 0)
    size = 0.5 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 2.0 * np.abs(c) + np.abs(bias)
    assert (np.abs(got - want) <= BOUND_FP32 * size).all(), float((np.abs(got - want) / size).max())


@pytest.mark.parametrize("M,N,K", [(1793, 3969, 545), (1665, 3009, 545)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_planes_single_products(hip, M, N, K, order):
    """Sums with one product that is not zero, of operands with all 24 bits: the left-out terms are at most 2^-24 of it, the matrix core's own addition
    truncates (2^-23), the others' are 2^-8 of that.  Any of the six products of terms left out would show as 2^-18 or more."""
    say("planes single products", M, N, K, order)
    rng = np.random.default_rng(K)
    a = np.zeros((M, K), np.float32)
    a[np.arange(M), rng.integers(0, K, M)] = rng.uniform(1, 2, M) * rng.choice([-1, 1], M)
    b = rng.uniform(1, 2, (K, N)).astype(np.float32)
    got, want = product(hip, a, b, order), a.astype(np.float64) @ b.astype(np.float64)
    assert "planes" in hip.last_kernel()
    err = np.abs(got - want) / np.abs(want) * 2.0 ** 24
    assert (err <= 3 + 7 / 64).all(), float(err.max())


@pytest.mark.parametrize("M,N,K", [(1793, 3969, 545), (1665, 3009, 545)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_planes_non_finite(hip, M, N, K, order):
    """Infinities, NaNs and values that round past the largest bf16 give what fp32 arithmetic gives, in the first and in the last tile and in the last k, and
    operands of 2^120 against 2^-20 are as accurate as others; rows and columns of other tiles are untouched."""
    say("planes non-finite", M, N, K, order)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    top = np.finfo(np.float32).max
    a[1, 7], a[2, 7], a[2, 30], a[4, K - 1] = np.inf, np.inf, -np.inf, np.nan
    a[5] = 0
    a[5, K - 1], b[K - 1, 2] = top, 1.0
    a[M - 1, K - 1] = -np.inf
    a[6] *= np.float32(2.0 ** 120)
    b[7, ::3] = 0
    got = product(hip, a, b, order)
    assert "planes" in hip.last_kernel()
    with np.errstate(invalid="ignore", over="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.array_equal(np.sign(got[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))
    assert got[5, 2] == top
    rows = np.setdiff1d(np.arange(M), [1, 2, 4, M - 1])
    size = np.abs(a[rows]).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got[rows] - ref[rows]) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("M,N,K", [(1793, 3969, 545), (1665, 3009, 545), (2000, 2432, 2016)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_error_is_that_of_the_staged_tiles_or_less(hip, monkeypatch, M, N, K, order):
    """No larger than what the tiles that planes stand before leave on the same operands; 1 % for the luck of the draw: over four million sums and more whose
    errors are independent a norm is known to some 0.05 %."""
    say("planes, error", M, N, K, order)
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    planes = np.linalg.norm(product(hip, a, b, order) - want)
    assert "planes" in hip.last_kernel()
    monkeypatch.setenv("AX_HIP_F32_NO_PLANES", "1")
    assert hip.L.axhip_tuning_reload() == 1
    try:
        staged = np.linalg.norm(product(hip, a, b, order) - want)
        assert hip.last_kernel().endswith("x3_staged") or hip.last_kernel() == "sgemm_splitk_x3"
    finally:
        monkeypatch.delenv("AX_HIP_F32_NO_PLANES")
        assert hip.L.axhip_tuning_reload() == 0
    assert planes <= 1.01 * staged, (planes, staged)
