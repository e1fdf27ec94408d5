"""Batches of A B with a narrow B on the kernels whose waves own 32 rows and all columns: edges of row blocks, column blocks and units of K,
rows off the 16-byte grid, and the inputs that bf16 terms cannot hold."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say

pytestmark = pytest.mark.gpu
KERNELS = ("sgemm_nn_rows128x3", "sgemm_nn_rows256x3")


def products(hip, a, b, alpha=1.0, pads=(0, 0, 0)):
    """alpha a @ b through buffers whose rows are longer by `pads` floats of NaN and whose operands begin `pads[0]` floats in."""
    (H, M, K), N = a.shape, b.shape[2]
    bufs = []
    for x, pad in ((a, pads[0]), (b, pads[1])):
        rows = np.full((H, x.shape[1], x.shape[2] + pad), np.nan, np.float32)
        rows[:, :, :x.shape[2]] = x
        bufs.append(hip.array(np.concatenate([np.full(pads[0], np.nan, np.float32), rows.ravel()])))
    dc = hip.array(np.full((H, M, N + pads[2]), np.nan, np.float32))
    hip.check(hip.L.axhip_sgemm_strided_batched(0, 0, M, N, K, alpha, bufs[0].ptr + 4 * pads[0], K + pads[0], M * (K + pads[0]),
                                                bufs[1].ptr + 4 * pads[0], N + pads[1], K * (N + pads[1]), 0.0, dc.ptr, N + pads[2],
                                                M * (N + pads[2]), H))
    assert hip.last_kernel() in KERNELS, hip.last_kernel()
    full = dc.numpy()
    assert np.isnan(full[:, :, N:]).all()
    return full[:, :, :N], hip.last_kernel()


KS = (64, 65, 95, 96, 128, 159, 256, 291)
# up to 32 columns, any alignment; more of them on the 16-byte grid (from 96 on with K >= 256 whole tiles only); off it where the staged tiles would be 128x128
FORMS = [(-(-400 // -(-M // 128)), M, N, K, pads) for pads in [(0, 0, 0), (1, 3, 5)] for M, N in [(96, 1), (128, 17), (129, 32), (300, 31)] for K in KS]
FORMS += [(-(-400 // -(-M // 128)), M, N, K, pads) for pads in [(0, 0, 0), (4, 8, 4)] for M, N in [(128, 80), (257, 96), (256, 128), (385, 72)] for K in KS
          if K % 4 == 0 and not (N > 96 and K < 256) and not (N >= 96 and K >= 256 and M % 128)]
FORMS += [(134, 338, 90, 146, (1, 3, 5)), (206, 345, 76, 133, (0, 0, 0)), (62, 966, 76, 210, (1, 3, 5)), (108, 458, 92, 286, (0, 0, 0))]


# K u sum |a||b| holds with room; with terms the left-out ones add at most 2^-24 of each product
@pytest.mark.parametrize("H,M,N,K,pads", FORMS)
def test_every_form(hip, H, M, N, K, pads):
    say("narrow batches", H, M, N, K, pads)
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = rng.uniform(-1, 1, (H, M, K)).astype(np.float32), rng.uniform(-1, 1, (H, K, N)).astype(np.float32)
    got, _ = products(hip, a, b, 0.5, pads)
    for h in {0, H // 2, H - 1}:
        want, size = 0.5 * (a[h].astype(np.float64) @ b[h].astype(np.float64)), 0.5 * (np.abs(a[h]).astype(np.float64) @ np.abs(b[h]).astype(np.float64))
        assert (np.abs(got[h] - want) <= BOUND_FP32 * size).all(), float((np.abs(got[h] - want) / size).max())
    sums = got.astype(np.float64).sum(axis=2) - 0.5 * np.matmul(a.astype(np.float64), b.astype(np.float64).sum(axis=2, keepdims=True))[:, :, 0]
    size = 0.5 * np.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64).sum(axis=2, keepdims=True))[:, :, 0]
    assert (np.abs(sums) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("H,M,N,K,taken", [
    (242, 175, 94, 134, False), (288, 227, 74, 199, False), (134, 338, 90, 146, True),     # off the grid, before 64x64 tiles in terms and before 128x128
    (146, 144, 4, 144, False), (200, 144, 4, 144, True), (192, 128, 20, 132, True), (191, 128, 20, 132, False),   # rows that exist, workgroups a CU
    (191, 100, 30, 66, False), (192, 100, 30, 66, True)])                                  # a K of three units, off the grid
def test_where_it_runs(hip, H, M, N, K, taken):
    """Both sides of the limits of the rule (256 CUs)."""
    say("narrow batches, limits", H, M, N, K)
    rng = np.random.default_rng(H + M + N)
    a, b = rng.normal(0, 1, (H, M, K)).astype(np.float32), rng.normal(0, 1, (H, K, N)).astype(np.float32)
    got = hip.sgemm_batched(hip.array(a), hip.array(b)).numpy()
    assert (hip.last_kernel() in KERNELS) == taken, hip.last_kernel()
    for h in (0, H - 1):
        want, size = a[h].astype(np.float64) @ b[h].astype(np.float64), np.abs(a[h]).astype(np.float64) @ np.abs(b[h]).astype(np.float64)
        assert (np.abs(got[h] - want) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("H,M,N,name", [(256, 128, 24, KERNELS[0]), (420, 128, 80, KERNELS[0]), (256, 250, 80, KERNELS[1])])
def test_four_waves_or_eight(hip, H, M, N, name):
    """The error is no larger than fp32 instructions leave (2^-24 a product and sqrt(K) roundings)."""
    say("narrow batches", H, M, N)
    K = 256
    rng = np.random.default_rng(H + M + N)
    a, b = rng.normal(0, 1, (H, M, K)).astype(np.float32), rng.normal(0, 1, (H, K, N)).astype(np.float32)
    got, kernel = products(hip, a, b)
    assert kernel == name
    want = np.matmul(a[::64].astype(np.float64), b[::64].astype(np.float64))
    assert np.linalg.norm(got[::64] - want) <= 2.0 ** -24 * (1 + np.sqrt(K) / 4) * np.linalg.norm(want)


@pytest.mark.parametrize("N,K", [(20, 132), (31, 131), (80, 200), (128, 256)])
def test_non_finite(hip, N, K):
    """Infinities and NaNs reach the rows and columns that hold them and no others; magnitudes up to the largest float come out."""
    say("narrow batches, non-finite", N, K)
    H, M = 400, 128
    rng = np.random.default_rng(K)
    a, b = rng.uniform(-1, 1, (H, M, K)).astype(np.float32), rng.uniform(-1, 1, (H, K, N)).astype(np.float32)
    a[1, 5, 3], a[1, 40, K - 1], b[2, 7, N - 1], b[2, K - 1, 3] = np.inf, np.nan, -np.inf, np.nan
    a[3] *= np.float32(2e36)
    b[4] *= np.float32(3e38)
    a[4] *= np.float32(2.0 ** -20)
    got, _ = products(hip, a, b)
    for h in range(6):
        with np.errstate(invalid="ignore", over="ignore"):
            want = a[h].astype(np.float64) @ b[h].astype(np.float64)
            size = np.abs(a[h]).astype(np.float64) @ np.abs(b[h]).astype(np.float64)
        held = np.isfinite(want) & (size < 3e38)
        assert held.mean() >= 0.9
        assert (np.abs(got[h][held] - want[held]) <= BOUND_FP32 * size[held]).all()
        assert np.array_equal(np.isnan(got[h]), np.isnan(want))
        inf = np.isinf(want)
        assert np.array_equal(got[h][inf], want[inf].astype(np.float32))
