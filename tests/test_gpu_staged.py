"""The register-staged tiles (products off the 16-byte grid or with K off the 32 grid: in bf16 terms from K = 64 on, on fp32 instructions
below and for batches of few columns; W8A32 at any alignment) against fp64, at the sizes where they can go wrong: one slab, a slab and one
value, ranges of K that end inside a slab, tiles that hang over by all but one row or column, every tile size, every storage order,
padded pitches and odd batch strides."""
import numpy as np
import pytest

from test_gpu_parity import BOUND_FP32, say

pytestmark = pytest.mark.gpu

# |sum in fp32 - sum in fp64| <= K u sum |a||b| for any order, u = 2^-24: BOUND_FP32 = 1e-5 covers K up to 168 for every order and,
# as sums of random signs grow with sqrt(K), the K used here by an order of magnitude


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("M,N,K", [(17, 17, 32), (33, 65, 33), (65, 129, 63), (64, 63, 64), (129, 257, 65), (41, 1113, 92), (61, 343, 551),
                                   (222, 434, 1376), (127, 11, 1023), (372, 2149, 257), (2001, 2003, 97), (17, 1, 4097), (2001, 2003, 32),
                                   (2033, 2003, 63)])
@pytest.mark.parametrize("order", ["nn", "nt", "tn"])
def test_staged_fp32(hip, M, N, K, order):
    say("staged", M, N, K, order)
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    pad_a, pad_b, pad_c = 3, 1, 5
    a = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    b = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    bias = rng.normal(0, 1, N).astype(np.float32)
    c = rng.uniform(-1, 1, (M, N)).astype(np.float32)

    def padded(x, pad):                                       # the columns past the matrix hold NaN: read or written, they show
        out = np.full((x.shape[0], x.shape[1] + pad), np.nan, np.float32)
        out[:, :x.shape[1]] = x
        return out
    sa, sb = padded(a.T if order[0] == "t" else a, pad_a), padded(b.T if order[1] == "t" else b, pad_b)
    da, db, dc, dbias = hip.array(sa), hip.array(sb), hip.array(padded(c, pad_c)), hip.array(bias)
    hip.check(hip.L.axhip_sgemm(int(order[0] == "t"), int(order[1] == "t"), M, N, K, 0.5, da.ptr, sa.shape[1], db.ptr, sb.shape[1], 2.0, dc.ptr,
                                N + pad_c, dbias.ptr, 1))
    kernel = hip.last_kernel()
    if K >= 64:
        assert kernel.endswith("x3_staged") or kernel == "sgemm_splitk_x3", kernel
    else:
        assert kernel == "sgemm_%s_%s_staged" % (order, "128x128k2" if M > 2000 else "64x64k2")
    full = dc.numpy()
    assert np.isnan(full[:, N:]).all()
    want = np.maximum(0.5 * (a.astype(np.float64) @ b.astype(np.float64)) + 2.0 * c + bias, 0)
    size = 0.5 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 2.0 * np.abs(c) + np.abs(bias)
    assert (np.abs(full[:, :N] - want) <= BOUND_FP32 * size).all(), float((np.abs(full[:, :N] - want) / size).max())


@pytest.mark.parametrize("Bn,M,N,K,transb", [(3, 103, 103, 32, 1), (9, 67, 64, 103, 0), (17, 130, 131, 33, 1), (2, 65, 33, 129, 0), (9, 700, 47, 300, 0),
                                             (16, 500, 501, 63, 1)])
def test_staged_batched(hip, Bn, M, N, K, transb):
    say("staged batched", Bn, M, N, K, transb)
    rng = np.random.default_rng(Bn + M + K)
    a = rng.uniform(-1, 1, (Bn, M, K)).astype(np.float32)
    b = rng.uniform(-1, 1, (Bn, N, K) if transb else (Bn, K, N)).astype(np.float32)
    got = hip.sgemm_batched(hip.array(a), hip.array(b), transb=bool(transb), alpha=0.25).numpy()
    assert hip.last_kernel().endswith("x3_staged" if K >= 64 and N >= 48 else "128x128k2_staged" if M == 500 else "64x64k2_staged")
    bt = b.astype(np.float64).transpose(0, 2, 1) if transb else b.astype(np.float64)
    want = 0.25 * (a.astype(np.float64) @ bt)
    size = 0.25 * (np.abs(a).astype(np.float64) @ np.abs(bt))
    assert (np.abs(got - want) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("M,N,K", [(17, 129, 64), (33, 127, 65), (9, 3, 127), (31, 2134, 1002), (65, 257, 191), (250, 1000, 2048), (129, 255, 1088),
                                   (516, 3200, 321), (834, 11009, 67), (100, 515, 2047)])
def test_staged_w8a32(hip, M, N, K):
    say("staged w8a32", M, N, K)
    rng = np.random.default_rng(M + N + K)
    a = (rng.uniform(-1, 1, (M, K)) * 10.0 ** rng.integers(-3, 4, (M, 1))).astype(np.float32)
    w = rng.integers(-128, 128, (N, K), dtype=np.int8)
    s = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    dout = hip.array(np.full((M + 1, N), np.nan, np.float32))          # a row past the output: never written
    da, dw, ds = hip.array(a), hip.array(w), hip.array(s)
    hip.check(hip.L.axhip_qgemm_w8a32(da.ptr, dw.ptr, ds.ptr, dout.ptr, M, N, K))
    kernel = hip.last_kernel()
    assert kernel.endswith("_staged") or kernel == "qgemm_w8a32_mfma_splitk", kernel
    full = dout.numpy()
    assert np.isnan(full[M]).all()
    want = (a.astype(np.float64) @ w.astype(np.float64).T) * s
    bound = BOUND_FP32 * (np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T) * s + 1e-30
    assert (np.abs(full[:M] - want) <= bound).all(), float((np.abs(full[:M] - want) / bound).max())


def test_staged_w8a32_non_finite(hip, oracle):
    """Infinities and NaNs pass through the cut into bf16 terms as through the reference's fp32 sum, a last slab included."""
    M, N, K = 41, 130, 321
    rng = np.random.default_rng(5)
    a = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    w[::3, 7] = 0
    a[1, 7], a[2, 320], a[3, 300], a[4, 0] = np.inf, -np.inf, np.nan, np.float32(3.0e38)
    a[5, 319] = np.array([0x7f800001], np.uint32).view(np.float32)[0]
    s = rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    got = hip.qgemm_w8a32(hip.array(a), hip.array(w), hip.array(s)).numpy()
    assert hip.last_kernel().endswith("_staged") or hip.last_kernel() == "qgemm_w8a32_mfma_splitk"
    with np.errstate(all="ignore"):
        ref = oracle.qgemm_w8a32(a, w, s)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    assert np.array_equal(np.sign(got[np.isinf(ref)]), np.sign(ref[np.isinf(ref)]))


@pytest.mark.parametrize("order,Bn,M,N,K,kernel", [
    ("nt", 176, 132, 131, 34, "sgemm_nt_64x64k2_staged"), ("nn", 30, 1168, 35, 32, "sgemm_nn_64x64k2_staged"), ("nt", 13, 543, 543, 32, "sgemm_nt_64x64k2_staged"),
    ("nt", 338, 294, 294, 65, "sgemm_nt_64x64x3_staged"), ("nt", 56, 447, 449, 69, "sgemm_nt_64x64x3_staged"), ("nn", 70, 800, 34, 96, "sgemm_nn_64x64k2_staged"),
    ("nn", 27, 1084, 85, 162, "sgemm_nn_128x128x3_staged")])
def test_tile_of_a_short_k(hip, order, Bn, M, N, K, kernel):
    """With a K of one to eight slabs first loads and write-back decide: 64x64 tiles, unless the large ones fill the CUs just once."""
    say("tile of a short k", order, Bn, M, N, K)
    rng = np.random.default_rng(Bn + M + N + K)
    a = rng.uniform(-1, 1, (Bn, M, K)).astype(np.float32)
    b = rng.uniform(-1, 1, (Bn, N, K) if order == "nt" else (Bn, K, N)).astype(np.float32)
    got = hip.sgemm_batched(hip.array(a), hip.array(b), transb=order == "nt", alpha=0.25).numpy()
    assert hip.last_kernel() == kernel
    for h in (0, Bn // 2, Bn - 1):
        bt = b[h].astype(np.float64).T if order == "nt" else b[h].astype(np.float64)
        want, size = 0.25 * (a[h].astype(np.float64) @ bt), 0.25 * (np.abs(a[h]).astype(np.float64) @ np.abs(bt))
        assert (np.abs(got[h] - want) <= BOUND_FP32 * size).all()


@pytest.mark.usefixtures("no_strips")
@pytest.mark.parametrize("order,M,N,K,kernel", [
    ("nn", 17, 576, 340, "sgemm_32x64k2_dma_edge"), ("nt", 160, 20, 472, "sgemm_32x64k2_dma_edge"), ("nt", 96, 3296, 392, "sgemm_32x64k2_dma_edge"),
    ("tn", 128, 672, 328, "sgemm_64x64k2_dma_edge"), ("nn", 249, 512, 376, "sgemm_nn_64x64x3_staged"), ("tn", 160, 32, 440, "sgemm_splitk_x3"),
    ("nn", 32, 1024, 540, "sgemm_splitk_x3"), ("nn", 685, 32, 960, "sgemm_splitk"),
    ("nt", 3100, 3004, 64, "sgemm_64x64_dma_edge"), ("nn", 4000, 2500, 32, "sgemm_64x64_dma_edge")])
def test_ranges_on_the_grid(hip, order, M, N, K, kernel):
    """Rows on the 16-byte grid with K off the 32 grid: ranges of K on the staged tiles only where K is long enough for what the
    direct-to-LDS tiles do in one launch.  A short K off the tile grid is one launch of theirs, however large the product."""
    say("ranges on the grid", order, M, N, K)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    da, db = hip.array(np.ascontiguousarray(a.T) if order[0] == "t" else a), hip.array(np.ascontiguousarray(b.T) if order[1] == "t" else b)
    got = hip.sgemm(da, db, transa=order[0] == "t", transb=order[1] == "t").numpy()
    assert hip.last_kernel() == kernel
    want, size = a.astype(np.float64) @ b.astype(np.float64), np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    assert (np.abs(got - want) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("M,N,K,transb", [(928, 43, 928, 0), (423, 41, 1023, 1), (361, 33, 777, 0)])
def test_batch_of_one_is_cut_like_a_product(hip, M, N, K, transb):
    say("batch of one", M, N, K, transb)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (1, M, K)).astype(np.float32), rng.uniform(-1, 1, (1, N, K) if transb else (1, K, N)).astype(np.float32)
    got = hip.sgemm_batched(hip.array(a), hip.array(b), transb=bool(transb), alpha=0.25).numpy()[0]
    assert hip.last_kernel() == "sgemm_splitk"
    bt = b[0].astype(np.float64).T if transb else b[0].astype(np.float64)
    want, size = 0.25 * (a[0].astype(np.float64) @ bt), 0.25 * (np.abs(a[0]).astype(np.float64) @ np.abs(bt))
    assert (np.abs(got - want) <= BOUND_FP32 * size).all()


@pytest.mark.parametrize("splits", [1, 3, 4096])
@pytest.mark.parametrize("M,N,K", [(372, 301, 2149), (65, 33, 257), (130, 1030, 1001)])
def test_forced_ranges(hip, monkeypatch, M, N, K, splits):
    """A forced number of K ranges (1: none) holds off the 16-byte grid too, for fp32 products and for int8 weights."""
    say("forced ranges", M, N, K, splits)
    rng = np.random.default_rng(M + N + K)
    a, b = rng.uniform(-1, 1, (M, K)).astype(np.float32), rng.uniform(-1, 1, (K, N)).astype(np.float32)
    w, s = rng.integers(-127, 128, (N, K), dtype=np.int8), rng.uniform(1e-3, 1e-2, N).astype(np.float32)
    da, db, dw, ds = hip.array(a), hip.array(b), hip.array(w), hip.array(s)
    monkeypatch.setenv("AX_HIP_F32_SPLITK", str(splits))
    assert hip.L.axhip_tuning_reload() == 1
    try:
        got, kernel = hip.sgemm(da, db).numpy(), hip.last_kernel()
        got8, kernel8 = hip.qgemm_w8a32(da, dw, ds).numpy(), hip.last_kernel()
    finally:
        monkeypatch.delenv("AX_HIP_F32_SPLITK")
        assert hip.L.axhip_tuning_reload() == 0
    if splits == 1:
        assert kernel == "sgemm_nn_64x64k2_staged" and kernel8.endswith("k2_staged"), (kernel, kernel8)
    else:
        assert kernel == "sgemm_splitk" and kernel8 == "qgemm_w8a32_mfma_splitk", (kernel, kernel8)
    size = np.abs(a).astype(np.float64)
    assert (np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= BOUND_FP32 * (size @ np.abs(b).astype(np.float64))).all()
    assert (np.abs(got8 - (a.astype(np.float64) @ w.astype(np.float64).T) * s) <= BOUND_FP32 * (size @ np.abs(w).astype(np.float64).T) * s).all()
