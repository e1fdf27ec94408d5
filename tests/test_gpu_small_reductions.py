"""Small column sums in one launch, and row kernels where a wave takes one short row: edges of their rules, against 64-bit sums."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.mark.parametrize("outer", [1, 3])
@pytest.mark.parametrize("axis", [1, 15, 63, 64, 127, 128, 129, 333, 1023, 1024, 1025])
@pytest.mark.parametrize("inner", [2, 3, 10, 64, 129, 1000, 1024, 2047])
def test_column_sums(hip, outer, axis, inner):
    say("column sums", outer, axis, inner)
    rng = np.random.default_rng(outer + axis * 7 + inner)
    x = rng.uniform(-1, 1, (outer, axis, inner)).astype(np.float32)
    dx, out = hip.array(x), hip.array(np.full(outer * inner + 1, np.nan, np.float32))
    hip.check(hip.L.axhip_sum_axis(dx.ptr, outer, axis, inner, out.ptr))
    got = out.numpy()
    assert np.isnan(got[-1])
    want, size = x.astype(np.float64).sum(axis=1), np.abs(x).astype(np.float64).sum(axis=1)
    # a value passes through at most 64 additions in a row of its own (16 a thread, 64 partial sums in a tree, slices) and a few more
    assert (np.abs(got[:-1].reshape(outer, inner) - want) <= 80 * EPS * size + 1e-37).all()
    hip.check(hip.L.axhip_reduce_axis(3, dx.ptr, outer, axis, inner, out.ptr))          # 0 sum, 1 mean, 2 max, 3 min
    assert np.array_equal(out.numpy()[:-1].reshape(outer, inner), x.min(axis=1))
    hip.check(hip.L.axhip_reduce_axis(2, dx.ptr, outer, axis, inner, out.ptr))
    assert np.array_equal(out.numpy()[:-1].reshape(outer, inner), x.max(axis=1))


def test_column_sums_non_finite(hip):
    x = np.random.default_rng(1).uniform(-1, 1, (130, 37)).astype(np.float32)
    x[3, 5], x[129, 5], x[7, 6], x[128, 7], x[0, 8], x[9, 8] = np.inf, 1.0, np.nan, -np.inf, np.inf, -np.inf
    dx, out = hip.array(x), hip.empty((37,))
    hip.check(hip.L.axhip_sum_axis(dx.ptr, 1, 130, 37, out.ptr))
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64).sum(axis=0)
    got = out.numpy()
    fine = np.isfinite(want)
    assert fine.sum() == 33 and np.abs(got - want)[fine].max() < 1e-4
    assert np.array_equal(got[~fine], want[~fine].astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 16383, 16384, 16385])
@pytest.mark.parametrize("cols", [1, 10, 63, 64, 65, 127, 128])
def test_short_rows(hip, rows, cols):
    say("short rows", rows, cols)
    rng = np.random.default_rng(rows + cols)
    x = rng.normal(0, 3, (rows, cols)).astype(np.float32)
    dx, out = hip.array(x), hip.array(np.full((rows + 1, cols), np.nan, np.float32))
    hip.check(hip.L.axhip_softmax_rows(dx.ptr, out.ptr, rows, cols))
    got = out.numpy()
    assert np.isnan(got[rows]).all()
    e = np.exp(x.astype(np.float64) - x.max(axis=1, keepdims=True))
    want = e / e.sum(axis=1, keepdims=True)
    assert (np.abs(got[:rows] - want) <= 4e-6 * want + 1e-37).all()       # |difference| up to 32: 32 * 2^-24, exp's and the sum's few units
    g, b = rng.normal(1, 0.2, cols).astype(np.float32), rng.normal(0, 1, cols).astype(np.float32)
    dg, db, dh, di = hip.array(g), hip.array(b), hip.empty((rows, cols)), hip.empty((rows,))
    hip.check(hip.L.axhip_layernorm_fwd(dx.ptr, dg.ptr, db.ptr, out.ptr, dh.ptr, di.ptr, rows, cols, 1e-5))
    got = out.numpy()
    assert np.isnan(got[rows]).all()
    x64 = x.astype(np.float64)
    inv = 1 / np.sqrt(x64.var(axis=1) + 1e-5)
    hat = (x64 - x64.mean(axis=1, keepdims=True)) * inv[:, None]
    # the variance as a difference of means of squares: its rounding over the variance, by how much the squares exceed it
    loss = 16 * EPS * (1 + (x64 ** 2).mean(axis=1) * inv ** 2)[:, None]
    bound = loss * (np.abs(hat) + np.abs(x64) * inv[:, None] + np.abs(x64.mean(axis=1) * inv)[:, None]) + 1e-6
    assert (np.abs(dh.numpy() - hat) <= bound).all()
    assert (np.abs(got[:rows] - (g * hat + b)) <= bound * np.abs(g) + 8 * EPS * (np.abs(g * hat) + np.abs(b))).all()
