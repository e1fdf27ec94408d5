"""Layer norm rows held in registers, four columns a load and one: edges of both, in place, and off the 16-byte grid."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
COLS = [129, 132, 252, 256, 260, 508, 511, 512, 516, 768, 1020, 1023, 1024, 1028, 2052, 4092, 4096, 4100, 6140, 6144]


@pytest.fixture(scope="module")
def hip():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from axiom_amd.hip import AxHip
    torch.zeros(1, device="cuda")
    h = AxHip()
    h.init()
    return h


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("cols", COLS)
def test_rows_against_64_bits(hip, cols, shift):
    import torch
    rows, eps = 7, 1e-5
    rng = np.random.default_rng(cols)
    x = rng.normal(0.5, 2.0, (rows, cols)).astype(np.float32)
    gamma, beta = rng.normal(1.0, 0.1, cols).astype(np.float32), rng.normal(0.0, 0.1, cols).astype(np.float32)

    def put(values):                                       # `shift` floats past the 16-byte grid
        room = torch.empty(values.size + shift + 8, device="cuda")
        room.fill_(7.0)
        room[shift:shift + values.size] = torch.from_numpy(values.reshape(-1)).cuda()
        return room

    bx, bg, bb, bo, bh = put(x), put(gamma), put(beta), put(np.zeros_like(x)), put(np.zeros_like(x))
    inv = torch.zeros(rows, device="cuda")
    at = lambda t: t.data_ptr() + 4 * shift
    hip.check(hip.L.axhip_layernorm_fwd(at(bx), at(bg), at(bb), at(bo), at(bh), inv.data_ptr(), rows, cols, eps))
    got = bo[shift:shift + x.size].cpu().numpy().reshape(x.shape)
    hat = bh[shift:shift + x.size].cpu().numpy().reshape(x.shape)
    for room in (bo, bh):
        assert torch.all(room[:shift] == 7.0) and torch.all(room[shift + x.size:] == 7.0)

    x64 = x.astype(np.float64)
    mean, var = x64.mean(1, keepdims=True), x64.var(1, keepdims=True)
    std = np.sqrt(var + np.float64(np.float32(eps)))
    want_hat = (x64 - mean) / std
    # at most 24 values a thread, six steps over a wave and two over four of them: 32 roundings of a sum, two more for squares and division
    dm = 34 * U * np.abs(x64).mean(1, keepdims=True)
    dv = 36 * U * (x64 ** 2).mean(1, keepdims=True) + 2 * np.abs(mean) * dm
    rel = dv / (2 * std ** 2) + 4 * U
    bound = np.abs(want_hat) * rel + (dm + U * np.abs(x64 - mean)) / std + U * np.abs(want_hat)
    assert np.all(np.abs(hat - want_hat) <= bound)
    assert np.all(np.abs(got - (gamma * want_hat + beta)) <= np.abs(gamma) * bound + U * np.abs(gamma * want_hat + beta))
    assert np.all(np.abs(inv.cpu().numpy() * std[:, 0] - 1) <= rel[:, 0])

    hip.check(hip.L.axhip_layernorm_fwd(at(bx), at(bg), at(bb), at(bx), None, None, rows, cols, eps))          # in place, neither kept
    assert np.array_equal(bx[shift:shift + x.size].cpu().numpy().reshape(x.shape), got)
