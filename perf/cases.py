"""The work that programs written against this framework give it, as timed cases.

Twelve listed cases and draw(), which gives more of the same ranges.  A case names one kind of program:

  mlp        forward of a Dense/ReLU classifier through ax_layer_forward
  train      one training step of a Dense/sigmoid classifier: forward, softmax cross-entropy gradient, backward, Adam (sigmoid and
             not ReLU: a ReLU whose input is zero up to rounding flips a whole gradient, which no tolerance of sums describes)
  encoder    forward of a stack of [LayerNorm, attention, LayerNorm, Dense, GELU, Dense] blocks through ax_layer_forward
  w8a32      one linear layer with int8 weights on fp32 activations (axhip_qgemm_w8a32)
  w8a8       one linear layer with int8 weights and activations, bias and activation in the write-back (axhip_qgemm_w8a8)
  gemm       one fp32 product in any of the three storage orders (axhip_sgemm)
  sdpa       fused attention forward (axhip_sdpa_fwd)
  products   attention as its two batched products with a row softmax between them, the probabilities kept

Device buffers that a program hands to the C ABI are torch tensors here; tensors of the layer API are the framework's own,
seen through torch.  Everything runs on the null stream.
"""
import ctypes as C
import math

import torch

from axiom_amd.axiom import DEVICE_HIP, TP, Axiom
from axiom_amd.hip import AxHip

DEV = "cuda:0"
_lib = {}


def _libs():
    """The two libraries, loaded and initialised once per process."""
    if not _lib:
        torch.zeros(1, device=DEV)
        hip = AxHip()
        hip.init()
        ax = Axiom()
        if ax.L.ax_init() != 0 or ax.L.ax_compute_init() != 0:
            raise RuntimeError("ax_init: %s" % (ax.err(),))
        _lib["hip"], _lib["ax"] = hip, ax
    return _lib["hip"], _lib["ax"]


# ---- the cases -------------------------------------------------------------------------------------------------------

def listed():
    return [
        # bs=1 inference of the 784-4096-4096-10 network of the benchmark: 80 MB of weights, latency
        {"name": "mlp_b1", "kind": "mlp", "batch": 1, "inputs": 784, "hidden": 4096, "outputs": 10},
        # the same network on a batch that is no multiple of any tile
        {"name": "mlp_b100", "kind": "mlp", "batch": 100, "inputs": 784, "hidden": 4096, "outputs": 10},
        # a training step of a smaller classifier on the usual mini-batch
        {"name": "train_b128_h1024", "kind": "train", "batch": 128, "inputs": 784, "hidden": 1024, "outputs": 10},
        # the encoder of the reference's bench_transformer.c: 6 blocks on [8, 128, 256], many small launches
        {"name": "encoder_8x128x256", "kind": "encoder", "batch": 8, "seq": 128, "width": 256, "heads": 4, "blocks": 6, "causal": False},
        # large causal blocks on a ragged sequence: the feed-forward shapes 1024-4096-1024 of the benchmark
        {"name": "encoder_4x500x1024", "kind": "encoder", "batch": 4, "seq": 500, "width": 1024, "heads": 16, "blocks": 2, "causal": True},
        # quantized weights, one token at a time
        {"name": "w8a32_1x4096x4096", "kind": "w8a32", "m": 1, "n": 4096, "k": 4096},
        # quantized weights, a prompt or a batch of tokens (the reference's quantized path at the size of its int8 benchmark)
        {"name": "w8a32_250x4096x4096", "kind": "w8a32", "m": 250, "n": 4096, "k": 4096},
        # int8 on both sides at the benchmark's two sizes
        {"name": "w8a8_256x4096x4096", "kind": "w8a8", "m": 256, "n": 4096, "k": 4096, "act": 0},
        {"name": "w8a8_8192x8192x8192", "kind": "w8a8", "m": 8192, "n": 8192, "k": 8192, "act": 0},
        # fp32 product at the benchmark's size
        {"name": "gemm_1024x1024x1024", "kind": "gemm", "m": 1024, "n": 1024, "k": 1024, "order": "nn"},
        # causal attention, ragged sequence, head size between the kernel's own
        {"name": "sdpa_causal_96x1000x80", "kind": "sdpa", "heads": 96, "seq": 1000, "dim": 80, "causal": True},
        # the benchmark's 32 x 16 heads of [512, 64] as separate products
        {"name": "products_512x512x64", "kind": "products", "heads": 512, "seq": 512, "dim": 64},
    ]


def _size(rng, lo, hi, grain):
    """Log-uniform in [lo, hi]; half of the draws on the grid of `grain` (sizes that models choose), half anywhere (sizes that data gives)."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if rng.random() < 0.5:
        v = round(v / grain) * grain
    return int(min(hi, max(lo, round(v))))


def draw(rng):
    kind = rng.choice(["mlp", "train", "encoder", "w8a32", "w8a8", "gemm", "sdpa", "products"])
    if kind in ("mlp", "train"):
        return {"kind": kind, "batch": _size(rng, 1 if kind == "mlp" else 16, 512, 16), "inputs": _size(rng, 256, 2048, 64),
                "hidden": _size(rng, 512, 4096 if kind == "mlp" else 2048, 64), "outputs": _size(rng, 10, 1000, 8)}
    if kind == "encoder":
        width = rng.choice([128, 256, 384, 512, 768, 1024])
        dim = rng.choice([32, 64])
        seq = _size(rng, 32, 512, 32)
        tokens = 2000 * (1024 / width)                       # no more work a block than the largest listed one
        batch = max(1, min(int(tokens / seq), _size(rng, 1, 32, 1)))
        blocks = rng.choice([1, 2, 2, 4, 6]) if width <= 512 else rng.choice([1, 2])
        return {"kind": kind, "batch": batch, "seq": seq, "width": width, "heads": width // dim, "blocks": blocks, "causal": rng.random() < 0.5}
    if kind == "w8a32":
        m = 1 if rng.random() < 0.2 else _size(rng, 1, 1024, 16)
        return {"kind": kind, "m": m, "n": _size(rng, 768, 11008, 64), "k": _size(rng, 768, 4096, 64)}
    if kind == "w8a8":
        return {"kind": kind, "m": _size(rng, 1, 4096, 32), "n": _size(rng, 768, 8192, 64), "k": _size(rng, 768, 8192, 64), "act": rng.choice([0, 1, 2])}
    if kind == "gemm":
        return {"kind": kind, "m": _size(rng, 32, 2048, 32), "n": _size(rng, 128, 4096, 32), "k": _size(rng, 64, 4096, 32),
                "order": rng.choice(["nn", "nt", "tn"])}
    if kind == "sdpa":
        seq = _size(rng, 32, 2048, 32)
        heads = max(1, min(int(512 * (512 / seq) ** 2), _size(rng, 4, 512, 4)))
        return {"kind": kind, "heads": heads, "seq": seq, "dim": rng.choice([32, 48, 64, 80, 96, 128]), "causal": rng.random() < 0.5}
    seq = _size(rng, 64, 1024, 32)
    return {"kind": kind, "heads": max(1, min(int(512 * (512 / seq) ** 2), _size(rng, 8, 512, 8))), "seq": seq, "dim": rng.choice([32, 64, 128])}


# ---- inputs ----------------------------------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7919 + 17)
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    return torch.empty(shape, device=DEV).normal_(mean, std, generator=g)


def _int8(g, shape):
    return torch.randint(-127, 128, shape, device=DEV, dtype=torch.int8, generator=g)


class _Memory:
    """Device memory of the framework, as torch reads it."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 3, "strides": None}


def _seen(t):
    """A contiguous fp32 ax_tensor_t as a torch tensor over the same memory."""
    c = t.contents
    return torch.as_tensor(_Memory(c.storage.contents.data + 4 * c.offset, tuple(c.shape[i] for i in range(c.ndim))), device=DEV)


def _on_device(fn, *args):
    """Runs a constructor with the GPU as the default device."""
    _, ax = _libs()
    before = ax.L.ax_get_default_device()
    ax.L.ax_set_default_device(DEVICE_HIP)
    made = fn(*args)
    ax.L.ax_set_default_device(before)
    if not made:
        raise RuntimeError("axiom: %s" % (ax.err(),))
    return made


class _Model:
    """A Sequential with its input tensor, as a serving program keeps them; the last result is given back when the next one is made."""

    def __init__(self, layers, x):
        _, self.ax = _libs()
        L = self.ax.L
        self.L = L
        self.seq = _on_device(L.ax_sequential_create)
        for make, args in layers:
            L.ax_sequential_add(self.seq, _on_device(getattr(L, make), *args))
        self.x = self.tensor(x)
        self.y, self.at, self.view = None, None, None

    def tensor(self, values):
        shape, ndim = self.ax.shape_arg(values.shape)
        t = _on_device(self.L.ax_tensor_create, shape, ndim, 0)
        _seen(t).copy_(values)
        return t

    def params(self):
        held = (TP * 256)()
        return [_seen(held[i]) for i in range(self.L.ax_layer_get_params(self.seq, held, 256))]

    def forward(self):
        if self.y:
            self.L.ax_tensor_destroy(self.y)
        self.y = self.L.ax_layer_forward(self.seq, self.x)
        if not self.y:
            raise RuntimeError("forward: %s" % (self.ax.err(),))
        at = self.y.contents.storage.contents.data
        if at != self.at:
            self.at, self.view = at, _seen(self.y)
        return self.view

    def __del__(self):
        self.ax.free(self.x, self.y)
        self.L.ax_layer_destroy(self.seq)


class _Trainer:
    """Weights, Adam moments, gradients and activations of a two-layer classifier, all tensors of the framework."""

    def __init__(self, c, g):
        _, self.ax = _libs()
        self.L = self.ax.L
        b, i, h, o = c["batch"], c["inputs"], c["hidden"], c["outputs"]
        self.batch = b
        self.t, self.seen = {}, {}
        for name, shape in (("x", (b, i)), ("target", (b, o)), ("h", (b, h)), ("z", (b, o)), ("dz", (b, o)), ("dh", (b, h)), ("slope", (b, h))):
            self.make(name, shape)
        for name, shape, std in (("w1", (i, h), math.sqrt(2 / i)), ("b1", (h,), 0.02), ("w2", (h, o), math.sqrt(2 / h)), ("b2", (o,), 0.02)):
            self.make(name, shape).copy_(_normal(g, shape, std))
            self.make("d" + name, shape).zero_()
            self.make("m" + name, shape).copy_(_normal(g, shape, 1e-3))
            self.make("v" + name, shape).copy_(_normal(g, shape, 1e-3).square_() + 1e-6)
        self.seen["x"].copy_(torch.rand((b, i), device=DEV, generator=g))
        self.seen["target"].copy_(torch.nn.functional.one_hot(torch.randint(0, o, (b,), device=DEV, generator=g), o).float())

    def make(self, name, shape):
        sh, nd = self.ax.shape_arg(shape)
        self.t[name] = _on_device(self.L.ax_tensor_create, sh, nd, 0)
        self.seen[name] = _seen(self.t[name])
        return self.seen[name]

    def step(self):
        L, t = self.L, self.t
        bad = L.ax_compute_gemm_bias_act(t["x"], t["w1"], t["b1"], 0, t["h"])
        bad |= L.ax_compute_sigmoid(t["h"], t["h"])
        bad |= L.ax_compute_gemm_bias_act(t["h"], t["w2"], t["b2"], 0, t["z"])
        bad |= L.ax_compute_softmax_rowwise(t["z"], t["dz"])
        bad |= L.ax_compute_sub(t["dz"], t["target"], t["dz"])
        bad |= L.ax_compute_mul_scalar(t["dz"], 1.0 / self.batch, t["dz"])
        bad |= L.ax_compute_gemm_tn(t["h"], t["dz"], t["dw2"])
        bad |= L.ax_compute_sum(t["dz"], 0, t["db2"])
        bad |= L.ax_compute_gemm_nt(t["dz"], t["w2"], t["dh"])
        bad |= L.ax_compute_square(t["h"], t["slope"])
        bad |= L.ax_compute_sub(t["h"], t["slope"], t["slope"])
        bad |= L.ax_compute_mul(t["dh"], t["slope"], t["dh"])
        bad |= L.ax_compute_gemm_tn(t["x"], t["dh"], t["dw1"])
        bad |= L.ax_compute_sum(t["dh"], 0, t["db1"])
        for p in ("w1", "b1", "w2", "b2"):
            bad |= L.ax_compute_adam_update(t[p], t["d" + p], t["m" + p], t["v" + p], 1e-3, 0.9, 0.999, 1e-8, 0.01, 0.65, 0.01, True)
        if bad:
            raise RuntimeError("training step: %s" % (self.ax.err(),))
        return {n: self.seen[n] for n in ("z", "dw1", "db1", "dw2", "db2", "w1", "b1", "w2", "b2", "mw1", "vw1", "mw2", "vw2")}

    def __del__(self):
        self.ax.free(*self.t.values())


def prepare(case, seed):
    hip, _ = _libs()
    g = _generator(seed)
    kind = case["kind"]
    s = {"case": case, "hip": hip, "L": hip.L}
    if kind == "mlp":
        x = torch.rand((case["batch"], case["inputs"]), device=DEV, generator=g)
        dims = (case["inputs"], case["hidden"], case["hidden"], case["outputs"])
        layers = []
        for i in range(3):
            layers.append(("ax_dense_create", (dims[i], dims[i + 1], True)))
            if i < 2:
                layers.append(("ax_relu_layer_create", ()))
        s["model"] = _Model(layers, x)
        for p in s["model"].params():                       # Kaiming weights; biases as training leaves them
            p.copy_(_normal(g, p.shape, 0.02 if p.dim() == 1 else math.sqrt(2 / p.shape[0])))
    elif kind == "train":
        s["trainer"] = _Trainer(case, g)
    elif kind == "encoder":
        d = case["width"]
        block = [("ax_layernorm_create", (d, 1e-5)), ("ax_mha_create", (d, case["heads"], True, case["causal"])),
                 ("ax_layernorm_create", (d, 1e-5)), ("ax_dense_create", (d, 4 * d, True)), ("ax_gelu_layer_create", ()),
                 ("ax_dense_create", (4 * d, d, True))]
        s["model"] = _Model(block * case["blocks"], _normal(g, (case["batch"], case["seq"], d)))
        params = s["model"].params()
        for i, p in enumerate(params):
            if p.dim() == 2:
                p.copy_(_normal(g, p.shape, 1 / math.sqrt(p.shape[0])))
            else:
                p.copy_(_normal(g, p.shape, 0.02))
        per = len(params) // case["blocks"]                  # gamma of a layer norm is near one
        for b in range(case["blocks"]):
            for i in (0, 10):
                params[b * per + i].add_(1.0)
    elif kind == "w8a32":
        m, n, k = case["m"], case["n"], case["k"]
        s.update(a=_normal(g, (m, k)), w=_int8(g, (n, k)), ws=torch.rand(n, device=DEV, generator=g) * 9e-3 + 1e-3, out=torch.empty((m, n), device=DEV))
    elif kind == "w8a8":
        m, n, k = case["m"], case["n"], case["k"]
        s.update(x=_int8(g, (m, k)), w=_int8(g, (n, k)), ws=torch.rand(n, device=DEV, generator=g) * 9e-3 + 1e-3, bias=_normal(g, (n,), 0.02),
                 out=torch.empty((m, n), device=DEV))
    elif kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        ta, tb = case["order"][0] == "t", case["order"][1] == "t"
        s.update(a=torch.rand((k, m) if ta else (m, k), device=DEV, generator=g) * 2 - 1,
                 b=torch.rand((n, k) if tb else (k, n), device=DEV, generator=g) * 2 - 1, c=torch.empty((m, n), device=DEV), ta=ta, tb=tb)
    elif kind in ("sdpa", "products"):
        shape = (case["heads"], case["seq"], case["dim"])
        s.update(q=_normal(g, shape), k=_normal(g, shape), v=_normal(g, shape), o=torch.empty(shape, device=DEV))
        if kind == "sdpa":
            s["lse"] = torch.empty(shape[:2], device=DEV)
        else:
            s["p"] = torch.empty((shape[0], shape[1], shape[1]), device=DEV)
    else:
        raise ValueError("unknown kind %r" % kind)
    return s


# ---- one pass --------------------------------------------------------------------------------------------------------

def run(s):
    case, hip, L = s["case"], s["hip"], s["L"]
    kind = case["kind"]
    if kind in ("mlp", "encoder"):
        return s["model"].forward()
    if kind == "train":
        return s["trainer"].step()
    if kind == "w8a32":
        hip.check(L.axhip_qgemm_w8a32(s["a"].data_ptr(), s["w"].data_ptr(), s["ws"].data_ptr(), s["out"].data_ptr(), case["m"], case["n"], case["k"]))
        return s["out"]
    if kind == "w8a8":
        hip.check(L.axhip_qgemm_w8a8(s["x"].data_ptr(), 0.02, s["w"].data_ptr(), s["ws"].data_ptr(), s["bias"].data_ptr(), case["act"],
                                     s["out"].data_ptr(), None, case["m"], case["n"], case["k"]))
        return s["out"]
    if kind == "gemm":
        hip.check(L.axhip_sgemm(int(s["ta"]), int(s["tb"]), case["m"], case["n"], case["k"], 1.0, s["a"].data_ptr(), s["a"].shape[1],
                                s["b"].data_ptr(), s["b"].shape[1], 0.0, s["c"].data_ptr(), case["n"], None, 0))
        return s["c"]
    bh, n, d = case["heads"], case["seq"], case["dim"]
    q, k, v, o = (s[x].data_ptr() for x in "qkvo")
    if kind == "sdpa":
        hip.check(L.axhip_sdpa_fwd(q, k, v, o, s["lse"].data_ptr(), bh, n, d, 1 / math.sqrt(d), int(case["causal"])))
        return s["o"], s["lse"]
    p = s["p"].data_ptr()
    hip.check(L.axhip_sgemm_strided_batched(0, 1, n, n, d, 1 / math.sqrt(d), q, d, n * d, k, d, n * d, 0.0, p, n, n * n, bh))
    hip.check(L.axhip_softmax_rows(p, p, bh * n, n))
    hip.check(L.axhip_sgemm_strided_batched(0, 0, n, d, n, 1.0, p, n, n * n, v, d, n * d, 0.0, o, d, n * d, bh))
    return s["o"], s["p"]


# ---- what a pass cannot do without, and how far two right answers may be apart ---------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "mlp":
        b, i, h, o = (case[x] for x in ("batch", "inputs", "hidden", "outputs"))
        weights = i * h + h * h + h * o
        return {"bytes": 4 * (weights + 2 * h + o + b * (i + o)), "flops": 2 * b * weights}
    if kind == "train":
        b, i, h, o = (case[x] for x in ("batch", "inputs", "hidden", "outputs"))
        weights = i * h + h * o + h + o
        # Adam reads and writes a weight and two moments; the gradients are outputs
        return {"bytes": 4 * (7 * weights + b * (i + 2 * o)), "flops": 2 * b * (2 * i * h + 3 * h * o)}
    if kind == "encoder":
        d, rows = case["width"], case["batch"] * case["seq"]
        seen = case["seq"] / 2 if case["causal"] else case["seq"]
        return {"bytes": 4 * (case["blocks"] * 12 * d * d + 2 * rows * d),
                "flops": case["blocks"] * (24 * rows * d * d + 4 * rows * seen * d)}
    if kind in ("w8a32", "w8a8", "gemm"):
        m, n, k = case["m"], case["n"], case["k"]
        a, b = {"w8a32": (4, 1), "w8a8": (1, 1), "gemm": (4, 4)}[kind]
        return {"bytes": a * m * k + b * n * k + 4 * m * n + (0 if kind == "gemm" else 4 * n), "flops": 2 * m * n * k}
    bh, n, d = case["heads"], case["seq"], case["dim"]
    if kind == "sdpa":
        return {"bytes": 4 * bh * n * (4 * d + 1), "flops": 4 * bh * n * n * d / (2 if case["causal"] else 1)}
    return {"bytes": 4 * bh * n * (4 * d + n), "flops": 4 * bh * n * n * d}


def tolerance(case):
    return TOLERANCE[case["kind"]]


#: About four times what a pass differs by from the same pass in 64 bits over listed and drawn cases (rel: 2-norms; max: largest
#: difference over the root mean square or the value).  Measured, rel / max: mlp 6.5e-7 / 2.9e-6, train 7.5e-7 / 3.6e-6,
#: encoder 2.5e-6 / 8.5e-6, w8a32 7.7e-7 / 7.4e-6, w8a8 4.4e-8 / 1.4e-7, gemm 6.5e-7 / 5.1e-6, sdpa 3.7e-7 / 7.0e-6,
#: products 6.7e-7 / 9.6e-6.
TOLERANCE = {
    "mlp": {"rel": 3e-6, "max": 1.5e-5},
    "train": {"rel": 3e-6, "max": 1.5e-5},
    "encoder": {"rel": 1e-5, "max": 4e-5},
    "w8a32": {"rel": 3e-6, "max": 3e-5},
    "w8a8": {"rel": 2e-7, "max": 1e-6},
    "gemm": {"rel": 3e-6, "max": 3e-5},
    "sdpa": {"rel": 2e-6, "max": 3e-5},
    "products": {"rel": 3e-6, "max": 4e-5},
}
