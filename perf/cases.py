"""Workloads of the DenseBlock path, timed and compared through its public entry points.

Every case drives soklyn_amd.devblock.DeviceBlock (one C-ABI call per step) on one
context with stream-ordered calls, as bench.py does.  The kinds of work:

  infer   one layer's forward of a network that is only used (not training)
  net     the whole forward of a network that is only used; returns its logits
  block   one layer's training step inside a larger model: forward, error from the
          upstream gradient, input gradient, weight gradient + optimiser
  hidden  a middle layer of an MLP's training step: forward, then the hidden error
          from the layer above with the weight gradient + optimiser
  head    an output layer's training step: forward, softmax cross-entropy, weight
          gradient + optimiser
  mlp     the whole training step of an MLP (forward of every layer, output error,
          backward from the last layer down, each weight updated before the error
          passes through it)

Activations with a kink (ReLU, LeakyReLU) are used only where the layer is small: on
millions of elements a few pre-activations lie within the rounding of a sum's order
of 0, and their slope then differs by all of it between two correct results.  Smooth
ones (SiLU, Mish, tanh) run through the same kernels.
"""
from __future__ import annotations

import math

import torch

from soklyn_amd import abi
from soklyn_amd.devblock import DeviceBlock

NORMS = {"none": abi.NORM_DISABLED, "rms": abi.NORM_RMS, "layer": abi.NORM_LAYER, "batch": abi.NORM_BATCH}
ACTS = {"identity": abi.ACT_IDENTITY, "relu": abi.ACT_RELU, "tanh": abi.ACT_TANH, "silu": abi.ACT_SILU,
        "mish": abi.ACT_MISH}
LOSS_SCALE = 512.0
DROP_P = 0.1
LR = {"f16": 1e-4, "f32": 1e-2}
MOMENTUM = 0.9
BETA1, BETA2, EPS = 0.9, 0.999, 1e-8


def listed():
    return [
        # one training step of a small digit classifier on a minibatch of 64: every
        # kernel is tiny, launches and host time count
        dict(name="mlp_784_128_10_f32_b64", kind="mlp", dtype="f32", batch=64, dims="784-128-10", norm="none",
             act="relu", dropout=False),
        # the same classifier family served: the whole forward of a 5-layer network
        # on a small request batch (RMSNorm + Mish as it was trained)
        dict(name="net_3072_2048x4_10_f16_b32", kind="net", dtype="f16", batch=32, dims="3072-2048-2048-2048-2048-10",
             norm="rms", act="mish", dropout=False),
        # one wide layer served to a handful of requests: the weights are read once
        dict(name="infer_4096_4096_f16_b16", kind="infer", dtype="f16", batch=16, inputs=4096, outputs=4096,
             norm="none", act="silu", dropout=False),
        # offline inference of a ragged fp32 layer on an ordinary batch
        dict(name="infer_777_1531_f32_b500", kind="infer", dtype="f32", batch=500, inputs=777, outputs=1531,
             norm="layer", act="tanh", dropout=False),
        # a middle layer trained on an ordinary minibatch of 512
        dict(name="hidden_2048_2048_f16_b512", kind="hidden", dtype="f16", batch=512, inputs=2048, outputs=2048,
             above=2048, norm="rms", act="mish", dropout=True),
        # a BatchNorm layer trained in fp16 on a minibatch of 2048
        dict(name="block_1024_1024_bn_f16_b2048", kind="block", dtype="f16", batch=2048, inputs=1024, outputs=1024,
             norm="batch", act="silu", dropout=False),
        # a classifier head of 1000 classes on a minibatch of 1024
        dict(name="head_2048_1000_f16_b1024", kind="head", dtype="f16", batch=1024, inputs=2048, outputs=1000,
             norm="none", act="identity", dropout=False),
        # the ten-class head under a very large batch: a stream over its input
        dict(name="head_2048_10_f16_b16384", kind="head", dtype="f16", batch=16384, inputs=2048, outputs=10,
             norm="none", act="identity", dropout=False),
        # the fp32 block of the benchmark
        dict(name="block_1024_1024_f32_b4096", kind="block", dtype="f32", batch=4096, inputs=1024, outputs=1024,
             norm="none", act="silu", dropout=False),
        # the ragged middle layer of the benchmark: no size a multiple of a tile
        dict(name="hidden_777_1531_f16_b12345", kind="hidden", dtype="f16", batch=12345, inputs=777, outputs=1531,
             above=3001, norm="layer", act="silu", dropout=False),
        # the large middle layer of the benchmark
        dict(name="hidden_2048_2048_f16_b16384", kind="hidden", dtype="f16", batch=16384, inputs=2048, outputs=2048,
             above=2048, norm="rms", act="mish", dropout=True),
        # the headline block of the benchmark
        dict(name="block_4096_4096_f16_b8192", kind="block", dtype="f16", batch=8192, inputs=4096, outputs=4096,
             norm="none", act="silu", dropout=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 64 (as widths are chosen), else any number."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 0.35 else max(64, (v + 32) // 64 * 64)


def draw(rng):
    kind = rng.choice(("infer", "infer", "net", "block", "block", "hidden", "hidden", "head", "mlp"))
    dtype = rng.choice(("f16", "f16", "f16", "f32"))
    norm = rng.choice(("none", "rms", "layer", "batch"))
    act = rng.choice(("tanh", "silu", "mish"))
    few = 32 if norm == "batch" else 2   # the statistics of a couple of rows say nothing
    if kind == "mlp":
        dims = [_width(rng, 64, 1024)] + [_width(rng, 64, 512) for _ in range(rng.randint(1, 2))] + [rng.randint(2, 16)]
        return dict(kind=kind, dtype=dtype, batch=_log(rng, 16, 1024), dims="-".join(map(str, dims)),
                    norm=rng.choice(("none", "rms", "layer")), act=act, dropout=rng.random() < 0.5)
    if kind == "net":
        dims = [_width(rng, 256, 3072)] + [_width(rng, 256, 2048) for _ in range(rng.randint(2, 4))] + [
            rng.randint(2, 16)]
        return dict(kind=kind, dtype=dtype, batch=_log(rng, few, 512), dims="-".join(map(str, dims)), norm=norm,
                    act=act, dropout=False)
    if kind == "infer":
        return dict(kind=kind, dtype=dtype, batch=_log(rng, few, 512), inputs=_width(rng, 128, 4096),
                    outputs=_width(rng, 128, 4096), norm=norm, act=act, dropout=False)
    c = dict(kind=kind, dtype=dtype, batch=_log(rng, 64, 16384), inputs=_width(rng, 128, 4096),
             outputs=_width(rng, 128, 4096), norm=norm, act=act, dropout=rng.random() < 0.5)
    if kind == "head":
        c.update(outputs=_log(rng, 2, 1024), norm="none", act="identity", dropout=False)
    if kind == "hidden":
        c["above"] = _width(rng, 128, 4096) if rng.random() < 0.8 else rng.randint(2, 16)
    # no more work than the listed cases: fp32 products run at a sixteenth of fp16's rate
    while _cost(c) > 0.4e-3 and c["batch"] > 64:
        c["batch"] = max(64, c["batch"] * 3 // 4)
    return c


def _cost(c):
    """Seconds of a pass at the card's nominal rates, both bounds added."""
    w = work(c)
    return w["bytes"] / 8e12 + w["flops"] / (2.5e15 if c["dtype"] == "f16" else 1.57e14)


# ---- the work of a pass -------------------------------------------------------------
def _dims(c):
    if "dims" in c:
        return [int(v) for v in c["dims"].split("-")]
    return [c["inputs"], c["outputs"]]


def _forward_work(c, k, n, norm, dropout):
    m, t = c["batch"], 2 if c["dtype"] == "f16" else 4
    caches = (3 if norm == "none" else 5) + (1 if dropout else 0)
    return t * (m * k + k * n + n + caches * m * n), 2.0 * m * k * n


def _update_work(c, k, n):
    # fp32 parameter and its moments read and written, and the fp16 copy written
    state = (8 + 8 + 8 + 2) if c["dtype"] == "f16" else (8 + 8)
    return state * k * n, 2.0 * c["batch"] * k * n


def _error_work(c, n, norm):
    # grad, d_prenorm (its fp16 copy) and the two norm gradients written
    return c["batch"] * n * (8 + (2 if c["dtype"] == "f16" else 0) + (8 if norm != "none" else 0))


def work(case):
    c = case
    m, t = c["batch"], 2 if c["dtype"] == "f16" else 4
    dims, b, f = _dims(c), 0.0, 0.0
    if c["kind"] in ("infer", "net", "mlp"):
        for i in range(len(dims) - 1):
            last = i == len(dims) - 2 and c["kind"] != "infer"
            norm = "none" if last else c["norm"]
            fb, ff = _forward_work(c, dims[i], dims[i + 1], norm, c["dropout"] and not last)
            b, f = b + fb - (t * m * dims[i] if i else 0), f + ff
            if c["kind"] == "mlp":
                ub, uf = _update_work(c, dims[i], dims[i + 1])
                b, f = b + ub + _error_work(c, dims[i + 1], norm), f + uf + (ff if i else 0)
        return {"bytes": b, "flops": f}
    k, n = dims
    fb, ff = _forward_work(c, k, n, c["norm"], c["dropout"])
    ub, uf = _update_work(c, k, n)
    b, f = fb + ub + _error_work(c, n, c["norm"]), ff + uf
    if c["kind"] == "block":     # the upstream gradient in, the input gradient out
        b, f = b + 4 * m * n + 4 * m * k, f + ff
    elif c["kind"] == "hidden":  # the layer above: its error and weights in
        b, f = b + t * (m + n) * c["above"], f + 2.0 * m * n * c["above"]
    else:                        # the targets in
        b += t * m * n
    return {"bytes": b, "flops": f}


def tolerance(case):
    # measured against exact(): about 4e-7 for fp32 layers, 3e-4 for one fp16 layer and
    # 1e-3 for a whole fp16 network (each cache is rounded to 11 bits)
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-2, "max": 0.4} if case["kind"] in ("net", "mlp") else {"rel": 5e-3, "max": 0.2}


# ---- inputs ---------------------------------------------------------------------------
_context = None


def _ctx():
    """One context for the whole program, its calls ordered on its stream (no wait per call)."""
    global _context
    if _context is None:
        _context = abi.Context(0, 16)
        _context.set_sync(False)
    return _context


def _tensors(case, seed):
    """The numbers a case starts from, on the GPU, from the seed alone: weights He-normal,
    biases small, inputs N(0, 1) (uniform for whole networks), gradients N(0, 1) times the
    loss scale, as fp16 where the block holds fp16."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    half = case["dtype"] == "f16"

    def normal(shape, std):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std

    dims, m = _dims(case), case["batch"]
    x = torch.rand((m, dims[0]), generator=g, device="cuda") if "dims" in case else normal((m, dims[0]), 1.0)
    t = {"x": x.half() if half else x}
    t["w"] = [normal((dims[i], dims[i + 1]), math.sqrt(2.0 / dims[i])) for i in range(len(dims) - 1)]
    t["b"] = [normal((1, n), 0.01) for n in dims[1:]]
    if case["kind"] == "block":
        t["s"] = normal((m, dims[1]), LOSS_SCALE)
    if case["kind"] == "hidden":
        t["w_above"] = normal((dims[1], case["above"]), math.sqrt(2.0 / dims[1]))
        t["dp_above"] = normal((m, case["above"]), LOSS_SCALE / 16)
    if case["kind"] in ("head", "mlp"):
        labels = torch.randint(0, dims[-1], (m,), generator=g, device="cuda")
        t["target"] = torch.nn.functional.one_hot(labels, dims[-1]).to(torch.float16 if half else torch.float32)
    return t


def _block(case, w, b, n_rows, last, training):
    half = case["dtype"] == "f16"
    wn = w.cpu().numpy()
    return DeviceBlock(_ctx(), w.shape[0], w.shape[1], n_rows, wn, half=half, master_w=wn if half else None,
                       b=b.cpu().numpy(), norm=NORMS["none" if last else case["norm"]],
                       act=ACTS["identity" if last else case["act"]], mask_coeff=DROP_P if case["dropout"] else 0.0,
                       is_training=training)


def prepare(case, seed):
    t = _tensors(case, seed)
    m, kind = case["batch"], case["kind"]
    training = kind not in ("infer", "net")
    whole = "dims" in case
    blocks = [_block(case, w, b, m, whole and i == len(t["w"]) - 1, training)
              for i, (w, b) in enumerate(zip(t["w"], t["b"]))]
    opt = abi.adam(BETA1, BETA2, EPS) if case["dtype"] == "f16" else abi.sgd(MOMENTUM)
    state = {"case": case, "x": t["x"], "blocks": blocks, "step": 0, "seed": int(seed),
             "train": abi.train_ctx(opt, opt, m, LR[case["dtype"]])}
    if kind == "block":
        state["s"] = t["s"]
        state["dx"] = torch.empty((m, blocks[0].inputs), device="cuda", dtype=torch.float32)
    if kind == "hidden":
        above = _block(dict(case, norm="none", act="identity", dropout=False), t["w_above"],
                       torch.zeros((1, case["above"])), m, True, True)
        above.d_prenorm.copy_(t["dp_above"])
        if above.d_prenorm_h is not None:
            above.d_prenorm_h.copy_(t["dp_above"])
        state["above"] = above
    if "target" in t:
        state["target"] = t["target"]
    return state


# ---- a pass -----------------------------------------------------------------------------
def _dropout_seed(seed, step, layer):
    return abi.load().skl_scramble_seed((seed + step) & 0xFFFFFFFF, 27 * layer)


def _forward_outputs(blk):
    o = {"out": blk.out, "predrop": blk.predrop, "preact": blk.preact}
    if blk.norm:
        o.update(prenorm=blk.prenorm, centered=blk.centered)
    return o


def _training_outputs(blk):
    o = {"out": blk.out, "preact": blk.preact, "grad": blk.grad, "d_prenorm": blk.d_prenorm, "w": blk.w, "b": blk.b, "dv_w": blk.dv_w,
         "dv_b": blk.dv_b}
    if blk.half:
        o.update(master_w=blk.master_w, dm_w=blk.dm_w)
    if blk.norm:
        o.update(norm_w=blk.norm_w, dv_norm_w=blk.dv_norm_w)
    return o


def run(state):
    case, blocks, x = state["case"], state["blocks"], state["x"]
    kind, m = case["kind"], case["batch"]
    state["step"] += 1
    step = state["step"]
    cur = x
    for i, blk in enumerate(blocks):
        drop = case["dropout"] and not ("dims" in case and i == len(blocks) - 1)
        cur = blk.forward(cur, m, drop, _dropout_seed(state["seed"], step, i) if drop else 0)
    if kind == "net":            # every layer's output, the logits last
        return {"out": [b.out for b in blocks]}
    if kind == "infer":
        return _forward_outputs(blocks[0])
    tc, blk = state["train"], blocks[-1]
    if kind == "block":
        blk.error_from_sum(state["s"], m)
        blk.input_grad(m, state["dx"])
        blk.backward(x, tc, step)
        return dict(_training_outputs(blk), dx=state["dx"])
    if kind == "hidden":
        blk.backward_hidden(state["above"], x, tc, step)
        return _training_outputs(blk)
    blk.output_error(state["target"], abi.LOSS_CE, abi.ACT_SOFTMAX)
    blk.backward(blocks[-2].out if len(blocks) > 1 else x, tc, step)
    for i in range(len(blocks) - 2, -1, -1):
        blocks[i].backward_hidden(blocks[i + 1], blocks[i - 1].out if i else x, tc, step)
    return [_training_outputs(b) for b in blocks]


# ---- the same in 64 bits ------------------------------------------------------------------
def _act64(act, z):
    if act == "relu":
        return z.clamp_min(0.0)
    if act == "tanh":
        return torch.tanh(z)
    if act == "silu":
        return z * torch.sigmoid(z)
    if act == "mish":
        return z * torch.tanh(torch.nn.functional.softplus(z))
    return z


def _slope64(act, z):
    if act == "relu":
        return (z > 0).double()
    if act == "tanh":
        return 1.0 - torch.tanh(z) ** 2
    if act == "silu":
        s = torch.sigmoid(z)
        return s + z * s * (1.0 - s)
    if act == "mish":
        t = torch.tanh(torch.nn.functional.softplus(z))
        return t + z * torch.sigmoid(z) * (1.0 - t * t)
    return torch.ones_like(z)


def _keep64(m, n, seed):
    """The dropout hash: True where element (row, column) is kept."""
    mask32 = 0xFFFFFFFF
    row = torch.arange(m, device="cuda", dtype=torch.int64)[:, None]
    col = torch.arange(n, device="cuda", dtype=torch.int64)[None, :]
    key = ((row * 1103515245) & mask32) ^ ((seed + row * 7) & mask32)
    s = key ^ ((col * 0x4C957F2D) & mask32)
    s = s ^ (s >> 17)
    s = (s * 1103515245 + 12345) & mask32
    s = s ^ (s >> 15)
    return s.float() / 4294967296.0 >= torch.tensor(DROP_P, dtype=torch.float32, device="cuda")


def _forward64(norm, act, x, w, b, keep):
    """One layer's forward; returns what its backward needs."""
    z = x @ w
    if norm != "batch":
        z = z + b
    f = {"prenorm": z, "x": x}
    if norm == "rms":
        f["rstd"] = ((z * z).mean(1, keepdim=True) + 1e-6).rsqrt()
        f["centered"] = z
    elif norm in ("layer", "batch"):
        d = 1 if norm == "layer" else 0
        f["centered"] = z - z.mean(d, keepdim=True)
        f["rstd"] = ((f["centered"] ** 2).mean(d, keepdim=True) + 1e-6).rsqrt()
    f["preact"] = z if norm == "none" else f["centered"] * f["rstd"]
    f["mask"] = torch.ones_like(z) if keep is None else keep.double() / (1.0 - DROP_P)
    f["out"] = _act64(act, f["preact"]) * f["mask"]
    return f


def _forward64_outputs(f, norm):
    o = {"out": f["out"], "predrop": f["out"], "preact": f["preact"]}   # no dropout
    if norm != "none":
        o.update(prenorm=f["prenorm"], centered=f["centered"])
    return o


def _error64(norm, f, e, scale):
    """The element-local norm gradient of the error e (a layer whose norm weight is 1)."""
    m, n = e.shape
    g = {"grad": e, "d_prenorm": e * scale}
    if norm != "none":
        p, r = f["centered"], f["rstd"]
        g["dnw"] = e * p * r
        if norm == "rms":
            g["d_prenorm"] = r * (e - r * r * p * p / n) * scale
        else:
            c = n if norm == "layer" else m
            g["d_prenorm"] = r * (e - e / c - r * r * p * p * e / c) * scale
    return g


def _step64(dtype, p, grad):
    """One optimiser step from zero moments: the parameter after it and the two moments."""
    lr = LR[dtype]
    if dtype == "f32":
        return p - lr * grad, grad, None
    return p - lr * grad / (grad.abs() + EPS), (1.0 - BETA2) * grad * grad, (1.0 - BETA1) * grad


def _update64(case, norm, f, g, w, b):
    c = 1.0 / (LOSS_SCALE * case["batch"])
    half = case["dtype"] == "f16"
    w1, dv, dm = _step64(case["dtype"], w, f["x"].t() @ g["d_prenorm"] * c)
    o = {"out": f["out"], "preact": f["preact"], "grad": g["grad"], "d_prenorm": g["d_prenorm"], "w": w1, "dv_w": dv}
    if norm == "batch":      # its bias is not used and not updated
        o["b"], o["dv_b"] = b, torch.zeros_like(b)
    else:
        o["b"], o["dv_b"], _ = _step64(case["dtype"], b, g["d_prenorm"].sum(0, keepdim=True) * c)
    if half:
        o.update(master_w=w1, dm_w=dm)
    if norm != "none":
        o["norm_w"], o["dv_norm_w"], _ = _step64(case["dtype"], torch.ones_like(b), g["dnw"].sum(0, keepdim=True) * c)
    return o


def exact(case, seed):
    t = _tensors(case, seed)
    half, m, kind = case["dtype"] == "f16", case["batch"], case["kind"]

    def held(v):                 # the value as the block holds it
        return (v.half() if half else v).double()

    masters = [w.double() for w in t["w"]]
    ws, bs = [held(w) for w in t["w"]], [held(b) for b in t["b"]]
    cur, fs, norms = held(t["x"]), [], []
    for i, (w, b) in enumerate(zip(ws, bs)):
        last = "dims" in case and i == len(ws) - 1
        norm, act = ("none", "identity") if last else (case["norm"], case["act"])
        keep = None
        if case["dropout"] and not last:
            keep = _keep64(m, w.shape[1], int(_dropout_seed(int(seed), 1, i)))
        f = _forward64(norm, act, cur, w, b, keep)
        fs.append(f)
        norms.append(norm)
        cur = f["out"]
    if kind == "net":
        return {"out": [f["out"] for f in fs]}
    if kind == "infer":
        return _forward64_outputs(fs[0], norms[0])
    f, norm = fs[-1], norms[-1]
    if kind == "block":
        g = _error64(norm, f, f["mask"] * _slope64(case["act"], f["preact"]) * t["s"].double(), 1.0)
        return dict(_update64(case, norm, f, g, masters[0], bs[0]), dx=g["d_prenorm"] @ ws[0].t())
    if kind == "hidden":
        s = held(t["dp_above"]) @ held(t["w_above"]).t()
        g = _error64(norm, f, f["mask"] * _slope64(case["act"], f["preact"]) * s, 1.0)
        return _update64(case, norm, f, g, masters[0], bs[0])
    f["out"] = torch.softmax(f["out"], 1)
    g = _error64("none", f, f["out"] - t["target"].double(), LOSS_SCALE)
    outs = [_update64(case, "none", f, g, masters[-1], bs[-1])]
    for i in range(len(ws) - 2, -1, -1):
        s = g["d_prenorm"] @ held(outs[0]["w"].float()).t()
        g = _error64(norms[i], fs[i], fs[i]["mask"] * _slope64(case["act"], fs[i]["preact"]) * s, 1.0)
        outs.insert(0, _update64(case, norms[i], fs[i], g, masters[i], bs[i]))
    return outs
