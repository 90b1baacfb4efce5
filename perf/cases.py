"""Performance cases: what a program that serves models with this framework calls.

Two kinds of entry point are covered.

* The compiled engine (``munet_amd.engine``): a model or a block is loaded and
  compiled once, its input is placed in the engine's device buffer and
  ``run_device()`` forwards it.  The KV-cache ``Decoder`` prefills a prompt and
  is stepped token by token.
* The capability calls (``munet_amd.backend.HipBackend``): MuNet's own modules
  reach the GPU through ``matmul``, ``add``, ``conv2d`` and the like, on
  weights in MuNet's layouts (Linear ``[in, out]``, convolution OIHW, NCHW
  activations).

``draw`` spans the same families: batch 1 to the largest, sequence lengths and
channel counts that are no multiple of any tile, head sizes 32 to 128 and the
three storage types.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

from munet_amd import models
from munet_amd.backend import BroadcastInfo, HipBackend, compute_broadcast, contiguous_strides
from munet_amd.engine import Decoder, Engine

DEV = "cuda"
TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # a classifier on one small batch: a few microseconds of work behind one
        # call (the repository's MLP workload)
        {"name": "mlp", "kind": "mlp", "dtype": "float32", "batch": 64, "sizes": "784,256,256,10"},
        # a small image classifier (the repository's CNN workload)
        {"name": "cnn", "kind": "cnn", "dtype": "float32", "batch": 32, "hw": 32, "c1": 32, "c2": 64, "hidden": 128},
        # segmentation of a batch of images (the repository's UNet workload)
        {"name": "unet", "kind": "unet", "dtype": "float16", "batch": 8, "h": 128, "w": 128, "base": 64, "levels": 4},
        # one encoder layer in half precision (the repository's encoder workload)
        {"name": "encoder_f16", "kind": "block", "dtype": "float16", "batch": 8, "t": 256, "heads": 8, "hd": 64,
         "ffn": 2048, "causal": False},
        # the same layer in single precision, on sentences of no round length
        {"name": "encoder_f32", "kind": "block", "dtype": "float32", "batch": 8, "t": 250, "heads": 8, "hd": 64,
         "ffn": 2048, "causal": False},
        # a decoder layer on one user's prompt: few rows, time to first token
        {"name": "prompt_block", "kind": "block", "dtype": "bfloat16", "batch": 1, "t": 237, "heads": 12, "hd": 64,
         "ffn": 3072, "causal": True},
        # a decoder layer of a larger model with 128-wide heads, long prompts
        {"name": "wide_block", "kind": "block", "dtype": "bfloat16", "batch": 2, "t": 1000, "heads": 16, "hd": 128,
         "ffn": 8192, "causal": True},
        # prefill of the 12-layer decoder: the repository's headline workload
        {"name": "prefill", "kind": "decoder", "dtype": "bfloat16", "batch": 4, "t": 1024, "heads": 12, "hd": 64,
         "ffn": 3072, "layers": 12, "vocab": 32000},
        # chat: a prompt, then one token after another with the KV cache
        {"name": "decode", "kind": "decode", "dtype": "bfloat16", "batch": 4, "t": 60, "steps": 16, "heads": 12, "hd": 64,
         "ffn": 3072, "layers": 12, "vocab": 32000, "max_len": 256},
        # a feed-forward layer as MuNet's modules call the backend: matmul on
        # the [in, out] weight, bias add, GELU, matmul, bias add, residual add
        {"name": "ffn_calls", "kind": "ffn", "dtype": "bfloat16", "m": 4096, "d": 1024, "ffn": 4096},
        # a convolution stage as MuNet's modules call it: NCHW conv2d, ReLU,
        # max-pool
        {"name": "conv_calls", "kind": "conv", "dtype": "float32", "batch": 16, "ic": 64, "oc": 128, "h": 56, "w": 56,
         "k": 3, "stride": 1, "pad": 1, "pool": 2},
        # a classification head in single precision: LayerNorm, matmul, bias
        # add, softmax over the classes
        {"name": "head_calls", "kind": "head", "dtype": "float32", "m": 1000, "d": 768, "classes": 5000},
    ]


def draw(rng):
    """One more case of the same ranges; never more work than the largest listed one."""
    while True:
        case = _draw(rng)
        w = work(case)
        slow = 16.0 if case["dtype"] == "float32" else 1.0  # single precision runs at about 1/16 of the 16-bit rate
        square = case["kind"] in ("block", "decoder") and case["batch"] * case["heads"] * case["t"] ** 2 * case["hd"] * case.get("layers", 1)
        if w["flops"] * slow <= 9e11 and w["bytes"] <= 1.2e9 and (square or 0) <= 4.1e9:
            return case


def _draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def mult(lo, hi, by):
        return max(by, log(lo, hi) // by * by)

    kind = rng.choice(["mlp", "cnn", "unet", "block", "block", "block", "decoder", "decode", "ffn", "conv", "head"])
    dtype = rng.choice(["float32", "float16", "bfloat16"])
    c = {"kind": kind, "dtype": dtype}
    if kind == "mlp":
        c.update(batch=log(1, 512), sizes="%d,%d,%d,%d" % (mult(64, 2048, 4), mult(32, 1024, 4), mult(32, 1024, 4), log(2, 1000)))
    elif kind == "cnn":
        c.update(batch=log(1, 128), hw=4 * log(4, 24), c1=mult(8, 64, 4), c2=mult(16, 128, 4), hidden=mult(32, 512, 4))
    elif kind == "unet":
        c.update(dtype=rng.choice(["float16", "bfloat16"]), batch=log(1, 8), h=8 * log(3, 20), w=8 * log(3, 20),
                 base=rng.choice([32, 64]), levels=4)
    elif kind == "block":
        hd = rng.choice([32, 48, 64, 64, 80, 96, 128])
        heads = log(2, 16)
        c.update(batch=log(1, 16), t=log(16, 2048), heads=heads, hd=hd, ffn=4 * heads * hd, causal=rng.random() < 0.5)
    elif kind == "decoder":
        heads, hd = rng.choice([4, 8, 12, 16]), rng.choice([32, 64, 64, 128])
        c.update(dtype=rng.choice(["float16", "bfloat16", "bfloat16"]), batch=log(1, 8), t=log(16, 1024), heads=heads, hd=hd,
                 ffn=4 * heads * hd, layers=rng.randint(1, 6), vocab=mult(500, 32000, 4))
    elif kind == "decode":
        heads, hd = rng.choice([4, 8, 12]), rng.choice([32, 64])
        c.update(dtype=rng.choice(["float16", "bfloat16"]), batch=log(1, 16), t=log(4, 200), steps=rng.randint(4, 24), heads=heads,
                 hd=hd, ffn=4 * heads * hd, layers=rng.randint(1, 12), vocab=mult(500, 32000, 4), max_len=256)
    elif kind == "ffn":
        d = mult(128, 2048, 4)
        c.update(m=log(1, 8192), d=d, ffn=4 * d)
    elif kind == "conv":
        c.update(batch=log(1, 32), ic=log(3, 256), oc=mult(8, 256, 4), h=log(14, 160), w=log(14, 160), k=rng.choice([1, 3, 3, 5]),
                 stride=rng.choice([1, 1, 2]), pad=1, pool=2)
    else:
        c.update(m=log(1, 4096), d=mult(64, 2048, 4), classes=log(10, 30000))
    return c


# ---- inputs --------------------------------------------------------------------

def _config(case):
    kind, dt = case["kind"], case["dtype"]
    if kind == "mlp":
        return models.mlp_config(tuple(int(s) for s in case["sizes"].split(",")), dt)
    if kind == "cnn":
        return models.cnn_config(dt, 3, case["hw"], case["c1"], case["c2"], case["hidden"])
    if kind == "unet":
        return models.unet_config(dt, 3, tuple(case["base"] << i for i in range(case["levels"])), 2)
    d = case["heads"] * case["hd"]
    if kind == "block":
        return models.block_config(d, case["heads"], case["ffn"], case["causal"], dt)
    return models.decoder_config(case["vocab"], max(case["t"], case.get("max_len", 0)), d, case["heads"], case["layers"],
                                 case["ffn"], dt, attention="textbook" if kind == "decode" else "munet")


def _input_shape(case):
    kind = case["kind"]
    if kind == "mlp":
        return (case["batch"], int(case["sizes"].split(",")[0]))
    if kind == "cnn":
        return (case["batch"], 3, case["hw"], case["hw"])
    if kind == "unet":
        return (case["batch"], 3, case["h"], case["w"])
    if kind == "block":
        return (case["batch"], case["t"], case["heads"] * case["hd"])
    return (case["batch"], case["t"])


def _made(case, seed):
    """(parameters by name, inputs by name), on the GPU and in the storage dtype."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt = TORCH[case["dtype"]]

    def normal(shape, std=1.0, mean=0.0):
        return (torch.randn(tuple(shape), device=DEV, generator=g) * std + mean).to(dt)

    kind = case["kind"]
    if kind == "ffn":
        m, d, f = case["m"], case["d"], case["ffn"]
        return ({"w1": normal((d, f), d ** -0.5), "b1": normal((f,), 0.1), "w2": normal((f, d), f ** -0.5),
                 "b2": normal((d,), 0.1)}, {"x": normal((m, d))})
    if kind == "conv":
        ic, oc, k = case["ic"], case["oc"], case["k"]
        return ({"w": normal((oc, ic, k, k), (2.0 / (ic * k * k)) ** 0.5), "b": normal((oc,), 0.1)},
                {"x": normal((case["batch"], ic, case["h"], case["w"]))})
    if kind == "head":
        m, d, n = case["m"], case["d"], case["classes"]
        return ({"g": normal((d,), 0.1, 1.0), "o": normal((d,), 0.1), "w": normal((d, n), 2.0 * d ** -0.5), "b": normal((n,), 0.1)},
                {"x": normal((m, d))})
    params = {}
    for name, shape, role, info in models.param_specs(_config(case)):
        if role == "ln_w":
            params[name] = normal(shape, 0.1, 1.0)
        elif role in ("ln_b", "bias"):
            params[name] = normal(shape, 0.05)
        elif role == "embed" or kind in ("decoder", "decode"):
            params[name] = normal(shape, 0.02)
        elif kind in ("cnn", "unet"):
            params[name] = normal(shape, (2.0 / info["fan_in"]) ** 0.5)
        else:
            params[name] = normal(shape, info["fan_in"] ** -0.5)
    if kind in ("decoder", "decode"):
        n = case["t"] + case.get("steps", 0)
        return params, {"ids": torch.randint(0, case["vocab"], (case["batch"], n), device=DEV, generator=g, dtype=torch.int32)}
    return params, {"x": normal(_input_shape(case))}


def _host(t):
    """A parameter as the engine's loader takes it: float32 values or 16-bit patterns."""
    t = t.cpu()
    return t.numpy() if t.dtype == torch.float32 else t.view(torch.int16).numpy().view(np.uint16)


class _Buffer:
    """Device memory of an engine, for torch to view; a view keeps the engine
    (which frees that memory when it goes) alive."""

    def __init__(self, engine, ptr, shape, typestr):
        self.engine = engine
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr, "version": 2}


def _view(engine, ptr, shape, dtype):
    typestr = "<i2" if dtype in (torch.float16, torch.bfloat16) else "<i4" if dtype == torch.int32 else "<f4"
    t = torch.as_tensor(_Buffer(engine, ptr, shape, typestr), device=DEV)
    return t.view(dtype) if typestr == "<i2" else t


def _empty(like, *shape):
    return torch.empty(shape, dtype=like.dtype, device=DEV)


def _bcast(a, b):
    return BroadcastInfo(*compute_broadcast(a, contiguous_strides(a), b, contiguous_strides(b)))


def prepare(case, seed):
    """What a serving program holds before the call: the compiled engine (or the
    weights and output buffers of the capability calls) and the input on the GPU."""
    params, x = _made(case, seed)
    kind = case["kind"]
    if kind in ("ffn", "conv", "head"):
        s = dict(case=case, be=HipBackend(), **params, **x)
        if kind == "ffn":
            m, d, f = case["m"], case["d"], case["ffn"]
            s.update(h=_empty(x["x"], m, f), h2=_empty(x["x"], m, f), y=_empty(x["x"], m, d), y2=_empty(x["x"], m, d),
                     bias_f=_bcast((m, f), (f,)), bias_d=_bcast((m, d), (d,)), same=_bcast((m, d), (m, d)))
        elif kind == "conv":
            oh, ow = _conv_out(case)
            p = case["pool"]
            s.update(y=_empty(x["x"], case["batch"], case["oc"], oh, ow), r=_empty(x["x"], case["batch"], case["oc"], oh, ow),
                     z=_empty(x["x"], case["batch"], case["oc"], (oh - p) // p + 1, (ow - p) // p + 1))
        else:
            m, n = case["m"], case["classes"]
            s.update(h=_empty(x["x"], m, case["d"]), y=_empty(x["x"], m, n), y2=_empty(x["x"], m, n), p=_empty(x["x"], m, n),
                     bias=_bcast((m, n), (n,)))
        return s
    eng = Engine().load(_config(case), {k: _host(v) for k, v in params.items()})
    shape = _input_shape(case)
    eng.compile(shape)
    if kind == "decode":
        ids = x["ids"].cpu().numpy()
        t0 = case["t"]
        s = dict(case=case, engine=eng, decoder=Decoder(eng, case["batch"], case["max_len"]),
                 prompt=np.ascontiguousarray(ids[:, :t0]), fed=[np.ascontiguousarray(ids[:, t0 + i]) for i in range(case["steps"])])
        s["decoder"].prefill(s["prompt"], logits=False)
        return s
    src = x["ids"] if kind == "decoder" else x["x"]
    _view(eng, eng.input_ptr(), shape, src.dtype).copy_(src)
    out = _view(eng, eng.output_ptr(), eng.out_shape, TORCH[case["dtype"]])
    return dict(case=case, engine=eng, out=out)


# ---- one pass --------------------------------------------------------------------

def _conv_out(case):
    k, s, p = case["k"], case["stride"], case["pad"]
    return (case["h"] + 2 * p - k) // s + 1, (case["w"] + 2 * p - k) // s + 1


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ffn":
        be, m, d, f = state["be"], case["m"], case["d"], case["ffn"]
        be.matmul(state["x"], state["w1"], state["h"], m, d, f)
        be.add(state["h"], state["b1"], state["h2"], state["bias_f"])
        be.gelu(state["h2"], state["h"], m * f)
        be.matmul(state["h"], state["w2"], state["y"], m, f, d)
        be.add(state["y"], state["b2"], state["y2"], state["bias_d"])
        be.add(state["x"], state["y2"], state["y"], state["same"])
        return state["y"]
    if kind == "conv":
        be, b, oc = state["be"], case["batch"], case["oc"]
        oh, ow = state["y"].shape[2:]
        be.conv2d(state["x"], state["w"], state["b"], state["y"], b, case["ic"], case["h"], case["w"], oc, case["k"], case["k"],
                  case["stride"], case["pad"])
        be.relu(state["y"], state["r"], state["y"].numel())
        be.max_pool2d(state["r"], state["z"], b, oc, oh, ow, case["pool"], case["pool"], 0)
        return state["r"], state["z"]
    if kind == "head":
        be, m, d, n = state["be"], case["m"], case["d"], case["classes"]
        be.layer_norm(state["x"], state["g"], state["o"], state["h"], m, d)
        be.matmul(state["h"], state["w"], state["y"], m, d, n)
        be.add(state["y"], state["b"], state["y2"], state["bias"])
        be.softmax(state["y2"], state["p"], m, n)
        return state["y2"], state["p"]
    if kind == "decode":
        dec = state["decoder"]
        dec.prefill(state["prompt"], logits=False)
        out = np.stack([dec.step(ids)[0] for ids in state["fed"]])
        return torch.from_numpy(out.view(np.int16)).view(TORCH[case["dtype"]])
    state["engine"].run_device()
    return state["out"]


# ---- the work of one pass, tolerance, and the result in 64 bits ---------------------

def work(case):
    kind, s = case["kind"], SIZE[case["dtype"]]
    if kind == "ffn":
        m, d, f = case["m"], case["d"], case["ffn"]
        return {"bytes": s * (2.0 * m * d + 2.0 * d * f + d + f), "flops": 4.0 * m * d * f}
    if kind == "conv":
        (oh, ow), b, k, p = _conv_out(case), case["batch"], case["k"], case["pool"]
        pixels = b * case["oc"] * (oh * ow + (oh // p) * (ow // p))
        return {"bytes": s * (float(b) * case["ic"] * case["h"] * case["w"] + case["oc"] * case["ic"] * k * k + pixels),
                "flops": 2.0 * b * oh * ow * case["oc"] * case["ic"] * k * k}
    if kind == "head":
        m, d, n = case["m"], case["d"], case["classes"]
        return {"bytes": s * (float(m) * d + d * n + n + 2.0 * m * n), "flops": 2.0 * m * d * n}
    cfg = _config(case)
    weights = float(sum(math.prod(shape) for _, shape, role, _ in models.param_specs(cfg) if role != "embed"))
    shape = _input_shape(case)
    if kind in ("mlp", "cnn", "unet"):
        flops, cells = _net_flops(case)
        return {"bytes": s * (weights + math.prod(shape) + cells), "flops": flops}
    b, t, d, f = case["batch"], case["t"], case["heads"] * case["hd"], case["ffn"]

    def block(rows, pairs):  # pairs: (query, key) pairs that attention has to score
        return 2.0 * rows * (4 * d * d + 2 * d * f) + 4.0 * pairs * d

    if kind == "block":
        return {"bytes": s * (weights + 2.0 * b * t * d), "flops": block(b * t, b * t * (t + 1) / 2 if case["causal"] else b * t * t)}
    n, v = case["layers"], case["vocab"]
    if kind == "decoder":
        return {"bytes": s * (weights + 2.0 * b * t * d + b * t * v), "flops": n * block(b * t, b * t * (t + 1) / 2) + 2.0 * b * t * d * v}
    k = case["steps"]
    ends = sum(t + i + 1 for i in range(k))  # keys seen by all steps
    return {"bytes": s * (weights * (k + 1) + n * (2.0 * b * ends * d + 2 * b * t * d) + b * k * v),
            "flops": n * (block(b * t, b * t * (t + 1) / 2) + block(b * k, b * ends)) + 2.0 * b * (t + k) * d * v}


def _net_flops(case):
    """(FLOPs, output values) of the MLP, CNN and UNet."""
    b = case["batch"]
    if case["kind"] == "mlp":
        z = [int(v) for v in case["sizes"].split(",")]
        return 2.0 * b * sum(i * o for i, o in zip(z, z[1:])), b * z[-1]
    if case["kind"] == "cnn":
        p = case["hw"] ** 2
        flat = case["c2"] * p // 16
        return 2.0 * b * (p * 27 * case["c1"] + p // 4 * 9 * case["c1"] * case["c2"] + flat * case["hidden"] + case["hidden"] * 10), b * 10
    total, res = 0.0, {}
    px = case["h"] * case["w"]
    for name, k, ic, oc, ks, stride, _ in models.unet_layers(_config(case)):
        level = int(name[-3] if "." in name else 0 if name == "head" else name[-1])
        if k == "convt":
            total += 2.0 * (px >> (2 * level)) * ic * oc
        else:
            total += 2.0 * (px >> (2 * (level + (stride == 2)))) * ic * oc * ks * ks
    return b * total, b * 2 * px


def tolerance(case):
    """About four times the distance of the outputs from the same sums in 64 bits
    that was measured: single precision differs by its summation order (5e-7,
    3e-6 after a softmax), the 16-bit types by one rounding per operation, which
    travels through the layers (single calls 2e-4 / 3e-3, a block 5e-4 / 4e-3,
    whole decoders 1e-2 in bfloat16)."""
    if case["dtype"] == "float32":
        return {"rel": 1.2e-5, "max": 1e-3}
    whole = case["kind"] in ("decoder", "decode")
    if case["dtype"] == "float16":
        return {"rel": 4e-3 if whole else 2e-3, "max": 0.2}
    return {"rel": 2.5e-2 if whole else 1.5e-2, "max": 0.9}


def exact(case, seed):
    """The pass in float64, in plain torch, from the same stored values."""
    params, x = _made(case, seed)
    p = {k: v.double() for k, v in params.items()}
    kind = case["kind"]
    c = float(torch.tensor(1.702, dtype=TORCH[case["dtype"]]))

    def gelu(v):  # nn::GELU: x sigmoid(1.702 x), the constant held in the dtype
        return v * torch.sigmoid(v * c)

    def linear(v, name):
        return v @ p[name + "weight"] + p[name + "bias"]

    def norm(v, g, o):
        mean = v.mean(-1, keepdim=True)
        var = ((v - mean) ** 2).mean(-1, keepdim=True)
        return (v - mean) / torch.sqrt(var + 1e-5) * g + o

    if kind == "ffn":
        v = x["x"].double()
        return v + (gelu(v @ p["w1"] + p["b1"]) @ p["w2"] + p["b2"])
    if kind == "conv":
        v = torch.relu(_conv(x["x"].double(), p["w"], p["b"], case["stride"], case["pad"]))
        return v, F.max_pool2d(v, case["pool"])
    if kind == "head":
        v = norm(x["x"].double(), p["g"], p["o"]) @ p["w"] + p["b"]
        return v, torch.softmax(v, -1)
    if kind == "mlp":
        v = x["x"].double()
        for i in (0, 2, 4):
            v = linear(v, "%d." % i)
            v = torch.relu(v) if i < 4 else v
        return v
    if kind == "cnn":
        v = x["x"].double()
        for i in (0, 3):
            v = F.max_pool2d(torch.relu(_conv(v, p["%d.weight" % i], p["%d.bias" % i], 1, 1)), 2)
        return linear(torch.relu(linear(v.flatten(1), "7.")), "9.")
    if kind == "unet":
        return _unet(x["x"].double(), p, case["levels"])

    heads, hd = case["heads"], case["hd"]
    scale = float(torch.tensor(1.0 / math.sqrt(hd), dtype=TORCH[case["dtype"]]))
    causal = case.get("causal", True)

    def attention(v, pre):
        b, t, d = v.shape
        q, k, u = (linear(v, pre + n).view(b, t, heads, hd).permute(0, 2, 1, 3).reshape(b * heads, t, hd).contiguous()
                   for n in ("q_proj.", "k_proj.", "v_proj."))
        if kind == "decode":
            keys = k.transpose(1, 2).contiguous()  # key j of a head is its row j
        else:  # MuNet reads k's buffer as a [hd, B H T] matrix
            keys = k.view(hd, b * heads, t).permute(1, 0, 2).contiguous()
        out = torch.empty_like(q)
        mask = torch.ones(t, t, dtype=torch.bool, device=DEV).triu(1) if causal else None
        for z in range(b * heads):
            s = (q[z] @ keys[z]) * scale
            if causal:
                s = s.masked_fill(mask, -math.inf)
            out[z] = torch.softmax(s, -1) @ u[z]
        return linear(out.view(b, heads, t, hd).permute(0, 2, 1, 3).reshape(b, t, d), pre + "out_proj.")

    def block(v, pre):
        v = v + attention(norm(v, p[pre + "ln1.weight"], p[pre + "ln1.bias"]), pre + "attn.")
        h = norm(v, p[pre + "ln2.weight"], p[pre + "ln2.bias"])
        return v + linear(gelu(linear(h, pre + "ff.0.")), pre + "ff.2.")

    if kind == "block":
        return block(x["x"].double(), "")
    ids = x["ids"].long()
    v = p["token_embed.weight"][ids] + p["pos_embed.weight"][: ids.shape[1]]
    for i in range(case["layers"]):
        v = block(v, "blocks.%d." % i)
    v = norm(v, p["ln_f.weight"], p["ln_f.bias"])
    if kind == "decode":
        v = v[:, case["t"]:].transpose(0, 1)
    return linear(v, "head.")


def _conv(v, w, b, stride, pad):
    """A convolution as one product over unfolded patches, image by image."""
    n, _, h, wd = v.shape
    oc, _, k, _ = w.shape
    oh, ow = (h + 2 * pad - k) // stride + 1, (wd + 2 * pad - k) // stride + 1
    wm = w.reshape(oc, -1)
    return torch.stack([wm @ F.unfold(v[i:i + 1], k, padding=pad, stride=stride)[0] + b[:, None] for i in range(n)]).view(n, oc, oh, ow)


def _unet(v, p, levels):
    def conv(v, name, stride=1, pad=1):
        return _conv(v, p[name + ".weight"], p[name + ".bias"], stride, pad)

    skips = []
    for i in range(levels):
        v = torch.relu(conv(torch.relu(conv(v, "enc%d.0" % i)), "enc%d.1" % i))
        if i < levels - 1:
            skips.append(v)
            v = torch.relu(conv(v, "down%d" % i, 2))
    for i in range(levels - 2, -1, -1):
        w, b = p["up%d.weight" % i], p["up%d.bias" % i]  # [iC, oC, 2, 2], stride 2: no overlap
        n, ic, h, wd = v.shape
        oc = w.shape[1]
        y = (v.permute(0, 2, 3, 1).reshape(-1, ic) @ w.reshape(ic, -1)).view(n, h, wd, oc, 2, 2)
        y = y.permute(0, 3, 1, 4, 2, 5).reshape(n, oc, 2 * h, 2 * wd) + b.view(1, -1, 1, 1)
        v = torch.cat([y, skips[i]], 1)
        v = torch.relu(conv(torch.relu(conv(v, "dec%d.0" % i)), "dec%d.1" % i))
    return conv(v, "head", 1, 0)
