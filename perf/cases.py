"""What this library is timed on: its operators as a training or serving program calls them.

A case is one layer (or a short chain of layers) with its sizes, storage type and activation.  `run` makes one pass
through the package's public API: forward and pullback for a training case, forward alone for a serving case.  Inputs
are torch tensors that the library borrows, results are handed back as torch tensors over the library's own memory, and
everything runs on torch's current stream, as in a program that uses both.
"""
import math
import random

import torch

from __graft_entry__ import load_package

lux = load_package()

EPS = 1e-5
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "bf16": 2}


# ------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # a small fully connected layer in training, the size at which launches and latency are the whole cost
        dict(name="dense_small_f32", kind="dense", train=True, dtype="f32", act="tanh", inp=128, out=256, batch=64),
        # a fully connected layer of an ordinary network: no size is a multiple of a tile or of a vector
        dict(name="dense_odd_f32", kind="dense", train=True, dtype="f32", act="gelu", inp=1023, out=517, batch=301),
        # serving: a few tokens at a time through a wide layer, which reads the weight once and does little else
        dict(name="dense_serving_bf16", kind="dense", train=False, dtype="bf16", act="gelu", inp=4096, out=11008, batch=3),
        # the feed-forward block of a transformer in training: layernorm, dense with gelu, dense
        dict(name="mlp_block_bf16", kind="mlp", dtype="bf16", width=4096, hidden=11008, tokens=8192),
        # batchnorm with running statistics, then bias and activation, in training
        dict(name="batchnorm_swish_f32", kind="batchnorm", dtype="f32", act="swish", w=32, h=32, c=64, n=128),
        # groupnorm with its activation in training, in both storage types: a large layer and an ordinary one whose
        # planes are no multiple of a vector
        dict(name="groupnorm_bf16", kind="groupnorm", dtype="bf16", act="swish", w=64, h=64, c=256, n=16, groups=32),
        dict(name="groupnorm_odd_f32", kind="groupnorm", dtype="f32", act="swish", w=35, h=35, c=96, n=24, groups=12),
        # layernorm over the features of every token in training, an odd number of features
        dict(name="layernorm_odd_f32", kind="layernorm", dtype="f32", act="identity", width=1023, tokens=6001),
        # a 3x3 convolution in the middle of a network, training, in both storage types
        dict(name="conv3x3_bf16", kind="conv", dtype="bf16", act="relu", w=56, h=56, cin=128, cout=128, k=3, stride=1, n=64),
        dict(name="conv3x3_f32", kind="conv", dtype="f32", act="swish", w=56, h=56, cin=128, cout=128, k=3, stride=1, n=64),
        # the first convolution of an image network: three channels in, a large window, stride two
        dict(name="conv_first_bf16", kind="conv", dtype="bf16", act="relu", w=224, h=224, cin=3, cout=64, k=7, stride=2, n=32),
        # causal self-attention in training
        dict(name="attention_bf16", kind="attention", dtype="bf16", width=128, heads=32, tokens=2048, batch=4, causal=True),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _even(rng, v, step):
    """Three times in five a multiple of `step`, as most layers have; otherwise v as it is."""
    return max(step, v // step * step) if rng.random() < 0.6 else v


def draw(rng: random.Random):
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(["dense", "serving", "mlp", "batchnorm", "groupnorm", "layernorm", "conv", "conv", "attention"])
    dtype = rng.choice(["f32", "bf16"])
    smooth = rng.choice(["identity", "tanh", "gelu", "swish"])
    if kind == "dense":
        return dict(kind="dense", train=True, dtype=dtype, act=smooth, inp=_even(rng, _log(rng, 32, 2048), 16),
                    out=_even(rng, _log(rng, 32, 2048), 16), batch=_even(rng, _log(rng, 16, 2048), 8))
    if kind == "serving":
        return dict(kind="dense", train=False, dtype=dtype, act=smooth, inp=_even(rng, _log(rng, 512, 12288), 64),
                    out=_even(rng, _log(rng, 512, 12288), 64), batch=_log(rng, 1, 16))
    if kind == "mlp":
        width = _even(rng, _log(rng, 512, 4096), 64)
        hidden = _even(rng, int(width * rng.uniform(2.0, 4.0)), 64)
        most = 8192 * 4096 * 11008 // (width * hidden)
        return dict(kind="mlp", dtype="bf16", width=width, hidden=hidden, tokens=_even(rng, _log(rng, 256, min(16384, most)), 64))
    if kind in ("batchnorm", "groupnorm"):
        w = _even(rng, _log(rng, 7, 64), 8)
        groups = rng.choice([4, 8, 12, 16, 32])
        c = groups * rng.choice([2, 3, 4, 8, 8, 16])
        n = _log(rng, 2, max(2, min(128, (1 << 24) // (w * w * c))))
        case = dict(kind=kind, dtype=dtype, act=smooth, w=w, h=w, c=c, n=n)
        return dict(case, groups=groups) if kind == "groupnorm" else case
    if kind == "layernorm":
        width = _even(rng, _log(rng, 64, 8192), 64)
        return dict(kind="layernorm", dtype=dtype, act=rng.choice(["identity", "gelu"]), width=width,
                    tokens=_log(rng, 64, (1 << 25) // width))
    if kind == "conv":
        k, stride = rng.choice([(1, 1), (3, 1), (3, 1), (3, 2), (5, 1), (7, 2)])
        cin = 3 if k == 7 else _even(rng, _log(rng, 16, 256), 16)
        cout = _even(rng, _log(rng, 16, 256), 16)
        w = _even(rng, _log(rng, 14, 224 if k == 7 else 112), 14)
        per = cin * cout * k * k * (-(-w // stride)) ** 2
        n = _log(rng, 1, max(1, min(64, 3 * 64 * 49 * 112 * 112 * 32 // per, (1 << 25) // (w * w * max(cin, cout)))))
        return dict(kind="conv", dtype=dtype, act="relu" if dtype == "bf16" else "swish", w=w, h=w, cin=cin, cout=cout, k=k,
                    stride=stride, n=n)
    width = rng.choice([32, 48, 64, 64, 80, 96, 128, 128])
    tokens = _even(rng, _log(rng, 64, 2048), 64)
    heads = rng.choice([2, 4, 8, 12, 16, 32])
    most = (128 * 2048 * 2048 * 32 * 4 // (16 if dtype == "f32" else 1)) // (width * tokens * tokens * heads)
    return dict(kind="attention", dtype=dtype, width=width, heads=heads, tokens=tokens, batch=_log(rng, 1, max(1, min(16, most))),
                causal=rng.random() < 0.5)


def _conv_sizes(case):
    pad = case["k"] // 2
    ow, oh = ((case[d] + 2 * pad - case["k"]) // case["stride"] + 1 for d in "wh")
    return pad, ow, oh


# ------------------------------------------------------------------------------------------------ torch <-> library
def _lend(t: torch.Tensor, shape):
    """The library's view of a torch tensor: `shape` is column-major, so a C-contiguous tensor has it reversed."""
    return lux.DeviceArray(shape, "bf16" if t.dtype == torch.bfloat16 else "f32", ptr=t.data_ptr(), base=t)


class _Memory:
    __slots__ = ("array", "__cuda_array_interface__")

    def __init__(self, a):
        self.array = a
        self.__cuda_array_interface__ = {"shape": a.shape[::-1], "typestr": "<f4" if a.dtype == "f32" else "<i2",
                                         "data": (a.ptr, False), "version": 2}


def _tensor(a):
    """A torch tensor over the memory of one of the library's arrays, which it keeps alive."""
    t = torch.as_tensor(_Memory(a), device="cuda")
    return t if a.dtype == "f32" else t.view(torch.bfloat16)


def _tensors(*arrays):
    return [_tensor(a) for a in arrays]


# ------------------------------------------------------------------------------------------------ preparation
def prepare(case, seed):
    lux.init(0, own_stream=False)
    lux.set_stream(torch.cuda.current_stream().cuda_stream)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    dt = TORCH[case["dtype"]]

    def normal(*shape, scale=1.0, shift=0.0):
        t = torch.empty(shape[::-1], dtype=torch.float32, device="cuda").normal_(shift, scale, generator=gen)
        return _lend(t.to(dt), shape)

    def uniform(*shape, lo=0.5, hi=1.5):
        t = torch.empty(shape[::-1], dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=gen)
        return _lend(t.to(dt), shape)

    kind, s = case["kind"], {"case": case}
    if kind == "dense":
        i, o, b = case["inp"], case["out"], case["batch"]
        s.update(w=normal(o, i, scale=math.sqrt(2.0 / (i + o))), x=normal(i, b), b=normal(o, scale=0.01))
        if case["train"]:
            s.update(d=normal(o, b))
    elif kind == "mlp":
        d, f, t = case["width"], case["hidden"], case["tokens"]
        std = math.sqrt(2.0 / (d + f))
        s.update(x=normal(d, t), g=uniform(d, 1), be=normal(d, 1, scale=0.1), w1=normal(f, d, scale=std), b1=normal(f, scale=0.01),
                 w2=normal(d, f, scale=std), b2=normal(d, scale=0.01), d=normal(d, t, scale=0.02))
    elif kind in ("batchnorm", "groupnorm"):
        shape, c = (case["w"], case["h"], case["c"], case["n"]), case["c"]
        s.update(x=normal(*shape, scale=2.0, shift=0.5), g=uniform(c), be=normal(c, scale=0.1), d=normal(*shape))
        if kind == "batchnorm":
            s.update(rm=normal(c, scale=0.1), rv=uniform(c), b2=normal(c, scale=0.1))
    elif kind == "layernorm":
        shape = (case["width"], case["tokens"])
        s.update(x=normal(*shape, scale=2.0, shift=0.5), g=uniform(shape[0], 1), be=normal(shape[0], 1, scale=0.1), d=normal(*shape))
    elif kind == "conv":
        pad, ow, oh = _conv_sizes(case)
        xs, ws = (case["w"], case["h"], case["cin"], case["n"]), (case["k"], case["k"], case["cin"], case["cout"])
        s.update(x=normal(*xs), w=normal(*ws, scale=math.sqrt(2.0 / (case["k"] ** 2 * case["cin"]))), b=normal(case["cout"], scale=0.01),
                 d=normal(ow, oh, case["cout"], case["n"]), dims=lux.DenseConvDims(xs, ws, stride=case["stride"], padding=pad))
    else:
        shape = (case["width"], case["heads"], case["tokens"], case["batch"])
        s.update(q=normal(*shape), k=normal(*shape), v=normal(*shape), d=normal(*shape))
    return s


# ------------------------------------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    act = case.get("act")
    if kind == "dense":
        if not case["train"]:
            return _tensors(lux.fused_dense_bias_activation(act, s["w"], s["x"], s["b"]))
        y, back = lux.pullback(lux.fused_dense_bias_activation, act, s["w"], s["x"], s["b"])
        return _tensors(y, *back(s["d"]))
    if kind == "mlp":
        h0, back0 = lux.pullback(lux.layernorm, s["x"], s["g"], s["be"], "identity", (1,), EPS)
        h1, back1 = lux.pullback(lux.fused_dense_bias_activation, "gelu", s["w1"], h0, s["b1"])
        y, back2 = lux.pullback(lux.fused_dense_bias_activation, "identity", s["w2"], h1, s["b2"])
        dw2, dh1, db2 = back2(s["d"])
        dw1, dh0, db1 = back1(dh1)
        dx, dg, dbe = back0(dh0)
        return _tensors(y, dw2, db2, dw1, db1, dx, dg, dbe)
    if kind == "batchnorm":
        (y1, stats), back1 = lux.pullback(lux.batchnorm, s["x"], s["g"], s["be"], s["rm"], s["rv"], True, "identity", 0.1, EPS)
        y, back2 = lux.pullback(lux.bias_activation, act, y1, s["b2"])
        dy1, db2 = back2(s["d"])
        return _tensors(y, stats["running_mean"], stats["running_var"], db2, *back1(dy1))
    if kind == "groupnorm":
        y, back = lux.pullback(lux.groupnorm, s["x"], s["g"], s["be"], case["groups"], act, EPS)
        return _tensors(y, *back(s["d"]))
    if kind == "layernorm":
        y, back = lux.pullback(lux.layernorm, s["x"], s["g"], s["be"], act, (1,), EPS)
        return _tensors(y, *back(s["d"]))
    if kind == "conv":
        y, back = lux.pullback(lux.fused_conv_bias_activation, act, s["w"], s["x"], s["b"], s["dims"])
        return _tensors(y, *back(s["d"]))
    (y, weights), back = lux.pullback(lux.scaled_dot_product_attention, s["q"], s["k"], s["v"], 1, 3, None, None,
                                      True if case["causal"] else None)
    return _tensors(y, weights, *back(s["d"]))


# ------------------------------------------------------------------------------------------------ work and tolerance
def work(case):
    kind, e = case["kind"], BYTES[case["dtype"]]
    if kind == "dense":
        i, o, b = case["inp"], case["out"], case["batch"]
        if not case["train"]:
            return {"bytes": e * (o * i + i * b + o + o * b), "flops": 2.0 * i * o * b}
        # forward: w, x, bias in, y out; pullback: delta in, dw, dx, dbias out
        return {"bytes": e * (2 * o * i + 2 * i * b + 2 * o * b + 2 * o), "flops": 3 * 2.0 * i * o * b}
    if kind == "mlp":
        d, f, t = case["width"], case["hidden"], case["tokens"]
        return {"bytes": e * (4 * d * t + 4 * d * f), "flops": 6 * 2.0 * d * f * t}
    if kind in ("batchnorm", "groupnorm", "layernorm"):
        size = case["width"] * case["tokens"] if kind == "layernorm" else case["w"] * case["h"] * case["c"] * case["n"]
        # the statistics need all of x before the first result, the pullback needs its sums before dx: x in, y out,
        # delta and x in, dx out
        return {"bytes": e * 5 * size, "flops": 30.0 * size}
    if kind == "conv":
        _, ow, oh = _conv_sizes(case)
        x, y = case["w"] * case["h"] * case["cin"] * case["n"], ow * oh * case["cout"] * case["n"]
        w = case["k"] ** 2 * case["cin"] * case["cout"]
        return {"bytes": e * (2 * x + 2 * y + 2 * w), "flops": 3 * 2.0 * w * ow * oh * case["n"]}
    tok, share = case["tokens"], (case["tokens"] + 1) / (2.0 * case["tokens"]) if case["causal"] else 1.0
    x = case["width"] * case["heads"] * tok * case["batch"]
    weights = tok * tok * case["heads"] * case["batch"]
    # q, k, v, delta in, out, dq, dk, dv out, the weights out; six products over the positions that count
    return {"bytes": e * (8 * x + weights), "flops": 6 * 2.0 * case["width"] * weights * share}


def tolerance(case):
    """Against torch in 64 bits the worst relative error of an output over the listed cases and 16 drawn ones was 3.7e-3
    in bf16 (gradients that pass three stored bf16 tensors) and 1.0e-6 in fp32 (contractions over 2000 terms)."""
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 5e-6}
