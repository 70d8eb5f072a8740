"""What this backend's performance is measured on: the work a program hands it, through the operator interface of
``tannic_amd.ops``, ``tannic_amd.decoder_layer`` and ``tannic_amd.Graph``.

A case is a dict of plain values.  ``listed()`` names twelve, ``draw(rng)`` gives one more of the same ranges; ``prepare``
makes what a program has in hand before the call (inputs and weights on the device, a recorded sequence where the
program would keep one), ``run`` is one pass, ``work`` what the pass cannot do without and ``tolerance`` how far another
correct implementation at the same precision may be off.

The kinds, and what they stand for:

    linear   one linear layer, ``X[M,K] . W[N,K]^T``, called eagerly: a token at a time, a batch of them, a prompt
    product  a plain matrix product of the front end's default type, both operands row-major
    chain    ``log(|X|+1) + Z*Z - exp(X) + 3*X`` with Z broadcast along two dims, one operator call a node; with
             integers an addition and a comparison, which gives bits
    reduce   one reduction along one dim of a three-dimensional tensor
    convs    the 53 convolutions (stem and sixteen bottleneck blocks with their shortcut additions) of a ResNet-50, batch
             normalisation folded into weights and bias; the backend has no pooling, so the blocks start from a map of their own
    prefill  one decoder layer over a prompt: the one-pass operators with packed projections, or the layer written with
             the front end's own operators only
    decode   one decoder layer over one new token of every sequence, keys and values of the earlier ones in a cache
"""
import math

import torch

import tannic_amd as ta
from tannic_amd import decoder_layer as dl
from tannic_amd import ops

_DTYPES = {"float16": ta.float16, "bfloat16": ta.bfloat16, "float32": ta.float32, "int32": ta.int32}
# (a 16-bit result is looked at as 16-bit integers first: the array interface has no bfloat16)
_TORCH = {"float16": ("<f2", None), "bfloat16": ("<i2", torch.bfloat16), "float32": ("<f4", None), "float64": ("<f8", None),
          "int32": ("<i4", None), "int64": ("<i8", None), "boolean": ("|u1", None)}

# hidden, heads, kv heads, head size, FFN of the decoder layers: the benchmark's, and two smaller of the same proportions
_LAYERS = {"large": (4096, 32, 8, 128, 14336), "middle": (2048, 16, 4, 128, 7168), "small": (1024, 16, 4, 64, 3584)}

# the bottleneck stages of a ResNet-50: blocks, inner width, stride of the first block
_STAGES = ((3, 64, 1), (4, 128, 2), (6, 256, 2), (3, 512, 2))


def listed():
    return [
        # one token through a square projection, called eagerly: the smallest call there is, launch and host count
        {"name": "linear-1-token", "kind": "linear", "dtype": "float16", "m": 1, "n": 4096, "k": 4096},
        # 128 tokens (a batch of sequences, one token each) through the same projection
        {"name": "linear-128-tokens", "kind": "linear", "dtype": "float16", "m": 128, "n": 4096, "k": 4096},
        # a prompt through the wide projection of a feed-forward block
        {"name": "linear-prompt", "kind": "linear", "dtype": "bfloat16", "m": 2048, "n": 14336, "k": 4096},
        # the fp32 product the reference's own CPU path can finish
        {"name": "product-fp32-512", "kind": "product", "dtype": "float32", "m": 512, "n": 512, "k": 512},
        # the broadcasting expression at its full size
        {"name": "chain-fp16", "kind": "chain", "dtype": "float16", "a": 64, "b": 4096, "c": 1024},
        # a sum over the middle dim of the same tensor
        {"name": "reduce-sum-fp32", "kind": "reduce", "dtype": "float32", "op": "sum", "axis": 1, "a": 64, "b": 4096, "c": 1024},
        # image classification in batches, 16-bit
        {"name": "convs-fp16-batch-32", "kind": "convs", "dtype": "float16", "batch": 32, "side": 224, "replay": False},
        # the same in the front end's default type
        {"name": "convs-fp32-batch-32", "kind": "convs", "dtype": "float32", "batch": 32, "side": 224, "replay": False},
        # one image at a time, recorded once: latency
        {"name": "convs-fp16-one-image", "kind": "convs", "dtype": "float16", "batch": 1, "side": 224, "replay": True},
        # a prompt through a decoder layer, one-pass operators, called eagerly
        {"name": "prefill-512", "kind": "prefill", "dtype": "bfloat16", "layer": "large", "seq": 512, "composed": False, "replay": False},
        # the same layer in the front end's own operators, recorded once
        {"name": "prefill-512-composed", "kind": "prefill", "dtype": "bfloat16", "layer": "large", "seq": 512, "composed": True, "replay": True},
        # one more token of one sequence behind a context of two thousand, recorded once
        {"name": "decode-1-sequence", "kind": "decode", "dtype": "bfloat16", "layer": "large", "batch": 1, "context": 2048},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _extent(rng, low, high):
    """Spread over the logarithm of the range; two of three times a multiple of 64 (or of 8 below that), else as it falls."""
    v = _log(rng, low, high)
    step = 64 if v >= 256 else 8 if v >= 16 else 1
    return max(low, v // step * step) if rng.random() < 0.67 else v


def draw(rng):
    kind = rng.choice(["linear", "linear", "product", "chain", "reduce", "convs", "convs", "prefill", "prefill", "decode"])
    if kind in ("linear", "product"):
        dtype = rng.choice(["float16", "bfloat16", "float32"]) if kind == "linear" else rng.choice(["float32", "float32", "float16"])
        while True:
            m, n, k = (_log(rng, 1, 4096), _extent(rng, 256, 16384), _extent(rng, 256, 16384)) if kind == "linear" else (_extent(rng, 32, 4096) for _ in range(3))
            if 2.0 * m * n * k <= (1.4e11 if dtype == "float32" else 4e11):
                return {"kind": kind, "dtype": dtype, "m": m, "n": n, "k": k}
    if kind in ("chain", "reduce"):
        while True:
            a, b, c = _log(rng, 1, 64), _log(rng, 16, 4096), _extent(rng, 16, 4096)
            if 1 << 14 <= a * b * c <= 1 << 28:
                break
        if kind == "chain":
            return {"kind": kind, "dtype": rng.choice(["float16", "bfloat16", "float32", "int32"]), "a": a, "b": b, "c": c}
        dtype = rng.choice(["float16", "bfloat16", "float32", "int32"])
        # (a mean of integers is not offered)
        op = rng.choice(["sum", "max", "argmax"] if dtype == "int32" else ["sum", "mean", "max", "argmax"])
        return {"kind": kind, "dtype": dtype, "op": op, "axis": rng.randrange(3), "a": a, "b": b, "c": c}
    if kind == "convs":
        while True:
            batch, side = _log(rng, 1, 32), rng.randrange(128, 321)
            if batch * side * side <= 32 * 224 * 224:
                side = side // 32 * 32 if rng.random() < 0.5 else side
                return {"kind": kind, "dtype": rng.choice(["float16", "bfloat16", "float32"]), "batch": batch, "side": side, "replay": rng.random() < 0.5}
    layer, dtype = rng.choice(["large", "large", "middle", "small"]), rng.choice(["bfloat16", "bfloat16", "float16"])
    if kind == "prefill":
        return {"kind": kind, "dtype": dtype, "layer": layer, "seq": _extent(rng, 16, 1024), "composed": rng.random() < 0.33, "replay": rng.random() < 0.5}
    return {"kind": kind, "dtype": dtype, "layer": layer, "batch": _log(rng, 1, 32), "context": _extent(rng, 64, 4096)}


# ---- tensors -------------------------------------------------------------------------------------------------------
class _Memory:
    """A tensor's memory as the array interface describes it; keeps the tensor."""

    def __init__(self, tensor, shape):
        self.tensor = tensor
        self.__cuda_array_interface__ = {"shape": shape, "typestr": _TORCH[tensor.dtype.name][0], "data": (tensor.address, False), "strides": None, "version": 2}


def _seen(tensor):
    """A contiguous tensor of the backend, seen by torch without a copy (booleans as their bytes of eight)."""
    shape = (tensor.nbytes,) if tensor.dtype is ta.boolean else tensor.shape
    view = torch.as_tensor(_Memory(tensor, shape), device=_DEVICE)
    as_type = _TORCH[tensor.dtype.name][1]
    return view if as_type is None else view.view(as_type)


_DEVICE = torch.device("cuda", 0)


class _Values:
    """Tensors filled from one seeded generator."""

    def __init__(self, seed):
        self.device = ta.Device(0)
        self.generator = torch.Generator(device=_DEVICE)
        self.generator.manual_seed(seed)

    def normal(self, dtype, shape, sigma=1.0):
        t = ta.Tensor(dtype, shape).initialize(self.device)
        _seen(t).normal_(0.0, sigma, generator=self.generator)
        return t

    def uniform(self, dtype, shape, low, high):
        t = ta.Tensor(dtype, shape).initialize(self.device)
        if dtype.is_integral:
            _seen(t).random_(int(low), int(high), generator=self.generator)
        else:
            _seen(t).uniform_(low, high, generator=self.generator)
        return t

    def ones(self, dtype, shape):
        t = ta.Tensor(dtype, shape).initialize(self.device)
        _seen(t).fill_(1.0)
        return t


# ---- the passes ------------------------------------------------------------------------------------------------------
def _linear(s):
    return ops.matmul(s["x"], s["w"])


def _chain(s):
    x, z = s["x"], s["z"]
    if x.dtype.is_integral:
        return ops.add(x, z), ops.gt(x, s["other"])
    t = ops.log(ops.add(ops.abs(x), s["one"]))
    t = ops.add(t, ops.mul(z, z))
    t = ops.sub(t, ops.exp(x))
    return ops.add(t, ops.scale(x, 3))


def _reduce(s):
    return s["op"](s["x"], s["axis"])


def _blocks(width_in=64):
    """(input width, inner width, stride, has a projection) of every bottleneck block."""
    out = []
    for blocks, width, stride in _STAGES:
        for i in range(blocks):
            out.append((width_in, width, stride if i == 0 else 1, i == 0))
            width_in = 4 * width
    return out


def _convs(s):
    stem = ops.convolve2d(s["image"], *s["stem"], 2, 3)
    x = s["map"]
    for reduce, spatial, expand, project, stride in s["blocks"]:
        y = ops.convolve2d(x, *reduce)
        y = ops.convolve2d(y, *spatial, stride, 1)
        y = ops.convolve2d(y, *expand)
        x = ops.add(y, x if project is None else ops.convolve2d(x, *project, stride))
    return stem, x


def _prefill(s):
    if s["composed"]:
        return dl.forward(s["shape"], s["weights"], s["x"], s["cos"], s["sin"], s["mask"], s["one"])
    return dl.forward_fused(s["shape"], s["weights"], s["x"], s["cos"], s["sin"], s["mask"])


def _decode(s):
    """x: [1, batch, hidden].  The new key and value are written behind the context; every query head of a group meets the
    group's keys in one product."""
    shape, w, x, at = s["shape"], s["weights"], s["x"], s["context"]
    batch, d = x.shape[1], shape.head_dim
    nq, nkv, group = shape.heads * d, shape.kv_heads * d, shape.heads // shape.kv_heads
    qkv = ops.matmul(ops.rms_norm(x, w["g1"], shape.eps), w["wqkv"].transpose()).view(batch, 1, nq + 2 * nkv)
    q = dl.split_heads(qkv[..., 0:nq], shape.heads)
    k = dl.split_heads(qkv[..., nq:nq + nkv], shape.kv_heads)
    v = dl.split_heads(qkv[..., nq + nkv:nq + 2 * nkv], shape.kv_heads)
    ops.copy_into(s["keys"][:, :, at:at + 1, :], ops.rope(k, s["cos"], s["sin"]))
    ops.copy_into(s["values"][:, :, at:at + 1, :], v)
    q = ops.rope(q, s["cos"], s["sin"]).view(batch, shape.kv_heads, group, d)
    scores = ops.matmul(q, s["keys"][:, :, 0:at + 1, :].transpose(-1, -2))
    p = ops.softmax(scores, None, 1.0 / math.sqrt(d))
    o = ops.matmul(p, s["values"][:, :, 0:at + 1, :]).view(1, batch, nq)
    h = ops.add(x, ops.matmul(o, w["wo"].transpose()))
    both = ops.matmul(ops.rms_norm(h, w["g2"], shape.eps), w["w13"].transpose())
    act = ops.swiglu(both[..., 0:shape.ffn], both[..., shape.ffn:2 * shape.ffn])
    return ops.add(h, ops.matmul(act, w["w2"].transpose()))


_PASSES = {"linear": _linear, "product": _linear, "chain": _chain, "reduce": _reduce, "convs": _convs, "prefill": _prefill, "decode": _decode}


# ---- the interface ---------------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind, dtype = case["kind"], _DTYPES[case["dtype"]]
    v = _Values(seed)
    s = {"kind": kind, "graph": None}
    if kind == "linear":        # activations N(0,1), weights N(0,0.02) stored [out, in]
        s["x"] = v.normal(dtype, (case["m"], case["k"]))
        s["w"] = v.normal(dtype, (case["n"], case["k"]), 0.02).transpose()
    elif kind == "product":
        s["x"] = v.uniform(dtype, (case["m"], case["k"]), -1.0, 1.0)
        s["w"] = v.uniform(dtype, (case["k"], case["n"]), -1.0, 1.0)
    elif kind == "chain":
        shape = (case["a"], case["b"], case["c"])
        s["x"] = v.uniform(dtype, shape, -4.0, 4.0)
        s["z"] = v.uniform(dtype, (1, case["b"], 1), -4.0, 4.0)
        if dtype.is_integral:
            s["other"] = v.uniform(dtype, shape, -4.0, 4.0)
        else:
            s["one"] = v.ones(dtype, (1,))
    elif kind == "reduce":
        s["x"] = v.uniform(dtype, (case["a"], case["b"], case["c"]), -4.0, 4.0)
        s["op"], s["axis"] = getattr(ops, case["op"]), case["axis"]
    elif kind == "convs":
        def weights(c, o, k):
            # (the variance that keeps the signal's, as there is no activation between the layers)
            return v.normal(dtype, (o, c, k, k), 1.0 / math.sqrt(c * k * k)), v.normal(dtype, (o,), 0.1)
        side = -(-case["side"] // 4)
        s["image"], s["stem"] = v.normal(dtype, (case["batch"], 3, case["side"], case["side"])), weights(3, 64, 7)
        s["map"] = v.normal(dtype, (case["batch"], 64, side, side))
        s["blocks"] = [(weights(c, width, 1), weights(width, width, 3), weights(width, 4 * width, 1), weights(c, 4 * width, 1) if project else None, stride)
                       for c, width, stride, project in _blocks()]
    else:
        hidden, heads, kv_heads, head_dim, ffn = _LAYERS[case["layer"]]
        s["shape"] = shape = dl.LayerShape(hidden, heads, kv_heads, head_dim, ffn)
        w = {name: v.ones(dtype, size) if name.startswith("g") else v.normal(dtype, size, 0.02) for name, size in dl.weight_shapes(shape).items()}
        s["weights"] = w
        if kind == "prefill":
            s["composed"] = case["composed"]
            if not case["composed"]:
                packed = dl.pack_weights(w)
                s["weights"] = {name: packed[name] for name in ("wqkv", "wo", "w13", "w2", "g1", "g2")}
            s["x"] = v.normal(dtype, (1, case["seq"], hidden))
            s["cos"], s["sin"] = dl.rotary_tables(shape, case["seq"], dtype, v.device)
            s["mask"], s["one"] = dl.causal_mask(case["seq"], dtype, v.device), v.ones(dtype, (1,))
        else:
            packed = dl.pack_weights(w)
            s["weights"] = {name: packed[name] for name in ("wqkv", "wo", "w13", "w2", "g1", "g2")}
            batch, at = case["batch"], case["context"]
            s["x"], s["context"] = v.normal(dtype, (1, batch, hidden)), at
            cos, sin = dl.rotary_tables(shape, at + 1, dtype, v.device)
            s["cos"], s["sin"] = cos[at:at + 1, :], sin[at:at + 1, :]
            # the cache has room for what the sequences may still grow by
            room = (at + 1 + 255) // 256 * 256
            s["keys"] = v.normal(dtype, (batch, kv_heads, room, head_dim), 1.28)
            s["values"] = v.normal(dtype, (batch, kv_heads, room, head_dim), 1.28)
    if kind == "decode" or case.get("replay"):
        # (once eagerly, as a program would before it records)
        _PASSES[kind](s)
        with ta.Graph(v.device) as graph:
            recorded = _PASSES[kind](s)
        s["recorded"] = recorded
        s["results"] = tuple(map(_seen, recorded)) if isinstance(recorded, tuple) else _seen(recorded)
        s["graph"] = graph
    return s


def run(state):
    if state["graph"] is not None:
        state["graph"].launch()
        out = state["results"]
    else:
        out = _PASSES[state["kind"]](state)
        out = tuple(map(_seen, out)) if isinstance(out, tuple) else _seen(out)
    if state["kind"] == "decode":
        return out, _seen(state["keys"]), _seen(state["values"])
    return out


def _map_sides(case):
    """The side of the map behind the first block of every stage."""
    side, out = -(-case["side"] // 4), []
    for _, _, stride in _STAGES:
        side = (side - 1) // stride + 1
        out.append(side)
    return out


def work(case):
    kind, size = case["kind"], 2 if case["dtype"] in ("float16", "bfloat16") else 4
    if kind in ("linear", "product"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": size * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    if kind == "chain":
        n = case["a"] * case["b"] * case["c"]
        if case["dtype"] == "int32":
            return {"bytes": 3 * size * n + n // 8, "flops": 2 * n}
        return {"bytes": 2 * size * n, "flops": 8 * n}
    if kind == "reduce":
        n = case["a"] * case["b"] * case["c"]
        return {"bytes": size * n + (8 if case["op"] == "argmax" else size) * n // (case["a"], case["b"], case["c"])[case["axis"]], "flops": n}
    if kind == "convs":
        batch, side = case["batch"], -(-case["side"] // 4)
        stem = ((case["side"] - 1) // 2 + 1) ** 2
        flops, weights = 2 * batch * stem * 64 * 147, 64 * 147
        sides = _map_sides(case)
        at, stage, left = side, 0, _STAGES[0][0]
        for c, width, stride, project in _blocks():
            after = sides[stage]
            flops += 2 * batch * (at * at * c * width + after * after * (9 * width * width + 4 * width * width + (c * 4 * width if project else 0)))
            weights += c * width + 13 * width * width + (c * 4 * width if project else 0)
            at, left = after, left - 1
            if left == 0 and stage + 1 < len(_STAGES):
                stage, left = stage + 1, _STAGES[stage + 1][0]
        moved = batch * (3 * case["side"] ** 2 + 64 * side * side + 64 * stem + 2048 * sides[-1] ** 2)
        return {"bytes": size * (moved + weights), "flops": flops}
    hidden, heads, kv_heads, d, ffn = _LAYERS[case["layer"]]
    shape = dl.LayerShape(hidden, heads, kv_heads, d, ffn)
    weights = sum(math.prod(v) for v in dl.weight_shapes(shape).values())
    if kind == "prefill":
        # attention is causal: half of the scores are ever used
        seq = case["seq"]
        return {"bytes": size * (weights + 2 * seq * hidden), "flops": dl.flop_count(shape, seq) - 2 * heads * seq * seq * d}
    batch, length = case["batch"], case["context"] + 1
    return {"bytes": size * (weights + 2 * batch * hidden + 2 * batch * kv_heads * length * d),
            "flops": 2 * batch * (weights + 2 * heads * length * d)}


# (rel, max) of another correct implementation: four times what the pass differs by from the same pass in the next wider
# type (16-bit against fp32, fp32 against fp64), the largest seen over the listed cases and ninety drawn ones; rel at most 0.03.
_TOLERANCES = {
    "linear": {"float16": (8e-4, 2e-3), "bfloat16": (7e-3, 1.6e-2), "float32": (2e-6, 1.6e-5)},
    "chain": {"float16": (2.3e-3, 1.4e-2), "bfloat16": (1.8e-2, 9e-2), "float32": (3e-7, 1.6e-6)},
    "reduce": {"float16": (8e-4, 2e-3), "bfloat16": (6e-3, 1.5e-2), "float32": (1.7e-6, 8e-6)},
    "convs": {"float16": (5.6e-3, 3.4e-2), "bfloat16": (3e-2, 2.6e-1), "float32": (1.1e-5, 6.4e-5)},
    "layer": {"float16": (3.6e-3, 2e-2), "bfloat16": (3e-2, 2.2e-1)},
}


def tolerance(case):
    if case["dtype"] == "int32" or case.get("op") in ("max", "argmax"):
        return "exact"
    kind = {"product": "linear", "prefill": "layer", "decode": "layer"}.get(case["kind"], case["kind"])
    rel, largest = _TOLERANCES[kind][case["dtype"]]
    return {"rel": rel, "max": largest}
