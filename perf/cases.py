"""The work whose time matters: what a program that runs language models, mixture-of-experts layers, vision encoders
and classifiers over weight-compressed FullyConnected nodes asks of this library.

A case is one layer's worth of calls through the public entry points on one request: the nodes are created once from
constants in OpenVINO's layout, the activations lie in device memory (in host memory for the classifier head), one pass
enqueues every call of the layer.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from openvino_amd import fc

# hidden size, width of k and of v, width of the gated MLP
_BLOCK_8B = {"hidden": 4096, "kv": 1024, "ffn": 14336}
_BLOCK_70B = {"hidden": 8192, "kv": 1024, "ffn": 28672}


def listed():
    return [
        # One token of one sequence: the decoder block of a chat at 4 bits, groups of 128, symmetric.
        {"name": "decode-1", "kind": "block", "rows": 1, **_BLOCK_8B, "weights": "i4", "group": 128, "zp": "none",
         "act": "f16"},
        # A dozen sequences decoding together, asymmetric 4-bit weights.
        {"name": "decode-12", "kind": "block", "rows": 12, **_BLOCK_8B, "weights": "u4", "group": 128, "zp": "u4",
         "act": "f16"},
        # A short prompt, at the finer group size that smaller models are exported with.
        {"name": "prompt-117-g64", "kind": "block", "rows": 117, **_BLOCK_8B, "weights": "i4", "group": 64,
         "zp": "none", "act": "f16"},
        # An ordinary prompt (or a chunk of a long one).
        {"name": "prompt-2048", "kind": "block", "rows": 2048, **_BLOCK_8B, "weights": "i4", "group": 128,
         "zp": "none", "act": "f16"},
        # A long document in one go: as many rows as the text has tokens, no multiple of anything.
        {"name": "prompt-5003", "kind": "block", "rows": 5003, **_BLOCK_8B, "weights": "u4", "group": 128, "zp": "u4",
         "act": "f16"},
        # One token of a larger model at 8 bits, one scale and zero-point per channel.
        {"name": "decode-1-w8", "kind": "block", "rows": 1, **_BLOCK_70B, "weights": "u8", "group": 0, "zp": "u8",
         "act": "f16"},
        # The same model serving two dozen sequences.
        {"name": "decode-24-w8", "kind": "block", "rows": 24, **_BLOCK_70B, "weights": "u8", "group": 0, "zp": "u8",
         "act": "f16"},
        # The same model reading a prompt with its activations quantised to int8 per token.
        {"name": "prompt-1024-w8a8", "kind": "block", "rows": 1024, **_BLOCK_70B, "weights": "u8", "group": 0,
         "zp": "u8", "act": "int8"},
        # The expert block of a mixture-of-experts layer over a batch of tokens, routed on the device.
        {"name": "experts-256", "kind": "experts", "rows": 256, "hidden": 4096, "ffn": 14336, "experts": 8, "top_k": 2,
         "weights": "u4", "group": 128, "zp": "u4"},
        # The same layer while a few sequences decode.
        {"name": "experts-6", "kind": "experts", "rows": 6, "hidden": 4096, "ffn": 14336, "experts": 8, "top_k": 2,
         "weights": "u4", "group": 128, "zp": "u4"},
        # A layer of a vision or text encoder (q/k/v, output, two MLP projections, biases) whose widths fit no tile.
        {"name": "encoder-577", "kind": "encoder", "rows": 577, "hidden": 1160, "ffn": 4300, "weights": "i8"},
        # The last layer of an image classifier, called with host tensors: the smallest call a program makes.
        {"name": "head-8", "kind": "head", "rows": 8, "classes": 1000, "features": 2048, "weights": "i8"},
    ]


_LARGEST_FLOPS = 2.0 * 5003 * (4096 * (2 * 4096 + 2 * 1024) + 3 * 4096 * 14336)


def _spread(rng, low, high):
    """A whole number of low .. high, even over its logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(["block", "block", "block", "block", "experts", "encoder", "head"])
    if kind == "block":
        hidden = 128 * rng.randint(16, 64)
        case = {"kind": kind, "rows": 0, "hidden": hidden,
                "kv": max(128, hidden // rng.choice([1, 2, 4, 8]) // 128 * 128),
                "ffn": 128 * round(hidden * rng.uniform(2.5, 4.0) / 128)}
        case["weights"], case["group"], case["zp"] = rng.choice([
            ("i4", 128, "none"), ("i4", 128, "none"), ("u4", 128, "u4"), ("u4", 128, "u4"), ("i4", 64, "none"),
            ("u4", 64, "u4"), ("i4", 32, "none"), ("u8", 0, "u8"), ("i8", 0, "none")])
        per_row = 2.0 * (hidden * (2 * hidden + 2 * case["kv"]) + 3 * hidden * case["ffn"])
        case["rows"] = _spread(rng, 1, min(5003, int(_LARGEST_FLOPS / per_row)))
        case["act"] = "int8" if case["weights"] in ("u8", "i8") and case["rows"] > 48 and rng.random() < 0.5 else "f16"
        return case
    if kind == "experts":
        hidden = 256 * rng.randint(8, 16)
        group, zp = rng.choice([(128, "u4"), (128, "none"), (64, "u4")])
        return {"kind": kind, "rows": _spread(rng, 1, 1024), "hidden": hidden, "ffn": 256 * rng.randint(8, 56),
                "experts": rng.choice([8, 8, 16]), "top_k": rng.choice([1, 2, 4]),
                "weights": "u4" if zp == "u4" else "i4", "group": group, "zp": zp}
    if kind == "encoder":
        hidden = 8 * rng.randint(48, 200)
        return {"kind": kind, "rows": _spread(rng, 16, 1500), "hidden": hidden,
                "ffn": rng.choice([4 * hidden, 2 * round(hidden * rng.uniform(1.4, 2.2))]),
                "weights": rng.choice(["i8", "i8", "u8"])}
    return {"kind": kind, "rows": _spread(rng, 1, 256), "classes": _spread(rng, 10, 4000),
            "features": 2 * _spread(rng, 256, 2048), "weights": rng.choice(["i8", "u8"])}


# ---- what a program keeps ------------------------------------------------------------------------------------------

_kept = []


def _session():
    """The device and the one request (stream) that a serving process keeps."""
    if not _kept:
        dev = fc.Device(0)
        _kept.append((dev, fc.InferRequest(dev)))
    return _kept[0]


class _State:
    """Nodes, tensors and the calls of one pass; gives the nodes back when it goes."""

    def __init__(self):
        self.nodes, self.tensors, self.calls, self.outputs = [], [], [], []

    def __del__(self):
        if self.nodes and _kept:
            _kept[0][1].sync()
            for node in self.nodes:
                node.close()


class _Source:
    """Seeded constants and activations."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed * 7919 + 11)

    def bytes(self, n, low=0, high=256):
        return torch.randint(low, high, (n,), generator=self.gen, device="cuda", dtype=torch.uint8).cpu().numpy()

    def nibbles(self, n, low, high):
        v = torch.randint(low, high, (2, (n + 1) // 2), generator=self.gen, device="cuda", dtype=torch.uint8)
        return (v[0] | (v[1] << 4)).cpu().numpy()

    def activations(self, *shape):
        """Normal values with one channel in a thousand twenty times larger, as normalised hidden states have."""
        x = torch.randn(shape, generator=self.gen, device="cuda")
        loud = torch.rand(shape[-1], generator=self.gen, device="cuda") < 1e-3
        return torch.where(loud, 20.0 * x, x).half()

    def node(self, dev, n, k, weights, group, zp, act="f16", glu=None, bias=False, out="f16"):
        """A node whose dequantised weights have a standard deviation of about 1 / sqrt(K)."""
        g = group or k
        four = weights in ("u4", "i4")
        # zero-points near the middle of the range, as an asymmetric quantiser leaves them
        w = self.bytes(n * k // 2 if four else n * k)
        step = 1.0 / ((4.6 if four else 74.0) * math.sqrt(k))
        s = (torch.rand((n, k // g), generator=self.gen, device="cuda") + 0.5) * step
        z = None
        if zp == "u4":
            z = self.nibbles(n * (k // g), 6, 11)
        elif zp == "u8":
            z = self.bytes(n * (k // g), 100, 157)
        b = torch.randn(n, generator=self.gen, device="cuda").half().cpu().numpy() if bias else None
        return fc.CompressedWeights(dev, w, s.half().cpu().numpy(), z, b, N=n, K=k, group_size=g, w_type=weights,
                                    zp_type=zp, output_type=out, glu=glu, dynamic_quantization=act == "int8")


def _mlp(src, dev, c, act):
    """gate/up with its gated linear unit and the down projection, as one node"""
    gate_up = src.node(dev, 2 * c["ffn"], c["hidden"], c["weights"], c["group"], c["zp"], act, glu="swish")
    down = src.node(dev, c["hidden"], c["ffn"], c["weights"], c["group"], c["zp"], act)
    node = fc.CompressedWeights.mlp(gate_up, down)
    gate_up.close()
    down.close()
    return node


def prepare(case, seed):
    dev, _ = _session()
    src, st, c, m = _Source(seed), _State(), case, case["rows"]
    if c["kind"] == "head":
        node = src.node(dev, c["classes"], c["features"], c["weights"], 0, "none", bias=True, out="f32")
        st.nodes.append(node)
        st.host = (node, src.activations(m, c["features"]).relu().cpu().numpy())
        return st
    if c["kind"] == "experts":
        e, h, f, k = c["experts"], c["hidden"], c["ffn"], c["top_k"]
        st.gate_up = [src.node(dev, 2 * f, h, c["weights"], c["group"], c["zp"], glu="swish") for _ in range(e)]
        st.down = [src.node(dev, h, f, c["weights"], c["group"], c["zp"]) for _ in range(e)]
        st.nodes += st.gate_up + st.down
        x = src.activations(m, h)
        score = torch.randn((m, e), generator=src.gen, device="cuda").softmax(-1)
        top, chosen = score.topk(k, dim=-1)
        routing, chosen = (top / top.sum(-1, keepdim=True)).half(), chosen.to(torch.int32).contiguous()
        y = torch.empty((m, h), dtype=torch.float16, device="cuda")
        st.tensors, st.outputs = [x, routing, chosen], [y]
        torch.cuda.synchronize()
        return st
    if c["kind"] == "encoder":
        h, f, w = c["hidden"], c["ffn"], c["weights"]
        nodes = [src.node(dev, n, k, w, 0, "none", bias=True) for n, k in ((3 * h, h), (h, h), (f, h), (h, f))]
    else:
        h, w, g, z, act = c["hidden"], c["weights"], c["group"], c["zp"], c["act"]
        nodes = [src.node(dev, h + 2 * c["kv"], h, w, g, z, act), src.node(dev, h, h, w, g, z, act),
                 _mlp(src, dev, c, act)]
    st.nodes = nodes
    for node in nodes:
        x = src.activations(m, node.K)
        y = torch.empty((m, node.N_out), dtype=torch.float16, device="cuda")
        st.tensors.append(x)
        st.outputs.append(y)
        st.calls.append((node, x.data_ptr(), y.data_ptr()))
    st.rows = m
    torch.cuda.synchronize()
    return st


def run(st):
    req = _kept[0][1]
    if hasattr(st, "host"):
        return req.infer(*st.host)
    if hasattr(st, "gate_up"):
        x, routing, chosen = st.tensors
        req.moe_routed_device(st.gate_up, st.down, x.data_ptr(), routing.data_ptr(), chosen.data_ptr(), x.shape[0],
                              chosen.shape[1], st.outputs[0].data_ptr())
        return st.outputs
    for node, x_ptr, y_ptr in st.calls:
        req.infer_device(node, x_ptr, y_ptr, st.rows)
    return st.outputs


def _node_bytes(n, k, weights, group, zp):
    """constants of a node as OpenVINO stores them"""
    groups = k // (group or k)
    return n * k * (0.5 if weights in ("u4", "i4") else 1) + n * groups * (2 + {"none": 0, "u4": 0.5, "u8": 1}[zp])


def work(case):
    c, m = case, case["rows"]
    if c["kind"] == "head":
        n, k = c["classes"], c["features"]
        return {"bytes": n * k + 4 * n + m * (2 * k + 4 * n), "flops": 2 * m * n * k}
    if c["kind"] == "encoder":
        shapes = ((3 * c["hidden"], c["hidden"]), (c["hidden"],) * 2, (c["ffn"], c["hidden"]), (c["hidden"], c["ffn"]))
        return {"bytes": sum(n * k + 4 * n + 2 * m * (n + k) for n, k in shapes),
                "flops": sum(2 * m * n * k for n, k in shapes)}
    h, f = c["hidden"], c["ffn"]
    w = (c["weights"], c["group"], c["zp"])
    mlp = _node_bytes(2 * f, h, *w) + _node_bytes(h, f, *w)
    if c["kind"] == "experts":
        # the experts that random routing reaches
        reached = c["experts"] * (1 - (1 - c["top_k"] / c["experts"]) ** m)
        return {"bytes": reached * mlp + m * (4 * h + 6 * c["top_k"]), "flops": 2 * m * c["top_k"] * 3 * h * f}
    n = h + 2 * c["kv"]
    return {"bytes": _node_bytes(n, h, *w) + _node_bytes(h, h, *w) + mlp + 2 * m * ((h + n) + 2 * h + 2 * h),
            "flops": 2 * m * (n * h + h * h + 3 * h * f)}


def tolerance(case):
    """Four times the distance from the same products in 64 bits: 4.3e-4 for f16 results (the rounding of the result, of
    the scaled weights and of the row between two projections), 7e-8 for f32 results, where a sum in another order
    moves the last bits.  int8 activations are quantised the same way by everyone who follows the definition."""
    return {"rel": 1e-6 if case["kind"] == "head" else 1.7e-3}
