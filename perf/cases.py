"""The work that a user has this framework do on one MI355X, as measurable cases.

A program compiles a graph once (``compile_graph``), keeps a ``HipExecutor``
with the weights on the device, writes its input there and runs the plan as
often as it has inputs. ``prepare`` does the first part, ``run`` one pass of
the plan; the outputs are views of the executor's own device buffers. The
one case that serves a single image goes through ``HipExecutor.run`` with
host arrays on both sides, as a request handler does.

Kinds: ``net`` (ResNet-18), ``gemm`` (Gemm + bias + ReLU), ``conv`` (Conv +
bias + ReLU, optionally with a residual add), ``dwconv`` (depthwise Conv +
Clip), ``qgemm`` (int8 Gemm, requantized), ``qblock`` (an int8 RepViT block:
quantized input, token mixer, 1x1, GELU lookup, 1x1, residual add).
"""

from __future__ import annotations

import math

import numpy as np
import torch

from mdlc_amd.codegen.hip.hip_executor import HipExecutor
from mdlc_amd.compiler import compile_graph
from mdlc_amd.tools.build_repvit_int8 import gelu_table
from mdlc_amd.tools.build_resnet18 import build_resnet18
from mdlc_amd.tools.graph_builder import GraphBuilder


def listed():
    return [
        # the headline workload: a batch of images through ResNet-18
        {"name": "resnet18_b32", "kind": "net", "batch": 32, "host": False},
        # one image served from host memory, logits back on the host
        {"name": "resnet18_b1_request", "kind": "net", "batch": 1, "host": True},
        # a large fused Gemm (throughput)
        {"name": "gemm_4096", "kind": "gemm", "M": 4096, "N": 4096, "K": 4096},
        # an odd-sized Gemm: no dimension a multiple of a tile, N and K odd
        {"name": "gemm_ragged", "kind": "gemm", "M": 1000, "N": 1511, "K": 777},
        # a classifier-sized Gemm with a deep K (latency; too few tiles to fill the chip)
        {"name": "gemm_small_deep", "kind": "gemm", "M": 49, "N": 512, "K": 4608},
        # a residual block's second 3x3 convolution
        {"name": "conv3x3_res", "kind": "conv", "batch": 32, "C": 128, "OC": 128, "H": 28, "W": 28,
         "k": 3, "s": 1, "res": True},
        # a strided 3x3 convolution on an odd plane (downsampling layer)
        {"name": "conv3x3_s2_odd", "kind": "conv", "batch": 8, "C": 192, "OC": 320, "H": 27, "W": 27,
         "k": 3, "s": 2, "res": False},
        # MobileNetV2's expanding 1x1 convolution
        {"name": "conv1x1_expand", "kind": "conv", "batch": 32, "C": 96, "OC": 576, "H": 14, "W": 14,
         "k": 1, "s": 1, "res": False},
        # MobileNetV2's depthwise 3x3 on a large plane (bandwidth)
        {"name": "dwconv_56", "kind": "dwconv", "batch": 32, "C": 144, "H": 56, "W": 56, "s": 1},
        # a large requantized int8 Gemm
        {"name": "qgemm_4096", "kind": "qgemm", "M": 4096, "N": 4096, "K": 4096},
        # a mid-sized int8 Gemm with ragged rows and columns
        {"name": "qgemm_ragged", "kind": "qgemm", "M": 700, "N": 1000, "K": 1536},
        # an int8 RepViT stage-3 block
        {"name": "qblock_14", "kind": "qblock", "batch": 32, "C": 192, "H": 14, "W": 14},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] >= 5e7 or w["bytes"] >= 1.5e7 or case["kind"] == "net":   # over a launch's own time
            return case


def _draw(rng):
    kind = rng.choice(["gemm", "gemm", "conv", "conv", "conv", "dwconv", "qgemm", "qblock", "net"])
    if kind == "net":
        return {"kind": "net", "batch": _log_int(rng, 1, 32), "host": False}
    if kind in ("gemm", "qgemm"):
        # rows from one image's classifier to a large batch, odd sizes among them
        M, N, K = _log_int(rng, 1, 4096), _log_int(rng, 48, 4096), _log_int(rng, 64, 4096)
        if rng.random() < 0.6:                  # most layers have channel counts in multiples of 16
            N, K = -(-N // 16) * 16, -(-K // 16) * 16
        if kind == "qgemm":
            K = -(-K // 16) * 16                # what the int8 Gemm accepts
        return {"kind": kind, "M": M, "N": N, "K": K}
    if kind == "qblock":
        return {"kind": "qblock", "batch": _log_int(rng, 1, 32), "C": 48 * rng.choice([1, 2, 4, 8]),
                "H": rng.choice([7, 14, 19, 28]), "W": rng.choice([7, 14, 19, 28])}
    H = rng.choice([7, 13, 14, 19, 28, 35, 56])
    W = H if rng.random() < 0.7 else rng.choice([9, 16, 27, 40])
    batch = _log_int(rng, 1, 32)
    if kind == "dwconv":
        return {"kind": "dwconv", "batch": batch, "C": _log_int(rng, 32, 512), "H": H, "W": W,
                "s": rng.choice([1, 1, 2])}
    C, OC = (_log_int(rng, 32, 512) for _ in range(2))
    if rng.random() < 0.7:
        C, OC = -(-C // 16) * 16, -(-OC // 16) * 16
    k = rng.choice([1, 3, 3])
    s = rng.choice([1, 1, 2])
    return {"kind": "conv", "batch": batch, "C": C, "OC": OC, "H": H, "W": W, "k": k, "s": s,
            "res": s == 1 and rng.random() < 0.4}


# ----- inputs and weights, from the seed ------------------------------------------

def _out(n, k, s):
    return (n + 2 * (k // 2) - k) // s + 1


def _operands(case, seed):
    """{name: array}: the runtime inputs and the weights of one case."""
    rng = np.random.default_rng(seed)

    def normal(*shape):
        return rng.standard_normal(shape, dtype=np.float32)

    k = case["kind"]
    if k == "net":
        return {"input": normal(case["batch"], 3, 224, 224)}
    if k == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        s = np.float32(1.0 / np.sqrt(K))
        return {"x": normal(M, K), "w": normal(K, N) * s, "b": normal(N) * np.float32(0.1)}
    if k in ("conv", "dwconv"):
        n, c, h, w = case["batch"], case["C"], case["H"], case["W"]
        oc, kk, icg = (case["OC"], case["k"], c) if k == "conv" else (c, 3, 1)
        d = {"x": normal(n, c, h, w), "w": normal(oc, icg, kk, kk) * np.float32(np.sqrt(2.0 / (icg * kk * kk))),
             "b": normal(oc) * np.float32(0.1)}
        if case.get("res"):
            d["r"] = normal(n, oc, h, w)
        return d
    if k == "qgemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"x": rng.integers(-127, 128, (M, K), dtype=np.int8),
                "w": rng.integers(-127, 128, (N, K), dtype=np.int8),
                "b": rng.integers(-1000, 1000, N, dtype=np.int32),
                "m": (rng.uniform(0.5, 1.0, N) * (60.0 / (5400.0 * np.sqrt(K)))).astype(np.float32)}
    n, c, h, w = case["batch"], case["C"], case["H"], case["W"]
    d = {"x": normal(n, c, h, w), "table": gelu_table(0.05, 0.03)}
    for name, oc, taps, shape in (("mix", c, 9, (c, 1, 3, 3)), ("up", 2 * c, c, (2 * c, c, 1, 1)),
                                  ("down", c, 2 * c, (c, 2 * c, 1, 1))):
        d[name + ".w"] = rng.integers(-127, 128, shape, dtype=np.int8)
        d[name + ".b"] = rng.integers(-1000, 1000, oc, dtype=np.int32)
        d[name + ".m"] = (rng.uniform(0.5, 1.0, oc) * (50.0 / (4000.0 * np.sqrt(taps)))).astype(np.float32)
    return d


def _conv_attrs(k, s, group=1):
    return dict(kernel_shape=[k, k], strides=[s, s], pads=[k // 2] * 4, dilations=[1, 1], group=group)


def _graph(case, d):
    k = case["kind"]
    if k == "net":
        return build_resnet18(batch=case["batch"])
    b = GraphBuilder(k)
    if k == "gemm":
        b.input("x", d["x"].shape)
        b.const("w", d["w"])
        b.const("b", d["b"])
        b.node("Gemm", ["x", "w", "b"], "pre")
        b.node("Relu", ["pre"], "y")
    elif k == "conv":
        b.input("x", d["x"].shape)
        b.const("w", d["w"])
        b.const("b", d["b"])
        y = b.node("Conv", ["x", "w", "b"], "pre", **_conv_attrs(case["k"], case["s"]))
        if case["res"]:
            b.input("r", d["r"].shape)
            y = b.node("Add", [y, "r"], "sum")
        b.node("Relu", [y], "y")
    elif k == "dwconv":
        b.input("x", d["x"].shape)
        b.const("w", d["w"])
        b.const("b", d["b"])
        b.const("lo", np.float32(0.0))
        b.const("hi", np.float32(6.0))
        b.node("Conv", ["x", "w", "b"], "pre", **_conv_attrs(3, case["s"], case["C"]))
        b.node("Clip", ["pre", "lo", "hi"], "y")
    elif k == "qgemm":
        b.input("x", d["x"].shape, dtype="int8")
        for n in "wbm":
            b.const(n, d[n])
        b.node("QGemm", ["x", "w", "b", "m"], "y", transB=1)
    else:
        b.input("x", d["x"].shape)
        for n, v in d.items():
            if n != "x":
                b.const(n, v)
        q = b.node("QuantizeLinear", ["x"], "q", inv_scale=32.0)
        t = b.node("QConv", [q, "mix.w", "mix.b", "mix.m"], "t", **_conv_attrs(3, 1, case["C"]))
        h = b.node("QConv", [t, "up.w", "up.b", "up.m"], "h", **_conv_attrs(1, 1))
        g = b.node("QLut", [h, "table"], "g")
        o = b.node("QConv", [g, "down.w", "down.b", "down.m"], "o", **_conv_attrs(1, 1))
        b.node("QAdd", [t, o], "y", ma=0.6, mb=0.5)
    b.output("y")
    return b.graph()


# ----- what a program keeps between calls -----------------------------------------

class _State:
    """A compiled graph on the device, with the inputs written there."""

    def __init__(self, case, seed):
        d = _operands(case, seed)
        g = _graph(case, d)
        self.host = bool(case.get("host"))
        self.feeds = {n: d[n] for n in g.inputs}
        c = compile_graph(g, feeds=self.feeds)
        self.ex = HipExecutor(c.module)
        self.names = list(c.module.graph.outputs)
        for n in self.feeds:
            self.ex.write(n, self.feeds[n])
        self.ex.ctx.synchronize()

    def __del__(self):
        ex = getattr(self, "ex", None)
        if ex is not None:
            ex.close()


class _DeviceArray:
    """An output buffer of an executor as torch reads it; keeps the executor."""

    def __init__(self, state, name):
        ex = state.ex
        shape = tuple(int(v) for v in ex.shapes[name])
        self.nhwc = ex.module.device_layout.get(name) == "NHWC" and len(shape) == 4
        if self.nhwc:
            shape = (shape[0], shape[2], shape[3], shape[1])
        self.state = state
        self.__cuda_array_interface__ = {"shape": shape, "typestr": np.dtype(ex.dtypes[name]).str,
                                         "data": (ex.ptr(name), False), "version": 2}

    def tensor(self):
        t = torch.as_tensor(self, device="cuda")
        return t.permute(0, 3, 1, 2) if self.nhwc else t


def prepare(case, seed):
    torch.cuda.init()
    state = _State(case, seed)
    if not state.host:
        outs = {n: _DeviceArray(state, n).tensor() for n in state.names}
        return {"plan": state.ex.plan, "outputs": outs}
    return {"executor": state, "feeds": state.feeds}


def run(state):
    if "executor" in state:
        return state["executor"].ex.run(state["feeds"])["outputs"]
    state["plan"].run(1)
    return state["outputs"]


# ----- what one pass cannot do without --------------------------------------------

_RESNET18_FLOPS = 3_628_146_688                 # convolutions and classifier of one image
_RESNET18_WEIGHTS = 11_689_512                  # parameters


def work(case):
    k = case["kind"]
    if k == "net":
        n = case["batch"]
        return {"bytes": 4 * (n * (3 * 224 * 224 + 1000) + _RESNET18_WEIGHTS), "flops": n * _RESNET18_FLOPS}
    if k in ("gemm", "qgemm"):
        M, N, K = case["M"], case["N"], case["K"]
        e = 4 if k == "gemm" else 1
        return {"bytes": e * (M * K + K * N + M * N) + 4 * N, "flops": 2 * M * N * K}
    n, c, h, w = case["batch"], case["C"], case["H"], case["W"]
    if k == "qblock":
        px = n * h * w
        return {"bytes": 5 * px * c + 9 * c + 4 * c * c + 32 * c, "flops": 2 * px * (9 * c + 4 * c * c)}
    s = case["s"]
    kk, oc, icg = (case["k"], case["OC"], c) if k == "conv" else (3, c, 1)
    px = n * _out(h, kk, s) * _out(w, kk, s)
    outs = px * oc * (2 if case.get("res") else 1)
    read = n * c * h * w if kk > 1 or s == 1 else px * c
    return {"bytes": 4 * (read + outs + oc * icg * kk * kk + oc), "flops": 2 * px * oc * icg * kk * kk}


def tolerance(case):
    if case["kind"] in ("qgemm", "qblock"):
        return "exact"                          # int8 codes from exact integer sums
    return {"rel": 4e-6}                        # measured against 64 bits: up to 1.1e-6 (K = 4096)


# ----- the same outputs in 64 bits --------------------------------------------------

def _conv64(x, w, b, s, group=1):
    """Conv with symmetric padding k // 2 in float64: one product per tap."""
    n, c, h, wd = x.shape
    oc, icg, k, _ = w.shape
    p = k // 2
    xp = torch.nn.functional.pad(x, (p, p, p, p))
    oh, ow = _out(h, k, s), _out(wd, k, s)
    y = torch.zeros((oc, n * oh * ow) if group == 1 else (n, oc, oh, ow), dtype=torch.float64, device=x.device)
    for i in range(k):
        for j in range(k):
            t = xp[:, :, i:i + (oh - 1) * s + 1:s, j:j + (ow - 1) * s + 1:s]
            if group == 1:
                y += w[:, :, i, j].contiguous() @ t.permute(1, 0, 2, 3).reshape(c, -1)
            else:
                y += w[:, 0, i, j].view(1, -1, 1, 1) * t
    if group == 1:
        y = y.view(oc, n, oh, ow).permute(1, 0, 2, 3)
    return y if b is None else y + b.view(1, -1, 1, 1)


def _net64(g, x):
    """ResNet-18's graph in float64."""
    dev = x.device
    v = {n: torch.from_numpy(np.asarray(a)).to(dev).double() for n, a in g.initializers.items()}
    v["input"] = x
    for n in g.topo_sort():
        i = [v[e] for e in n.inputs]
        if n.op_type == "Identity":
            y = i[0]
        elif n.op_type == "Conv":
            y = _conv64(i[0], i[1], None, n.attrs["strides"][0])
        elif n.op_type == "BatchNormalization":
            sc, sh, mu, var = (t.view(1, -1, 1, 1) for t in i[1:5])
            y = (i[0] - mu) / torch.sqrt(var + n.attrs["epsilon"]) * sc + sh
        elif n.op_type == "Relu":
            y = i[0].clamp(min=0)
        elif n.op_type == "Add":
            y = i[0] + i[1]
        elif n.op_type == "MaxPool":
            t = torch.nn.functional.pad(i[0], (1, 1, 1, 1), value=-math.inf)
            oh, ow = _out(i[0].shape[2], 3, 2), _out(i[0].shape[3], 3, 2)
            y = None
            for a in range(3):
                for b in range(3):
                    q = t[:, :, a:a + 2 * oh - 1:2, b:b + 2 * ow - 1:2]
                    y = q if y is None else torch.maximum(y, q)
        elif n.op_type == "GlobalAveragePool":
            y = i[0].mean(dim=(2, 3), keepdim=True)
        elif n.op_type == "Flatten":
            y = i[0].flatten(1)
        else:                                   # Gemm, transB = 1
            y = i[0] @ i[1].T.contiguous() + i[2]
        v[n.outputs[0]] = y
    return v["logits"]


def exact(case, seed):
    k = case["kind"]
    if k in ("qgemm", "qblock"):
        return None                             # whole codes: compared as they are
    d = _operands(case, seed)
    t = {n: torch.from_numpy(np.asarray(a)).cuda().double() for n, a in d.items()}
    if k == "net":
        return {"logits": _net64(build_resnet18(batch=case["batch"]), t["input"])}
    if k == "gemm":
        return {"y": (t["x"] @ t["w"] + t["b"]).clamp(min=0)}
    if k == "dwconv":
        return {"y": _conv64(t["x"], t["w"], t["b"], case["s"], case["C"]).clamp(0, 6)}
    y = _conv64(t["x"], t["w"], t["b"], case["s"])
    return {"y": (y + t["r"] if "r" in t else y).clamp(min=0)}
