"""The split-bf16 fp32 GEMM, convolution and Winograd convolution
(``split_fp32``) on the device.

Every tile shape at sizes that leave remainders in each dimension, against
float64. The bound is the kernel's own: each of the six accumulations a
16-deep k step makes (and each slice of a K split) rounds by at most 2^-24 of
a partial sum, itself at most sum |a||b|, and the three products left out are
below 3 * 2^-25 of sum |a||b|; the epilogue adds a few more roundings.
Infinities, NaNs and values next to FLT_MAX come out as float32 gives them.
"""

from __future__ import annotations

import numpy as np
import pytest

from gpu_util import device_run
from mdlc_amd.codegen.hip import emit
from mdlc_amd.codegen.schedule import CONV_X3_STEP_US, X3_TILES, conv_x3_tile
from mdlc_amd.tools.graph_builder import GraphBuilder
from oracle.reference import run_reference

pytestmark = pytest.mark.gpu


def _bound(K, mag, slices=1):
    return (6 * -(-K // 16) + slices + 8) * 2.0 ** -24 * mag + 1e-30


def _gemm(M, N, K, act=True, seed=0):
    rng = np.random.default_rng(seed)
    b = GraphBuilder("g")
    b.input("x", (M, K))
    w = rng.standard_normal((K, N)).astype(np.float32)
    c = rng.standard_normal(N).astype(np.float32)
    b.const("w", w)
    b.const("c", c)
    b.node("Gemm", ["x", "w", "c"], "p" if act else "y")
    if act:
        b.node("Relu", ["p"], "y")
    b.output("y")
    return b.graph(), rng.standard_normal((M, K)).astype(np.float32), w, c


@pytest.mark.parametrize("tile", X3_TILES, ids=lambda t: t.key())
@pytest.mark.parametrize("shape", [(1, 48, 16, 1), (33, 65, 17, 1), (257, 300, 95, 1), (130, 129, 400, 3),
                                   (300, 520, 777, 2)], ids=lambda s: "x".join(map(str, s)))
def test_gemm_tiles(tile, shape, hip_ctx, monkeypatch):
    import dataclasses

    M, N, K, sk = shape
    monkeypatch.setattr(emit, "x3_schedule", lambda *a: (dataclasses.replace(tile, SK=sk), 0.0))
    g, x, w, c = _gemm(M, N, K)
    cm, got, _ = device_run(g, {"x": x}, ctx=hip_ctx, split_fp32=True)
    assert "x3" in cm.module.plan[0].kernel_name
    want = np.maximum(x.astype(np.float64) @ w + c, 0)
    mag = np.abs(x).astype(np.float64) @ np.abs(w) + np.abs(c)
    assert np.all(np.abs(got["y"] - want) <= _bound(K, mag, sk))


def _conv(n, C, H, W, OC, k, s, d, pads, residual, act=True, seed=0):
    rng = np.random.default_rng(seed)
    b = GraphBuilder("c")
    b.input("x", (n, C, H, W))
    w = rng.standard_normal((OC, C) + tuple(k)).astype(np.float32)
    b.const("w", w)
    b.const("c", rng.standard_normal(OC).astype(np.float32))
    y = b.node("Conv", ["x", "w", "c"], "p" if act else "y", kernel_shape=list(k), strides=list(s), dilations=list(d),
               pads=list(pads), group=1)
    if residual:
        oh = (H + pads[0] + pads[2] - d[0] * (k[0] - 1) - 1) // s[0] + 1
        ow = (W + pads[1] + pads[3] - d[1] * (k[1] - 1) - 1) // s[1] + 1
        b.input("r", (n, OC, oh, ow))
        y = b.node("Add", [y, "r"], "q")
    if act:
        b.node("Relu", [y], "y")
    b.output("y")
    feeds = {"x": rng.standard_normal((n, C, H, W)).astype(np.float32)}
    if residual:
        feeds["r"] = rng.standard_normal((n, OC, oh, ow)).astype(np.float32)
    return b.graph(), feeds, w


def _conv64(x, w, s, d, pads):
    """Float64 correlation, one product per tap."""
    x = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (pads[0], pads[2]), (pads[1], pads[3])))
    kh, kw = w.shape[2:]
    oh = (x.shape[2] - d[0] * (kh - 1) - 1) // s[0] + 1
    ow = (x.shape[3] - d[1] * (kw - 1) - 1) // s[1] + 1
    y = np.zeros((x.shape[0], w.shape[0], oh, ow))
    for i in range(kh):
        for j in range(kw):
            t = x[:, :, i * d[0]:i * d[0] + (oh - 1) * s[0] + 1:s[0], j * d[1]:j * d[1] + (ow - 1) * s[1] + 1:s[1]]
            y += np.einsum("oc,nchw->nohw", w[:, :, i, j].astype(np.float64), t)
    return y


CONVS = [  # n, C, H, W, OC, kernel, strides, dilations, pads, slices, residual
    (3, 24, 9, 11, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 1, True),     # images inside a tile
    (2, 37, 15, 13, 130, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1), 3, False),  # stride 2, ragged channels, slices
    (1, 16, 20, 18, 33, (5, 3), (2, 3), (1, 2), (0, 2, 1, 1), 1, False),   # uneven window, strides, padding
    (5, 48, 7, 7, 100, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 2, True),     # 1x1 across images
    (2, 20, 9, 10, 70, (1, 1), (2, 2), (1, 1), (0, 0, 0, 0), 1, False),    # 1x1 strided
    (1, 8, 30, 5, 16, (3, 3), (1, 1), (3, 1), (3, 1, 3, 1), 1, False),     # dilated
]


@pytest.mark.parametrize("tile", sorted(CONV_X3_STEP_US), ids=lambda t: "w%dx%dn%d" % t)
@pytest.mark.parametrize("case", CONVS, ids=lambda c: "x".join(map(str, c[:6])).replace(" ", ""))
def test_conv_tiles(tile, case, hip_ctx, monkeypatch):
    n, C, H, W, OC, k, s, d, pads, sk, residual = case
    monkeypatch.setattr(emit, "conv_x3_schedule", lambda geo: (conv_x3_tile(geo, *tile, sk), 0.0))
    g, feeds, w = _conv(n, C, H, W, OC, k, s, d, pads, residual)
    cm, got, _ = device_run(g, feeds, ctx=hip_ctx, split_fp32=True, winograd=False)
    assert "x3" in cm.module.plan[0].kernel_name and (len(cm.module.plan) > 1) == (sk > 1)
    c = g.initializers["c"].reshape(1, -1, 1, 1).astype(np.float64)
    r = feeds.get("r", 0.0)
    want = np.maximum(_conv64(feeds["x"], w, s, d, pads) + c + r, 0)
    mag = _conv64(np.abs(feeds["x"]), np.abs(w), s, d, pads) + np.abs(c) + np.abs(r)
    assert np.all(np.abs(got["y"] - want) <= _bound(C * k[0] * k[1] + 32 * k[0] * k[1], mag, sk))


@pytest.mark.parametrize("kind", ["gemm", "conv"])
def test_infinities_and_nans_are_float32s(kind, hip_ctx):
    """Rows (pixels) that read an infinity, a NaN, a float next to FLT_MAX or
    overflow get what float32 arithmetic gives; the others keep the bound."""
    if kind == "gemm":
        g, x, w, _ = _gemm(70, 90, 64, act=False)
        x[3, 5], x[10, 0], x[20, 63], x[40] = np.inf, np.nan, -np.inf, 0
        x[40, 7], x[41, 1] = 3.4e38, -3.39e38
        w[5, 8] = 0.0                                      # inf * 0
        w[2, 77], w[9, 30] = np.inf, np.nan                # a whole column
    else:
        g, feeds, w = _conv(2, 16, 8, 9, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), False, act=False)
        x = feeds["x"]
        x[0, 3, 0, 0], x[1, 15, 7, 8], x[1, 0, 3, 3] = np.inf, np.nan, 3.4e38
        w[7, 2, 1, 1] = -np.inf
        g.initializers["w"] = w
    if kind == "gemm":
        g.initializers["w"] = w
    feeds = {"x": x}
    cm, got, _ = device_run(g, feeds, ctx=hip_ctx, split_fp32=True, winograd=False)
    assert "x3" in cm.module.plan[0].kernel_name
    with np.errstate(all="ignore"):
        want = run_reference(cm.graph, feeds)["y"]
    np.testing.assert_array_equal(np.isnan(got["y"]), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got["y"]), np.isposinf(want))
    np.testing.assert_array_equal(np.isneginf(got["y"]), np.isneginf(want))
    fin = np.isfinite(want)
    scale = np.abs(want[fin & (np.abs(want) < 1e6)]).max()
    ok = np.abs(got["y"][fin].astype(np.float64) - want[fin]) <= 1e-5 * np.maximum(np.abs(want[fin]), scale)
    assert ok.all()


WINOS = [  # n, C, H, W, OC, pads, slices, residual
    (3, 24, 9, 11, 40, (1, 1, 1, 1), 1, True),        # images inside a tile, odd sizes, half a chunk
    (2, 37, 15, 13, 130, (0, 1, 2, 0), 1, False),     # ragged channels, uneven padding, three channel blocks
    (5, 170, 7, 7, 70, (1, 1, 1, 1), 4, True),        # slices, the last one short
    (1, 9, 30, 6, 64, (2, 2, 2, 2), 1, False),        # one chunk
    (2, 48, 24, 56, 33, (1, 1, 1, 1), 1, True),       # even sizes: whole tiles, three chunks
    (4, 32, 12, 64, 16, (1, 1, 1, 1), 1, False),      # the largest patches
]


def _wino_mag(x, w, pads):
    """Sum over channels and positions of |U||V| (V with |B|), through |A|."""
    U = np.abs(emit.wino_filter_transform(w)).astype(np.float64).reshape(4, 4, w.shape[0], w.shape[1])
    x = np.pad(np.abs(x).astype(np.float64), ((0, 0), (0, 0), (pads[0], pads[2] + 1), (pads[1], pads[3] + 1)))
    oh, ow = x.shape[2] - 3, x.shape[3] - 3
    B = np.array([[1, 0, 1, 0], [0, 1, 1, 0], [0, 1, 1, 0], [0, 1, 0, 1]], np.float64)
    A = np.array([[1, 1, 1, 0], [0, 1, 1, 1]], np.float64)
    y = np.zeros((x.shape[0], w.shape[0], oh, ow))
    for i in range(0, oh, 2):
        for j in range(0, ow, 2):
            d = np.pad(x[:, :, i:i + 4, j:j + 4], ((0, 0), (0, 0), (0, max(0, i + 4 - x.shape[2])),
                                                   (0, max(0, j + 4 - x.shape[3]))))
            v = np.einsum("ar,ncrk,bk->ncab", B, d, B)
            m = np.einsum("aboc,ncab->noab", U, v)
            t = np.einsum("ia,noab,jb->noij", A, m, A)
            y[:, :, i:i + 2, j:j + 2] = t[:, :, :oh - i, :ow - j]
    return y


@pytest.mark.parametrize("case", WINOS, ids=lambda c: "x".join(map(str, c[:5])))
def test_winograd(case, hip_ctx, monkeypatch):
    """The GEMM's bound at the magnitude of Winograd's sums; U and V carry
    three roundings more, the output transform four."""
    n, C, H, W, OC, pads, sk, residual = case
    monkeypatch.setattr(emit, "wino_x3_slices", lambda *a: (sk, 0.0))
    g, feeds, w = _conv(n, C, H, W, OC, (3, 3), (1, 1), (1, 1), pads, residual)
    cm, got, _ = device_run(g, feeds, ctx=hip_ctx, split_fp32=True, winograd=True)
    assert "wino_x3" in cm.module.plan[0].kernel_name and (len(cm.module.plan) > 1) == (sk > 1)
    c = g.initializers["c"].reshape(1, -1, 1, 1).astype(np.float64)
    r = feeds.get("r", 0.0)
    want = np.maximum(_conv64(feeds["x"], w, (1, 1), (1, 1), pads) + c + r, 0)
    mag = _wino_mag(feeds["x"], w, pads) + np.abs(c) + np.abs(r)
    assert np.all(np.abs(got["y"] - want) <= _bound(C + 16, mag, sk + 7))


@pytest.mark.parametrize("sk", [1, 2])
def test_winograd_infinities_and_nans_are_the_fp32_kernels(sk, hip_ctx, monkeypatch):
    monkeypatch.setattr(emit, "wino_x3_slices", lambda *a: (sk, 0.0))
    g, feeds, w = _conv(2, 70, 9, 14, 70, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), False, act=False)
    x = feeds["x"]
    x[0, 3, 0, 0], x[1, 69, 8, 13], x[1, 0, 3, 3], x[0, 40, 5, 9] = np.inf, np.nan, 3.4e38, -np.inf
    w[67, 2, 1, 1], w[7, 50, 0, 0] = np.inf, np.nan
    g.initializers["w"] = w
    cm, got, _ = device_run(g, feeds, ctx=hip_ctx, split_fp32=True, winograd=True)
    assert "wino_x3" in cm.module.plan[0].kernel_name
    _, want, _ = device_run(g, feeds, ctx=hip_ctx, split_fp32=False, winograd=True)
    got, want = got["y"], want["y"]
    assert not np.isfinite(want).all() and np.isfinite(want).any()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    scale = np.abs(want[fin & (np.abs(want) < 1e6)]).max()
    assert (np.abs(got[fin].astype(np.float64) - want[fin]) <= 1e-5 * np.maximum(np.abs(want[fin]), scale)).all()
