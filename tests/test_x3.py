"""Host side of the split-bf16 GEMM and convolution, on the CPU: the packed
constant is the float32 matrix exactly, the patch bound covers every position
the kernel's lanes can read, and the rule that picks the kernel."""

from __future__ import annotations

import numpy as np
import pytest

from mdlc_amd.codegen.hip.emit import WINO_X3_SIGN, wino_x3_pack, x3_pack
from mdlc_amd.codegen.schedule import (CONV_X3_MAX_STEPS, CONV_X3_STEP_US, conv_x3_patch, conv_x3_schedule,
                                       conv_x3_tile, wino_patch, wino_x3_slices, x3_schedule)
from mdlc_amd.compiler import compile_graph
from mdlc_amd.tools.graph_builder import GraphBuilder


@pytest.mark.parametrize("rows,K", [(1, 1), (40, 50), (32, 16), (65, 4097)])
def test_packed_terms_sum_to_the_float(rows, K):
    rng = np.random.default_rng(rows)
    w = (rng.standard_normal((rows, K)) * np.exp2(rng.integers(-90, 90, (rows, K)))).astype(np.float32)
    special = np.array([np.inf, -np.inf, 0.0, -0.0, 3.4028235e38, -3.3999e38, 1.0, 2.0 ** -100], np.float32)
    flat = w.reshape(-1)
    flat[:min(flat.size, 8)] = special[:flat.size]
    if flat.size > 20:
        flat.view(np.uint32)[9:11] = 0x7f800001, 0xffffffff      # a signalling and a negative NaN
    img, kp = x3_pack(w)
    assert kp == -(-K // 16) * 16 and img.shape == (-(-rows // 32), kp // 16, 3, 2, 32, 8)
    t = (img.astype(np.uint32) << 16).view(np.float32)
    v = (t[:, :, 0] + (t[:, :, 1] + t[:, :, 2])).transpose(0, 3, 1, 2, 4).reshape(-1, kp)
    np.testing.assert_array_equal(v[:rows, :K], w)
    assert not v[rows:].any() and not v[:, K:].any()


GEOS = [dict(N=n, C=32, H=h, W=w, OC=64, KH=kh, KW=kw, SH=sh, SW=sw, DH=dh, DW=dw, group=1,
             OH=(h + 2 - dh * (kh - 1) - 1) // sh + 1, OW=(w + 2 - dw * (kw - 1) - 1) // sw + 1)
        for n, h, w, kh, kw, sh, sw, dh, dw in
        [(3, 9, 11, 3, 3, 1, 1, 1, 1), (2, 15, 13, 3, 3, 2, 2, 1, 1), (1, 40, 18, 5, 3, 2, 3, 1, 2),
         (7, 5, 4, 3, 3, 1, 2, 1, 1), (1, 57, 56, 3, 3, 2, 1, 1, 1), (5, 7, 7, 1, 1, 1, 1, 1, 1)]]


@pytest.mark.parametrize("geo", GEOS)
@pytest.mark.parametrize("bn", [64, 128])
def test_patch_covers_every_window(geo, bn):
    """The kernel's own index arithmetic, for every workgroup, pixel and tap:
    the position read lies in the patch and is the position that staged the
    tap's input element."""
    OH, OW, SH, SW, P = geo["OH"], geo["OW"], geo["SH"], geo["SW"], geo["N"] * geo["OH"] * geo["OW"]
    ONE = geo["KH"] * geo["KW"] == 1
    size = conv_x3_patch(geo, bn)
    WP = (OW - 1) * SW + (geo["KW"] - 1) * geo["DW"] + 1
    WPH = -(-WP // SW)
    WR, FR = WPH * SW, (OH - 1) * SH + (geo["KH"] - 1) * geo["DH"] + 1
    for n0 in range(0, P, bn):
        last = min(n0 + bn, P) - 1
        nf, nl = n0 // (OH * OW), last // (OH * OW)
        rlo = (n0 - nf * OH * OW) // OW * SH
        rlast = (last - nl * OH * OW) // OW * SH + (geo["KH"] - 1) * geo["DH"] + 1
        rows0 = (rlast if nl == nf else FR) - rlo
        PS = (rows0 + ((nl - nf - 1) * FR + rlast if nl > nf else 0)) * WR
        assert ONE or PS <= size
        for p in range(n0, last + 1):
            r = p - nf * OH * OW
            s1, s = divmod(r, OH * OW)
            oh, ow = divmod(s, OW)
            at = p - n0 if ONE else ((oh * SH - rlo) if s1 == 0 else rows0 + (s1 - 1) * FR + oh * SH) * WR + ow
            for kh in range(geo["KH"]):
                for kw in range(geo["KW"]):
                    toff = 0 if ONE else (kh * geo["DH"] * WR + kw * geo["DW"] % SW * WPH + kw * geo["DW"] // SW)
                    e = at + toff
                    assert 0 <= e < size
                    if ONE:
                        continue
                    q, c = divmod(e, WR)
                    n, row = nf, rlo + q
                    if q >= rows0:
                        n, row = nf + 1 + (q - rows0) // FR, (q - rows0) % FR
                    col = c % WPH * SW + c // WPH
                    assert (n, row, col) == (nf + s1, oh * SH + kh * geo["DH"], ow * SW + kw * geo["DW"])


@pytest.mark.parametrize("OC,C,OCP,CP", [(5, 3, 64, 16), (70, 40, 128, 64)])
def test_winograd_filter_image_sums_to_the_floats(OC, C, OCP, CP):
    u = np.random.default_rng(OC).standard_normal((16, OC, C)).astype(np.float32)
    t = (wino_x3_pack(u, OCP, CP).astype(np.uint32) << 16).view(np.float32)
    v = t[:, :, :, :, 0] + (t[:, :, :, :, 1] + t[:, :, :, :, 2])        # ocb, chunk, xi, blk, lk, li, j
    v = v.transpose(2, 0, 3, 5, 1, 4, 6).reshape(16, OCP, CP)
    np.testing.assert_array_equal(v[:, :OC, :C] * WINO_X3_SIGN.reshape(16, 1, 1), u)
    assert not v[:, OC:].any() and not v[:, :, C:].any()


@pytest.mark.parametrize("N,H,W,PT,PL,OH,OW", [(3, 9, 11, 1, 1, 9, 11), (2, 15, 13, 0, 1, 15, 12), (5, 7, 7, 1, 1, 7, 7),
                                               (1, 30, 5, 2, 2, 32, 7), (2, 24, 56, 1, 1, 24, 56), (40, 2, 1, 1, 0, 2, 1)])
def test_winograd_patch_planes_hold_every_window(N, H, W, PT, PL, OH, OW):
    """The kernel's layout: where a tile's window position is read, the pixel
    that was loaded there."""
    TH, TW = -(-OH // 2), -(-OW // 2)
    TT, P, WP, SR, PW = TH * TW, N * TH * TW, 2 * TW + 2, 2 * TH + 2, TW + 1
    size = -(-wino_patch(N, H, W, PT, OH, OW) // 64) * 64
    for t0 in range(0, P, 64):
        last = min(t0 + 63, P - 1)
        nf, nl = t0 // TT, last // TT
        rlo0, rhil = 2 * (t0 % TT // TW) - PT, 2 * (last % TT // TW) + 3 - PT
        rows0 = (rhil if nl == nf else 2 * TH + 1 - PT) - rlo0 + 1
        PS = rows0 * WP + ((nl - nf - 1) * SR * WP + (rhil + PT + 1) * WP if nl > nf else 0)
        PP = PS >> 2
        assert PS % (2 * WP) == 0 and rows0 % 2 == 0 and PS <= size
        for t in range(t0, last + 1):
            n, ty, tx = t // TT, t % TT // TW, t % TW
            row = 2 * ty - PT - rlo0 if n == nf else rows0 + (n - nf - 1) * SR + 2 * ty
            for r in range(4):
                for k in range(4):
                    e = (row >> 1) * PW + tx + (r & 1) * 2 * PP + (r >> 1) * PW + (k & 1) * PP + (k >> 1)
                    pl, f = divmod(e, PP)
                    q, col = 2 * (f // PW) + (pl >> 1), 2 * (f % PW) + (pl & 1)
                    seg, h = (0, rlo0 + q) if q < rows0 else (1 + (q - rows0) // SR, (q - rows0) % SR - PT)
                    assert 0 <= e < PS and (nf + seg, h, col - PL) == (n, 2 * ty - PT + r, 2 * tx - PL + k)


def test_winograd_or_direct():
    """Winograd where its estimate is below the direct convolution's, with
    slices that leave two chunks each."""
    def kernel(C, OC, H, W, batch, **kw):
        b = GraphBuilder("g")
        b.input("x", (batch, C, H, W))
        b.const("w", np.ones((OC, C, 3, 3), np.float32))
        b.node("Conv", ["x", "w"], "y", kernel_shape=[3, 3], strides=[1, 1], dilations=[1, 1], pads=[1, 1, 1, 1], group=1)
        b.output("y")
        return compile_graph(b.graph(), feeds={"x": np.zeros((batch, C, H, W), np.float32)}, **kw).module.plan[0].kernel_name

    assert "wino_x3" in kernel(256, 128, 28, 28, 32) and "wino_x3" in kernel(128, 128, 28, 28, 32)
    assert "conv_x3" in kernel(144, 80, 27, 40, 9) and "wino" not in kernel(128, 128, 28, 28, 8)
    assert "wino" in kernel(144, 80, 27, 40, 9, split_fp32=False) and "x3" not in kernel(128, 128, 28, 28, 32, split_fp32=False)
    for oc, tiles, c in [(64, 16, 16), (64, 16, 33), (512, 512, 512), (512, 16, 2048)]:
        s, us = wino_x3_slices(oc, tiles, c)
        assert us > 0 and (s == 1 or -(-(-(-c // 16)) // s) >= 2)


def test_schedules_cover_k_and_fit():
    for M, N, K in [(1, 1000, 512), (16, 333, 1000), (4096, 4096, 4096), (1000, 1511, 777), (5, 48, 16)]:
        s, us = x3_schedule(M, N, K)
        assert s.valid() and us > 0
    for geo in GEOS:
        got = conv_x3_schedule(dict(geo, N=geo["N"] * 8))
        assert got is not None
        s = got[0]
        stages = -(-geo["C"] // (16 * s.KS))
        assert s.lds_bytes() <= 160 * 1024 and -(-stages // s.SK) * s.KS * geo["KH"] * geo["KW"] <= CONV_X3_MAX_STEPS
    assert conv_x3_schedule(dict(GEOS[0], C=4)) is None and conv_x3_schedule(dict(GEOS[0], group=2)) is None
    wide = dict(GEOS[0], H=3, W=4000, OH=3, OW=4000)            # a patch no tile's LDS holds
    assert all(conv_x3_tile(wide, *t) is None for t in CONV_X3_STEP_US) and conv_x3_schedule(wide) is None


def test_the_split_is_taken_by_default_and_never_with_callers_schedules():
    rng = np.random.default_rng(0)
    b = GraphBuilder("g")
    b.input("x", (300, 200))
    b.const("w", rng.standard_normal((200, 111)).astype(np.float32))
    b.node("MatMul", ["x", "w"], "y")
    b.output("y")

    def kernel(**kw):
        return compile_graph(b.graph(), feeds={"x": np.zeros((300, 200), np.float32)}, **kw).module.plan[0].kernel_name

    from mdlc_amd.codegen.schedule import default_schedule

    assert "x3" in kernel() and "x3" in kernel(split_fp32=True)
    for kw in (dict(split_fp32=False), dict(winograd=False), dict(schedule_fn=lambda n, mnk: default_schedule(*mnk))):
        assert "x3" not in kernel(**kw)
    with pytest.raises(ValueError, match="split_fp32"):
        kernel(split_fp32="yes")
