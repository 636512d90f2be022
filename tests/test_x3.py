"""Host side of the split-bf16 GEMM and convolution, on the CPU: the packed
constant is the float32 matrix exactly, the patch bound covers every position
the kernel's lanes can read, and the rule that picks the kernel."""

from __future__ import annotations

import numpy as np
import pytest

from mdlc_amd.codegen.hip.emit import x3_pack
from mdlc_amd.codegen.schedule import (CONV_X3_MAX_STEPS, CONV_X3_STEP_US, conv_x3_patch, conv_x3_schedule,
                                       conv_x3_tile, x3_schedule)
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
