"""The streaming pointwise kernel's whole-line stores (conv_pw.hip): rows that start anywhere in a 128-byte line, images
that end inside a block, ranges that end inside an image, filters past a 64-filter group, and an output that itself starts
inside a line. Sampled outputs are compared with the oracle, every output with the kernel that stores each tile by itself,
and no byte outside y may change."""
import ctypes

import numpy as np
import pytest

import gie
import oracle as O
from gpu_helpers import Bundle

pytestmark = pytest.mark.gpu

CASES = [
    # (B, C, H, W, O, precision, bias, relu): ranges of 4 and more blocks throughout
    (90, 16, 28, 28, 70, "fp16", True, True),     # rows start at 32-byte steps
    (250, 72, 8, 25, 24, "bf16", True, True),     # 200 pixels: three whole blocks at most between image ends
    (700, 136, 8, 9, 12, "fp16", True, False),    # 72 pixels: a block is rarely whole, never two in a row
    (300, 8, 16, 16, 9, "bf16", False, True),     # rows on whole lines: nothing waits
    (80, 200, 10, 100, 300, "fp16", False, False),  # two filter blocks, the second mostly past the filters
]


@pytest.mark.parametrize("yoff", [0, 8, 16, 96])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5])) + f"-{c[5]}")
def test_pws_whole_line_stores(case, yoff):
    B, C, H, W, Oc, prec, bias, relu = case
    p = gie.Problem(B, C, H, W, Oc, 1, 1, 1, 1, 0, 0, precision=prec, has_bias=bias, relu=relu)
    b = Bundle(p, 0x77 + C, O.NORMAL, full_reference=False, sample=4096)
    g = p.geom(C)
    n = int(np.prod(p.y_shape()))
    ybuf = gie.DeviceBuffer(2 * n + 512)
    gie.check_hip(gie.hip().gie_hip_fill_u16(ybuf.addr, n + 256, 0xFFFF, None), "fill")
    gie.check_hip(gie.hip().gie_hip_conv_pws(gie.PRECISIONS[prec], ctypes.byref(g), b.t.dx.addr, b.t.dw.addr,
                                             b.t.bias_addr(), ybuf.addr + 256 + yoff, None), "conv_pws")
    gie.synchronize()
    raw = ybuf.download(np.uint16, n + 256)
    at = (256 + yoff) // 2
    assert (raw[:at] == 0xFFFF).all() and (raw[at + n:] == 0xFFFF).all()
    y = raw[at:at + n]
    m = b.compare(gie.storage_to_float(y, prec).reshape(p.y_shape()))
    assert m.passed(), m.summary()
    # every element, against a kernel that stores each tile by itself
    gie.check_hip(gie.hip().gie_hip_conv_pw(gie.PRECISIONS[prec], ctypes.byref(g), b.t.dx.addr, b.t.dw.addr,
                                            b.t.bias_addr(), b.t.dy.addr, None), "conv_pw")
    gie.synchronize()
    a, r = gie.storage_to_float(y, prec), b.t.y().reshape(-1)
    # both sum the same FP32 products in another order and round once: one last place of the larger value, and the
    # FP32 difference of C products of magnitude ~1 where they cancel
    ulp = 2.0 ** (-10 if prec == "fp16" else -7)
    assert (np.abs(a - r) <= ulp * np.maximum(np.abs(a), np.abs(r)) + C * 2.0 ** -20).all()
