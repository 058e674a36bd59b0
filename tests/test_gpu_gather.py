"""GPU parity of the gathering pointwise kernel (conv_gather.hip: 1x1, any stride) through its C-ABI, every
configuration, against the oracle's double reference under the reference's tolerance
(tests/conv_test_common.h:83-127).

Cases sit where it can go wrong: every load width (images of a multiple of 4, 2 and 1 pixels, strides), images smaller
than a store's eight pixels (chunks over several images), tiles partly past the filters and pixels, one step and many,
channels that end inside a step, inside a 16-byte chunk and after one whole step, padding, and tensors aligned to less
than the wide loads need.
"""
import ctypes

import numpy as np
import pytest

import gie
import oracle as O
from gpu_helpers import Bundle

pytestmark = pytest.mark.gpu

CASES = [
    # (B, C, H, W, O, stride, pad)
    (3, 64, 8, 8, 70, 1, 0),       # 4-pixel loads, one whole step
    (2, 130, 14, 14, 64, 1, 0),    # 196 pixels: 8-pixel chunks straddle images; 130 = two steps and 2 channels
    (5, 128, 6, 7, 130, 1, 0),     # 42 pixels: pairs
    (4, 72, 7, 7, 33, 1, 0),       # odd images: one pixel per load
    (40, 192, 1, 1, 20, 1, 0),     # one-pixel images: every chunk spans eight of them
    (9, 66, 1, 3, 300, 1, 0),      # images smaller than a chunk
    (2, 320, 15, 13, 96, 2, 0),    # stride 2, odd sides, five steps
    (1, 1030, 9, 8, 258, 2, 0),    # many steps, 6 channels past a step, filters past two tiles
    (2, 16, 5, 6, 40, 3, 1),       # padding: output pixels outside the image
    (1, 2, 20, 20, 8, 1, 0),       # two channels
]


def _conv(config, p, t, x, w, y):
    g = p.geom(p.in_channels)
    gie.check_hip(gie.hip().gie_hip_conv_gather(config, gie.PRECISIONS[p.precision], ctypes.byref(g), x, w, t.bias_addr(),
                                                y, None), "conv_gather")
    gie.synchronize()


@pytest.mark.parametrize("prec", ["fp16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_gather_kernel_through_cabi(case, prec):
    i = CASES.index(case)
    B, C, H, W, Oc, S, P = case
    p = gie.Problem(B, C, H, W, Oc, 1, 1, S, S, P, P, precision=prec, has_bias=i % 3 != 2, relu=i % 2 == 0)
    b = Bundle(p, 0x6A + i, O.NORMAL)
    t = b.t
    bufs = {n: gie.DeviceBuffer(getattr(t, n).nbytes + 16) for n in ("dx", "dw", "dy")}
    for config in range(gie.hip().gie_hip_gather_config_count()):
        lds = ctypes.c_int(0)
        assert gie.hip().gie_hip_gather_check(config, ctypes.byref(p.geom(C)), ctypes.byref(lds)) == 0
        assert 0 < lds.value <= 160 * 1024
        t.poison()
        _conv(config, p, t, t.dx.addr, t.dw.addr, t.dy.addr)
        y = t.y()
        m = b.compare(y)
        assert m.passed(), f"config {config}: {m.summary()}"
        # x and y 2-byte, w 4-byte aligned: narrower loads, the same sums
        for n, off in (("dx", 2), ("dw", 4), ("dy", 2)):
            gie.check(gie.capi().gie_memcpy_d2d_async(bufs[n].addr + off, getattr(t, n).addr, getattr(t, n).nbytes, None))
        _conv(config, p, t, bufs["dx"].addr + 2, bufs["dw"].addr + 4, bufs["dy"].addr + 2)
        raw = np.frombuffer(bufs["dy"].download(np.uint8, t.dy.nbytes, 2).tobytes(), np.uint16)
        assert np.array_equal(np.nan_to_num(gie.storage_to_float(raw, prec).reshape(y.shape)), np.nan_to_num(y)), config


@pytest.mark.parametrize("prec", ["fp16", "bf16"])
def test_gather_entry_with_weights_aligned_to_one_element(prec):
    """The registry entry takes 2-byte aligned weights by running the small-convolution kernel."""
    p = gie.Problem(2, 48, 9, 9, 40, 1, 1, 2, 2, 0, 0, precision=prec, has_bias=True, relu=True)
    b = Bundle(p, 0x6E, O.UNIFORM)
    t = b.t
    plan = gie.Plan(p, f"gather_{prec}_1x1_64x64_t128")
    assert plan.workspace_bytes == 0
    w = gie.DeviceBuffer(t.dw.nbytes + 16)
    gie.check(gie.capi().gie_memcpy_d2d_async(w.addr + 2, t.dw.addr, t.dw.nbytes, None))
    t.poison()
    plan.execute_raw(t.dx.addr, w.addr + 2, t.bias_addr(), t.dy.addr, None, 0)
    gie.synchronize()
    m = b.compare(t.y())
    assert m.passed(), m.summary()


@pytest.mark.parametrize("c,h,w,stride", [(66, 6, 8, 1), (130, 7, 7, 1), (70, 9, 9, 2), (2, 4, 6, 1)],
                         ids=lambda v: str(v))
def test_gather_ignores_what_lies_past_the_reduction(c, h, w, stride):
    """Channels end inside a 16-byte chunk of weights that runs into the next filter. Every second filter and the next
    image are infinite: nothing of them may reach the others' sums, not even times the zeros that x is past its channels."""
    p = gie.Problem(2, c, h, w, 20, 1, 1, stride, stride, precision="fp16", has_bias=False, relu=False)
    b = Bundle(p, 0x6D, O.UNIFORM)
    x, wt = b.x.copy(), b.w.copy()
    x[1] = np.inf
    wt[1::2] = np.inf
    t = gie.ConvTensors(p, x, wt, None)
    for config in range(gie.hip().gie_hip_gather_config_count()):
        _conv(config, p, b.t, b.t.dx.addr, b.t.dw.addr, b.t.dy.addr)
        ref = b.t.y()
        t.poison()
        _conv(config, p, t, t.dx.addr, t.dw.addr, t.dy.addr)
        y = t.y()
        assert np.isfinite(y[0, ::2]).all() and np.array_equal(y[0, ::2], ref[0, ::2]), config


def test_gather_takes_outputs_smaller_than_the_image():
    """A geometry whose output leaves out the last rows and columns of a stride-1 layer: output pixels are no longer runs
    of input pixels, whatever the image size allows."""
    p = gie.Problem(2, 64, 8, 8, 40, 1, 1, precision="fp16", has_bias=True, relu=False)
    b = Bundle(p, 0x6F, O.UNIFORM)
    t, g = b.t, p.geom(64)
    g.out_h, g.out_w = 5, 6
    n = 2 * 40 * 5 * 6
    for config in range(gie.hip().gie_hip_gather_config_count()):
        _conv(config, p, t, t.dx.addr, t.dw.addr, t.dy.addr)  # every pixel, by wide loads
        full = t.y()
        t.poison()
        gie.check_hip(gie.hip().gie_hip_conv_gather(config, gie.PRECISIONS["fp16"], ctypes.byref(g), t.dx.addr, t.dw.addr,
                                                    t.bias_addr(), t.dy.addr, None), "conv_gather")
        gie.synchronize()
        y = gie.storage_to_float(t.dy.download(np.uint16, n), "fp16").reshape(2, 40, 5, 6)
        assert np.array_equal(y, full[:, :, :5, :6]), config


def test_gather_argument_checks():
    h = gie.hip()
    ok = gie.Problem(1, 16, 5, 5, 16, 1, 1, precision="fp16")
    g, d = ok.geom(16), gie.DeviceBuffer(1 << 16)
    assert h.gie_hip_gather_check(h.gie_hip_gather_config_count(), ctypes.byref(g), None) == -1
    for bad in (gie.Problem(1, 16, 5, 5, 16, 3, 3, 1, 1, 1, 1, precision="fp16"),   # 3x3
                gie.Problem(1, 15, 5, 5, 16, 1, 1, precision="fp16"),               # odd channels
                gie.Problem(64, 1024, 224, 224, 16, 1, 1, precision="fp16")):       # 6.6 GB of input
        assert h.gie_hip_gather_check(0, ctypes.byref(bad.geom(bad.in_channels)), None) == -2
    assert h.gie_hip_conv_gather(0, 0, ctypes.byref(g), d.addr, d.addr, None, d.addr, None) == -2      # fp32
    assert h.gie_hip_conv_gather(0, 1, ctypes.byref(g), d.addr, d.addr + 2, None, d.addr, None) == -2  # w 2-byte aligned
    assert h.gie_hip_conv_gather(0, 1, ctypes.byref(g), d.addr + 1, d.addr, None, d.addr, None) == -1
    assert h.gie_hip_conv_gather(0, 1, ctypes.byref(g), None, d.addr, None, d.addr, None) == -1
