"""GPU parity of the small-convolution kernel (conv_mini.hip: any filter, the whole reduction in one workgroup) through
its C-ABI, every configuration, against the oracle's double reference under the reference's tolerance
(tests/conv_test_common.h:83-127).

Cases sit where it can go wrong: tiles partly past the filters and past the pixels, images smaller than a tile, odd
pixel counts (no pair stores), reductions that end inside an operand chunk at the very end of the weights, odd
reductions (weights element by element), fewer supersteps than waves, many supersteps per wave, padding wider than the
image, strides, filters of 2 to 49 taps (the table form) and caller tensors aligned to one element only.
"""
import ctypes

import numpy as np
import pytest

import gie
import oracle as O
from gpu_helpers import Bundle

pytestmark = pytest.mark.gpu

CASES = [
    # (B, C, H, W, O, KH, KW, stride, PH, PW)
    (1, 1, 1, 1, 1, 1, 1, 1, 0, 0),
    (2, 72, 7, 7, 33, 1, 1, 1, 0, 0),      # odd pixel count, a filter past the tile
    (1, 100, 9, 8, 40, 1, 1, 2, 0, 0),     # reduction of 100: the last chunk is half inside
    (3, 13, 5, 6, 17, 1, 1, 1, 0, 0),      # odd reduction
    (1, 1040, 4, 4, 16, 1, 1, 1, 0, 0),    # several supersteps per wave
    (3, 130, 9, 11, 70, 3, 3, 1, 1, 1),    # 1170 = 146 chunks and 2
    (2, 5, 6, 5, 20, 3, 3, 2, 1, 1),       # odd reduction, below one superstep
    (1, 256, 14, 14, 48, 3, 3, 1, 1, 1),
    (2, 32, 3, 2, 31, 3, 3, 1, 2, 3),      # padding wider than the image
    (1, 600, 5, 5, 18, 3, 3, 1, 0, 0),     # many supersteps per wave
    (2, 9, 12, 11, 24, 5, 5, 2, 2, 2),
    (1, 24, 9, 9, 40, 1, 7, 1, 0, 3),
    (1, 3, 20, 17, 32, 7, 7, 2, 3, 3),     # 49 taps: beyond a 32-bit tap mask
]


def _run(config, p, t, off=0):
    """conv_mini through the C-ABI; off: bytes that every tensor starts past its allocation."""
    g = p.geom(p.in_channels)
    dt = gie.PRECISIONS[p.precision]
    lds = ctypes.c_int(0)
    assert gie.hip().gie_hip_mini_check(config, dt, ctypes.byref(g), ctypes.byref(lds)) == 0
    assert 0 < lds.value <= 160 * 1024
    t.poison()
    if off == 0:
        gie.check_hip(gie.hip().gie_hip_conv_mini(config, dt, ctypes.byref(g), t.dx.addr, t.dw.addr, t.bias_addr(),
                                                  t.dy.addr, None), "conv_mini")
        gie.synchronize()
        return t.y()
    bufs = {n: gie.DeviceBuffer(getattr(t, n).nbytes + 16) for n in ("dx", "dw", "dy")}
    for n in ("dx", "dw", "dy"):
        gie.check(gie.capi().gie_memcpy_d2d_async(bufs[n].addr + off, getattr(t, n).addr, getattr(t, n).nbytes, None))
    gie.check_hip(gie.hip().gie_hip_conv_mini(config, dt, ctypes.byref(g), bufs["dx"].addr + off, bufs["dw"].addr + off,
                                              t.bias_addr(), bufs["dy"].addr + off, None), "conv_mini")
    gie.synchronize()
    raw = np.frombuffer(bufs["dy"].download(np.uint8, t.dy.nbytes, off).tobytes(), np.uint16 if p.esize == 2 else np.uint32)
    return gie.storage_to_float(raw, p.precision).reshape(p.y_shape())


@pytest.mark.parametrize("prec", ["fp16", "bf16", "fp32", "tf32"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_mini_kernel_through_cabi(case, prec):
    i = CASES.index(case)
    B, C, H, W, Oc, KH, KW, S, PH, PW = case
    p = gie.Problem(B, C, H, W, Oc, KH, KW, S, S, PH, PW, precision=prec, has_bias=i % 3 != 2, relu=i % 2 == 0)
    b = Bundle(p, 0x313 + i, O.NORMAL)
    for config in range(gie.hip().gie_hip_mini_config_count()):
        y = _run(config, p, b.t)
        m = b.compare(y)
        assert m.passed(), f"config {config}: {m.summary()}"
        # the same sums in the same order, by element loads where the pointers are not 4-byte aligned
        shifted = _run(config, p, b.t, off=2 if p.esize == 2 else 4)
        assert np.array_equal(np.nan_to_num(y), np.nan_to_num(shifted)), config


def test_mini_ignores_what_lies_past_the_reduction():
    """Weights of the next filter and pixels of the next image are infinite: nothing of them may reach a finite sum."""
    p = gie.Problem(2, 10, 5, 5, 20, 3, 3, 1, 1, 1, 1, precision="fp16", has_bias=False, relu=False)
    b = Bundle(p, 0x1F, O.UNIFORM)
    x, w = b.x.copy(), b.w.copy()
    x[1] = np.inf
    w[1::2] = np.inf
    t = gie.ConvTensors(p, x, w, None)
    for config in range(gie.hip().gie_hip_mini_config_count()):
        y = _run(config, p, t)
        ref = _run(config, p, b.t)
        assert np.array_equal(y[0, ::2], ref[0, ::2]), config


def test_mini_argument_checks():
    h = gie.hip()
    ok = gie.Problem(1, 16, 5, 5, 16, 3, 3, 1, 1, 1, 1, precision="fp16")
    g, d = ok.geom(16), gie.DeviceBuffer(1 << 16)
    assert h.gie_hip_mini_check(h.gie_hip_mini_config_count(), 1, ctypes.byref(g), None) == -1
    assert h.gie_hip_mini_check(0, 4, ctypes.byref(g), None) == -2
    big = gie.Problem(1, 4, 20, 20, 16, 9, 9, 1, 1, 4, 4, precision="fp16")      # 81 taps
    assert h.gie_hip_mini_check(0, 1, ctypes.byref(big.geom(4)), None) == -2
    far = gie.Problem(64, 1024, 224, 224, 16, 1, 1, precision="fp16")            # 6.6 GB of input
    assert h.gie_hip_mini_check(0, 1, ctypes.byref(far.geom(1024)), None) == -2
    assert h.gie_hip_conv_mini(0, 1, ctypes.byref(g), None, d.addr, None, d.addr, None) == -1
    assert h.gie_hip_conv_mini(0, 1, ctypes.byref(g), d.addr, d.addr + 1, None, d.addr, None) == -1
    assert h.gie_hip_conv_mini(0, 0, ctypes.byref(g), d.addr, d.addr, None, d.addr + 2, None) == -1
