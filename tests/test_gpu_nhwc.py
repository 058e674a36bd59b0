"""GPU parity of the padded-NHWC kernels (conv_nhwc.hip): the repack bit for bit against numpy, and the convolution
through the registry entries against the oracle's double reference under the reference's tolerance
(tests/conv_test_common.h:83-127).

Cases sit where they can go wrong: odd image sizes (pixel groups that end inside an image), channels that are no multiple
of 8 or of 32, filter runs that end inside a step and inside its first chunk, asymmetric padding and filters, strides,
images smaller than a store's eight pixels, tiles partly past the filters and pixels, a filter too large for the repack's
LDS, split-K, and inputs whose padding neighbours are infinite.
"""
import ctypes

import numpy as np
import pytest

import gie
import oracle as O
from gpu_helpers import Bundle, run_plan

pytestmark = pytest.mark.gpu

CASES = [
    # (B, C, H, W, O, KH, KW, stride, PH, PW)
    (2, 64, 14, 14, 70, 3, 3, 1, 1, 1),     # a run of exactly three steps
    (3, 13, 9, 11, 40, 3, 3, 1, 1, 1),      # 16 padded channels: a run of 48
    (2, 136, 7, 7, 130, 3, 3, 2, 1, 1),     # a run of 408: the last step ends after three chunks
    (5, 24, 6, 5, 66, 5, 5, 1, 2, 2),
    (1, 40, 17, 9, 33, 1, 7, 1, 0, 3),
    (2, 72, 3, 2, 64, 7, 1, 1, 3, 0),       # padding on one axis only, taller than the image
    (30, 16, 2, 1, 20, 3, 3, 1, 1, 1),      # two-pixel images
    (1, 8, 20, 20, 300, 3, 3, 3, 0, 0),     # no padding, stride 3
    (1, 2048, 4, 4, 40, 3, 3, 1, 1, 1),     # 18432 elements per filter
    (2, 64, 1, 1, 64, 1, 1, 1, 0, 0),
]


def _problem(case, prec):
    i = CASES.index(case)
    B, C, H, W, Oc, KH, KW, S, PH, PW = case
    return gie.Problem(B, C, H, W, Oc, KH, KW, S, S, PH, PW, precision=prec, has_bias=i % 3 != 2, relu=i % 2 == 0)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_nhwc_repack_is_bit_exact(case):
    B, C, H, W, Oc, KH, KW, S, PH, PW = case
    p = _problem(case, "fp16")
    rng = np.random.default_rng(7)
    x = rng.integers(0, 1 << 16, p.x_shape(), dtype=np.uint16)
    w = rng.integers(0, 1 << 16, p.w_shape(), dtype=np.uint16)
    g = p.geom(C)
    xb, wb = ctypes.c_longlong(), ctypes.c_longlong()
    assert gie.hip().gie_hip_nhwc_check(0, 1, ctypes.byref(g), ctypes.byref(xb), ctypes.byref(wb), None, None) == 0
    cp = (C + 7) // 8 * 8
    run = (KW * cp + 63) // 64 * 64
    assert xb.value == 2 * B * (H + 2 * PH) * (W + 2 * PW) * cp and wb.value == 2 * Oc * KH * run
    for off in (0, 2):  # source tensors aligned to one element
        dx, dw = gie.DeviceBuffer(x.nbytes + 16), gie.DeviceBuffer(w.nbytes + 16)
        dx.upload(x, off)
        dw.upload(w, off)
        xp, wp = gie.DeviceBuffer(xb.value), gie.DeviceBuffer(wb.value)
        xp.fill(0xFF)
        wp.fill(0xFF)
        gie.check_hip(gie.hip().gie_hip_repack_nhwc(1, dx.addr + off, xp.addr, dw.addr + off, wp.addr, ctypes.byref(g), None),
                      "repack")
        gie.synchronize()
        want = np.zeros((B, H + 2 * PH, W + 2 * PW, cp), np.uint16)
        want[:, PH:PH + H, PW:PW + W, :C] = x.transpose(0, 2, 3, 1)
        assert np.array_equal(xp.download(np.uint16, want.size).reshape(want.shape), want)
        rows = np.zeros((Oc, KH, KW, cp), np.uint16)
        rows[..., :C] = w.transpose(0, 2, 3, 1)
        want = np.zeros((Oc, KH, run), np.uint16)
        want[:, :, :KW * cp] = rows.reshape(Oc, KH, KW * cp)
        assert np.array_equal(wp.download(np.uint16, want.size).reshape(want.shape), want)


@pytest.mark.parametrize("prec", ["fp16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_nhwc_entries(case, prec):
    p = _problem(case, prec)
    b = Bundle(p, 0x9C + CASES.index(case), O.NORMAL)
    ran = 0
    for k in gie.registry():
        if not k.startswith(f"nhwc_{prec}_"):
            continue
        y, why = run_plan(k, b, repeats=2)
        if y is None:
            assert "too short" in why, why
            continue
        m = b.compare(y)
        assert m.passed(), f"{k}: {m.summary()}"
        ran += 1
    assert ran >= 5


def test_nhwc_pads_a_run_with_zeros_on_both_sides():
    """Pixels past a filter row's run are infinite: the last step of the run must not multiply them, even by zero."""
    p = gie.Problem(1, 24, 5, 16, 16, 3, 3, 1, 1, 1, 1, precision="fp16", has_bias=False, relu=False)
    b = Bundle(p, 0x2F, O.UNIFORM)
    x = b.x.copy()
    x[:, :, :, 8:] = np.inf
    t = gie.ConvTensors(p, x, b.w, None)
    plan = gie.Plan(p, "nhwc_fp16_64x64x64_sk1")
    ws = gie.DeviceBuffer(plan.workspace_bytes)
    plan.execute(t, ws)
    ref, _ = run_plan("nhwc_fp16_64x64x64_sk1", b)
    gie.synchronize()
    assert np.array_equal(t.y()[:, :, :, :7], ref[:, :, :, :7])


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_nhwc_fp32(case):
    """Both FP32 tiles and a split through the C-ABI, every tensor one element into its allocation."""
    p = _problem(case, "fp32")
    b = Bundle(p, 0x3F + CASES.index(case), O.NORMAL)
    g, h, n = p.geom(p.in_channels), gie.hip(), int(np.prod(p.y_shape()))
    dx, dw, db, y = (gie.DeviceBuffer(v + 16) for v in (b.x.nbytes, b.w.nbytes, 4 * p.out_channels, 4 * n))
    dx.upload(b.x.astype(np.float32), 4)
    dw.upload(b.w.astype(np.float32), 4)
    if b.b is not None:
        db.upload(b.b.astype(np.float32), 4)
    bias = db.addr + 4 if p.has_bias else None
    for config in (0, 2):
        xb, wb, steps = ctypes.c_longlong(), ctypes.c_longlong(), ctypes.c_int()
        assert h.gie_hip_nhwc_check(config, 0, ctypes.byref(g), ctypes.byref(xb), ctypes.byref(wb), ctypes.byref(steps),
                                    None) == 0
        xp, wp, part = gie.DeviceBuffer(xb.value), gie.DeviceBuffer(wb.value), gie.DeviceBuffer(8 * n)
        for split in (1, 2):
            if steps.value < split:
                continue
            for d in (xp, wp, part, y):
                d.fill(0xFF)
            gie.check_hip(h.gie_hip_repack_nhwc(0, dx.addr + 4, xp.addr, dw.addr + 4, wp.addr, ctypes.byref(g), None), "r")
            gie.check_hip(h.gie_hip_conv_nhwc(config, 0, ctypes.byref(g), xp.addr, wp.addr, bias, y.addr + 4,
                                              part.addr if split > 1 else None, split, None), "conv")
            if split > 1:
                gie.check_hip(h.gie_hip_splitk_reduce(0, part.addr, bias, y.addr + 4, n, split, p.out_channels,
                                                      p.out_h * p.out_w, int(p.relu), None), "reduce")
            gie.synchronize()
            m = b.compare(y.download(np.float32, n + 1)[1:].reshape(p.y_shape()))
            assert m.passed(), f"config {config} split {split}: {m.summary()}"


FP32_LAYERS = [(32, 128, 28, 28, 128, 3, 3, 1, 1, 1), (8, 3, 112, 112, 64, 7, 7, 2, 3, 3), (2, 24, 9, 9, 32, 3, 3, 1, 1, 1)]


def _align(n):
    return (n + 255) // 256 * 256


@pytest.mark.parametrize("case", FP32_LAYERS, ids=lambda c: "x".join(map(str, c)))
def test_nhwc_fp32_entries(case):
    """The FP32 entries run these kernels (bit for bit the C-ABI's repack, convolution and reduce) in a workspace of their
    copies and partials alone."""
    p = gie.Problem(*case[:8], case[7], *case[8:], precision="fp32", has_bias=True, relu=True)
    b = Bundle(p, 0x8E, O.NORMAL, full_reference=False, sample=4096)
    g, h, n, t = p.geom(p.in_channels), gie.hip(), int(np.prod(p.y_shape())), b.t
    ran = 0
    for name in (k for k in gie.registry() if k.startswith("nhwc_fp32_")):
        config, split = (0 if "_64x64x" in name else 2), int(name.rsplit("_sk", 1)[1])
        y, why = run_plan(name, b, repeats=2)
        if y is None:
            assert "too short" in why, why
            continue
        m = b.compare(y)
        assert m.passed(), f"{name}: {m.summary()}"
        xb, wb = ctypes.c_longlong(), ctypes.c_longlong()
        assert h.gie_hip_nhwc_check(config, 0, ctypes.byref(g), ctypes.byref(xb), ctypes.byref(wb), None, None) == 0
        part_bytes = 4 * n * split if split > 1 else 0
        assert gie.Plan(p, name).workspace_bytes == _align(xb.value) + _align(wb.value) + _align(part_bytes)
        xp, wp = gie.DeviceBuffer(xb.value), gie.DeviceBuffer(wb.value)
        part = gie.DeviceBuffer(part_bytes) if split > 1 else None
        t.poison()
        gie.check_hip(h.gie_hip_repack_nhwc(0, t.dx.addr, xp.addr, t.dw.addr, wp.addr, ctypes.byref(g), None), "repack")
        gie.check_hip(h.gie_hip_conv_nhwc(config, 0, ctypes.byref(g), xp.addr, wp.addr, t.bias_addr(), t.dy.addr,
                                          part.addr if part else None, split, None), "conv")
        if part:
            gie.check_hip(h.gie_hip_splitk_reduce(0, part.addr, t.bias_addr(), t.dy.addr, n, split, p.out_channels,
                                                  p.out_h * p.out_w, int(p.relu), None), "reduce")
        gie.synchronize()
        assert np.array_equal(y, t.y()), name
        ran += 1
    assert ran >= 2


@pytest.mark.parametrize("case", FP32_LAYERS, ids=lambda c: "x".join(map(str, c)))
def test_fp32_split_8_entry_runs_its_own_kernel(case):
    """Bit for bit gie_hip_conv_f32 with 128 filters a tile and eight splits, in a workspace of eight partials."""
    name = "implicit_gemm_fp32_128x128x16_mfma_sk8"
    p = gie.Problem(*case[:8], case[7], *case[8:], precision="fp32", has_bias=True, relu=True)
    b = Bundle(p, 0x8E, O.NORMAL, full_reference=False, sample=4096)
    g, h, n, t = p.geom(p.in_channels), gie.hip(), int(np.prod(p.y_shape())), b.t
    assert gie.Plan(p, name).workspace_bytes == _align(8 * 4 * n)
    y, why = run_plan(name, b, repeats=2)
    assert y is not None, why
    m = b.compare(y)
    assert m.passed(), m.summary()
    (config,) = [c for c in range(h.gie_hip_f32_config_count()) if h.gie_hip_f32_config_tile_m(c) == 128]
    part = gie.DeviceBuffer(8 * 4 * n)
    t.poison()
    gie.check_hip(h.gie_hip_conv_f32(config, 0, ctypes.byref(g), t.dx.addr, t.dw.addr, t.bias_addr(), t.dy.addr, part.addr,
                                     8, None), "conv_f32")
    gie.check_hip(h.gie_hip_splitk_reduce(0, part.addr, t.bias_addr(), t.dy.addr, n, 8, p.out_channels, p.out_h * p.out_w,
                                          int(p.relu), None), "reduce")
    gie.synchronize()
    assert np.array_equal(y, t.y())


def test_nhwc_argument_checks():
    h = gie.hip()
    ok = gie.Problem(1, 16, 5, 5, 16, 3, 3, 1, 1, 1, 1, precision="fp16")
    g, d = ok.geom(16), gie.DeviceBuffer(1 << 20)
    assert h.gie_hip_nhwc_check(h.gie_hip_nhwc_config_count(), 1, ctypes.byref(g), None, None, None, None) == -1
    far = gie.Problem(64, 1024, 224, 224, 16, 3, 3, 1, 1, 1, 1, precision="fp16")
    assert h.gie_hip_nhwc_check(0, 1, ctypes.byref(far.geom(1024)), None, None, None, None) == -2
    assert h.gie_hip_conv_nhwc(0, 3, ctypes.byref(g), d.addr, d.addr, None, d.addr, None, 1, None) == -2   # tf32
    assert h.gie_hip_nhwc_check(1, 0, ctypes.byref(g), None, None, None, None) == -2  # fp32: 64x64 and 128x128 only
    assert h.gie_hip_conv_nhwc(0, 1, ctypes.byref(g), d.addr + 8, d.addr, None, d.addr, None, 1, None) == -1
    assert h.gie_hip_conv_nhwc(0, 1, ctypes.byref(g), d.addr, d.addr, None, d.addr, None, 2, None) == -1   # no partials
    assert h.gie_hip_conv_nhwc(0, 1, ctypes.byref(g), d.addr, d.addr, None, d.addr, d.addr, 4, None) == -2  # 3 steps
    assert h.gie_hip_repack_nhwc(1, d.addr + 1, d.addr, d.addr, d.addr, ctypes.byref(g), None) == -1
