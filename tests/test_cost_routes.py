"""The cost model's order inside and between families where measurements separate them (no GPU needed): each case names
the entry or family that was measured faster and the one it must stay ahead of."""
import pytest

import gie

P = gie.Problem


def _us(p):
    return dict(gie.model_rank(p))


@pytest.mark.parametrize("p,first,second", [
    # the split form of a 14-row slab beats the full form of the same slab: 9.1 and 16.0 us
    (P(32, 256, 14, 14, 256, 3, 3, 1, 1, 1, 1, precision="fp16"), "slab_fp16_3x3_32x14r16_k32_s3_ld_sk1",
     "slab_fp16_3x3_32x14r16_k32_s3_sk1"),
    # a reduce over 1.2 million outputs costs more than split-K gains: 15.6 and 21.5 us
    (P(22, 288, 12, 12, 367, 3, 3, 1, 1, 1, 1, precision="fp16"), "slab_fp16_3x3_32x14r16_k32_s3_ld_sk1",
     "slab_fp16_3x3_32x14r16_k32_s3_ld_sk2"),
    # 56-pixel rows leave a 64-position band's stores short: 28.7 and 56.5 us; halo 48.3
    (P(32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1, precision="bf16"), "nhwc_bf16_64x128x64_sk1",
     "band_bf16_3x3_32x256x32_s3_sk1"),
    (P(32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1, precision="bf16"), "nhwc_bf16_64x128x64_sk1",
     "halo_bf16_3x3_64x128x32_s2_sk1"),
    # strided rows of x: 28.7 and 38.0 us
    (P(32, 256, 56, 56, 512, 1, 1, 2, 2, 0, 0, precision="fp16"), "gather_fp16_1x1_256x128_t512",
     "gather_fp16_1x1_128x128_t256"),
    (P(53, 544, 29, 29, 32, 1, 1, 2, 2, 0, 0, precision="bf16"), "mini_bf16_32x32_k16w", "mini_bf16_16x16_k8w"),
    # the gathering kernel's whole and ragged channel steps: 22.3 and 43.1 us, 6.7 and 10.5, 6.9 and 10.7
    (P(16, 704, 17, 17, 1408, 1, 1, precision="bf16"), "gather_bf16_1x1_256x128_t512", "nhwc_bf16_128x256x64_sk1"),
    (P(11, 192, 27, 27, 96, 1, 1, precision="fp16"), "gather_fp16_1x1_64x64_t128", "mini_fp16_32x32_k8w"),
    (P(19, 128, 30, 30, 128, 1, 1, 2, 2, precision="bf16"), "gather_bf16_1x1_64x64_t128", "mini_bf16_32x32_k8w"),
    # the padded-NHWC kernel's rounds, stores and odd images: 28.8 and 48.7 us, 24.9 and 40.3, 19.0 and 25.5
    (P(39, 32, 36, 36, 1024, 1, 1, precision="fp16"), "pw_fp16_1x1_256x64x16_s4_wreg", "nhwc_fp16_256x256x64_sk1"),
    (P(24, 48, 36, 56, 1024, 1, 1, precision="fp16"), "pw_fp16_1x1_256x64x16_s4_wreg", "nhwc_fp16_256x256x64_sk1"),
    (P(11, 416, 15, 15, 1664, 1, 1, precision="bf16"), "gather_bf16_1x1_256x128_t512", "nhwc_bf16_128x128x64_sk1"),
    # the halo kernel's rounds, repack and odd images: 24.9 and 33.8 us, 32.2 and 42.7
    (P(4, 160, 53, 53, 160, 3, 3, 1, 1, 1, 1, precision="bf16"), "nhwc_bf16_128x128x64_sk1", "halo_bf16_3x3_64x128x32_s2_sk1"),
    (P(6, 256, 39, 39, 256, 3, 3, 1, 1, 1, 1, precision="fp16"), "nhwc_fp16_128x128x64_sk1", "halo_fp16_3x3_64x128x32_s2_sk1"),
    # a band's input pixels: 58.7 and 110.5 us, 15.2 and 22.8 (stride 2)
    (P(15, 352, 32, 32, 272, 3, 3, 1, 1, 1, 1, precision="bf16", has_bias=False, relu=False), "nhwc_bf16_128x256x64_sk1",
     "band_bf16_3x3_32x224x32_s4_sk1"),
    (P(6, 256, 33, 33, 64, 3, 3, 2, 2, 1, 1, precision="bf16"), "nhwc_bf16_64x64x64_sk4", "band_bf16_3x3_32x256x32_s3_sk4"),
    # the implicit GEMM over images of no multiple of four pixels: 20.3 and 31.2 us, 47.2 and 78.3; its rounds: 46.8 and
    # 68.0, 22.5 and 28.6
    (P(4, 3, 225, 225, 96, 7, 7, 2, 2, 3, 3, precision="fp16"), "nhwc_fp16_128x256x64_sk1", "mfma_fp16_64x64x32_w2x2_s4_sk1"),
    (P(14, 3, 225, 225, 96, 7, 7, 2, 2, 3, 3, precision="fp16"), "nhwc_fp16_128x256x64_sk1", "mfma_fp16_64x128x32_w2x2_s4_sk1"),
    (P(2, 464, 46, 46, 464, 3, 3, 1, 1, 1, 1, precision="bf16"), "nhwc_bf16_128x128x64_sk1", "mfma_bf16_128x64x128_w4x2_s2_sk1"),
    (P(11, 130, 44, 15, 288, 3, 3, 1, 1, 1, 1, precision="bf16"), "nhwc_bf16_128x128x64_sk1", "mfma_bf16_64x128x64_w2x4_s4_sk1"),
    # large strided 1x1 layers are no small convolutions: 18.1 and 27.4 us, 26.5 and 40.2
    (P(59, 744, 23, 23, 33, 1, 1, 2, 2, precision="bf16"), "gather_bf16_1x1_64x64_t128", "mini_bf16_32x32_k16w"),
    (P(42, 836, 14, 30, 224, 1, 1, 2, 2, precision="fp16"), "gather_fp16_1x1_64x64_t128", "mini_fp16_32x32_k16w"),
    # strided rows that every filter tile reads again: 18.7 and 31.9 us, 35.2 and 56.2
    (P(4, 1408, 24, 24, 1408, 1, 1, 2, 2, precision="bf16"), "mfma_bf16_64x64x64_w4x2_s4_sk1", "gather_bf16_1x1_64x64_t128"),
    (P(4, 1920, 34, 34, 1920, 1, 1, 2, 2, precision="fp16"), "nhwc_fp16_128x128x64_sk1", "gather_fp16_1x1_64x64_t128"),
    # small convolutions in whole rounds of workgroups: 7.1 and 10.1 us, 12.9 and 19.7, 6.4 and 9.6
    (P(16, 32, 12, 12, 128, 1, 3, 1, 1, 0, 1, precision="bf16", relu=False), "nhwc_bf16_64x64x64_sk1", "mini_bf16_32x32_k8w"),
    (P(26, 416, 33, 33, 32, 1, 1, precision="fp16"), "gather_fp16_1x1_64x128_t256", "mini_fp16_32x32_k8w"),
    (P(8, 39, 27, 27, 16, 3, 3, 1, 1, 1, 1, precision="bf16"), "mini_bf16_32x32_k8w", "nhwc_bf16_64x64x64_sk1"),
    # the FP32 tile kernel's rounds, stages and reduce: 55.6 and 78.7 us, 19.6 and 25.8
    (P(23, 352, 18, 14, 176, 3, 1, 1, 1, 1, 0, precision="tf32", has_bias=False, relu=False), "mfma_tf32_64x128x16_sk8",
     "mfma_tf32_64x128x16_sk2"),
    (P(33, 32, 52, 52, 256, 1, 1, 2, 2, precision="fp32"), "implicit_gemm_fp32_64x128x16_mfma_sk1",
     "implicit_gemm_fp32_128x128x16_mfma_sk1"),
])
def test_measured_order(p, first, second):
    us = _us(p)
    assert us[first] < us[second], (us[first], us[second])


@pytest.mark.parametrize("side,batch", [(28, 8), (28, 16), (28, 32), (28, 64), (20, 16), (20, 32), (20, 64)])
@pytest.mark.parametrize("prec", ["fp16", "bf16"])
def test_wide_pointwise_layers_take_the_streaming_form(prec, side, batch):
    """256 -> 1024 channels: 10.1 to 54 us where the tiled form takes 10.8 to 93 (FP16 28x28, batch 64: 53.7 and 83.9)."""
    p = P(batch, 256, side, side, 1024, 1, 1, precision=prec, has_bias=True, relu=True)
    assert gie.model_rank(p)[0][0] == f"pw_{prec}_1x1_256x64x16_s4_wreg"


@pytest.mark.parametrize("case", [(32, 512, 28, 28, 128), (13, 592, 24, 24, 296), (11, 448, 48, 39, 96), (16, 512, 28, 28, 256)],
                         ids=lambda c: "x".join(map(str, c)))
def test_pointwise_layers_of_many_channels_take_the_tiled_form(case):
    """Channels past the streaming form's 256: 10.3, 10.3, 8.7 and 10.1 us, the gathering kernel 1.26 to 1.43 times
    those."""
    p = P(*case, 1, 1, precision="fp16", has_bias=True, relu=True)
    assert gie.model_rank(p)[0][0] == "pw_fp16_1x1_128x128x32_s4_sk1"


def test_pointwise_tensors_the_cache_holds_are_not_priced_at_hbm_rates():
    """256 -> 128 over 56x56, batch 32: 19.2 and 19.5 us on the two pointwise forms, 23.0 on the gathering kernel; 77 MB at
    their families' HBM rates would be 20.1 and 19.3."""
    p = P(32, 256, 56, 56, 128, 1, 1, precision="fp16", has_bias=True, relu=True)
    assert gie.model_rank(p)[0][0].startswith("pw_")


def test_tiled_pointwise_entry_counts_tiles_per_image():
    """784 pixels are seven tiles of 128 in every image, whatever the batch makes of them in a row."""
    p = P(64, 256, 28, 28, 1024, 1, 1, precision="fp16")
    assert gie.model_estimate("pw_fp16_1x1_128x128x32_s4_sk1", p)["tile_efficiency"] == 784 / (7 * 128)
    assert gie.model_estimate("pw_fp16_1x1_256x64x16_s4_wreg", p)["tile_efficiency"] == 1.0


@pytest.mark.parametrize("kh,kw,c,prec,measured", [
    (1, 3, 32, "bf16", {4: 5.6, 6: 5.7, 8: 5.7, 9: 10.0, 12: 10.1, 16: 10.2, 17: 14.5, 20: 14.5, 24: 14.8}),
    (3, 3, 64, "bf16", {4: 5.2, 6: 5.2, 8: 5.2, 9: 9.0, 12: 9.0, 16: 9.2, 17: 13.0, 20: 13.0, 24: 13.4})])
def test_small_convolutions_run_in_whole_rounds_of_workgroups(kh, kw, c, prec, measured):
    """32 -> 32 or 64 -> 32 over 32x32: 32 workgroups an image, one on each of 256 CUs at a time. The time steps between
    256 and 288 workgroups and again past 512, and is flat between; the estimate follows it."""
    for batch, us in measured.items():
        p = P(batch, c, 32, 32, 32, kh, kw, 1, 1, kh // 2, kw // 2, precision=prec)
        est = gie.model_estimate(f"mini_{prec}_32x32_k8w", p)["time_us"]
        assert abs(est / us - 1) < 0.08, (batch, est, us)


def test_large_fp32_layers_take_entries_that_describe_what_runs():
    """3x3 128 -> 128 over 28x28, batch 32: the padded-NHWC kernel (90 us; the tile kernel 118) under a name, launches and
    tiles of its own, and the split-8 tile entry priced as the tile kernel with its eight partials on any device."""
    p = P(32, 128, 28, 28, 128, 3, 3, 1, 1, 1, 1, precision="fp32", has_bias=True, relu=True)
    assert gie.model_rank(p)[0][0] == "nhwc_fp32_128x128x32_sk1"
    d = gie.kernel_describe("nhwc_fp32_128x128x32_sk1")
    assert (d["backend"], d["launches"], d["threads"], d["tile_m"], d["tile_n"]) == ("implicit_gemm", 2, 512, 128, 128)
    assert gie.kernel_describe("nhwc_fp32_64x64x32_sk2")["launches"] == 3
    partials = 2 * 8 * 4 * 32 * 128 * 28 * 28
    for cus in (64, 128, 256):
        e = gie.model_estimate("implicit_gemm_fp32_128x128x16_mfma_sk8", p, dict(cus=cus, hbm_gbs=8000.0))
        assert e["memory_us"] > partials / 8e6


@pytest.mark.parametrize("kernel,p,bound", [
    ("gather_fp16_1x1_64x64_t128", P(1, 8, 4, 4, 8, 1, 1, precision="fp16"), "launch"),
    ("gather_fp16_1x1_64x64_t128", P(32, 8, 224, 224, 8, 1, 1, precision="fp16"), "bandwidth"),
    ("band_fp16_3x3_32x256x32_s3_sk1", P(1, 8, 8, 8, 8, 3, 3, 1, 1, 1, 1, precision="fp16"), "launch"),
    ("halo_fp16_3x3_64x128x32_s2_sk1", P(1, 8, 8, 8, 8, 3, 3, 1, 1, 1, 1, precision="fp16"), "launch"),
    ("nhwc_bf16_256x256x64_sk1", P(16, 256, 56, 56, 256, 3, 3, 1, 1, 1, 1, precision="bf16"), "compute"),
])
def test_estimates_name_what_bounds_a_call(kernel, p, bound):
    """Entries timed by a formula of their own keep the roofline's parts: a formula's fixed costs are not arithmetic."""
    assert gie.model_estimate(kernel, p)["bound"] == bound


@pytest.mark.parametrize("prec", ["fp32", "tf32", "fp16", "bf16"])
def test_every_estimate_is_finite_and_positive(prec):
    for p in (P(1, 8, 1, 1, 8, 1, 1, 1, 1, 0, 0, precision=prec), P(3, 7, 33, 31, 9, 3, 3, 2, 1, 0, 2, precision=prec),
              P(64, 2048, 56, 56, 2048, 3, 3, 1, 1, 1, 1, precision=prec),
              P(2, 5, 40, 3, 6, 11, 3, 3, 3, 5, 1, precision=prec)):
        us = gie.model_rank(p)
        assert us and all(0.0 < u < 1e7 for _, u in us), us[:3]
