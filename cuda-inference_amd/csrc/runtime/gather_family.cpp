// The gathering pointwise family (conv_gather.hip: 1x1 filters of any stride, image size and even channel count straight
// from NCHW / OIHW) as registry entries gather_<p>_1x1_<filters>x<pixels>_t<threads>, in the role of the reference's tcmma registration
// (src/kernels/tensor_core_mma.cu:264-395): one launch, no repack of either operand, no workspace.
//   * capability filter: fp16/bf16, a gfx950 device, a 1x1 filter, an even channel count, offsets, LDS and grid within
//     gie_hip_gather_check's limits;
//   * weights that are only 2-byte aligned run the small-convolution kernel instead (conv_mini.hip: element loads).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "gie_hip.h"
#include "gpu_inference/kernel_registry.h"
#include "mini_family.h"

namespace gie {
namespace {

gie_conv_geom geom_of(const ConvProblem& prob) {
  const Conv2DParams& p = prob.p;
  gie_conv_geom g;
  g.batch = p.batch;
  g.in_channels = p.in_channels;
  g.in_h = p.in_h;
  g.in_w = p.in_w;
  g.out_channels = p.out_channels;
  g.kernel_h = p.kernel_h;
  g.kernel_w = p.kernel_w;
  g.stride_h = p.stride_h;
  g.stride_w = p.stride_w;
  g.pad_h = p.pad_h;
  g.pad_w = p.pad_w;
  g.out_h = p.out_h();
  g.out_w = p.out_w();
  g.c_pad = p.in_channels;
  g.relu = prob.activation == Activation::kReLU ? 1 : 0;
  return g;
}

int dtype_of(Precision p) { return p == Precision::kFp16 ? GIE_HIP_FP16 : GIE_HIP_BF16; }

struct Tile {
  int m = 1, n = 1, threads = 64;
};
Tile tile_of(int config) {
  Tile t;
  (void)gie_hip_gather_config_get(config, &t.m, &t.n, &t.threads);
  return t;
}

template <int Config, Precision P>
struct Fns {
  static bool supports(const ConvProblem& prob, const DeviceInfo& dev, std::string* why) {
    auto no = [&](const std::string& m) {
      if (why) *why = m;
      return false;
    };
    if (prob.precision != P) return no(std::string("kernel is ") + to_string(P) + " only");
    if (!dev.is_gfx950()) return no("needs gfx950 matrix cores; device is " + dev.gcn_arch);
    const gie_conv_geom g = geom_of(prob);
    int lds = 0;
    if (gie_hip_gather_check(Config, &g, &lds) != GIE_HIP_OK || mini_best_config(prob, dev.sm_count, nullptr) < 0)
      return no("gathering kernel: 1x1 filter, even in_channels, offsets and grid within its limits");
    if (size_t(lds) > dev.smem_per_block_optin) return no("needs more LDS than a workgroup may use");
    return true;
  }
  static size_t workspace(const ConvProblem&) { return 0; }
  static size_t lds(const ConvProblem& prob) {
    const gie_conv_geom g = geom_of(prob);
    int bytes = 0;
    return gie_hip_gather_check(Config, &g, &bytes) == GIE_HIP_OK ? size_t(bytes) : 0;
  }
  static int64_t blocks(const ConvProblem& prob) {
    const Tile t = tile_of(Config);
    return (prob.p.gemm_n() + t.n - 1) / t.n * ((prob.p.out_channels + t.m - 1) / t.m);
  }
  static int occupancy(const ConvProblem& prob) {
    return std::max<int>(1, std::min<int>(2048 / 2 / tile_of(Config).threads, int(160 * 1024 / std::max<size_t>(lds(prob), 1))));
  }
  // A workgroup takes `start` us and each 64-channel step `step` us plus a share of its vector loads (16 clocks each: a
  // wave's x loads cover 64 pixel groups, its w loads 8 rows); one workgroup alone on a CU is bound by latency (`alone`).
  // Fitted per tile to 58 layers on one MI355X (7 to 56 a side, 14 to 1992 channels, both strides): 11-15 % rms.
  static double busy_us(const ConvProblem& prob, int cus) {
    struct Fit {
      double fixed, start, step, step_load, alone, alone_load;
    };
    constexpr Fit kFit[] = {{3.4, 0.46, 0.18, 0.93, 0.0, 2.1}, {3.2, 1.33, 0.16, 0.84, 0.23, 1.18},
                            {4.4, 1.62, 0.69, 0.72, 0.35, 1.19}, {4.0, 4.83, 0.19, 1.52, 0.0, 1.5}};
    const Fit& f = kFit[Config];
    const Conv2DParams& p = prob.p;
    const Tile t = tile_of(Config);
    const int64_t hw = int64_t(p.in_h) * p.in_w;
    const bool flat = p.stride_h == 1 && p.stride_w == 1 && p.pad_h == 0 && p.pad_w == 0;
    const int px = std::min(flat && hw % 4 == 0 ? 4 : flat && hw % 2 == 0 ? 2 : 1, t.m == 256 ? 2 : 4);
    // a strided row of x takes twice the cache lines (256 -> 512, 56x56 /2, batch 32: 38 us at 128x128)
    const double spread = p.stride_w > 1 ? 1.35 : 1.0;
    const double loads = (spread * double(t.n) / px + t.m / 8.0) * 16.0 / 2400.0;  // us of a step's vector loads
    const double steps = double((p.in_channels + 63) / 64), share = double(blocks(prob)) / std::max(cus, 1);
    return f.fixed + std::max(steps * (f.alone + f.alone_load * loads),
                              share * (f.start + steps * (f.step + f.step_load * loads)));
  }
  static void launch(const LaunchArgs& la) {
    if (la.only_stage >= 0 && la.only_stage != 1) return;  // one stage: the convolution itself
    if (reinterpret_cast<uintptr_t>(la.w) & 3u) {
      mini_launch(mini_best_config(*la.problem, la.dev->sm_count, nullptr), *la.problem, la.x, la.w, la.bias, la.y,
                  la.stream);
      return;
    }
    const gie_conv_geom g = geom_of(*la.problem);
    check_kernel_status(gie_hip_conv_gather(Config, dtype_of(P), &g, la.x, la.w, la.bias, la.y, la.stream),
                        "gathering MFMA convolution (NCHW / OIHW direct)");
  }
};

template <int Config, Precision P>
KernelDesc make_entry() {
  using F = Fns<Config, P>;
  const Tile t = tile_of(Config);
  KernelDesc k;
  k.backend = Backend::kTensorCore;
  k.name = std::string("gather_") + to_string(P) + "_1x1_" + std::to_string(t.m) + "x" + std::to_string(t.n) + "_t" +
           std::to_string(t.threads);
  k.version = 1;
  k.params = {{"block_m", t.m}, {"block_n", t.n}, {"block_k", 64}, {"split_k", 1}};
  k.threads_per_block = t.threads;
  k.tile_m = t.m;
  k.tile_n = t.n;
  k.tile_k = 16;
  k.uses_tensor_cores = true;
  k.launches = 1;
  k.supports = &F::supports;
  k.workspace_bytes = &F::workspace;
  k.dynamic_smem_bytes = &F::lds;
  k.num_blocks = &F::blocks;
  k.blocks_per_cu = &F::occupancy;
  k.busy_us = &F::busy_us;
  k.launch = &F::launch;
  return k;
}

template <Precision P>
void add_precision(std::vector<KernelDesc>& out) {
  out.push_back(make_entry<0, P>());
  out.push_back(make_entry<1, P>());
  out.push_back(make_entry<2, P>());
  out.push_back(make_entry<3, P>());
}

}  // namespace

void register_gather_family(std::vector<KernelDesc>& out) {
  if (gie_hip_gather_config_count() != 4) throw Error(StatusCode::kInternal, "gathering tile table changed");
  add_precision<Precision::kFp16>(out);
  add_precision<Precision::kBf16>(out);
}

}  // namespace gie
