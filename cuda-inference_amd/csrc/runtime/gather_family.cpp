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
  // A fixed cost (more where images are no multiple of a store's eight pixels), then each 64-channel step at one
  // workgroup's latency (`alone`) plus, beyond 0.75 workgroups a CU, its share of them (`step`); both grow with the step's
  // vector loads (16 clocks each: a wave's x loads cover 64 pixel groups, its w loads 8 rows) and where channels end
  // inside a step (`part`); then the output stores, and more for each MB of x and y past the 80 that stay in the
  // Infinity Cache over a few sets of tensors (`spill`, `spill_lines` where image rows of y share 128-byte lines). A strided
  // row of x takes twice the cache lines: dearer loads alone and shared (`lines`), and each filter tile reads the rows'
  // lines again (`again`, per MB: 1920 -> 1920 over 33x33, batch 7, 58 us; without it 38). Fitted per tile to 2366-2699
  // layers on one MI355X (7 to 56 a side, 16 to 2000 channels, both strides): 8-11 % rms, 8-11 % on 523-535 others.
  static double busy_us(const ConvProblem& prob, int cus) {
    struct Fit {
      double fixed, alone, alone_load, step, step_load, out, odd, part, spill, spill_lines, lines, lines_shared, again;
    };
    constexpr Fit kFit[] = {{2.10, 0.291, 0.776, 0.155, 0.267, 0.331, 0.96, 0.55, 0.34, 0.28, 0.15, 0.00, 0.077},
                            {2.25, 0.416, 0.529, 0.294, 0.379, 0.225, 1.14, 0.18, 0.25, 0.20, 0.61, 0.37, 0.068},
                            {3.09, 0.568, 0.553, 0.461, 0.433, 0.238, 1.66, 0.14, 0.26, 0.13, 0.67, 1.51, 0.038},
                            {3.13, 0.579, 0.613, 0.196, 1.667, 0.268, 1.52, 0.16, 0.14, 0.16, 0.72, 0.68, 0.048}};
    const Fit& f = kFit[Config];
    const Conv2DParams& p = prob.p;
    const Tile t = tile_of(Config);
    const int64_t hw = int64_t(p.in_h) * p.in_w, ohw = int64_t(p.out_h()) * p.out_w();
    const bool flat = p.stride_h == 1 && p.stride_w == 1 && p.pad_h == 0 && p.pad_w == 0;
    const int px = std::min(flat && hw % 4 == 0 ? 4 : flat && hw % 2 == 0 ? 2 : 1, t.m == 256 ? 2 : 4);
    const double strided = p.stride_w > 1 ? 1.0 : 0.0;
    const double x_loads = double(t.n) / px * 16.0 / 2400.0, w_loads = t.m / 8.0 * 16.0 / 2400.0;  // us of a step's loads
    const double steps = double((p.in_channels + 63) / 64), share = double(blocks(prob)) / std::max(cus, 1);
    const double y = double(p.output_shape().numel()) * 2.0 / 1e6;
    const double x = double(p.input_shape().numel()) * 2.0 / 1e6 / p.stride_h;  // MB of the rows that are read
    const double spill = std::max(0.0, x + y - 80.0) * (f.spill + (ohw % 64 != 0 ? f.spill_lines : 0.0));
    const double step = f.alone + f.alone_load * (x_loads * (1.0 + f.lines * strided) + w_loads) +
                        std::max(0.0, share - 0.75) *
                            (f.step + f.step_load * (x_loads * (1.0 + f.lines_shared * strided) + w_loads));
    const double part = p.in_channels % 64 != 0 ? 1.0 + f.part : 1.0;
    const double again = strided * f.again * x * double((p.out_channels + t.m - 1) / t.m);
    return f.fixed + (ohw % 8 != 0 ? f.odd : 0.0) + steps * step * part + f.out * y + again + spill;
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
