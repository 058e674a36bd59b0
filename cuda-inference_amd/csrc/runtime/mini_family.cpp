// The small-convolution family (conv_mini.hip: any filter of at most 64 taps straight from NCHW / OIHW, the whole
// reduction in one workgroup) as registry entries, for the layers whose time is latency and launches: one launch, no
// repack, no split-K reduce, no workspace, any channel count and any element-aligned pointers.
//   * FP16 / BF16 entries are mini_<p>_<tile>x<tile>_k<waves>w (Backend::kTensorCore); FP32 and TF32 problems reach the
//     kernel through the split-1 entry of the FP32 family (f32_family.cpp).
//   * capability filter: the entry's precision, a gfx950 device, offsets and LDS within gie_hip_mini_check's limits.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
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

int dtype_of(Precision p) {
  return p == Precision::kFp16   ? GIE_HIP_FP16
         : p == Precision::kBf16 ? GIE_HIP_BF16
         : p == Precision::kTf32 ? GIE_HIP_TF32
                                 : GIE_HIP_FP32;
}

int tile_of(int config) {
  int t = 32, w = 1;
  (void)gie_hip_mini_config_get(config, &t, &w);
  return t;
}
int waves_of(int config) {
  int t = 32, w = 1;
  (void)gie_hip_mini_config_get(config, &t, &w);
  return w;
}
bool half_precision(Precision p) { return p == Precision::kFp16 || p == Precision::kBf16; }
int64_t blocks_of(int config, const ConvProblem& prob) {
  const int t = tile_of(config);
  return (prob.p.gemm_n() + t - 1) / t * ((prob.p.out_channels + t - 1) / t);
}

}  // namespace

// One workgroup runs on a CU at a time, so a launch takes whole rounds of them: 1x3 32 -> 32 over 32x32, BF16, takes
// 5.7 us at 128 to 256 workgroups, 10.0 to 10.2 at 288 to 512, 14.5 at 544 to 640. A round costs `start` (pixel set-up,
// partial tiles, stores), each operand load of a lane `load` and each superstep of the longest wave's share `step`; with
// 16x16 tiles over few channels the rounds overlap in part. Strided rows of x take more cache lines (`strided`), which
// every filter tile of a 1x1 layer reads `again`; odd 16-bit rows of weights take element loads (`ragged`). 1x1 layers, up
// to 2000 channels of tens of images, are priced for their MB of x and y too. Fitted per type, filter and tile to 95-4835
// timings on one MI355X: 5-13 % rms, 5-13 % on 19-1024 others.
double mini_busy_us(int config, const ConvProblem& prob, int cus) {
  struct Fit {
    double start, load, step, overlap, strided, ragged, again, x, y;
  };
  constexpr Fit kFit[2][3][2] = {  // 16 / 32 bits; 1x1, 3x3, other filters; 16x16, 32x32 tiles
      {{{1.33, 0.0052, 0.191, 0.47, 0.00, 2.04, 0.043, 0.325, 0.00}, {1.34, 0.0052, 0.298, 0.00, 0.23, 1.80, 0.042, 0.139, 0.30}},
       {{1.44, 0.0079, 0.082, 0.11, 0.21, 1.37, 0.0, 0.0, 0.0}, {1.48, 0.0073, 0.068, 0.04, 0.31, 1.51, 0.0, 0.0, 0.0}},
       {{1.63, 0.0061, 0.854, 0.00, 0.00, 1.90, 0.0, 0.0, 0.0}, {2.23, 0.0059, 1.431, 0.00, 0.00, 1.30, 0.0, 0.0, 0.0}}},
      {{{1.24, 0.0058, 0.445, 0.45, 0.07, 0.00, 0.012, 0.255, 0.00}, {1.14, 0.0088, 0.747, 0.11, 0.12, 0.00, 0.042, 0.076, 0.40}},
       {{1.81, 0.0096, 0.616, 0.08, 0.24, 0.00, 0.0, 0.0, 0.0}, {2.10, 0.0098, 0.867, 0.09, 0.24, 0.00, 0.0, 0.0, 0.0}},
       {{1.86, 0.0113, 0.280, 0.00, 0.73, 0.00, 0.0, 0.0, 0.0}, {2.60, 0.0136, 0.455, 0.00, 0.46, 0.00, 0.0, 0.0, 0.0}}}};
  const Conv2DParams& p = prob.p;
  const bool k16 = half_precision(prob.precision), one = p.kernel_h * p.kernel_w == 1;
  const bool nine = p.kernel_h == 3 && p.kernel_w == 3;
  const int ck = k16 ? 8 : 4, t = tile_of(config), nw = waves_of(config);
  const Fit& f = kFit[k16 ? 0 : 1][one ? 0 : nine ? 1 : 2][t == 16 ? 0 : 1];
  // supersteps of the reduction (3x3: 9 chunks of each lane group, else 64 k in 16 bits) and a lane's operand loads
  const int64_t ss = nine ? 9 * (64 / t) * ck : 8 * ck, steps = (p.gemm_k() + ss - 1) / ss;
  const double loads = double(steps * ss) / (ck * (64 / t)) * (ck + 1);
  const double share = std::max(1.0, double(blocks_of(config, prob)) / std::max(cus, 1));
  const double rounds = f.overlap * share + (1.0 - f.overlap) * std::ceil(share);
  const double spread = p.stride_w > 1 ? 1.0 + f.strided : 1.0, ragged = k16 && p.gemm_k() % 2 != 0 ? 1.0 + f.ragged : 1.0;
  // sixteen waves on the same supersteps: 3x3 1 % faster (their stores spread over more threads), 1 % slower where they set
  // up a table of taps
  const double wide = nw != 16 || one ? 0.0 : nine ? -0.04 : 0.08;
  const double es = k16 ? 2.0 : 4.0, y = double(p.output_shape().numel()) * es / 1e6;
  const double x = double(p.input_shape().numel()) * es / 1e6 / (one ? p.stride_h : 1);  // MB of the rows that are read
  const double again = p.stride_w > 1 ? f.again * x * double((p.out_channels + t - 1) / t) : 0.0;
  return rounds * (f.start + wide + loads * f.load * spread * ragged + double((steps + nw - 1) / nw) * f.step) + f.x * x +
         f.y * y + again;
}

int mini_best_config(const ConvProblem& prob, int cus, double* us) {
  const gie_conv_geom g = geom_of(prob);
  int best = -1;
  double best_us = 0;
  for (int c = 0; c < gie_hip_mini_config_count(); ++c) {
    if (gie_hip_mini_check(c, dtype_of(prob.precision), &g, nullptr) != GIE_HIP_OK) continue;
    const double t = mini_busy_us(c, prob, cus);
    if (best < 0 || t < best_us) best = c, best_us = t;
  }
  if (us) *us = best_us;
  return best;
}

void mini_launch(int config, const ConvProblem& prob, const void* x, const void* w, const void* bias, void* y,
                 void* stream) {
  const gie_conv_geom g = geom_of(prob);
  check_kernel_status(gie_hip_conv_mini(config, dtype_of(prob.precision), &g, x, w, bias, y, stream),
                      "small MFMA convolution (NCHW / OIHW direct)");
}

namespace {

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
    if (gie_hip_mini_check(Config, dtype_of(P), &g, &lds) != GIE_HIP_OK)
      return no("more than 64 filter taps, or offsets, grid or reduction past the kernel's limits");
    if (size_t(lds) > dev.smem_per_block_optin) return no("needs more LDS than a workgroup may use");
    return true;
  }
  static size_t workspace(const ConvProblem&) { return 0; }
  static size_t lds(const ConvProblem& prob) {
    const gie_conv_geom g = geom_of(prob);
    int bytes = 0;
    return gie_hip_mini_check(Config, dtype_of(P), &g, &bytes) == GIE_HIP_OK ? size_t(bytes) : 0;
  }
  static int64_t blocks(const ConvProblem& prob) { return blocks_of(Config, prob); }
  static int occupancy(const ConvProblem&) { return std::max(1, 8 / waves_of(Config)); }
  static double busy_us(const ConvProblem& prob, int cus) { return mini_busy_us(Config, prob, cus); }
  static void launch(const LaunchArgs& la) {
    if (la.only_stage >= 0 && la.only_stage != 1) return;  // one stage: the convolution itself
    mini_launch(Config, *la.problem, la.x, la.w, la.bias, la.y, la.stream);
  }
};

template <int Config, Precision P>
KernelDesc make_entry() {
  using F = Fns<Config, P>;
  const int t = tile_of(Config), nw = waves_of(Config);
  KernelDesc k;
  k.backend = Backend::kTensorCore;
  k.name = std::string("mini_") + to_string(P) + "_" + std::to_string(t) + "x" + std::to_string(t) + "_k" +
           std::to_string(nw) + "w";
  k.version = 1;
  k.params = {{"block_m", t}, {"block_n", t}, {"block_k", 64}, {"waves", nw}, {"split_k", 1}};
  k.threads_per_block = 64 * nw;
  k.tile_m = t;
  k.tile_n = t;
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
}

}  // namespace

void register_mini_family(std::vector<KernelDesc>& out) {
  if (gie_hip_mini_config_count() != 3) throw Error(StatusCode::kInternal, "small-convolution tile table changed");
  add_precision<Precision::kFp16>(out);
  add_precision<Precision::kBf16>(out);
}

}  // namespace gie
