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

// A CU works through its share of the workgroups at a fixed cost each (pixel set-up, partial tiles, stores) plus a
// cost for each operand load of its waves. Fitted on one MI355X, 16-bit: 1x1 960 workgroups x 432 loads 17.4 us,
// x 108 loads 9.9 us; 3x3 1568 x 1296 loads 86 us, 56 x 1296 13.1 us; 7x7 50176 x 108 loads 984 us; FP32 3x3
// 196 x 360 loads 6.7 us, 3136 x 720 loads 126 us. In FP32 sixteen waves hide the loads of long 1x1 reductions better
// (800 channels, 15925 pixels: 26 us against 42).
double mini_busy_us(int config, const ConvProblem& prob, int cus) {
  const Conv2DParams& p = prob.p;
  const bool k16 = half_precision(prob.precision), one = p.kernel_h * p.kernel_w == 1;
  const bool nine = p.kernel_h == 3 && p.kernel_w == 3;
  const int ck = k16 ? 8 : 4, t = tile_of(config);
  // operand loads of a lane over the reduction's whole supersteps (3x3: 9 chunks of each lane group, else 64 k)
  const int64_t ss = nine ? 9 * (64 / t) * ck : 8 * ck;
  const double loads = double((p.gemm_k() + ss - 1) / ss * ss) / (ck * (64 / t)) * (ck + 1);
  double per_load = !one && !nine ? (t == 16 ? 0.014 : k16 ? 0.0105 : 0.022) : !k16 ? 0.012 : t == 16 && one ? 0.0057 : 0.0085;
  const double wave = std::max(1.0, double(blocks_of(config, prob)) / std::max(cus, 1));
  if (waves_of(config) == 16 && (one || nine || wave <= 1.0))
    per_load *= !one && !nine ? 0.85 : k16 ? 1.0 : one ? 0.7 : 0.95;
  // weights element by element (3x3, 331 channels: 44 us)
  if (k16 && p.gemm_k() % 2 != 0) per_load *= one || nine ? 3.5 : 1.4;
  // strided rows of x take twice the cache lines (1x1 544 -> 32, 29x29 /2, batch 53: 37 us at 16x16)
  // FP32: 1x1 466 -> 384, 22x22 /2, batch 60: 85 us, twice the unstrided rate's
  if ((one || (k16 && nine)) && p.stride_w > 1 && wave > 1.0) per_load *= k16 ? 1.6 : 2.0;
  const double share = k16 ? 0.5 * (wave + std::ceil(wave)) : wave;  // the last wave of workgroups is partly empty
  // a CU with a single workgroup is bound by its latency, not by its load path (1024 -> 256, 196 pixels: 5.7 us)
  if (k16 && one && t == 32) per_load -= 0.0038 * std::max(0.0, 2.0 - share);
  // filters without an unrolled form set up their taps for each workgroup, which a CU with one hides in part (1x3 32 ->
  // 143 over 43x43: 15 us); 3x3 workgroups beyond two a CU queue on the load path
  double start = t != 16 ? 1.0 : k16 && one ? 0.7 : 1.3;
  if (k16 && t == 32 && !one && !nine) start = wave > 1.0 ? 3.6 : 2.2;
  if (k16 && t == 32 && nine && wave > 2.0) start *= 1.3, per_load *= 1.15;
  return 0.5 + share * (start + loads * per_load) + (t == 16 ? 0.7 * (share - 1.0) : 0.0);
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
