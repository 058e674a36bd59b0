// The padded-NHWC implicit-GEMM family (conv_nhwc.hip: any filter, stride and padding) as registry entries
// nhwc_<p>_<filters>x<pixels>_sk<S>, in the role of the reference's tcmma registration
// (src/kernels/tensor_core_mma.cu:264-395): one repack dispatch, the GEMM, and a reduce when split-K.
// FP32 entries (nhwc_fp32_<filters>x<pixels>x32_sk<S>) carry Backend::kImplicitGemm, the reference's FP32 backend, beside the
// tile kernel's of f32_family.cpp.
//   * capability filter: fp16/bf16/fp32, a gfx950 device, offsets, grid and steps within gie_hip_nhwc_check's limits, LDS,
//     workspace at most a quarter of device memory;
//   * workspace = [padded NHWC x | 256-B align][repacked w | align][split * |Y| FP32 partials | align]. Caller tensors
//     need only their element's alignment.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "gie_hip.h"
#include "gpu_inference/kernel_registry.h"

namespace gie {
namespace {

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

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
  return p == Precision::kFp16 ? GIE_HIP_FP16 : p == Precision::kBf16 ? GIE_HIP_BF16 : GIE_HIP_FP32;
}

struct Tile {
  int m = 1, n = 1, threads = 64;
};
Tile tile_of(int config) {
  Tile t;
  (void)gie_hip_nhwc_config_get(config, &t.m, &t.n, &t.threads);
  return t;
}

struct Plan {  // what the kernels need for a problem; ok: the configuration takes it
  bool ok = false;
  size_t x_bytes = 0, w_bytes = 0;
  int steps = 0, lds = 0;
};
Plan plan_of(int config, const ConvProblem& prob) {
  const gie_conv_geom g = geom_of(prob);
  long long xb = 0, wb = 0;
  Plan p;
  p.ok = gie_hip_nhwc_check(config, dtype_of(prob.precision), &g, &xb, &wb, &p.steps, &p.lds) == GIE_HIP_OK;
  p.x_bytes = size_t(xb), p.w_bytes = size_t(wb);
  return p;
}

// One call: repack, GEMM, reduce where split; `ws` holds [x | w | partials], each 256-byte aligned.
void run(int config, int split, const LaunchArgs& la) {
  const ConvProblem& prob = *la.problem;
  const gie_conv_geom g = geom_of(prob);
  const Plan pl = plan_of(config, prob);
  char* ws = static_cast<char*>(la.workspace);
  void* wp = ws + align256(pl.x_bytes);
  float* part = split > 1 ? reinterpret_cast<float*>(ws + align256(pl.x_bytes) + align256(pl.w_bytes)) : nullptr;
  const int dt = dtype_of(prob.precision);
  const auto stage = [&](int k) { return la.only_stage < 0 || la.only_stage == k; };
  record_stage_event(la, 0);
  if (stage(0))
    check_kernel_status(gie_hip_repack_nhwc(dt, la.x, ws, la.w, wp, &g, la.stream), "repack (padded NHWC, filter runs)");
  record_stage_event(la, 1);
  if (stage(1))
    check_kernel_status(gie_hip_conv_nhwc(config, dt, &g, ws, wp, la.bias, la.y, part, split, la.stream),
                        "padded-NHWC MFMA convolution");
  record_stage_event(la, 2);
  if (split > 1 && stage(2))
    check_kernel_status(gie_hip_splitk_reduce(dt, part, la.bias, la.y, prob.p.output_shape().numel(), split,
                                              prob.p.out_channels, g.out_h * g.out_w, g.relu, la.stream),
                        "split-K reduce");
}

template <int Config, int Split, Precision P>
struct Fns {
  static bool supports(const ConvProblem& prob, const DeviceInfo& dev, std::string* why) {
    auto no = [&](const std::string& m) {
      if (why) *why = m;
      return false;
    };
    if (prob.precision != P) return no(std::string("kernel is ") + to_string(P) + " only");
    if (!dev.is_gfx950()) return no("needs gfx950 matrix cores; device is " + dev.gcn_arch);
    const Plan pl = plan_of(Config, prob);
    if (!pl.ok) return no("padded copies or grid exceed 32-bit offsets");
    if (Split > 1 && pl.steps < 4 * Split) return no("reduction too short for this split-K factor");
    if (size_t(pl.lds) > dev.smem_per_block_optin) return no("needs more LDS than a workgroup may use");
    if (workspace(prob) > dev.global_mem_bytes / 4) return no("workspace exceeds a quarter of device memory");
    return true;
  }
  static size_t part_bytes(const ConvProblem& prob) {
    return Split > 1 ? align256(size_t(Split) * size_t(prob.p.output_shape().numel()) * 4) : 0;
  }
  static size_t workspace(const ConvProblem& prob) {
    const Plan pl = plan_of(Config, prob);
    return align256(pl.x_bytes) + align256(pl.w_bytes) + part_bytes(prob);
  }
  static size_t lds(const ConvProblem& prob) { return size_t(plan_of(Config, prob).lds); }
  static int64_t blocks(const ConvProblem& prob) {
    const Tile t = tile_of(Config);
    return (prob.p.gemm_n() + t.n - 1) / t.n * ((prob.p.out_channels + t.m - 1) / t.m) * Split;
  }
  static int occupancy(const ConvProblem& prob) {
    return std::max<int>(1, std::min<int>(2048 / tile_of(Config).threads, int(160 * 1024 / std::max<size_t>(lds(prob), 1))));
  }
  // Fixed cost (two launches' set-up and drain, dispatch aside; more where images of x are no multiple of four pixels or
  // images of y of eight), the repack of x and w, the output and the reduce at their traffic, then one workgroup's latency
  // or each CU's share of the workgroups (the last round partly empty) at a start-up cost and a cost for each step of 64
  // 16-bit units. Fitted per tile to 894-4825 timings on one MI355X: 6-8 % rms, 6-8 % on held-out layers (11-17 % without
  // the odd images and the rounds). FP32: 555 and 467 timings, 8 % and 6 %.
  static double busy_us(const ConvProblem& prob, int cus) {
    struct Fit {
      double fixed, alone, alone_step, start, step, x, w, reduce, out, odd_x, odd_y;
    };
    constexpr Fit kFit[] = {{3.06, 0.49, 0.272, 1.01, 0.198, 0.254, 0.87, 0.252, 0.164, 0.86, 0.71},
                            {3.97, 0.43, 0.346, 0.80, 0.308, 0.247, 0.94, 0.266, 0.204, 0.91, 1.01},
                            {2.98, 1.73, 0.434, 2.28, 0.533, 0.235, 0.98, 0.257, 0.222, 0.92, 1.25},
                            {3.48, 2.82, 0.733, 3.13, 0.989, 0.217, 1.19, 0.000, 0.152, 0.90, 2.27},
                            {3.52, 4.79, 1.188, 4.69, 1.483, 0.206, 1.75, 0.000, 0.145, 1.41, 4.03}};
    constexpr Fit kFp32[] = {{3.35, 0.78, 0.642, 1.08, 0.597, 0.187, 0.79, 0.248, 0.120, 0.0, 0.0},
                             {3.07, 2.44, 2.043, 2.92, 2.107, 0.187, 1.17, 0.286, 0.196, 0.0, 0.0}};
    constexpr bool f32 = P == Precision::kFp32;
    const Fit& f = f32 ? kFp32[Config == 0 ? 0 : 1] : kFit[Config];
    const Conv2DParams& p = prob.p;
    const Plan pl = plan_of(Config, prob);
    const double es = double(dtype_size(prob.dtype()));
    const double steps = double(pl.steps) / Split, rounds = double(blocks(prob)) / std::max(cus, 1);
    const double whole = f32 ? 0.87 : 0.5;  // weight of whole rounds: FP32 steps keep the matrix cores busy
    const double share = (1.0 - whole) * rounds + whole * std::ceil(rounds);
    const double x = (double(pl.x_bytes) + double(p.input_shape().numel()) * es) / 1e6, w = 2.0 * double(pl.w_bytes) / 1e6;
    const double y = double(p.output_shape().numel()) * es / 1e6;
    const double partials = Split > 1 ? (Split + 1) * double(p.output_shape().numel()) * 4.0 / 1e6 : 0.0;  // MB, as the above
    const bool odd_x = int64_t(p.in_h) * p.in_w % 4 != 0, odd_y = int64_t(p.out_h()) * p.out_w() % 8 != 0;
    return f.fixed + (odd_x ? f.odd_x : 0.0) + (odd_y ? f.odd_y : 0.0) + f.x * x + f.w * w + f.out * y + f.reduce * partials +
           std::max(f.alone + steps * f.alone_step, share * (f.start + steps * f.step));
  }
  static void launch(const LaunchArgs& la) { run(Config, Split, la); }
};

template <int Config, int Split, Precision P>
KernelDesc make_entry() {
  using F = Fns<Config, Split, P>;
  const Tile t = tile_of(Config);
  KernelDesc k;
  const bool f32 = P == Precision::kFp32;
  const int bk = f32 ? 32 : 64;  // channels of a step
  k.backend = f32 ? Backend::kImplicitGemm : Backend::kTensorCore;
  k.name = std::string("nhwc_") + to_string(P) + "_" + std::to_string(t.m) + "x" + std::to_string(t.n) + "x" +
           std::to_string(bk) + "_sk" + std::to_string(Split);
  k.version = 1;
  k.params = {{"block_m", t.m}, {"block_n", t.n}, {"block_k", bk}, {"split_k", Split}};
  k.threads_per_block = t.threads;
  k.tile_m = t.m;
  k.tile_n = t.n;
  k.tile_k = bk;
  k.uses_tensor_cores = !f32;  // FP32 is priced against the FP32 ceiling, which the FP32 MFMA rate equals
  k.launches = 2 + (Split > 1 ? 1 : 0);
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
  out.push_back(make_entry<0, 1, P>());
  out.push_back(make_entry<1, 1, P>());
  out.push_back(make_entry<2, 1, P>());
  out.push_back(make_entry<3, 1, P>());
  out.push_back(make_entry<4, 1, P>());
  out.push_back(make_entry<0, 2, P>());
  out.push_back(make_entry<1, 2, P>());
  out.push_back(make_entry<0, 4, P>());
  out.push_back(make_entry<1, 4, P>());
  out.push_back(make_entry<2, 2, P>());
}

// FP32: the tiles whose four accumulators fit the registers
void add_fp32(std::vector<KernelDesc>& out) {
  constexpr Precision P = Precision::kFp32;
  out.push_back(make_entry<0, 1, P>());
  out.push_back(make_entry<2, 1, P>());
  out.push_back(make_entry<0, 2, P>());
  out.push_back(make_entry<2, 2, P>());
  out.push_back(make_entry<0, 4, P>());
  out.push_back(make_entry<2, 4, P>());
}

}  // namespace

void register_nhwc_family(std::vector<KernelDesc>& out) {
  if (gie_hip_nhwc_config_count() != 5) throw Error(StatusCode::kInternal, "padded-NHWC tile table changed");
  add_precision<Precision::kFp16>(out);
  add_precision<Precision::kBf16>(out);
  add_fp32(out);
}

}  // namespace gie
