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
  // Fixed cost (two launches' set-up and drain, dispatch aside), the repack and the reduce at their traffic, then each
  // CU's share of the workgroups at a start-up cost and a cost for each 64-element step, or one workgroup's latency
  // where there are fewer than CUs. Fitted per tile to 120-229 layers on one MI355X: 9-13 % rms.
  static double busy_us(const ConvProblem& prob, int cus) {
    struct Fit {
      double fixed, alone, alone_step, start, step;
    };
    constexpr Fit kFit[] = {{5.2, 0.0, 0.288, 1.09, 0.248}, {6.2, 0.0, 0.368, 1.24, 0.376}, {6.2, 0.4, 0.467, 2.86, 0.654},
                            {6.7, 1.9, 0.750, 4.60, 1.028}, {8.1, 4.2, 1.241, 3.99, 1.865}};
    const Plan pl = plan_of(Config, prob);
    const double steps = double(pl.steps) / Split, share = double(blocks(prob)) / std::max(cus, 1);
    const double moved = double(pl.x_bytes) + double(prob.p.input_shape().numel()) * double(dtype_size(prob.dtype())) +
                         2.0 * double(pl.w_bytes);
    const double partials = Split > 1 ? (Split + 1) * double(prob.p.output_shape().numel()) * 4 / 1e6 : 0.0;  // MB
    if (P == Precision::kFp32) {
      // whole rounds of workgroups on CUs that the matrix cores keep busy; fitted to 75 layers (4-7 % rms)
      constexpr double kFp32[][4] = {{5.2, 0.617, 0.8, 0.526}, {4.5, 1.945, 2.95, 1.945}};  // fixed, alone, start, step
      const auto& q = kFp32[Config == 0 ? 0 : 1];
      return q[0] + moved / 4.3e6 + 0.27 * partials + std::max(steps * q[1], std::ceil(share) * (q[2] + steps * q[3]));
    }
    const Fit& f = kFit[Config];
    return f.fixed + moved / 4.3e6 + partials / 5.0 + std::max(f.alone + steps * f.alone_step, share * (f.start + steps * f.step));
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
