// Pointwise convolution (1x1 filter) of any stride, padding, image size and even channel count straight from NCHW x and
// OIHW w on the 16-bit matrix cores (v_mfma_f32_32x32x16_{f16,bf16}, FP32 accumulation): one launch, no repack, no
// workspace. (conv_pw.hip's kernels need 16-byte pixel chunks: stride 1 and images of a multiple of 8 pixels.)
//
// What bounded these layers before: the repack (X read and written, read again by the GEMM, a launch of its own), for
// strided layers of four times the pixels that are needed, and a GEMM that stored its output as 32-byte runs. Here the
// GEMM (pixels x filters over channels) gathers its activation tile itself:
//   * X: each thread owns PX neighbouring pixels (4 or 2 at stride 1 where image size and alignment allow 8- or 4-byte
//     loads, else 1) and a fixed set of 8-channel chunks of the tile; it loads each channel's pixels (the lanes of a
//     wave cover neighbouring pixels, the channel is a scalar offset), transposes in registers (one byte permute for two
//     elements) and writes whole 16-byte chunks to LDS rows [pixel][channel]. A vector load costs the CU's address path
//     16 clocks whatever its width, so the loads' width is what the rate of small tiles hangs on;
//   * W: OIHW rows are channel-contiguous: 16-byte loads to registers, [filter][channel] rows in LDS;
//   * two LDS stages and the loads of the next two steps in flight in registers while a step multiplies, one barrier
//     per step; two or three workgroups per CU cover each other's waits. (One step in flight: 37 us against 32 for 996
//     -> 1992 over 53x53; three leave registers for fewer workgroups.)
//   * epilogue: bias + ReLU + one rounding into an LDS tile [filter][pixel], which leaves as rows of 16-byte stores
//     (at any 2-byte alignment; element by element only where 8 pixels straddle two images), so runs are as long as
//     the tile.
// Grid: the filter tiles of one pixel tile run one after another on one XCD (slot mod 8), so its X comes from HBM once.
// Measured: 256 -> 512 stride 2 over 56x56, batch 16: 29.5 -> 15.9 us (batch 32: 45.0 -> 28.7); 996 -> 1992 over 53x53,
// one image: 49.0 -> 31.7; 896 -> 448 over 10x10, batch 41: 22.0 -> 13.8.
#include <algorithm>

#include "tile_epilogue.h"

namespace gie_hip {
namespace {

constexpr int kGaOut = int(0x80000000u);  // past any buffer range: loads return zeros
constexpr int kGaWord3 = 0x00020000;

struct GatherGeom {
  int C, H, W, O, SH, SW, PH, PW, OW;
  int HW, OHW, N;
  int T;  // 64-channel steps
  int n_pt, n_ot;
  int x_bytes, w_bytes;
  int relu;
};

constexpr int kGaBK = 64;  // channels per step: rows of 128 bytes in LDS
// 16-byte chunk c of row r sits at slot c ^ swz(r), which spreads 16 consecutive rows over the 64 banks (a wave's
// writes and an operand's reads alike)
__device__ __forceinline__ int ga_swz(int row) { return (row >> 1) & 7; }

// Barrier between a step's LDS writes and the next step's reads: drains this wave's LDS accesses only, the prefetches
// stay in flight (__syncthreads would wait for every one of them).
__device__ __forceinline__ void ga_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vmcnt and expcnt unconstrained
  asm volatile("s_barrier" ::: "memory");
}

// TO x TP: filters x pixels of the tile, WO x WP waves, PX pixels per thread and load. EXACT: whole 64-channel steps.
template <typename E, int TO, int TP, int WO, int WP, int PX, bool EXACT>
__global__ __launch_bounds__(WO * WP * 64) void gather_kernel(const uint16_t* __restrict__ x,
                                                              const uint16_t* __restrict__ w,
                                                              const uint16_t* __restrict__ bias,
                                                              uint16_t* __restrict__ y, GatherGeom g) {
  constexpr int NT = WO * WP * 64;
  constexpr int BK = kGaBK, CPR = BK / 8, ROWB = BK * 2;
  constexpr int TPG = TP / PX;                     // threads that cover the tile's pixels once
  constexpr int GX = NT / TPG, CPT = CPR / GX;     // thread groups along the channels, chunks per thread
  constexpr int NE = CPT * 8;                      // x loads per thread per step
  constexpr int XW = PX == 4 ? 2 : 1;              // registers per load
  constexpr int WL = TO * CPR / NT;                // w chunks per thread per step
  constexpr int STG = (TO + TP) * ROWB;            // bytes per stage: x rows, then w rows
  constexpr int WTP = TP / WP, WTO = TO / WO, FP = WTP / 32, FO = WTO / 32;
  static_assert(GX * TPG == NT && CPT * GX == CPR && CPT >= 1, "chunks divide over the thread groups");
  static_assert(WL * NT == TO * CPR && WL >= 1, "weight chunks divide over the threads");
  static_assert(WTP % 32 == 0 && WTO % 32 == 0, "wave tiles are whole 32 x 32 blocks");
  extern __shared__ __attribute__((aligned(16))) unsigned char ga_lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wp = wave / WO, wo = wave % WO;
  const int L = int(blockIdx.x), xcd = L & 7, rr = L >> 3;
  const int ot = rr % g.n_ot, pt = (rr / g.n_ot) * 8 + xcd;
  if (pt >= g.n_pt) return;  // workgroup-uniform: padding slots of the last group
  const int o0 = ot * TO, n0 = pt * TP;

  // ---- x: the thread's pixels (of one image: an image is a multiple of PX pixels) and chunks ----
  const int xp = (tid % TPG) * PX, xg = tid / TPG, e0 = xg * NE;  // first pixel of the tile, first channel of the step
  const int n = n0 + xp;
  const bool n_ok = n < g.N;
  const int b = (n_ok ? n : 0) / g.OHW, p = (n_ok ? n : 0) - b * g.OHW;
  const int oh = p / g.OW, ow = p - oh * g.OW;
  const int ih = oh * g.SH - g.PH, iw = ow * g.SW - g.PW;
  const bool in = n_ok & (unsigned(ih) < unsigned(g.H)) & (unsigned(iw) < unsigned(g.W));
  const int vo = in ? ((b * g.C + e0) * g.HW + ih * g.W + iw) * 2 : kGaOut;
  unsigned x_dst[PX][CPT];
#pragma unroll
  for (int a = 0; a < PX; ++a)
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      x_dst[a][c] = unsigned((xp + a) * ROWB + (((xg * CPT + c) ^ ga_swz(xp + a)) << 4));
  // ---- w: chunk e of the tile is row e / CPR, chunk e % CPR ----
  int w_off[WL], w_k[WL];
  unsigned w_dst[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int e = tid + i * NT, row = e / CPR, c = e - row * CPR;
    w_off[i] = o0 + row < g.O ? ((o0 + row) * g.C + c * 8) * 2 : kGaOut;
    w_k[i] = c * 8;
    w_dst[i] = unsigned(TP * ROWB + row * ROWB + ((c ^ ga_swz(row)) << 4));
  }

  constexpr int PF = 2;  // steps in flight, each in a register set of its own
  struct Set {
    uint32_t xe[NE][XW];
    u32x4 we[WL];
  };
  Set set[PF];
  // Loads of step t. Steps past the last one go through resources of length zero, so every turn of the loop issues the
  // same loads without a branch and the compiler's wait counting stays exact.
  auto load = [&](int t, Set& r) __attribute__((always_inline)) {
    const int k0 = t * BK;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0,
                                                                        t < g.T ? g.x_bytes : 0, kGaWord3);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w), 0,
                                                                        t < g.T ? g.w_bytes : 0, kGaWord3);
#pragma unroll
    for (int i = 0; i < WL; ++i)
      r.we[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                              wr, !EXACT && k0 + w_k[i] >= g.C ? kGaOut : w_off[i], k0 * 2, 0));
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int off = !EXACT && k0 + e0 + i >= g.C ? kGaOut : vo, soff = (k0 + i) * g.HW * 2;
      if constexpr (PX == 4) {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xr, off, soff, 0));
        r.xe[i][0] = v.x, r.xe[i][XW - 1] = v.y;
      } else if constexpr (PX == 2) {
        r.xe[i][0] = __builtin_amdgcn_raw_buffer_load_b32(xr, off, soff, 0);
      } else {
        r.xe[i][0] = __builtin_amdgcn_raw_buffer_load_b16(xr, off, soff, 0);
      }
    }
  };
  // step t from its registers into stage t % 2; w chunks that run past the last channel are cleared behind it
  auto store = [&](int t, Set& r) __attribute__((always_inline)) {
    unsigned char* base = ga_lds + (t & 1) * STG;
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      if constexpr (!EXACT) {
        const int left = g.C - (t * BK + w_k[i]);
#pragma unroll
        for (int d = 0; d < 4; ++d)
          r.we[i][d] = 2 * d + 1 < left ? r.we[i][d] : 2 * d < left ? r.we[i][d] & 0xffffu : 0u;
      }
      *reinterpret_cast<u32x4*>(base + w_dst[i]) = r.we[i];
    }
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
#pragma unroll
      for (int a = 0; a < PX; ++a) {
        u32x4 v;
#pragma unroll
        for (int d = 0; d < 4; ++d)  // pixel a of channels 2d, 2d + 1
          v[d] = __builtin_amdgcn_perm(r.xe[8 * c + 2 * d + 1][a >> 1], r.xe[8 * c + 2 * d][a >> 1],
                                       a & 1 ? 0x07060302u : 0x05040100u);
        *reinterpret_cast<u32x4*>(base + x_dst[a][c]) = v;
      }
    }
  };

  // ---- operands: A = pixels (rows), B = filters (columns); lane: row lane % 32, k-chunk 2 kk + lane / 32 ----
  const int fr = lane & 31, fc = lane >> 5;
  const int swz = ga_swz(fr);  // wave tiles start at multiples of 32 rows, where the swizzle repeats
  const unsigned a_row = unsigned((wp * WTP + fr) * ROWB), b_row = unsigned((TP + wo * WTO + fr) * ROWB);
  f32x16 acc[FP][FO];
#pragma unroll
  for (int i = 0; i < FP; ++i)
#pragma unroll
    for (int j = 0; j < FO; ++j) acc[i][j] = f32x16{};
  auto compute = [&](int st) __attribute__((always_inline)) {
    const unsigned char* base = ga_lds + st * STG;
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      const unsigned col = unsigned(((2 * kk + fc) ^ swz) << 4);
      u32x4 af[FP], bf[FO];
#pragma unroll
      for (int i = 0; i < FP; ++i) af[i] = *reinterpret_cast<const u32x4*>(base + a_row + i * 32 * ROWB + col);
#pragma unroll
      for (int j = 0; j < FO; ++j) bf[j] = *reinterpret_cast<const u32x4*>(base + b_row + j * 32 * ROWB + col);
#pragma unroll
      for (int i = 0; i < FP; ++i)
#pragma unroll
        for (int j = 0; j < FO; ++j) acc[i][j] = E::mfma32(af[i], bf[j], acc[i][j]);
    }
  };

  // ---- steps: step t multiplies from stage t % 2 while steps t + 1 .. t + PF load; one barrier per step. Step k's
  // registers are set k % PF; set t % PF has just been stored when step t starts ----
#pragma unroll
  for (int k = 0; k < PF; ++k) load(k, set[k]);
  store(0, set[0]);
  ga_barrier();
  for (int t0 = 0; t0 < g.T; t0 += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int t = t0 + u;
      if (u == 0 || t < g.T) {
        load(t + PF, set[u]);
        compute(t & 1);
        store(t + 1, set[(u + 1) % PF]);
        ga_barrier();
      }
    }
  }

  // ---- every wave has finished its last step (the barrier above): the stages become the output tile ----
  tile_to_y<E, TO, TP, WO, WP>(acc, ga_lds, bias, y, tid, o0, n0, g.O, g.OHW, g.N, g.relu);
}

// ---- configurations: filters x pixels of the tile, threads ----
struct GatherConfig {
  int to, tp, threads;
};
constexpr GatherConfig kGatherConfigs[] = {
    {64, 64, 128}, {64, 128, 256}, {128, 128, 256}, {256, 128, 512},
};
constexpr int kGatherCount = int(sizeof(kGatherConfigs) / sizeof(kGatherConfigs[0]));

using GatherFn = void (*)(const uint16_t*, const uint16_t*, const uint16_t*, uint16_t*, GatherGeom);

template <typename E, int PX, bool X>
GatherFn gather_fn(int config) {
  switch (config) {
    case 0: return &gather_kernel<E, 64, 64, 1, 2, PX, X>;
    case 1: return &gather_kernel<E, 64, 128, 2, 2, PX, X>;
    case 2: return &gather_kernel<E, 128, 128, 2, 2, PX, X>;
    default: return &gather_kernel<E, 256, 128, 4, 2, PX < 4 ? PX : 2, X>;  // 512 threads cover 128 pixels in pairs
  }
}

int gather_prepare(int config, const gie_conv_geom* gg, GatherGeom* g, int* lds, long long* blocks) {
  if (!gg || config < 0 || config >= kGatherCount) return GIE_HIP_EINVAL;
  if (gg->batch <= 0 || gg->in_channels <= 0 || gg->in_h <= 0 || gg->in_w <= 0 || gg->out_channels <= 0 ||
      gg->kernel_h <= 0 || gg->kernel_w <= 0 || gg->stride_h <= 0 || gg->stride_w <= 0 || gg->pad_h < 0 ||
      gg->pad_w < 0 || gg->out_h <= 0 || gg->out_w <= 0)
    return GIE_HIP_EINVAL;
  // 16-byte weight loads need 4-byte aligned rows
  if (gg->kernel_h != 1 || gg->kernel_w != 1 || gg->in_channels % 2 != 0) return GIE_HIP_EUNSUPPORTED;
  const GatherConfig& gc = kGatherConfigs[config];
  const long long c = gg->in_channels, hw = 1LL * gg->in_h * gg->in_w, ohw = 1LL * gg->out_h * gg->out_w;
  const long long t = (c + kGaBK - 1) / kGaBK, n = ohw * gg->batch;
  const long long xb = hw * gg->batch * c * 2, wb = c * gg->out_channels * 2;
  if (xb + 4 * kGaBK * hw >= 0x7fffffffLL || wb + 4096 >= 0x7fffffffLL || n >= 0x7fffffffLL - 512)
    return GIE_HIP_EUNSUPPORTED;
  if (1LL * gg->out_h * gg->stride_h > (1 << 24) || 1LL * gg->out_w * gg->stride_w > (1 << 24))
    return GIE_HIP_EUNSUPPORTED;
  *lds = std::max(2 * (gc.to + gc.tp) * kGaBK * 2, gc.to * (gc.tp * 2 + 16));
  const long long n_pt = (n + gc.tp - 1) / gc.tp, n_ot = (gg->out_channels + gc.to - 1) / gc.to;
  *blocks = (n_pt + 7) / 8 * 8 * n_ot;
  if (*blocks > 0x7fffffffLL) return GIE_HIP_EUNSUPPORTED;
  g->C = gg->in_channels;
  g->H = gg->in_h;
  g->W = gg->in_w;
  g->O = gg->out_channels;
  g->SH = gg->stride_h;
  g->SW = gg->stride_w;
  g->PH = gg->pad_h;
  g->PW = gg->pad_w;
  g->OW = gg->out_w;
  g->HW = int(hw);
  g->OHW = int(ohw);
  g->N = int(n);
  g->T = int(t);
  g->n_pt = int(n_pt);
  g->n_ot = int(n_ot);
  g->x_bytes = int(xb);
  g->w_bytes = int(wb);
  g->relu = gg->relu ? 1 : 0;
  return GIE_HIP_OK;
}

}  // namespace
}  // namespace gie_hip

using namespace gie_hip;

extern "C" int gie_hip_gather_config_count(void) { return kGatherCount; }

extern "C" int gie_hip_gather_config_get(int config, int* tile_m, int* tile_n, int* threads) {
  if (config < 0 || config >= kGatherCount || !tile_m || !tile_n || !threads) return GIE_HIP_EINVAL;
  *tile_m = kGatherConfigs[config].to;
  *tile_n = kGatherConfigs[config].tp;
  *threads = kGatherConfigs[config].threads;
  return GIE_HIP_OK;
}

extern "C" int gie_hip_gather_check(int config, const gie_conv_geom* gg, int* lds_bytes) {
  GatherGeom g;
  int lds = 0;
  long long blocks = 0;
  const int rc = gather_prepare(config, gg, &g, &lds, &blocks);
  if (rc == GIE_HIP_OK && lds_bytes) *lds_bytes = lds;
  return rc;
}

extern "C" int gie_hip_conv_gather(int config, int dtype, const gie_conv_geom* gg, const void* x, const void* w,
                                   const void* bias, void* y, void* stream) {
  if (!x || !w || !y) return GIE_HIP_EINVAL;
  if (dtype != GIE_HIP_FP16 && dtype != GIE_HIP_BF16) return GIE_HIP_EUNSUPPORTED;
  GatherGeom g;
  int lds = 0;
  long long blocks = 0;
  if (int rc = gather_prepare(config, gg, &g, &lds, &blocks)) return rc;
  const auto off = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; };
  if (off(x, 2) || off(w, 2) || off(y, 2) || off(bias, 2)) return GIE_HIP_EINVAL;
  if (off(w, 4)) return GIE_HIP_EUNSUPPORTED;
  // several pixels per load: output pixels are the input's (stride 1, no padding, no row or column left out), whole groups
  // per image, aligned rows
  const bool flat = g.SH == 1 && g.SW == 1 && g.PH == 0 && g.PW == 0 && gg->out_h == g.H && g.OW == g.W;
  const int px = flat && g.HW % 4 == 0 && !off(x, 8) ? 4 : flat && g.HW % 2 == 0 && !off(x, 4) ? 2 : 1;
  const auto pick = [&](auto e) -> GatherFn {
    using E = decltype(e);
    if (g.C % kGaBK == 0)
      return px == 4 ? gather_fn<E, 4, true>(config) : px == 2 ? gather_fn<E, 2, true>(config) : gather_fn<E, 1, true>(config);
    return px == 4 ? gather_fn<E, 4, false>(config) : px == 2 ? gather_fn<E, 2, false>(config) : gather_fn<E, 1, false>(config);
  };
  const GatherFn fn = dtype == GIE_HIP_FP16 ? pick(Fp16{}) : pick(Bf16{});
  if (lds > 64 * 1024)
    if (int rc = lds_opt_in(reinterpret_cast<const void*>(fn), 160 * 1024)) return rc;
  hipLaunchKernelGGL(fn, dim3(unsigned(blocks)), dim3(unsigned(kGatherConfigs[config].threads)), size_t(lds),
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w),
                     static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(y), g);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GIE_HIP_OK : int(e);
}
