// Small convolutions straight from NCHW x and OIHW w in one launch, any filter of at most 64 taps, any stride and
// padding, any channel count: the whole reduction inside one workgroup, operands straight from memory to registers.
//
// What bounds the layers this is for (one image, or a few small ones) is latency and launches, not bytes or FLOPs:
// a repack, a convolution of a few dozen workgroups and a split-K reduce take 12-15 us for work worth 0.1 us. Here a
// workgroup owns one 16x16 or 32x32 tile (filters x output pixels) and its NW waves split the reduction between them,
// so a layer of 196 pixels x 256 filters is 208 workgroups x 8 waves with every load of a wave's share in flight at
// once:
//   * one MFMA block per wave, A = filters, B = pixels. The reduction runs in OIHW order, k = c * RS + tap, so a lane's A
//     operand (one filter, consecutive k) is one 16-byte load of the caller's weights, and its B operand (one pixel,
//     the same k) is one element load for each k, 16 or 32 lanes reading neighbouring pixels;
//   * the element loads cost no address arithmetic for the two common filters. 1x1: the channel is a scalar offset.
//     3x3: 9 per-lane offsets (one for each tap, out of range where the tap lies in the padding, so the load returns
//     zero) and a scalar channel offset; a superstep of 9 operand chunks of each lane group covers whole channels, so
//     which tap an element is follows from its position alone (each group holds its nine offsets rotated by where its
//     chunks start). Other filters read (offset, tap) for each k from a table in LDS;
//   * no LDS and no barrier in the reduction. At the end the waves' partial tiles are added in LDS in wave
//     order (so the sum does not depend on timing), then bias, ReLU, one rounding and stores of pixel pairs.
// Partly filled last supersteps take a masked copy of the loop body (both operands, so nothing past the end of a
// filter's weights enters the sum, not even times zero).
// FP32 and TF32 run the same way with the FP32 MFMAs (32x32x2, 16x16x4: four of them for each 16-byte chunk); TF32
// rounds both operands in registers as conv_f32.hip does.
// Which tile: 16x16 doubles the element loads for each product but quarters the work of a workgroup, so it wins while
// its workgroups fit the 256 CUs once (196 pixels x 1024 -> 256, 1x1: 4.2 us against 5.7; 3x3 x 256: 8.2 against 13.1)
// and loses beyond (196 pixels x 256 -> 1024: 8.2 against 3.7 us). Before, repack + implicit GEMM (+ reduce): 10.6,
// 9.5 (slab, split 4) and 7.9 us; FP32 3x3 64 -> 64 over 56x56, one image: 18.3 -> 6.6 us (FP32 kernel, split 8).
#include <algorithm>

#include "device_common.h"

namespace gie_hip {
namespace {

constexpr int kMiniOut = int(0x80000000u);  // past any buffer range: loads return zeros, stores are dropped
constexpr int kMiniWord3 = 0x00020000;
// floats per row of a partial tile: the lane groups' rows, 4 apart, fall on disjoint parts of the 64 banks
constexpr int mini_pitch(int t) { return t == 32 ? 40 : 20; }
// operand chunks of each lane group per superstep: 3x3 covers whole channels, the others spread 64 k over the groups
constexpr int mini_chunks(int rsk, int t) { return rsk == 9 ? 9 : t == 32 ? 4 : 2; }
template <int T>
struct MiniAcc {
  typedef f32x4 type;
};
template <>
struct MiniAcc<32> {
  typedef f32x16 type;
};

struct MiniGeom {
  int C, H, W, O, KH, KW, SH, SW, PH, PW, OW;
  int HW, OHW, RS, K, N;
  int S;        // supersteps of the reduction
  int n_ot;     // filter blocks
  int x_shift;  // elements the x resource starts before x (the padding's share of the smallest tap offset)
  int x_bytes, w_bytes;
  int relu, y_pairs;
};

struct MiniF32 {
  static constexpr int kDtype = GIE_HIP_FP32;
};
struct MiniTf32 {
  static constexpr int kDtype = GIE_HIP_TF32;
};

template <typename E>
struct MiniTraits {
  static constexpr bool k16 = E::kDtype == GIE_HIP_FP16 || E::kDtype == GIE_HIP_BF16;
  static constexpr int ES = k16 ? 2 : 4;
  static constexpr int CK = 16 / ES;  // elements of a 16-byte operand chunk
};

__device__ __forceinline__ uint32_t mini_tf32(uint32_t u) {
  if ((u & 0x7f800000u) != 0x7f800000u) u = (u + 0x1000u) & 0xffffe000u;  // Inf/NaN pass through
  return u;
}

// RSK: 1 or 9 taps (unpadded offsets known at compile time), 0 any filter (table in LDS). T: tile side, 16 or 32.
// WVEC: weights by 16-byte loads (rows of whole 4-byte words), else element by element.
template <typename E, int RSK, int NW, int T, bool WVEC>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(NW / 4, NW / 4))) void mini_kernel(
    const void* __restrict__ x, const void* __restrict__ w, const void* __restrict__ bias, void* __restrict__ y,
    MiniGeom g) {
  using Tr = MiniTraits<E>;
  using Acc = typename MiniAcc<T>::type;
  constexpr int CK = Tr::CK, ES = Tr::ES;
  constexpr int G = 64 / T;                           // lane groups, each with its own operand chunk
  constexpr int MM = mini_chunks(RSK, T);             // chunks of each group per superstep
  constexpr int SS = MM * G * CK;                     // reduction elements per superstep
  constexpr int CPS = RSK == 0 ? 0 : SS / (RSK == 9 ? 9 : 1);  // whole channels per superstep
  constexpr int NV = RSK == 9 ? 9 : 1;
  constexpr int MB = RSK != 9 ? MM : !WVEC ? (NW == 16 ? 1 : 3) : Tr::k16 && NW == 16 ? 3 : 9;  // chunks loaded together
  constexpr int PITCH = mini_pitch(T), TILE = T * PITCH;
  extern __shared__ __attribute__((aligned(16))) unsigned char mini_lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int px = lane % T, h = lane / T;
  const int ot = int(blockIdx.x) % g.n_ot, pt = int(blockIdx.x) / g.n_ot;
  const int o0 = ot * T, n0 = pt * T;

  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(x)) - static_cast<long long>(g.x_shift) * ES, 0, g.x_bytes, kMiniWord3);
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(w), 0, g.w_bytes, kMiniWord3);

  // ---- table of the general form: byte displacement and tap of every k (past the reduction: out of range) ----
  int2* lut = reinterpret_cast<int2*>(mini_lds);
  if constexpr (RSK == 0) {
    const int kp = g.S * SS;
    for (int k = tid; k < kp; k += NW * 64) {
      const int c = k / g.RS, t = k - c * g.RS, r = t / g.KW, s = t - r * g.KW;
      lut[k] = k < g.K ? int2{(c * g.HW + r * g.W + s) * ES, t} : int2{kMiniOut, 0};
    }
    __syncthreads();
  }

  // ---- the lane's pixel ----
  const int n = n0 + px;
  const bool n_ok = n < g.N;
  const int b = (n_ok ? n : 0) / g.OHW, p = (n_ok ? n : 0) - b * g.OHW;
  const int oh = p / g.OW, ow = p - oh * g.OW;
  const int ih0 = oh * g.SH - g.PH, iw0 = ow * g.SW - g.PW;
  const int pbase = (b * g.C * g.HW + ih0 * g.W + iw0 + g.x_shift) * ES;  // tap (0, 0), channel 0 of the resource
  int vo[NV];
  unsigned long long bad = 0;  // general form: taps outside the image
  if constexpr (RSK == 9) {
    // element q of the group's chunks is k = h * CK + q: with u = q % 9, tap (h * CK + u) % 9 of the channel
    // (h * CK + u) / 9 later than q / 9
#pragma unroll
    for (int u = 0; u < 9; ++u) {
      const int k = h * CK + u, c = (k * 57) >> 9, t = k - 9 * c, r = (t * 11) >> 5, s = t - 3 * r;  // k < 33
      const bool ok = n_ok & (unsigned(ih0 + r) < unsigned(g.H)) & (unsigned(iw0 + s) < unsigned(g.W));
      vo[u] = ok ? pbase + (c * g.HW + r * g.W + s) * ES : kMiniOut;
    }
  } else if constexpr (RSK == 1) {
    const bool ok = n_ok & (unsigned(ih0) < unsigned(g.H)) & (unsigned(iw0) < unsigned(g.W));
    vo[0] = ok ? pbase + h * CK * g.HW * ES : kMiniOut;
  } else {
    vo[0] = pbase;
    unsigned cols = 0;
    for (int s = 0; s < g.KW; ++s) cols |= unsigned(unsigned(iw0 + s) < unsigned(g.W)) << s;
    unsigned long long good = 0;
    for (int r = 0; r < g.KH; ++r)
      if (n_ok && unsigned(ih0 + r) < unsigned(g.H)) good |= static_cast<unsigned long long>(cols) << (r * g.KW);
    bad = ~good;
  }
  const int wo = o0 + px < g.O ? ((o0 + px) * g.K + h * CK) * ES : kMiniOut;

  Acc acc = {};
  auto superstep = [&](int s, auto tail_c) __attribute__((always_inline)) {
    constexpr bool TAIL = decltype(tail_c)::value;
#pragma unroll
    for (int m0 = 0; m0 < MM; m0 += MB) {
      if constexpr (MB < MM) __builtin_amdgcn_sched_barrier(0);  // or the compiler hoists every batch's loads
      uint32_t xe[MB][CK], we[MB][WVEC ? 1 : CK];
      u32x4 wf[MB];
#pragma unroll
      for (int m = m0; m < m0 + MB; ++m) {
        const int kb = s * SS + (G * m + h) * CK;   // the lane's first k of the chunk
        const int left = g.K - kb;                  // TAIL: its elements inside the reduction
        const int wsoff = (s * SS + G * m * CK) * ES;
        if constexpr (WVEC) {
          wf[m - m0] = __builtin_bit_cast(
              u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, TAIL && left <= 0 ? kMiniOut : wo, wsoff, 0));
        } else {
#pragma unroll
          for (int i = 0; i < CK; ++i)
            we[m - m0][i] = __builtin_amdgcn_raw_buffer_load_b16(
                wr, (TAIL && i >= left) || wo == kMiniOut ? kMiniOut : wo + i * ES, wsoff, 0);
        }
#pragma unroll
        for (int i = 0; i < CK; ++i) {
          const int q = G * m * CK + i;
          int off, soff;
          if constexpr (RSK == 0) {
            const int2 l = lut[kb + i];
            off = (bad >> l.y) & 1u ? kMiniOut : int(unsigned(vo[0]) + unsigned(l.x));
            soff = 0;
          } else {
            off = TAIL && i >= left ? kMiniOut : vo[RSK == 9 ? q % 9 : 0];
            soff = (s * CPS + (RSK == 9 ? q / 9 : q)) * g.HW * ES;
          }
          if constexpr (Tr::k16) xe[m - m0][i] = __builtin_amdgcn_raw_buffer_load_b16(xr, off, soff, 0);
          else xe[m - m0][i] = __builtin_amdgcn_raw_buffer_load_b32(xr, off, soff, 0);
        }
      }
      // every load of the batch goes out before the first is waited for
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = m0; m < m0 + MB; ++m) {
        u32x4 a, v;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          if constexpr (WVEC) a[d] = wf[m - m0][d];
          else a[d] = we[m - m0][2 * d] | (we[m - m0][2 * d + 1] << 16);
          if constexpr (Tr::k16) v[d] = xe[m - m0][2 * d] | (xe[m - m0][2 * d + 1] << 16);
          else v[d] = xe[m - m0][d];
        }
        if constexpr (TAIL && WVEC) {  // the chunk may run into the next filter's weights
          const int left = g.K - (s * SS + (G * m + h) * CK);
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            if constexpr (Tr::k16) a[d] = 2 * d + 1 < left ? a[d] : 2 * d < left ? a[d] & 0xffffu : 0u;
            else a[d] = d < left ? a[d] : 0u;
          }
        }
        if constexpr (Tr::k16) {
          if constexpr (T == 32) acc = E::mfma32(a, v, acc);
          else acc = E::mfma(a, v, acc);
        } else {
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const float av = __uint_as_float(E::kDtype == GIE_HIP_TF32 ? mini_tf32(a[d]) : a[d]);
            const float xv = __uint_as_float(E::kDtype == GIE_HIP_TF32 ? mini_tf32(v[d]) : v[d]);
            if constexpr (T == 32) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, xv, acc, 0, 0, 0);
            else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, xv, acc, 0, 0, 0);
          }
        }
      }
    }
  };

  // ---- the wave's share of the supersteps ----
  const int active = min(NW, g.S);
  if (wave < active) {
    const int s_end = g.S * (wave + 1) / active;
    for (int s = g.S * wave / active; s < s_end; ++s) {
      if ((s + 1) * SS <= g.K) superstep(s, std::false_type{});
      else superstep(s, std::true_type{});
    }
  }

  // ---- partial tiles to LDS, added in wave order ----
  if constexpr (RSK == 0) __syncthreads();  // the table's space is reused
  float* red = reinterpret_cast<float*>(mini_lds);
  if (wave < active) {
#pragma unroll
    for (int r = 0; r < T * T / 64; ++r)  // 32: rows 8 (r / 4) + 4 h + r % 4; 16: rows 4 h + r
      red[wave * TILE + (8 * (r >> 2) + 4 * h + (r & 3)) * PITCH + px] = acc[r];
  }
  __syncthreads();
  for (int i = tid; i < T * T / 2; i += NW * 64) {
    const int row = i / (T / 2), c2 = (i % (T / 2)) * 2, o = o0 + row, nn = n0 + c2;
    if (o >= g.O || nn >= g.N) continue;
    float v0 = 0.f, v1 = 0.f;
    for (int a = 0; a < active; ++a) {
      const f32x2 t = *reinterpret_cast<const f32x2*>(red + a * TILE + row * PITCH + c2);
      v0 += t.x;
      v1 += t.y;
    }
    if (bias != nullptr) {
      float bv;
      if constexpr (Tr::k16) bv = E::to_f32(static_cast<const uint16_t*>(bias)[o]);
      else bv = static_cast<const float*>(bias)[o];
      v0 += bv;
      v1 += bv;
    }
    if (g.relu) {
      v0 = fmaxf(v0, 0.f);
      v1 = fmaxf(v1, 0.f);
    }
    const int b0 = nn / g.OHW, p0 = nn - b0 * g.OHW;
    const long long e0 = (static_cast<long long>(b0) * g.O + o) * g.OHW + p0;
    if (g.y_pairs) {  // an even number of pixels per image, y aligned for pairs
      if constexpr (Tr::k16)
        *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(y) + e0) = uint32_t(E::from_f32(v0)) | (uint32_t(E::from_f32(v1)) << 16);
      else
        *reinterpret_cast<f32x2*>(static_cast<float*>(y) + e0) = f32x2{v0, v1};
      continue;
    }
    const bool wrap = p0 + 1 == g.OHW;  // the second pixel is the next image's first
    const long long e1 = wrap ? (static_cast<long long>(b0 + 1) * g.O + o) * g.OHW : e0 + 1;
    if constexpr (Tr::k16) {
      static_cast<uint16_t*>(y)[e0] = E::from_f32(v0);
      if (nn + 1 < g.N) static_cast<uint16_t*>(y)[e1] = E::from_f32(v1);
    } else {
      static_cast<float*>(y)[e0] = v0;
      if (nn + 1 < g.N) static_cast<float*>(y)[e1] = v1;
    }
  }
}

// ---- configurations: tile side and waves ----
struct MiniConfig {
  int t, nw;
};
constexpr MiniConfig kMiniConfigs[] = {{16, 8}, {32, 8}, {32, 16}};
constexpr int kMiniCount = int(sizeof(kMiniConfigs) / sizeof(kMiniConfigs[0]));

using MiniFn = void (*)(const void*, const void*, const void*, void*, MiniGeom);

template <typename E, int RSK, bool WVEC>
MiniFn mini_fn(int config) {
  switch (config) {
    case 0: return &mini_kernel<E, RSK, 8, 16, WVEC>;
    case 1: return &mini_kernel<E, RSK, 8, 32, WVEC>;
    default: return &mini_kernel<E, RSK, 16, 32, WVEC>;
  }
}
template <typename E>
MiniFn mini_fn(int config, int rsk, bool wvec) {
  if constexpr (MiniTraits<E>::k16) {  // rows of 32-bit words always take 16-byte loads
    if (!wvec)
      return rsk == 1 ? mini_fn<E, 1, false>(config) : rsk == 9 ? mini_fn<E, 9, false>(config) : mini_fn<E, 0, false>(config);
  }
  return rsk == 1 ? mini_fn<E, 1, true>(config) : rsk == 9 ? mini_fn<E, 9, true>(config) : mini_fn<E, 0, true>(config);
}

// the geometry the kernel takes: any filter of at most 64 taps whose offsets fit 32 bits and whose table fits the LDS
int mini_prepare(int config, int dtype, const gie_conv_geom* gg, MiniGeom* g, int* rsk, int* lds, long long* blocks) {
  if (!gg || config < 0 || config >= kMiniCount) return GIE_HIP_EINVAL;
  if (dtype < GIE_HIP_FP32 || dtype > GIE_HIP_TF32) return GIE_HIP_EUNSUPPORTED;
  if (gg->batch <= 0 || gg->in_channels <= 0 || gg->in_h <= 0 || gg->in_w <= 0 || gg->out_channels <= 0 ||
      gg->kernel_h <= 0 || gg->kernel_w <= 0 || gg->stride_h <= 0 || gg->stride_w <= 0 || gg->pad_h < 0 ||
      gg->pad_w < 0 || gg->out_h <= 0 || gg->out_w <= 0)
    return GIE_HIP_EINVAL;
  const MiniConfig& mc = kMiniConfigs[config];
  const bool k16 = dtype == GIE_HIP_FP16 || dtype == GIE_HIP_BF16;
  const int es = k16 ? 2 : 4, ck = 16 / es;
  const long long rs = 1LL * gg->kernel_h * gg->kernel_w;
  if (rs > 64 || gg->kernel_w > 32) return GIE_HIP_EUNSUPPORTED;
  *rsk = rs == 1 ? 1 : gg->kernel_h == 3 && gg->kernel_w == 3 ? 9 : 0;
  const int ss = mini_chunks(*rsk, mc.t) * (64 / mc.t) * ck;
  const long long k = rs * gg->in_channels, hw = 1LL * gg->in_h * gg->in_w, ohw = 1LL * gg->out_h * gg->out_w;
  const long long s = (k + ss - 1) / ss, n = ohw * gg->batch;
  const long long shift = 1LL * gg->pad_h * gg->in_w + gg->pad_w;
  const long long xb = (hw * gg->batch * gg->in_channels + shift) * es, wb = k * gg->out_channels * es;
  // offsets of whole supersteps, a lane half and a chunk further than the data, and of taps past the last row
  const long long slack = (1LL * (ss + 4 * ck) * hw + 1LL * (gg->kernel_h + gg->pad_h) * (gg->in_w + gg->pad_w)) * es;
  if (xb + slack >= 0x7fffffffLL || wb + 2 * ss * es >= 0x7fffffffLL || n >= 0x7fffffffLL - 64 ||
      n * gg->out_channels >= (1LL << 40))
    return GIE_HIP_EUNSUPPORTED;
  // the tallest and widest reach of a tap past the image must not leave the 32-bit range either
  if (1LL * (gg->out_h - 1) * gg->stride_h + gg->kernel_h > (1 << 24) ||
      1LL * (gg->out_w - 1) * gg->stride_w + gg->kernel_w > (1 << 24))
    return GIE_HIP_EUNSUPPORTED;
  const long long table = *rsk == 0 ? s * ss * 8 : 0;
  const long long red = 1LL * std::min<long long>(mc.nw, s) * mc.t * mini_pitch(mc.t) * 4;
  if (std::max(table, red) > 128 * 1024) return GIE_HIP_EUNSUPPORTED;
  *lds = int(std::max(table, red));
  const long long n_ot = (gg->out_channels + mc.t - 1) / mc.t;
  *blocks = (n + mc.t - 1) / mc.t * n_ot;
  if (*blocks > 0x7fffffffLL) return GIE_HIP_EUNSUPPORTED;
  g->C = gg->in_channels;
  g->H = gg->in_h;
  g->W = gg->in_w;
  g->O = gg->out_channels;
  g->KH = gg->kernel_h;
  g->KW = gg->kernel_w;
  g->SH = gg->stride_h;
  g->SW = gg->stride_w;
  g->PH = gg->pad_h;
  g->PW = gg->pad_w;
  g->OW = gg->out_w;
  g->HW = int(hw);
  g->OHW = int(ohw);
  g->RS = int(rs);
  g->K = int(k);
  g->N = int(n);
  g->S = int(s);
  g->n_ot = int(n_ot);
  g->x_shift = int(shift);
  g->x_bytes = int(xb);
  g->w_bytes = int(wb);
  g->relu = gg->relu ? 1 : 0;
  g->y_pairs = 0;
  return GIE_HIP_OK;
}

}  // namespace
}  // namespace gie_hip

using namespace gie_hip;

extern "C" int gie_hip_mini_config_count(void) { return kMiniCount; }

extern "C" int gie_hip_mini_config_get(int config, int* tile, int* waves) {
  if (config < 0 || config >= kMiniCount || !tile || !waves) return GIE_HIP_EINVAL;
  *tile = kMiniConfigs[config].t;
  *waves = kMiniConfigs[config].nw;
  return GIE_HIP_OK;
}

extern "C" int gie_hip_mini_check(int config, int dtype, const gie_conv_geom* gg, int* lds_bytes) {
  MiniGeom g;
  int rsk = 0, lds = 0;
  long long blocks = 0;
  const int rc = mini_prepare(config, dtype, gg, &g, &rsk, &lds, &blocks);
  if (rc == GIE_HIP_OK && lds_bytes) *lds_bytes = lds;
  return rc;
}

extern "C" int gie_hip_conv_mini(int config, int dtype, const gie_conv_geom* gg, const void* x, const void* w,
                                 const void* bias, void* y, void* stream) {
  if (!x || !w || !y) return GIE_HIP_EINVAL;
  MiniGeom g;
  int rsk = 0, lds = 0;
  long long blocks = 0;
  if (int rc = mini_prepare(config, dtype, gg, &g, &rsk, &lds, &blocks)) return rc;
  const bool k16 = dtype == GIE_HIP_FP16 || dtype == GIE_HIP_BF16;
  const uintptr_t es = k16 ? 2 : 4;
  const auto off = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; };
  if (off(x, es) || off(w, es) || off(y, es) || off(bias, es)) return GIE_HIP_EINVAL;
  // 16-byte buffer loads need 4-byte aligned addresses: rows of an even number of halves, w itself aligned
  const bool wvec = (1LL * g.K * int(es)) % 4 == 0 && !off(w, 4);
  g.y_pairs = g.OHW % 2 == 0 && !off(y, 2 * es) ? 1 : 0;
  MiniFn fn;
  switch (dtype) {
    case GIE_HIP_FP16: fn = mini_fn<Fp16>(config, rsk, wvec); break;
    case GIE_HIP_BF16: fn = mini_fn<Bf16>(config, rsk, wvec); break;
    case GIE_HIP_FP32: fn = mini_fn<MiniF32>(config, rsk, true); break;
    default: fn = mini_fn<MiniTf32>(config, rsk, true); break;
  }
  if (lds > 64 * 1024)
    if (int rc = lds_opt_in(reinterpret_cast<const void*>(fn), 128 * 1024)) return rc;
  hipLaunchKernelGGL(fn, dim3(unsigned(blocks)), dim3(unsigned(kMiniConfigs[config].nw * 64)), size_t(lds),
                     static_cast<hipStream_t>(stream), x, w, bias, y, g);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GIE_HIP_OK : int(e);
}
