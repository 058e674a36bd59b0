// Convolution of any filter, stride and padding on the 16-bit matrix cores (v_mfma_f32_32x32x16_{f16,bf16}, FP32
// accumulation) over a spatially padded NHWC copy of x, both operands by direct-to-LDS loads: two launches.
//
// What bounded the layers this takes (3x3 at stride 2 and over images too wide for the slab kernel's rows, 5x5, 1x7):
// the implicit GEMM of conv_mfma.hip loads through registers with a bounds test for each row and tap, keeps too little
// in flight for its tile sizes and stores its output as 32-byte runs; gathering straight from NCHW costs one vector load
// (16 clocks of a CU's address path) for every 64 elements of the unrolled matrix. Here:
//   * repack, one dispatch: x to [image][H + 2 PH][W + 2 PW][Cp] with the padding as real zeros (Cp = channels rounded up
//     to 8), w to [filter][KH][run], run = KW * Cp rounded up to 64. With the padding in memory no load needs a bounds
//     test: tap row r of a pixel is one contiguous run of KW * Cp elements, whatever the stride, so the reduction is KH
//     runs of 64-element steps, a step's whole address is a per-lane constant plus a scalar, and the loop has no address
//     arithmetic. Reads take four pixels of eight channels at any alignment, a register transpose, 16-byte stores;
//   * GEMM: TO filters x TP pixels per workgroup, NST stages of LDS rows [pixel or filter][64 k] filled by 16-byte
//     direct-to-LDS loads (16-byte chunk c of row r in slot c ^ ((r >> 1) & 7): 16 rows of an operand read cover the 64
//     banks; the permutation is in the lanes' source addresses), NST - 1 steps in flight, counted waits, one barrier
//     per step, the next fragments read while the current ones multiply. Where a run is no multiple of 64, the lanes past
//     its end load zeros in its last step (the weights there are zeros too, but x could be infinite);
// What bounds it now: LDS, at about 85 bytes per clock and CU for operand reads and direct loads together (neither more
// stages, nor unpermuted loads, nor fragments read a step ahead change a step's time), hence the 256 x 256 tile for the
// largest layers. Measured (both launches): BF16 3x3 256 -> 256 over 56x56, batch 16: 118.9 -> 71.8 us; FP16 3x3 64 -> 64 over
// 56x56, batch 32: 33.8 -> 26 (best of the other kernels; 53 for the one the dispatcher took); 3x3 stride 2 128 -> 128
// over 56x56, batch 32: 32.6 -> 26.
//   * output through an LDS tile as whole rows (tile_epilogue.h), or FP32 partials for split-K (splitk_reduce.hip sums
//     them in order).
#include <algorithm>

#include "lds_pipe.h"
#include "slab_common.h"
#include "tile_epilogue.h"

namespace gie_hip {
namespace {

// FP32 (v_mfma_f32_32x32x2_f32): the same kernel on twice the 16-bit units, a 16-byte fragment being four channels and
// so four MFMAs, each with an accumulator of its own: no MFMA waits for the one before. Every 16 steps (512 channels) the
// four are added into the tile's sums, so that no sum runs over more than 128 products and the error does not grow with
// the reduction (3x3 512 channels: 1.4e-7 of the norm, 4.0e-7 for one chain). Here the matrix cores bound: a step runs at
// 0.81 (64 x 64) and 0.88 (128 x 128) of their rate, the rest is the last round of tiles and the repack. Measured: 3x3
// 128 -> 128 over 28x28, batch 32: 118.7 -> 90.0 us; 64 -> 64 over 56x56, batch 32: 148 -> 97; 7x7 stride 2 3 -> 64 over
// 224x224, batch 8: 119 -> 50.
struct NhF32 {
  static constexpr int kDtype = GIE_HIP_FP32, kAcc = 4;
  template <int N>
  static __device__ __forceinline__ void mma(u32x4 a, u32x4 b, f32x16 (&c)[N]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      c[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(f32x4, a)[e], __builtin_bit_cast(f32x4, b)[e], c[e],
                                                  0, 0, 0);
  }
};
template <typename E16>
struct NhHalf : E16 {
  static constexpr int kAcc = 1;
  template <int N>
  static __device__ __forceinline__ void mma(u32x4 a, u32x4 b, f32x16 (&c)[N]) {
    c[0] = E16::mfma32(a, b, c[0]);
  }
};

// Cp, Kp and the 64-unit steps count 16-bit units: an FP32 channel is two.
struct NhwcGeom {
  int C, H, W, O, KH, KW, SH, SW, PH, PW, OW, OHW, N;
  int Cp, Hp, Wp;
  int run_steps;  // 64-element steps per filter row
  int tail;       // 16-byte chunks of a run's last step that hold data
  int Kp;         // elements of a repacked filter
  int T;          // steps of the reduction
  int n_pt, n_ot, split;
  int xp_bytes, wp_bytes;
  int relu;
  long long total;  // |Y| (partial stride)
};

// ---- repack ----
constexpr int kNhThreads = 256;
constexpr int kNhFilter = 32768;  // bytes of a filter staged in LDS

template <typename T>
struct NhwcRepack {  // Cp, Kp and run in elements
  const T* x;
  const T* w;
  T* xp;
  T* wp;
  int B, C, H, W, HW, Cp, Hp, Wp, PH, PW, O, KH, KW, Kp, run;  // run: elements per filter row, padded
  int gpi, cgs;           // four-pixel groups per image rounded up to 16, groups of four 16-byte chunks of channels
  long long x_waves;      // wave items: (image, 16 pixel groups, channel group)
  long long x_blocks, border, b_blocks;  // border: 16-byte chunks of padding
};

// Four pixels of one channel at any alignment; past the end of the channel's row of pixels: zeros.
__device__ __forceinline__ u32x2 nh_load4(const uint16_t* p, int left) {
  u32x2 v = {0u, 0u};
  if (left >= 4) {
    __builtin_memcpy(&v, p, 8);
  } else {
    uint32_t e[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) e[i] = i < left ? p[i] : 0u;
    v = u32x2{e[0] | (e[1] << 16), e[2]};
  }
  return v;
}
__device__ __forceinline__ u32x4 nh_load4(const uint32_t* p, int left) {
  u32x4 v = {0u, 0u, 0u, 0u};
  if (left >= 4) {
    __builtin_memcpy(&v, p, 16);
  } else {
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] = i < left ? p[i] : 0u;
  }
  return v;
}

template <typename T>
__global__ __launch_bounds__(kNhThreads) void nhwc_repack_kernel(NhwcRepack<T> j) {
  constexpr int CH = 16 / int(sizeof(T)), FL = kNhFilter / int(sizeof(T));  // channels of a 16-byte chunk, staged elements
  __shared__ __attribute__((aligned(16))) T buf[FL];
  const int tid = threadIdx.x, lane = tid & 63;
  long long blk = blockIdx.x;
  if (blk < j.x_blocks) {
    // a wave: 16 lanes along pixels (4 each) x 4 lane groups along channels (CH each)
    const long long item = blk * (kNhThreads / 64) + (tid >> 6);
    if (item >= j.x_waves) return;
    const int cg = int(item % j.cgs);
    const long long rest = item / j.cgs;
    const int per = j.gpi / 16, b = int(rest / per), p = (int(rest - static_cast<long long>(b) * per) * 16 + (lane & 15)) * 4;
    const int c8 = (cg * 4 + (lane >> 4)) * CH;
    if (p >= j.HW || c8 >= j.Cp) return;
    const T* src = j.x + (static_cast<long long>(b) * j.C + c8) * j.HW + p;
    decltype(nh_load4(src, 0)) in[CH];
#pragma unroll
    for (int r = 0; r < CH; ++r)
      in[r] = nh_load4(src + static_cast<long long>(r) * j.HW, c8 + r < j.C ? j.HW - p : 0);
    int h = p / j.W, w = p - h * j.W;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (p + q < j.HW) {
        u32x4 v;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          v[d] = CH == 4 ? in[d][q]
                         : __builtin_amdgcn_perm(in[(2 * d + 1) % CH][q >> 1], in[(2 * d) % CH][q >> 1],
                                                 q & 1 ? 0x07060302u : 0x05040100u);
        const long long px = (static_cast<long long>(b) * j.Hp + h + j.PH) * j.Wp + w + j.PW;
        *reinterpret_cast<u32x4*>(j.xp + px * j.Cp + c8) = v;
      }
      if (++w == j.W) w = 0, ++h;
    }
    return;
  }
  blk -= j.x_blocks;
  if (blk < j.b_blocks) {
    // padding: rows above, rows below, then the columns left and right of each image row
    const long long i = blk * kNhThreads + tid;
    if (i >= j.border) return;
    const int cv = j.Cp / CH, c8 = int(i % cv) * CH;
    const long long cell = i / cv;
    const int top = j.PH * j.Wp, side = j.Wp - j.W, per = 2 * top + j.H * side;
    const int b = int(cell / per), e = int(cell - static_cast<long long>(b) * per);
    int row, col;
    if (e < top) {
      row = e / j.Wp, col = e - row * j.Wp;
    } else if (e < 2 * top) {
      const int f = e - top, r = f / j.Wp;
      row = j.H + j.PH + r, col = f - r * j.Wp;
    } else {
      const int f = e - 2 * top, r = f / side, s = f - r * side;
      row = j.PH + r, col = s < j.PW ? s : j.W + s;
    }
    *reinterpret_cast<u32x4*>(j.xp + ((static_cast<long long>(b) * j.Hp + row) * j.Wp + col) * j.Cp + c8) = u32x4{0u, 0u, 0u, 0u};
    return;
  }
  // weights: one filter per workgroup, through LDS where it fits
  const int o = int(blk - j.b_blocks), rs = j.KH * j.KW, n = j.C * rs;
  const T* src = j.w + static_cast<long long>(o) * n;
  const bool staged = n <= FL;
  if (staged) {
    const int n8 = n & ~(CH - 1);
    for (int i = tid * CH; i < n8; i += kNhThreads * CH) __builtin_memcpy(buf + i, src + i, 16);
    for (int i = n8 + tid; i < n; i += kNhThreads) buf[i] = src[i];
    __syncthreads();
  }
  T* dst = j.wp + static_cast<long long>(o) * j.Kp;
  for (int t = tid; t < j.Kp / CH; t += kNhThreads) {
    const int r = (t * CH) / j.run, k = t * CH - r * j.run, s = k / j.Cp, c8 = k - s * j.Cp;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (s < j.KW) {
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        const int c = c8 + q, at = c * rs + r * j.KW + s;
        const uint32_t e = c < j.C ? (staged ? buf[at] : src[at]) : 0u;
        if (CH == 4) v[q % 4] = e;
        else v[q / 2] |= e << (16 * (q & 1));
      }
    }
    *reinterpret_cast<u32x4*>(dst + t * CH) = v;
  }
}

// ---- GEMM ----
template <typename E, int TO, int TP, int WO, int WP, int NST>
__global__ __launch_bounds__(WO * WP * 64, E::kAcc == 4 && TO == 64 ? 3 : 1)
void nhwc_kernel(const uint16_t* __restrict__ xp, const uint16_t* __restrict__ wk, const void* __restrict__ bias,
                 void* __restrict__ y, float* __restrict__ partial, NhwcGeom g) {
  constexpr int NW = WO * WP, ROWB = 128, STG = (TO + TP) * ROWB;
  constexpr int LX = TP / 8 / NW, LW = TO / 8 / NW, NI = LX + LW;  // direct loads (8 rows each) per wave and step
  constexpr int WTP = TP / WP, WTO = TO / WO, FP = WTP / 32, FO = WTO / 32;
  static_assert(LX * NW * 8 == TP && LW * NW * 8 == TO, "every wave issues the same loads");
  static_assert(NST * NI < 64, "loads in flight fit the vmcnt counter");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wp = wave / WO, wo = wave % WO;
  // the filter tiles (and K ranges) of one pixel tile run one after another on one XCD (slot mod 8)
  const int L = int(blockIdx.x), xcd = L & 7, rr = L >> 3, per = g.n_ot * g.split;
  const int sub = rr % per, pt = (rr / per) * 8 + xcd;
  if (pt >= g.n_pt) return;  // workgroup-uniform: padding slots of the last group
  const int z = sub / g.n_ot, ot = sub - z * g.n_ot;
  const int o0 = ot * TO, n0 = pt * TP;
  const int t_beg = int(static_cast<long long>(g.T) * z / g.split), t_end = int(static_cast<long long>(g.T) * (z + 1) / g.split);
  const v4i xr = make_vsharp(xp, g.xp_bytes), wr = make_vsharp(wk, g.wp_bytes);
  const v4i x0 = make_vsharp(xp, 0), w0 = make_vsharp(wk, 0);  // every offset out of range: loads give zeros
  const unsigned lds0 = lds_addr(lds);

  // load i of the wave covers rows 8 * (wave + NW * i) .. +7: lane = (row, slot), source chunk slot ^ swz(row)
  int x_off[LX], x_tail[LX], w_off[LW];
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int row = 8 * (wave + NW * i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7), n = n0 + row;
    const int nc = min(n, g.N - 1), b = nc / g.OHW, p = nc - b * g.OHW, oh = p / g.OW, ow = p - oh * g.OW;
    const int off = (((b * g.Hp + oh * g.SH) * g.Wp + ow * g.SW) * g.Cp + c * 8) * 2;
    x_off[i] = n < g.N ? off : kOut;
    x_tail[i] = n < g.N && c < g.tail ? off : kOut;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = 8 * (wave + NW * i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
    w_off[i] = o0 + row < g.O ? ((o0 + row) * g.Kp + c * 8) * 2 : kOut;
  }
  // cursor of the next step to load: filter row, step of its run
  int t_ld = t_beg, r_ld = t_beg / g.run_steps, j_ld = t_beg - r_ld * g.run_steps, st_ld = 0;
  auto issue = [&]() __attribute__((always_inline)) {
    const bool real = t_ld < t_end, last = j_ld + 1 == g.run_steps;
    const v4i xs = real ? xr : x0, ws = real ? wr : w0;
    const int xo = real ? (r_ld * g.Wp * g.Cp + j_ld * 64) * 2 : 0, wof = real ? t_ld * 128 : 0;
    const unsigned base = lds0 + unsigned(st_ld * STG);
#pragma unroll
    for (int i = 0; i < LX; ++i) dma16s(xs, base + unsigned((wave + NW * i) * 1024), last ? x_tail[i] : x_off[i], xo);
#pragma unroll
    for (int i = 0; i < LW; ++i) dma16s(ws, base + unsigned(TP * ROWB + (wave + NW * i) * 1024), w_off[i], wof);
    ++t_ld;
    j_ld = last ? 0 : j_ld + 1;
    r_ld += last ? 1 : 0;
    st_ld = st_ld + 1 == NST ? 0 : st_ld + 1;
  };
#pragma unroll
  for (int k = 0; k < NST; ++k) issue();

  // operands: A = pixels (rows), B = filters (columns); lane: row lane % 32, k-chunk 2 kk + lane / 32
  const int fr = lane & 31, fc = lane >> 5, swz = (fr >> 1) & 7;
  const unsigned a_row = unsigned((wp * WTP + fr) * ROWB), b_row = unsigned((TP + wo * WTO + fr) * ROWB);
  constexpr int NA = E::kAcc;
  f32x16 sum[FP][FO][NA];
#pragma unroll
  for (int i = 0; i < FP; ++i)
#pragma unroll
    for (int j = 0; j < FO; ++j)
#pragma unroll
      for (int a = 0; a < NA; ++a) sum[i][j][a] = f32x16{};

  // Fragments of 16-element step kk + 1 are read while step kk multiplies, across steps too: the last kk of a step meets
  // the barrier first (the next step has landed for every wave, and every wave has read the last of this step's stage,
  // which the loads of step t + NST then take) and reads the next step's first fragments before its own MFMAs.
  f32x16 acc[FP][FO];
#pragma unroll
  for (int i = 0; i < FP; ++i)
#pragma unroll
    for (int j = 0; j < FO; ++j) acc[i][j] = f32x16{};
  auto add_up = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FP; ++i)
#pragma unroll
      for (int j = 0; j < FO; ++j) {
        if constexpr (NA == 4) acc[i][j] += (sum[i][j][0] + sum[i][j][1]) + (sum[i][j][2] + sum[i][j][3]);
        else acc[i][j] = sum[i][j][0];
#pragma unroll
        for (int a = 0; a < NA; ++a) sum[i][j][a] = f32x16{};
      }
  };
  u32x4 af[2][FP], bf[2][FO];
  auto rd = [&](int set, int stage, int kk) __attribute__((always_inline)) {
    const unsigned base = lds0 + unsigned(stage * STG), col = unsigned(((2 * kk + fc) ^ swz) << 4);
#pragma unroll
    for (int i = 0; i < FP; ++i) af[set][i] = rd16(base + a_row + unsigned(i * 32 * ROWB) + col);
#pragma unroll
    for (int j = 0; j < FO; ++j) bf[set][j] = rd16(base + b_row + unsigned(j * 32 * ROWB) + col);
  };
  auto mm = [&](int set) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FP; ++i)
#pragma unroll
      for (int j = 0; j < FO; ++j) E::mma(af[set][i], bf[set][j], sum[i][j]);
  };
  wait_vmcnt<(NST - 1) * NI>();
  stage_barrier();
  rd(0, 0, 0);
  int st = 0;
  for (int t = t_beg; t < t_end; ++t) {
    const int nx = st + 1 == NST ? 0 : st + 1;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (kk < 3) {
        rd((kk + 1) & 1, st, kk + 1);
      } else {
        wait_vmcnt<(NST - 2) * NI>();
        stage_barrier();
        rd(0, nx, 0);
        issue();
      }
      __builtin_amdgcn_sched_barrier(0);
      mm(kk & 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    st = nx;
    if (NA > 1 && (t - t_beg) % 16 == 15) add_up();
  }
  wait_vmcnt<0>();  // loads past the last step still target the stages
  __syncthreads();
  add_up();
  float* part = partial + static_cast<long long>(z) * g.total;
  const bool last = g.split == 1;
  if constexpr (E::kDtype == GIE_HIP_FP32) {
    if (last) {
      part = static_cast<float*>(y);
#pragma unroll
      for (int j = 0; j < FO; ++j) {
        const int o = o0 + wo * WTO + j * 32 + fr;
        const float bv = bias != nullptr && o < g.O ? static_cast<const float*>(bias)[o] : 0.0f;
#pragma unroll
        for (int i = 0; i < FP; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            acc[i][j][e] += bv;
            if (g.relu) acc[i][j][e] = fmaxf(acc[i][j][e], 0.0f);
          }
      }
    }
  } else if (last) {
    tile_to_y<E, TO, TP, WO, WP>(acc, lds, static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(y), tid, o0, n0, g.O,
                                 g.OHW, g.N, g.relu);
    return;
  }
#pragma unroll
  for (int i = 0; i < FP; ++i) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = n0 + wp * WTP + i * 32 + 8 * q + 4 * fc;  // four consecutive pixels
      const int b = min(n, g.N - 1) / g.OHW, p = n - b * g.OHW;
      const bool whole = n + 4 <= g.N && p + 4 <= g.OHW;
#pragma unroll
      for (int j = 0; j < FO; ++j) {
        const int o = o0 + wo * WTO + j * 32 + fr;
        if (o >= g.O) continue;
        float* d = part + (static_cast<long long>(b) * g.O + o) * g.OHW + p;
        if (whole) {
          const f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          __builtin_memcpy(d, &v, 16);
        } else {
          int pp = p;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (n + e < g.N) *d = acc[i][j][4 * q + e];
            ++d;
            if (++pp == g.OHW) pp = 0, d += static_cast<long long>(g.O - 1) * g.OHW;
          }
        }
      }
    }
  }
}

// ---- configurations: filters x pixels of the tile, threads, stages ----
struct NhwcConfig {
  int to, tp, threads, stages;
  bool f32;  // four accumulators fit the registers two workgroups share
};
constexpr NhwcConfig kNhwcConfigs[] = {
    {64, 64, 256, 4, true},    {64, 128, 256, 3, false},  {128, 128, 512, 3, true},
    {128, 256, 512, 3, false}, {256, 256, 512, 2, false},
};
constexpr int kNhwcCount = int(sizeof(kNhwcConfigs) / sizeof(kNhwcConfigs[0]));

using NhwcFn = void (*)(const uint16_t*, const uint16_t*, const void*, void*, float*, NhwcGeom);

template <typename E>
NhwcFn nhwc_fn(int config) {
  switch (config) {
    case 0: return &nhwc_kernel<E, 64, 64, 2, 2, 4>;
    case 1: return &nhwc_kernel<E, 64, 128, 2, 2, 3>;
    case 2: return &nhwc_kernel<E, 128, 128, 2, 4, 3>;
    case 3: return &nhwc_kernel<E, 128, 256, 2, 4, 3>;
    default: return &nhwc_kernel<E, 256, 256, 4, 2, 2>;
  }
}

NhwcFn nhwc_fn32(int config) {
  return config == 0 ? &nhwc_kernel<NhF32, 64, 64, 2, 2, 4> : &nhwc_kernel<NhF32, 128, 128, 2, 4, 3>;
}

int nhwc_prepare(int config, int dtype, const gie_conv_geom* gg, int split, NhwcGeom* g, int* lds, long long* blocks) {
  if (!gg || config < 0 || config >= kNhwcCount || split < 1 || split > 64) return GIE_HIP_EINVAL;
  if (dtype != GIE_HIP_FP16 && dtype != GIE_HIP_BF16 && (dtype != GIE_HIP_FP32 || !kNhwcConfigs[config].f32))
    return GIE_HIP_EUNSUPPORTED;
  const int unit = dtype == GIE_HIP_FP32 ? 2 : 1;  // 16-bit units of an element
  if (gg->batch <= 0 || gg->in_channels <= 0 || gg->in_h <= 0 || gg->in_w <= 0 || gg->out_channels <= 0 ||
      gg->kernel_h <= 0 || gg->kernel_w <= 0 || gg->stride_h <= 0 || gg->stride_w <= 0 || gg->pad_h < 0 ||
      gg->pad_w < 0 || gg->out_h <= 0 || gg->out_w <= 0)
    return GIE_HIP_EINVAL;
  const NhwcConfig& nc = kNhwcConfigs[config];
  const long long cp = (1LL * gg->in_channels * unit + 7) / 8 * 8, hp = gg->in_h + 2LL * gg->pad_h, wp = gg->in_w + 2LL * gg->pad_w;
  if ((gg->out_h - 1LL) * gg->stride_h + gg->kernel_h > hp || (gg->out_w - 1LL) * gg->stride_w + gg->kernel_w > wp)
    return GIE_HIP_EINVAL;
  const long long run = gg->kernel_w * cp, steps = (run + 63) / 64, kp = steps * 64 * gg->kernel_h;
  const long long xb = hp * wp * cp * gg->batch * 2, wb = kp * gg->out_channels * 2;
  const long long ohw = 1LL * gg->out_h * gg->out_w, n = ohw * gg->batch;
  if (xb + 4096 >= 0x7fffffffLL || wb + 4096 >= 0x7fffffffLL || n >= 0x7fffffffLL - 512 || kp >= (1 << 30))
    return GIE_HIP_EUNSUPPORTED;
  const long long t = steps * gg->kernel_h;
  if (t < split) return GIE_HIP_EUNSUPPORTED;
  *lds = std::max(nc.stages * (nc.to + nc.tp) * 128, unit == 1 ? nc.to * (nc.tp * 2 + 16) : 0);
  const long long n_pt = (n + nc.tp - 1) / nc.tp, n_ot = (gg->out_channels + nc.to - 1) / nc.to;
  *blocks = (n_pt + 7) / 8 * 8 * n_ot * split;
  if (*blocks > 0x7fffffffLL) return GIE_HIP_EUNSUPPORTED;
  g->C = gg->in_channels, g->H = gg->in_h, g->W = gg->in_w, g->O = gg->out_channels;
  g->KH = gg->kernel_h, g->KW = gg->kernel_w, g->SH = gg->stride_h, g->SW = gg->stride_w;
  g->PH = gg->pad_h, g->PW = gg->pad_w, g->OW = gg->out_w;
  g->OHW = int(ohw), g->N = int(n);
  g->Cp = int(cp), g->Hp = int(hp), g->Wp = int(wp);
  g->run_steps = int(steps), g->tail = int((run - (steps - 1) * 64) / 8), g->Kp = int(kp), g->T = int(t);
  g->n_pt = int(n_pt), g->n_ot = int(n_ot), g->split = split;
  g->xp_bytes = int(xb), g->wp_bytes = int(wb);
  g->relu = gg->relu ? 1 : 0;
  g->total = n * gg->out_channels;
  return GIE_HIP_OK;
}

bool off_by(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; }

template <typename T>
int repack_nhwc(const NhwcGeom& g, int batch, const void* x, void* xp, const void* w, void* wp, void* stream) {
  constexpr int unit = int(sizeof(T)) / 2;
  NhwcRepack<T> j;
  j.x = static_cast<const T*>(x), j.w = static_cast<const T*>(w);
  j.xp = static_cast<T*>(xp), j.wp = static_cast<T*>(wp);
  j.B = batch, j.C = g.C, j.H = g.H, j.W = g.W, j.HW = g.H * g.W, j.Cp = g.Cp / unit, j.Hp = g.Hp, j.Wp = g.Wp;
  j.PH = g.PH, j.PW = g.PW, j.O = g.O, j.KH = g.KH, j.KW = g.KW, j.Kp = g.Kp / unit, j.run = g.run_steps * 64 / unit;
  j.gpi = ((j.HW + 3) / 4 + 15) / 16 * 16;
  j.cgs = (g.Cp + 31) / 32;
  j.x_waves = 1LL * batch * (j.gpi / 16) * j.cgs;
  j.x_blocks = (j.x_waves + 3) / 4;
  j.border = 1LL * batch * (1LL * g.Hp * g.Wp - j.HW) * (g.Cp / 8);
  j.b_blocks = (j.border + kNhThreads - 1) / kNhThreads;
  const long long total = j.x_blocks + j.b_blocks + g.O;
  if (total > 0x7fffffffLL) return GIE_HIP_EUNSUPPORTED;
  hipLaunchKernelGGL(nhwc_repack_kernel<T>, dim3(unsigned(total)), dim3(kNhThreads), 0, static_cast<hipStream_t>(stream), j);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GIE_HIP_OK : int(e);
}

}  // namespace
}  // namespace gie_hip

using namespace gie_hip;

extern "C" int gie_hip_nhwc_config_count(void) { return kNhwcCount; }

extern "C" int gie_hip_nhwc_config_get(int config, int* tile_m, int* tile_n, int* threads) {
  if (config < 0 || config >= kNhwcCount || !tile_m || !tile_n || !threads) return GIE_HIP_EINVAL;
  *tile_m = kNhwcConfigs[config].to;
  *tile_n = kNhwcConfigs[config].tp;
  *threads = kNhwcConfigs[config].threads;
  return GIE_HIP_OK;
}

extern "C" int gie_hip_nhwc_check(int config, int dtype, const gie_conv_geom* gg, long long* x_bytes, long long* w_bytes,
                                  int* steps, int* lds_bytes) {
  NhwcGeom g;
  int lds = 0;
  long long blocks = 0;
  const int rc = nhwc_prepare(config, dtype, gg, 1, &g, &lds, &blocks);
  if (rc != GIE_HIP_OK) return rc;
  if (x_bytes) *x_bytes = g.xp_bytes;
  if (w_bytes) *w_bytes = g.wp_bytes;
  if (steps) *steps = g.T;
  if (lds_bytes) *lds_bytes = lds;
  return GIE_HIP_OK;
}

extern "C" int gie_hip_repack_nhwc(int dtype, const void* x, void* xp, const void* w, void* wp, const gie_conv_geom* gg,
                                   void* stream) {
  if (!x || !xp || !w || !wp) return GIE_HIP_EINVAL;
  NhwcGeom g;
  int lds = 0;
  long long blocks = 0;
  if (int rc = nhwc_prepare(0, dtype, gg, 1, &g, &lds, &blocks)) return rc;
  const uintptr_t es = dtype == GIE_HIP_FP32 ? 4 : 2;
  if (off_by(x, es) || off_by(w, es) || off_by(xp, 16) || off_by(wp, 16)) return GIE_HIP_EINVAL;
  return dtype == GIE_HIP_FP32 ? repack_nhwc<uint32_t>(g, gg->batch, x, xp, w, wp, stream)
                               : repack_nhwc<uint16_t>(g, gg->batch, x, xp, w, wp, stream);
}

extern "C" int gie_hip_conv_nhwc(int config, int dtype, const gie_conv_geom* gg, const void* xp, const void* wp,
                                 const void* bias, void* y, float* partial, int split, void* stream) {
  if (!xp || !wp || (split == 1 && !y) || (split > 1 && !partial)) return GIE_HIP_EINVAL;
  NhwcGeom g;
  int lds = 0;
  long long blocks = 0;
  if (int rc = nhwc_prepare(config, dtype, gg, split, &g, &lds, &blocks)) return rc;
  const uintptr_t es = dtype == GIE_HIP_FP32 ? 4 : 2;
  if (off_by(xp, 16) || off_by(wp, 16) || off_by(y, es) || off_by(bias, es) || off_by(partial, 4)) return GIE_HIP_EINVAL;
  const NhwcFn fn = dtype == GIE_HIP_FP16   ? nhwc_fn<NhHalf<Fp16>>(config)
                    : dtype == GIE_HIP_BF16 ? nhwc_fn<NhHalf<Bf16>>(config)
                                            : nhwc_fn32(config);
  if (int rc = set_lds_limit(reinterpret_cast<const void*>(fn), lds)) return rc;
  hipLaunchKernelGGL(fn, dim3(unsigned(blocks)), dim3(unsigned(kNhwcConfigs[config].threads)), size_t(lds),
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(xp), static_cast<const uint16_t*>(wp),
                     bias, y, partial, g);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GIE_HIP_OK : int(e);
}
