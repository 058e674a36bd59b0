// Output stage shared by the kernels that multiply pixels (MFMA rows) x filters (columns) in 32x32 blocks (conv_gather,
// conv_nhwc): bias + ReLU + one rounding into an LDS tile [filter][pixel], whole rows of y out of it. Private to
// csrc/kernels.
#pragma once

#include "device_common.h"

namespace gie_hip {

// The workgroup's TO x TP tile (filters o0 .., output pixels n0 .. of the flat batch * OHW axis). A lane of wave (wo, wp)
// holds, for 32x32 block (i, j), pixels 8q + 4 * (lane / 32) + 0..3 of column lane % 32. `lds`: TO * (TP * 2 + 16) bytes
// no wave still reads (the caller has met a barrier). Rows leave as 16-byte stores at any 2-byte alignment; only eight
// pixels that straddle two images go element by element.
template <typename E, int TO, int TP, int WO, int WP, int FP, int FO>
__device__ __forceinline__ void tile_to_y(const f32x16 (&acc)[FP][FO], unsigned char* lds, const uint16_t* __restrict__ bias,
                                          uint16_t* __restrict__ y, int tid, int o0, int n0, int O, int OHW, int N,
                                          int relu) {
  constexpr int NT = WO * WP * 64, WTO = TO / WO, WTP = TP / WP, YROW = TP * 2 + 16;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wp = wave / WO, wo = wave % WO, fr = lane & 31, fc = lane >> 5;
#pragma unroll
  for (int j = 0; j < FO; ++j) {
    const int oc = wo * WTO + j * 32 + fr;
    const float bv = bias != nullptr && o0 + oc < O ? E::to_f32(bias[o0 + oc]) : 0.0f;
#pragma unroll
    for (int i = 0; i < FP; ++i) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[i][j][4 * q + e] + bv;
          if (relu) v[e] = fmaxf(v[e], 0.0f);
        }
        const int px = wp * WTP + i * 32 + 8 * q + 4 * fc;  // four consecutive pixels
        *reinterpret_cast<u32x2*>(lds + oc * YROW + px * 2) = u32x2{E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
      }
    }
  }
  __syncthreads();
  constexpr int CK = TP / 8, RPP = NT / CK, NP = TO / RPP;  // 16-byte chunks per row, rows per pass, passes
  static_assert(NT % CK == 0 && NP * RPP == TO, "a thread keeps its chunk column");
  const int ck = tid % CK, r0 = tid / CK;
  const int nn = n0 + ck * 8, b0 = nn / OHW, p0 = nn - b0 * OHW;
  const bool whole = nn + 8 <= N && p0 + 8 <= OHW;  // the eight pixels lie in one image
  uint16_t* const y0 = y + static_cast<long long>(b0) * O * OHW + p0;
  if (whole) {
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int r = r0 + q * RPP;
      const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * YROW + ck * 16);
      if (o0 + r < O) __builtin_memcpy(y0 + static_cast<long long>(o0 + r) * OHW, &v, 16);
    }
    return;
  }
  for (int r = r0; r < TO && o0 + r < O; r += RPP) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * YROW + ck * 16);
    uint16_t* d = y0 + static_cast<long long>(o0 + r) * OHW;
    int pp = p0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (nn + q < N) *d = uint16_t(v[q >> 1] >> (16 * (q & 1)));
      ++d;
      if (++pp == OHW) {  // on to the same filter of the next image
        pp = 0;
        d += static_cast<long long>(O - 1) * OHW;
      }
    }
  }
}

}  // namespace gie_hip
