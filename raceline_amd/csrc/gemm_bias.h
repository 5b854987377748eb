// The bias product of the prefill GEMM for kernels whose waves read its operands from memory
// (gemm_mid.hip, gemm_few.hip); gemm4_kernel stages them in the LDS.
#pragma once

#include "q4_tile.h"

namespace rlq {

// C steps st0 .. of the bias product sum_g b[n][g] gsum[m][g] (see gemm4_kernel, whose steps
// and order these are) for MT row tiles of 32: bias_load requests the pieces of the wave's
// rows and its 32 features' scale quads, all at once, straight from memory; steps from st1
// on load zeros and add nothing. bias_mul adds the products to acc.
struct BiasSrc {
  __amdgpu_buffer_rsrc_t rgs, rsb;
  uint32_t svoff;
  int M, gs_stride, G4, m0, c32, h;
};

template <int SD, int MT, int C>
__device__ __forceinline__ void bias_load(const BiasSrc &b, u32x4 (&bv)[C], u32x4 (&ba)[C][MT], int st0, int st1) {
#pragma unroll
  for (int u = 0; u < C; ++u) {
    const int st = st0 + u, q = SD == 0 ? 2 * st + b.h : st;            // quad of groups 4q .. 4q+3
    bv[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                          b.rsb, st < st1 && q < b.G4 ? b.svoff + 256u * q : kFarOffset, 0, 0));
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = b.m0 + 32 * mt + b.c32;
      const uint32_t off = (uint32_t)(((size_t)m * b.gs_stride + 16 * st + 8 * b.h) * 2);
      ba[u][mt] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(b.rgs, st < st1 && m < b.M ? off : kFarOffset, 0, 0));
    }
  }
}

template <int SD, int MT, int C>
__device__ __forceinline__ void bias_mul(const u32x4 (&bv)[C], const u32x4 (&ba)[C][MT], int h, f32x16 (&acc)[MT]) {
#pragma unroll
  for (int u = 0; u < C; ++u) {
    u32x4 d;
    if constexpr (SD == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) d[e] = (bv[u][e] >> 16) * 0x10001u;       // (b, b): times hi and lo
    } else {
      const uint32_t b0 = (h ? bv[u][2] : bv[u][0]) >> 16, b1 = (h ? bv[u][3] : bv[u][1]) >> 16;
      d[0] = d[1] = b0 * 0x10001u;                                          // b of group 4q + 2h, four times
      d[2] = d[3] = b1 * 0x10001u;                                          // and of group 4q + 2h + 1
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if constexpr (SD == 0)
        acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, ba[u][mt]),
                                                        __builtin_bit_cast(half8, d), acc[mt], 0, 0, 0);
      else
        acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ba[u][mt]),
                                                         __builtin_bit_cast(bf16x8, d), acc[mt], 0, 0, 0);
    }
  }
}

}  // namespace rlq
