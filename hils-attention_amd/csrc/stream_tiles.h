// Helper for kernels in which one operand side streams through LDS in 64-row tiles, stored row-major, PITCH bytes apart
// (D * 2 + 32: the 16-byte reads of 16 rows that a score product makes take 4 cycles, 8 at D * 2 + 16).
#pragma once
#include "common.h"

// Gradient product of one wavefront: acc[rt][dt] += T^T (16 features of dt x 64 streamed) * P[rt] (64 streamed x 16 owned),
// the features by the transposing LDS load: a 16-lane group addresses a
// 4 x 16 block, lane l row l/4 and columns 4(l%4).., and receives column l of it; with rows 4j.. of two neighbouring
// 16-row tiles that is the order in which the score accumulators hold p (lane: owned row = lane & 15, streamed rows
// 4*(lane>>4)+i of tile tt).  A lane's accumulators are features 16 dt + 4*(lane>>4)+i of its owned row or, with COLS, the
// product taken the other way round, feature 16 dt + (lane & 15) of the owned rows 4*(lane>>4)+i.
template <int D, int NT, int PITCH, bool COLS = false>
__device__ __forceinline__ void lzm_grad_product_rows(const unsigned char* rows, const float (&p)[NT][4][4],
                                                      f32x4_t (&acc)[NT][D / 16], int col, int j) {
  typedef short lz_s4 __attribute__((ext_vector_type(4)));
  typedef short lz_s8 __attribute__((ext_vector_type(8)));
  typedef unsigned lz_u4 __attribute__((ext_vector_type(4)));
  const unsigned char* t_addr = rows + (4 * j + (col >> 2)) * PITCH + (col & 3) * 8;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    bf16x8_t a[NT];
#pragma unroll
    for (int rt = 0; rt < NT; ++rt) {
      lz_u4 u;
      u.x = pack_bf2(p[rt][2 * h][0], p[rt][2 * h][1]);
      u.y = pack_bf2(p[rt][2 * h][2], p[rt][2 * h][3]);
      u.z = pack_bf2(p[rt][2 * h + 1][0], p[rt][2 * h + 1][1]);
      u.w = pack_bf2(p[rt][2 * h + 1][2], p[rt][2 * h + 1][3]);
      a[rt] = __builtin_bit_cast(bf16x8_t, u);
    }
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) {
      const unsigned char* p0 = t_addr + (2 * h * 16) * PITCH + dt * 32;
      const lz_s4 b0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lz_s4*)p0);
      const lz_s4 b1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) lz_s4*)(p0 + 16 * PITCH));
      const bf16x8_t b = __builtin_bit_cast(bf16x8_t, (lz_s8)__builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
        acc[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(COLS ? a[rt] : b, COLS ? b : a[rt], acc[rt][dt], 0, 0, 0);
    }
  }
}
