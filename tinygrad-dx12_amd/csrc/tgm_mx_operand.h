// FP4 / FP6 panels in LDS for the scaled MFMA (32x32x64): operand type codes, rows of one 128-element K step
// with their 16-byte columns permuted against bank conflicts, and one lane's 32 codes of a row.
#pragma once

#include "tgm_mfma_common.h"

namespace tgm {

constexpr int kMxK = 128;  // K step

// v_mfma_scale_f32_32x32x64_f8f6f4 operand type codes (cbsz / blgp) of the FP6 / FP4 formats
constexpr int kOpE2M3 = 2, kOpE3M2 = 3, kOpE2M1 = 4;

template <int T>
struct F8F6F4 {
  static constexpr int bits = T <= kOpE3M2 ? 6 : 4;
  static constexpr int RB = 128 * bits / 8;  // bytes per row and 128-element step
  static constexpr int C = RB / 16;          // 16-byte columns per row and step
  static constexpr int L = 4 * bits;         // bytes of one lane's 32 values
};

template <int C>
__device__ __forceinline__ int col_phys(int r, int c) {
  if constexpr (C == 4) return c ^ ((r >> 2) & 3);
  else return (c + ((r >> 3) & 1)) % 6;
}
template <int C>
__device__ __forceinline__ int col_logical(int r, int pc) {
  if constexpr (C == 4) return pc ^ ((r >> 2) & 3);
  else return (pc + 6 - ((r >> 3) & 1)) % 6;
}

// One lane's 32 values of row r (panel at ``panel``) for block kb (0..3) of a step.
template <int T>
__device__ __forceinline__ i32x8 read_block(const unsigned char* panel, int r, int kb) {
  using O = F8F6F4<T>;
  const unsigned char* row = panel + r * O::RB;
  i32x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
  if constexpr (O::bits == 4) {
    const u32x4 q = *(const u32x4*)(row + 16 * col_phys<O::C>(r, kb));
    v[0] = (int)q[0]; v[1] = (int)q[1]; v[2] = (int)q[2]; v[3] = (int)q[3];
  } else {  // 24 bytes at 24 kb: three 8-byte pieces, each inside one 16-byte column
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int b = 24 * kb + 8 * i;
      const u32x2 q = *(const u32x2*)(row + 16 * col_phys<O::C>(r, b >> 4) + (b & 15));
      v[2 * i] = (int)q[0];
      v[2 * i + 1] = (int)q[1];
    }
  }
  return v;
}

}  // namespace tgm
