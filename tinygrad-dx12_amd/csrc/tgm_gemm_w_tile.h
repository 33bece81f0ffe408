// Packed-weight GEMM over one output tile per workgroup, with the tile, the split of K inside the
// workgroup and the depth of the load pipeline chosen per product (tgm_gemm_w for products whose
// 128 x 256 tiles would leave compute units idle, and every INT4 / UINT4 product).
//
//   C[m, n] = sum_k A[m, k] * deq(W)[n, k]
//
// What bounds it.  With 17 to a few hundred activation rows the products are short: at 64 x 14336 x
// 4096 the weights take 5 us of HBM time and the MFMAs 3 us.  One 128 x 256 tile per workgroup leaves
// 56 workgroups, each a serial chain of 32 K steps whose loads are one step ahead.  Here
//
//  * a tile is 32 FA activation rows x 32 WN weight rows, and the waves of a workgroup are WN x WK:
//    each wave owns 32 weight rows and every WK-th 128-wide K step, so short products still put waves
//    on every SIMD; the WK partial tiles meet in LDS in wave order (deterministic);
//  * every weight code is decoded by one wave only and used for FA MFMAs;
//  * NBUF stages of WK K steps are in LDS or on their way there (buffer_load ... lds); a wave waits
//    only for its share of the stage it computes next (vmcnt counts down in issue order), so NBUF - 1
//    stages of loads cover the memory latency.  One barrier per stage;
//  * a stage's load instructions are issued one after each MFMA: in one burst behind the barrier they
//    hold up the MFMAs behind them by the time the L1 takes for the panel (FP4 512 x 4096 x 14336 on
//    128 x 128 tiles: 94 us in a burst, 80 us spread).
//
// Measured against the 128 x 256-tile kernels that took these products before (us, K = 4096 unless noted):
//
//   FP4   64 x 14336: 42 -> 15      17 x 4096: 39 -> 7.2     512 x 4096: 43 -> 21     512 x 4096 x 14336: 134 -> 66
//   E2M3  64 x 14336: 51 -> 17      200 x 3000 x 2304: 33 -> 13
//   INT4 g128  512 x 6144: 74 -> 39     64 x 14336: 68 -> 18     4096 x 4096: 160 -> 139     2048 x 14336: 301 -> 256
//   INT4 g32   512 x 4096: 96 -> 36     4096 x 4096: 195 -> 173
//
// The INT4 products are bound by VALU work beside the MFMAs (12 instructions per 8 codes, and 16 FMAs per
// MFMA tile and scale group) and by the clock that both together leave: at 4096 x 4096 the MFMA pipe is busy
// 45 % (profiles/one_tile_products.txt) at about 2.06 GHz; the 64 x 64-per-wave kernel before, which decoded every
// code twice, 34 % at 2.38 GHz.  At 512 x 6144 it is 22 % in one and a half rounds of 64 x 128 tiles.
//
// Operand layout in LDS, per K step: the A panel as rows of 256 bytes with 16-byte columns
// XOR-swizzled by row % 16; the W panel as rows of 64 bytes (FP4, INT4; 16-byte chunks swizzled by
// (row / 4) % 4) or 96 bytes (FP6, dense).  The scales of a wave's 32 rows are one dword per row and
// step (E8M0) or one zero-extended value per row and group (INT4), loaded straight to LDS as well: an
// ordinary load would make the compiler wait for every load in flight.
//
// K order: for FP4 / FP6, lane half h owns K [64 h, 64 h + 64) of a step and MFMA j (32x32x16) takes
// [64 h + 8 j, + 8) of it, so a lane's codes are contiguous.  INT4 takes [16 j + 8 h, + 8): no MFMA spans
// two groups of 32 or 64, and every group size (and none) sums K in ascending order, so that a rounding
// does not depend on how a weight's scales are grouped.  (Groups of 128 in the contiguous order, whose
// codes are two LDS reads instead of four, are 3 % faster, 134 against 139 us at 4096 x 4096 x 4096, and change
// the last place of the sums, which the attention of a two-layer decoder prompt grows to 2.4e-3 of its logits.)
// INT4 codes become exact f16 values, the MFMAs of a group sum in fp32 and the sum times the group's fp32
// scale is added to the accumulator.
#pragma once

#include "tgm_mfma_common.h"

namespace tgm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 wt_bf16x8;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 wt_bf16x2;
typedef __attribute__((__vector_size__(32 * sizeof(__bf16)))) __bf16 wt_bf16x32;
typedef __attribute__((__vector_size__(6 * sizeof(int)))) int wt_i32x6;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 wt_f16x8;
typedef _Float16 wt_half2 __attribute__((ext_vector_type(2)));

// Weight kinds: an FP4 / FP6 format (scales E8M0 per 32, or none), or 4-bit integers with scales per
// 32, 64 or 128 K-elements or none (kKindI4 + group, + 1 when the scales are fp32 and not 16-bit).
constexpr int kKindI4 = 1000;
constexpr bool kind_is_i4(int kind) { return kind >= kKindI4; }
constexpr int kind_group(int kind) { return (kind - kKindI4) & ~1; }
constexpr int kind_scale_bytes(int kind) { return kind & 1 ? 4 : 2; }

constexpr int kWtK = 128;  // K step

struct WTileArgs {
  const uint8_t* a;
  const uint8_t* w;
  const uint8_t* scales;  // E8M0 bytes [N, K / 32] or INT4 group scales [N, K / G] of dtype sdt; null = unscaled
  void* c;
  int64_t ldc;
  unsigned lda_bytes;
  int M, N, K, cdt, sdt, is_signed;
  int steps_per_split;  // > 0: blockIdx.y takes that many K steps and writes its fp32 product to part [splits][M][N]
  float* part;
  int swiglu;  // rows of W interleave gate and up: C has N / 2 columns, silu(gate) * up
};

// 16-bit values to LDS, one zero-extended dword per lane.
__device__ __forceinline__ void lds_dma2(i32x4v rsrc, unsigned lds_addr, unsigned voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_ushort %1, %2, 0 offen lds" : : "s"(lds_addr), "v"(voff), "s"(rsrc) : "memory");
}

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// Workgroup barrier that orders LDS accesses only: the loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Eight nibbles as exact f16 values, 12 instructions: per byte a v_perm puts the byte in both halves, one
// v_bitop3 keeps the low nibble of one and the high nibble of the other under the f16 pattern 0x6400
// (1024 + n and 1024 + 16 n, with the sign bits flipped for int4) and one packed f16 FMA removes the
// offset and the 16 (exact: every value on the way is an integer below 2048 / 16).
struct NibbleConsts {
  unsigned pattern;   // 0x64006400 ^ sign flips
  wt_half2 offset;    // {-1024, -64}, or {-1032, -72} for signed codes
};
__device__ __forceinline__ wt_f16x8 decode_nibbles(unsigned v, const NibbleConsts& c) {
  const wt_half2 mul = {(_Float16)1.0f, (_Float16)0.0625f};
  wt_half2 p[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const unsigned t = (__builtin_amdgcn_perm(v, v, 0x0C000C00u | (unsigned)(b | (b << 16))) & 0x00F0000Fu) ^ c.pattern;
    p[b] = __builtin_elementwise_fma(__builtin_bit_cast(wt_half2, t), mul, c.offset);
  }
  return wt_f16x8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// MX block blk (0 or 1) of a lane's 64 codes to the operands of MFMAs 4 blk .. 4 blk + 3, times 2^(e - 127).
template <int KIND>
__device__ __forceinline__ void decode_mx_block(const unsigned* raw, int blk, unsigned e8, wt_bf16x8 out[4]) {
  const float s = __builtin_bit_cast(float, e8 << 23);
  if constexpr (KIND == TGM_FMT_FP4_E2M1) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const unsigned v = raw[4 * blk + d];
      const wt_bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, s, 0);
      const wt_bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, s, 1);
      const wt_bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, s, 2);
      const wt_bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, s, 3);
      out[d] = wt_bf16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
  } else {
    wt_i32x6 v;
#pragma unroll
    for (int q = 0; q < 6; ++q) v[q] = (int)raw[6 * blk + q];
    wt_bf16x32 d;
    if constexpr (KIND == TGM_FMT_FP6_E2M3) d = __builtin_amdgcn_cvt_scalef32_pk32_bf16_fp6(v, s);
    else d = __builtin_amdgcn_cvt_scalef32_pk32_bf16_bf6(v, s);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      out[j] = wt_bf16x8{d[8 * j], d[8 * j + 1], d[8 * j + 2], d[8 * j + 3], d[8 * j + 4], d[8 * j + 5], d[8 * j + 6],
                         d[8 * j + 7]};
  }
}

template <int KIND, int FA, int WN, int WK, int NBUF>
struct WTile {
  static constexpr bool kI4 = kind_is_i4(KIND);
  static constexpr int kG = kI4 ? kind_group(KIND) : 32;      // scale group (0: unscaled INT4)
  static constexpr int kWaves = WN * WK, kThreads = 64 * kWaves;
  static constexpr int kBM = 32 * FA, kBN = 32 * WN;
  static constexpr int kRow = kI4 || KIND == TGM_FMT_FP4_E2M1 ? 64 : 96;  // packed bytes per W row and step
  static constexpr int kA = kBM * kWtK * 2, kW = kBN * kRow;  // panel bytes per step
  static constexpr int kNS = kI4 ? (kG ? kWtK / kG : 0) : 1;  // scale dwords per row and step
  static constexpr int kS = kNS * 256;                        // scale bytes per wave and step (64 lanes of a dword)
  static constexpr int kStep = kA + kW + WN * kS;             // LDS bytes per K step
  static constexpr int kStage = WK * kStep;
  static constexpr int kLoadsA = 8 * FA / WN, kLoadsW = kRow / 32;  // load instructions per wave and stage
  static constexpr int kLoads = kLoadsA + kLoadsW + kNS;
  // Pieces of a stage's loads by substep: issued from the substep that frees the buffer on, spread over a
  // stage's time where a further stage in flight covers their latency (NBUF > 2), over half of it otherwise.
  static constexpr int kPD = FA >= 4 ? 1 : 2;
  static constexpr int kSpread = NBUF > 2 ? 8 : 4;
  static constexpr int slot(int j) { return (j + kPD) % 8; }  // substep 8 - kPD comes first
  static constexpr int first_piece(int j) { return slot(j) < kSpread ? slot(j) * kLoads / kSpread : kLoads; }
  static constexpr int end_piece(int j) { return slot(j) < kSpread ? (slot(j) + 1) * kLoads / kSpread : kLoads; }
  static constexpr int kEpi = (WK - 1) * WN * FA * 4096 + WN * 32 * 36 * 4;  // partial tiles, store blocks
  static constexpr int kLds = NBUF * kStage > kEpi ? NBUF * kStage : kEpi;
  // waves per SIMD that fit by LDS; told to the compiler, which otherwise halves the registers into VGPRs
  // and AGPRs and copies partial sums between them
  static constexpr int kOccupancy = kWaves / 4 * (160 * 1024 / kLds < 1 ? 1 : 160 * 1024 / kLds);
  static constexpr bool kFits = 8 * FA % WN == 0 && kLoads * (NBUF - 1) < 64 && kLds <= 160 * 1024;
};

template <int KIND, int FA, int WN, int WK, int NBUF>
__global__ void __launch_bounds__(64 * WN * WK) 
__attribute__((amdgpu_waves_per_eu(WTile<KIND, FA, WN, WK, NBUF>::kOccupancy, WTile<KIND, FA, WN, WK, NBUF>::kOccupancy)))
gemm_w_tile(WTileArgs p) {
  using T = WTile<KIND, FA, WN, WK, NBUF>;
  constexpr bool I4 = T::kI4;
  constexpr int G = T::kG;
  __shared__ __attribute__((aligned(16))) unsigned char lds[T::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int tiles_m = (p.M + T::kBM - 1) / T::kBM, tiles_n = (p.N + T::kBN - 1) / T::kBN;
  int tm, tn;
  tile_of_ranges(blockIdx.x, p.K, tiles_m, tiles_n, 8, tm, tn);
  const int m0 = tm * T::kBM, n0 = tn * T::kBN;
  // split K (WK == 1 shapes only): steps s_begin .. of this workgroup
  const int s_begin = WK == 1 && p.part ? (int)blockIdx.y * p.steps_per_split : 0;
  const int nsteps = WK == 1 && p.part ? min(p.steps_per_split, p.K / kWtK - s_begin) : p.K / kWtK;
  const int nstages = (nsteps + WK - 1) / WK;
  const unsigned kbw = (unsigned)p.K / 8u * (T::kRow == 64 ? 4u : 6u);  // packed bytes per W row
  const i32x4v ra = buffer_rsrc(p.a, (unsigned)(p.M - 1) * p.lda_bytes + (unsigned)p.K * 2u);
  const i32x4v rw = buffer_rsrc(p.w, (unsigned)p.N * kbw);
  constexpr unsigned ssize = (unsigned)kind_scale_bytes(KIND);                   // INT4 scale bytes
  const unsigned srow = I4 ? (G ? (unsigned)(p.K / (G ? G : 1)) * ssize : 0u) : (unsigned)p.K / 32u;  // scale bytes per W row
  const i32x4v rs = buffer_rsrc(p.scales, p.scales ? (unsigned)p.N * srow : 0u);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;

  // Loads: the WN waves of K group wk fill the panels of its step.  A instruction i = wn + WN q covers
  // rows 4 i .. 4 i + 3 (lane l: row 4 i + l / 16, logical 16-byte column (l % 16) ^ (row % 16)); W
  // instruction i = wn + WN q fills bytes [1024 i, + 1024) of the W panel.
  unsigned voa[T::kLoadsA], vow[T::kLoadsW];
#pragma unroll
  for (int q = 0; q < T::kLoadsA; ++q) {
    const int row = 4 * (wn + WN * q) + (lane >> 4);
    voa[q] = (unsigned)(m0 + row) * p.lda_bytes + (unsigned)(((lane & 15) ^ (row & 15)) * 16 + wk * kWtK * 2);
  }
#pragma unroll
  for (int q = 0; q < T::kLoadsW; ++q) {
    const int i = wn + WN * q;
    if constexpr (T::kRow == 64) {
      const int row = 16 * i + (lane >> 2);
      vow[q] = (unsigned)(n0 + row) * kbw + (unsigned)(((lane & 3) ^ ((row >> 2) & 3)) * 16 + wk * T::kRow);
    } else {
      const int f = 1024 * i + 16 * lane;
      vow[q] = (unsigned)(n0 + f / 96) * kbw + (unsigned)(f % 96 + wk * T::kRow);
    }
  }
  const unsigned vos = (unsigned)(n0 + 32 * wn + (lane & 31)) * srow +
                       (I4 ? (unsigned)(wk * T::kNS) * ssize : (unsigned)(wk * 4));
  // Load piece q (< kLoads) of stage st into buffer buf: the A instructions, then W's, then the scales.
  auto load_piece = [&](int st, int buf, int q) __attribute__((always_inline)) {
    st = st < nstages ? st : nstages - 1;  // past the end: the last stage again, so that every wave's count stays
    const unsigned base = lds_base + (unsigned)(buf * T::kStage + wk * T::kStep);
    const unsigned s0 = (unsigned)(s_begin + st * WK);
    // a step past K loads zeros for A and the scales (an offset past the operand), so that its products
    // add nothing: the next row's scale could be infinite or NaN
    const bool inside = WK == 1 || (int)s0 + wk < nsteps;
    if (q < T::kLoadsA) {
      const unsigned dst = base + (unsigned)(wn + WN * q) * 1024u;
      lds_dma16(ra, dst, inside ? voa[q < T::kLoadsA ? q : 0] + s0 * (kWtK * 2) : 0xFFFFFFF0u);
    } else if (q < T::kLoadsA + T::kLoadsW) {
      const int i = q - T::kLoadsA;
      lds_dma16(rw, base + (unsigned)T::kA + (unsigned)(wn + WN * i) * 1024u,
                vow[i >= 0 && i < T::kLoadsW ? i : 0] + s0 * (unsigned)T::kRow);
    } else {
      const unsigned g = (unsigned)(q - T::kLoadsA - T::kLoadsW);
      const unsigned dst = base + (unsigned)(T::kA + T::kW + wn * T::kS) + g * 256u;
      const unsigned off = inside ? vos + (I4 ? (s0 * T::kNS + g) * ssize : s0 * 4u) : 0xFFFFFFF0u;
      if constexpr (!I4 || ssize == 4) lds_dma4(rs, dst, off);
      else lds_dma2(rs, dst, off);
    }
  };

  const int half = lane >> 5, l32 = lane & 31;
  NibbleConsts nib;
  nib.pattern = p.is_signed ? 0x64006400u ^ 0x00800008u : 0x64006400u;
  nib.offset = p.is_signed ? wt_half2{(_Float16)-1032.0f, (_Float16)-72.0f} : wt_half2{(_Float16)-1024.0f, (_Float16)-64.0f};
  const unsigned sshift = p.sdt == TGM_BF16 ? 16u : 0u;
  constexpr int JPG = I4 && G ? G / 16 : 8;              // MFMAs per scale group
  constexpr int RAW = T::kRow / 8;                       // dwords of a lane's 64 codes
  const int w_row = 32 * wn + l32;
  f32x16 acc[FA];
  constexpr int PD = T::kPD, SL = 2 * PD;       // A is read PD substeps ahead (4 MFMAs of time)
  u32x4 fa[SL][FA];                                       // A fragments of substeps j (slot j % SL)
  unsigned raw[RAW], rawn[RAW];                           // packed codes of this step and the next
  unsigned sbits[T::kNS ? T::kNS : 1], sbitsn[T::kNS ? T::kNS : 1];  // scale words of this step and the next
  wt_bf16x8 wd[I4 ? 1 : 8];                               // decoded MX weights
  wt_f16x8 wi[2];                                         // decoded nibbles of substeps j (slot j % 2)
#pragma unroll
  for (int t = 0; t < FA; ++t) {
    acc[t] = f32x16{};
  }
  auto read_a = [&](int buf, int j, u32x4 (&dst)[FA]) __attribute__((always_inline)) {
    const int col = (I4 ? 2 * j + half : 8 * half + j) ^ (l32 & 15);
#pragma unroll
    for (int t = 0; t < FA; ++t)
      dst[t] = *(const u32x4*)(lds + buf * T::kStage + wk * T::kStep + (32 * t + l32) * 256 + col * 16);
  };
  auto read_w = [&](int buf, unsigned (&r)[RAW], unsigned (&sb)[T::kNS ? T::kNS : 1]) __attribute__((always_inline)) {
    const unsigned char* pw = lds + buf * T::kStage + wk * T::kStep + T::kA;
    if constexpr (I4) {  // dword 2 j + h of the row
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const unsigned* c = (const unsigned*)(pw + w_row * 64 + ((q ^ ((w_row >> 2) & 3)) * 16) + 4 * half);
        r[2 * q] = c[0];
        r[2 * q + 1] = c[2];
      }
    } else {
#pragma unroll
      for (int q = 0; q < RAW / 4; ++q) {
        const u32x4 v = T::kRow == 96 ? *(const u32x4*)(pw + w_row * 96 + 48 * half + 16 * q)
                                      : *(const u32x4*)(pw + w_row * 64 + (((2 * half + q) ^ ((w_row >> 2) & 3)) * 16));
#pragma unroll
        for (int e = 0; e < 4; ++e) r[4 * q + e] = v[e];
      }
    }
    {
      const unsigned* ps = (const unsigned*)(pw + T::kW + wn * T::kS) + l32;
#pragma unroll
      for (int g = 0; g < T::kNS; ++g) sb[g] = ps[64 * g];
    }
  };
  auto mx_block = [&](const unsigned (&r)[RAW], unsigned sb, int blk) __attribute__((always_inline)) {
    if constexpr (!I4) {
      const unsigned e8 = p.scales ? (sb >> (16 * half + 8 * blk)) & 0xFFu : 127u;  // block 2 h + blk
      decode_mx_block<KIND>(r, blk, e8, wd + 4 * blk);
    }
  };

  // One stage from buffer cur.  On entry fa holds A of substeps 0 and 1, raw and sbits the stage's weights,
  // and substep 0's weights are decoded.  Substep j reads A of j + 2 and decodes ahead; before substep 6,
  // when every LDS read of the stage is done, the wave waits for its share of the next stage, the barrier
  // publishes it and frees this buffer, and substeps 6 and 7 cover the refill's issue, the next stage's
  // first reads and its first decode.
  auto stage = [&](int st, int prv, int cur, int nxt) __attribute__((always_inline)) {
    f32x16 part[FA];  // the sums of the current scale group
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      if (j == 8 - PD) {
        wait_loads<(NBUF - 2) * T::kLoads>();
        lds_barrier();
        read_w(nxt, rawn, sbitsn);
        read_a(nxt, 0, fa[0]);

      } else if (j > 8 - PD) {
        read_a(nxt, j + PD - 8, fa[j + PD - 8]);
      } else {
        read_a(cur, j + PD, fa[(j + PD) % SL]);
      }
      // this substep's share of the loads, one after each MFMA: stage st + NBUF into this buffer from substep
      // 8 - PD on, the rest of stage st + NBUF - 1 into the previous stage's buffer before
      auto pieces = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < T::kLoads; ++q)
          if (q >= T::first_piece(j) && q < T::end_piece(j) && (q - T::first_piece(j)) % FA == t) {
            __builtin_amdgcn_sched_barrier(0);
            if (j >= 8 - PD) load_piece(st + NBUF, cur, q);
            else load_piece(st + NBUF - 1, prv, q);
            __builtin_amdgcn_sched_barrier(0);
          }
      };
      if constexpr (I4) {
        if (j < 7) wi[(j + 1) & 1] = decode_nibbles(raw[j + 1], nib);
#pragma unroll
        for (int t = 0; t < FA; ++t) {
          const wt_f16x8 a = __builtin_bit_cast(wt_f16x8, fa[j % SL][t]);
          if constexpr (G == 0) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, wi[j & 1], acc[t], 0, 0, 0);
          else part[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, wi[j & 1], j % JPG ? part[t] : f32x16{}, 0, 0, 0);
          pieces(t);
        }
        if (j == 7) wi[0] = decode_nibbles(rawn[0], nib);
        if (G != 0 && j % JPG == JPG - 1) {
          const unsigned bits = sbits[j / JPG];
          const float sv = ssize == 2 && p.sdt == TGM_F16 ? (float)__builtin_bit_cast(_Float16, (unsigned short)bits)
                                                          : __builtin_bit_cast(float, bits << sshift);
#pragma unroll
          for (int t = 0; t < FA; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[t][v] += part[t][v] * sv;
          // pins these sums here: left to itself the compiler collects every group's at the stage's end,
          // and with them every group's 16 FA partial sums (G = 32: 512 registers)
#pragma unroll
          for (int t = 0; t < FA; ++t) asm volatile("" : "+v"(acc[t]));
        }
      } else {
        if (j == 2) mx_block(raw, sbits[0], 1);
#pragma unroll
        for (int t = 0; t < FA; ++t) {
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(wt_bf16x8, fa[j % SL][t]), wd[j], acc[t], 0, 0, 0);
          pieces(t);
        }
        if (j == 7) mx_block(rawn, sbitsn[0], 0);
      }
    }
#pragma unroll
    for (int i = 0; i < RAW; ++i) raw[i] = rawn[i];
#pragma unroll
    for (int g = 0; g < T::kNS; ++g) {
      sbits[g] = sbitsn[g];
    }
  };

#pragma unroll
  for (int s = 0; s < NBUF; ++s)
#pragma unroll
    for (int q = 0; q < T::kLoads; ++q)
      if (s < NBUF - 1 || q < T::first_piece(0)) load_piece(s, s, q);
  wait_loads<(NBUF - 2) * T::kLoads + T::first_piece(0)>();
  lds_barrier();
  read_w(0, raw, sbits);
#pragma unroll
  for (int j = 0; j < PD; ++j) read_a(0, j, fa[j]);
  if constexpr (I4) wi[0] = decode_nibbles(raw[0], nib);
  else mx_block(raw, sbits[0], 0);
  int prv = NBUF - 1, cur = 0;
#pragma unroll 1
  for (int st = 0; st < nstages; ++st) {
    const int nxt = cur + 1 < NBUF ? cur + 1 : 0;
    stage(st, prv, cur, nxt);
    prv = cur;
    cur = nxt;
  }
  wait_loads<0>();
  __syncthreads();  // the epilogue reuses the LDS

  float* parts = (float*)lds;
  if constexpr (WK > 1) {
    if (wk > 0) {
#pragma unroll
      for (int t = 0; t < FA; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) parts[((((wk - 1) * WN + wn) * FA + t) * 16 + v) * 64 + lane] = acc[t][v];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int k = 1; k < WK; ++k)
#pragma unroll
      for (int t = 0; t < FA; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] += parts[((((k - 1) * WN + wn) * FA + t) * 16 + v) * 64 + lane];
  }
  float* ep = parts + (WK - 1) * WN * FA * 1024 + wn * 32 * 36;
#pragma unroll
  for (int t = 0; t < FA; ++t) {
    if (WK == 1 && p.part)
      store_tile32(acc[t], ep, lane, m0 + 32 * t, n0 + 32 * wn, p.M, p.N, p.part + (int64_t)blockIdx.y * p.M * p.N, TGM_F32,
                   p.N);
    else if (!I4 && p.swiglu)
      store_tile32_swiglu(acc[t], ep, lane, m0 + 32 * t, n0 + 32 * wn, p.M, p.N, p.c, p.cdt, p.ldc);
    else store_tile32(acc[t], ep, lane, m0 + 32 * t, n0 + 32 * wn, p.M, p.N, p.c, p.cdt, p.ldc);
  }
}

template <int KIND, int FA, int WN, int WK, int NBUF>
int launch_w_tile(const WTileArgs& p, int splits, hipStream_t stream) {
  using T = WTile<KIND, FA, WN, WK, NBUF>;
  static_assert(T::kFits, "tile shape");
  const int64_t tiles = (int64_t)((p.M + T::kBM - 1) / T::kBM) * ((p.N + T::kBN - 1) / T::kBN);
  hipLaunchKernelGGL((gemm_w_tile<KIND, FA, WN, WK, NBUF>), dim3((unsigned)tiles, (unsigned)splits), dim3(T::kThreads), 0,
                     stream, p);
  return launch_status("tgm_gemm_w");
}

// The choice of tile.  A shape's time is that of the rounds of workgroups it takes: `lo` us for a first
// round of few workgroups and `hi` for one on every compute unit (measured at K = 4096), and lo2 .. hi2 for
// two (less than twice where two workgroups fit a compute unit's LDS).  `fixed` is the share of that time
// that does not grow with K (launch, prologue, epilogue), where shapes that compete differ in it; the others
// leave it 0, and only their ratios count.  The smallest estimate wins, so a product takes the smallest tile
// that still gives every compute unit one workgroup, and larger tiles, which read less per MFMA, as it grows.
// Shapes that split K over wk waves want two K steps for each; shorter products go to the others.
struct TileCost {
  int bm, bn, wk;
  float lo, hi, lo2, hi2, fixed;
};
inline float tile_estimate(const TileCost& t, int64_t m, int64_t n, int64_t k, int64_t cus) {
  const int64_t w = ((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
  const int64_t pairs = w / (2 * cus), rest = w - pairs * 2 * cus;
  const float f = (float)(rest % cus ? rest % cus : cus) / (float)cus;
  const float tail = rest == 0 ? 0.f : rest <= cus ? t.lo + (t.hi - t.lo) * f : t.lo2 + (t.hi2 - t.lo2) * f;
  return ((float)pairs * t.hi2 + tail) * (t.fixed + (1.f - t.fixed) * (float)k / 4096.f);
}
template <int COUNT>
int cheapest_tile(const TileCost (&table)[COUNT], int64_t m, int64_t n, int64_t k, int cus) {
  int best = -1;
  float least = 0.f;
  for (int i = 0; i < COUNT; ++i) {
    if (table[i].wk > 1 && k / kWtK < 2 * table[i].wk) continue;
    const float e = tile_estimate(table[i], m, n, k, cus > 0 ? cus : 256);
    if (best < 0 || e < least) {
      best = i;
      least = e;
    }
  }
  return best;
}

// What an entry point launches for a product (the tgm_*_tile queries): rows and columns of C per workgroup,
// wave groups that share its K steps, and the kind of kernel.
constexpr int kOneTile = 0, kLargeTile = 1, kPersistent = 2;
struct TileChoice {
  int rows, cols, k_groups, kernel;
};
inline int tell_tile(const TileChoice& t, int64_t* tile) {
  tile[0] = t.rows;
  tile[1] = t.cols;
  tile[2] = t.k_groups;
  tile[3] = t.kernel;
  return TGM_OK;
}

// One-tile products by format; tgm_gemm_w_tile_mx.hip and tgm_gemm_w_tile_i4.hip.  cus: compute units of
// the stream's device (0 if unknown).
int launch_gemm_w_tile_mx(const WTileArgs& p, int fmt, int cus, hipStream_t stream);
int launch_gemm_w_tile_i4(const WTileArgs& p, int64_t block_size, int splits, int cus, hipStream_t stream);
TileChoice w_tile_mx(int fmt, int64_t m, int64_t n, int64_t k, int cus);
TileChoice w_tile_i4(int64_t group, int64_t m, int64_t n, int64_t k, int cus);

}  // namespace tgm
