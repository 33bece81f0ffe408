// bf16 / f16 GEMM over one output tile per workgroup, for products whose 128 x 256 tiles leave compute units idle.
//
//   C[m, n] = sum_k A[m, k] * B[n, k]      both K-contiguous
//
// What bounds it.  64 x 4096 x 4096 takes 6 us of HBM time and 1 us of MFMAs; on 128 x 256 tiles it has 16 workgroups,
// each a serial chain of 64 K steps whose loads are one step ahead: 0.7 us a step.  The schedule is that of the packed
// pairs' tiles (tgm_gemm_mx_tile.h): WM x WN x WK waves of 32 FA x 32 FB, the WK groups taking every WK-th K step (their
// sums meet in LDS in group order); NBUF stages of WK steps in LDS or on their way, a wave waiting only for its share of
// the next stage; the next stage's fragments read while the current one's are multiplied, and the freed buffer's refill
// issued between the MFMAs.
//
// Measured against the 128 x 256-tile kernel that took these products before (bf16, us, K = 4096 unless noted):
//
//   17 x 1024: 43.6 -> 10.2    64 x 4096: 48.2 -> 12.2    128 x 8192: 50.9 -> 16.6    512 x 4096: 51.3 -> 24.0
//   1024 x 4096: 52.5 -> 34.8  2048 x 4096: 64.0 -> 62.5  700 x 2048 x 8192: 90 -> 37  333 x 520 x 512: 11.6 -> 5.6
//
// The 128 x 128 shape with four waves has four stages in flight; eight waves that split K have two and are slower
// (1024 x 4096: 34.8 against 40.2), eight waves of 64 x 32 read half as much again from LDS (36.9).
#pragma once

#include <type_traits>

#include "tgm_gemm_w_tile.h"

namespace tgm {

constexpr int kDtK = 64, kDtRow = 2 * kDtK;  // K step and its bytes per row

struct DenseTileArgs {
  const uint8_t *a, *b;
  void* c;
  int64_t ldc;
  unsigned lda, ldb;  // bytes between rows
  int M, N, K, cdt;
};

template <int FA, int FB, int WM, int WN, int WK, int NBUF>
struct DenseTile {
  static constexpr int kW = WM * WN, kThreads = 64 * kW * WK;
  static constexpr int kBM = 32 * FA * WM, kBN = 32 * FB * WN;
  static constexpr int kPA = kBM * kDtRow, kPB = kBN * kDtRow;  // panel bytes of one K step
  static constexpr int kStep = kPA + kPB, kStage = WK * kStep;
  static constexpr int kQA = kPA / 1024 / kW, kQB = kPB / 1024 / kW, kLoads = kQA + kQB;  // loads per wave and stage
  static constexpr int kEpi = (WK - 1) * kW * FA * FB * 4096 + kW * 32 * 36 * 4;
  static constexpr int kLds = NBUF * kStage > kEpi ? NBUF * kStage : kEpi;
  static constexpr int kByLds = kW * WK * (160 * 1024 / kLds) / 4, kByRegs = FA * FB == 1 ? 4 : 2;
  static constexpr int kOccupancy = kByLds < kByRegs ? kByLds : kByRegs;  // waves per SIMD
  static constexpr bool kFits = kLds <= 160 * 1024 && kLoads * (NBUF - 1) < 64 && kPA % (1024 * kW) == 0 &&
                                kPB % (1024 * kW) == 0 && NBUF >= 2;
};

template <int T16, int FA, int FB, int WM, int WN, int WK, int NBUF>
__global__ void __launch_bounds__(64 * WM * WN * WK)
__attribute__((amdgpu_waves_per_eu(DenseTile<FA, FB, WM, WN, WK, NBUF>::kOccupancy,
                                   DenseTile<FA, FB, WM, WN, WK, NBUF>::kOccupancy)))
gemm_dense_tile(DenseTileArgs p) {
  using T = DenseTile<FA, FB, WM, WN, WK, NBUF>;
  __shared__ __attribute__((aligned(16))) unsigned char lds[T::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / T::kW, w = wave % T::kW, wm = w / WN, wn = w % WN;
  const int tiles_m = (p.M + T::kBM - 1) / T::kBM, tiles_n = (p.N + T::kBN - 1) / T::kBN;
  int tm, tn;
  tile_of_ranges(blockIdx.x, p.K, tiles_m, tiles_n, 8, tm, tn);
  const int m0 = tm * T::kBM, n0 = tn * T::kBN;
  const int nsteps = p.K / kDtK, nstages = (nsteps + WK - 1) / WK;
  const i32x4v ra = buffer_rsrc(p.a, (unsigned)(p.M - 1) * p.lda + (unsigned)p.K * 2u);
  const i32x4v rb = buffer_rsrc(p.b, (unsigned)(p.N - 1) * p.ldb + (unsigned)p.K * 2u);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;

  // Load instruction i of a panel fills rows 8 i .. 8 i + 7: lane l writes slot l % 8 of row 8 i + l / 8, which
  // holds logical 16-byte column (l % 8) ^ ((row >> 1) & 7).  Rows past M or N read zeros (buffer bounds).
  unsigned voa[T::kQA], vob[T::kQB];
#pragma unroll
  for (int q = 0; q < T::kQA; ++q) {
    const int r = 8 * (w + T::kW * q) + (lane >> 3);
    voa[q] = (unsigned)(m0 + r) * p.lda + (unsigned)(((lane & 7) ^ ((r >> 1) & 7)) * 16 + wk * kDtRow);
  }
#pragma unroll
  for (int q = 0; q < T::kQB; ++q) {
    const int r = 8 * (w + T::kW * q) + (lane >> 3);
    vob[q] = (unsigned)(n0 + r) * p.ldb + (unsigned)(((lane & 7) ^ ((r >> 1) & 7)) * 16 + wk * kDtRow);
  }
  auto load_piece = [&](int st, int buf, int q) __attribute__((always_inline)) {
    const unsigned base = lds_base + (unsigned)(buf * T::kStage + wk * T::kStep);
    const int sc = st < nstages ? st : nstages - 1;  // past the end: the last stage again, into a free buffer
    const unsigned s0 = (unsigned)(sc * WK) * (unsigned)kDtRow;
    const bool inside = WK == 1 || sc * WK + wk < nsteps;  // a step past K loads zeros
    if (q < T::kQA)
      lds_dma16(ra, (unsigned)__builtin_amdgcn_readfirstlane((int)(base + (unsigned)(w + T::kW * q) * 1024u)),
                inside ? voa[q < T::kQA ? q : 0] + s0 : 0xFFFFFFF0u);
    else {
      const int i = q - T::kQA;
      lds_dma16(rb, (unsigned)__builtin_amdgcn_readfirstlane((int)(base + (unsigned)T::kPA + (unsigned)(w + T::kW * i) * 1024u)),
                inside ? vob[i >= 0 && i < T::kQB ? i : 0] + s0 : 0xFFFFFFF0u);
    }
  };

  const int half = lane >> 5, sw = (lane >> 1) & 7;  // (row >> 1) & 7 of every row this lane reads
  const int ar = (wm * FA * 32 + (lane & 31)) * kDtRow, br = (wn * FB * 32 + (lane & 31)) * kDtRow;
  struct Frags {
    u32x4 a[4][FA], b[4][FB];  // by MFMA: j takes K [16 j + 8 h, + 8) of the step for lane half h
  };
  auto read = [&](Frags& f, int buf) __attribute__((always_inline)) {
    const unsigned char* pa = lds + buf * T::kStage + wk * T::kStep;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = ((2 * j + half) ^ sw) * 16;
#pragma unroll
      for (int t = 0; t < FA; ++t) f.a[j][t] = *(const u32x4*)(pa + ar + col + t * 32 * kDtRow);
#pragma unroll
      for (int t = 0; t < FB; ++t) f.b[j][t] = *(const u32x4*)(pa + T::kPA + br + col + t * 32 * kDtRow);
    }
  };
  f32x16 acc[FA][FB];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) acc[i][j] = f32x16{};

#pragma unroll
  for (int s = 0; s < NBUF; ++s)
#pragma unroll
    for (int q = 0; q < T::kLoads; ++q) load_piece(s, s, q);
  wait_loads<(NBUF - 1) * T::kLoads>();
  lds_barrier();
  // Stage st, its fragments in f: wait for this wave's loads of the next stage; behind the barrier that stage is
  // complete and this stage's buffer free; the next fragments are read and the buffer's refill is issued between
  // the MFMAs.
  int cur = 0;
  auto stage = [&](const Frags& f, Frags& g, int st) __attribute__((always_inline)) {
    using V = typename std::conditional<T16 == TGM_F16, wt_f16x8, wt_bf16x8>::type;
    const int nxt = cur + 1 < NBUF ? cur + 1 : 0;
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // f is read: its buffer may be overwritten
    wait_loads<(NBUF - 2) * T::kLoads>();
    lds_barrier();
    read(g, nxt);
    __builtin_amdgcn_sched_barrier(0);
    constexpr int kMfmas = 4 * FA * FB;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j) {
          const int idx = (u * FA + i) * FB + j;
          const V va = __builtin_bit_cast(V, f.a[u][i]), vb = __builtin_bit_cast(V, f.b[u][j]);
          if constexpr (T16 == TGM_F16) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, vb, acc[i][j], 0, 0, 0);
          else acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, vb, acc[i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < T::kLoads; ++q)
            if (q * kMfmas / T::kLoads == idx) load_piece(st + NBUF, cur, q);
          __builtin_amdgcn_sched_barrier(0);
        }
    cur = nxt;
  };
  Frags f0, f1;
  read(f0, 0);
#pragma unroll 1
  for (int st = 0; st < nstages; st += 2) {
    stage(f0, f1, st);
    if (st + 1 < nstages) stage(f1, f0, st + 1);
  }
  wait_loads<0>();
  __syncthreads();  // the epilogue reuses the LDS

  float* parts = (float*)lds;
  if constexpr (WK > 1) {
    if (wk > 0) {
#pragma unroll
      for (int t = 0; t < FA * FB; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) parts[((((wk - 1) * T::kW + w) * FA * FB + t) * 16 + v) * 64 + lane] = acc[t / FB][t % FB][v];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int k = 1; k < WK; ++k)
#pragma unroll
      for (int t = 0; t < FA * FB; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t / FB][t % FB][v] += parts[((((k - 1) * T::kW + w) * FA * FB + t) * 16 + v) * 64 + lane];
  }
  float* ep = parts + (WK - 1) * T::kW * FA * FB * 1024 + w * 32 * 36;
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j)
      store_tile32(acc[i][j], ep, lane, m0 + (wm * FA + i) * 32, n0 + (wn * FB + j) * 32, p.M, p.N, p.c, p.cdt, p.ldc);
}

template <int T16, int FA, int FB, int WM, int WN, int WK, int NBUF>
int launch_dense_tile(const DenseTileArgs& p, hipStream_t s) {
  using T = DenseTile<FA, FB, WM, WN, WK, NBUF>;
  static_assert(T::kFits, "tile shape");
  const int64_t tiles = (int64_t)((p.M + T::kBM - 1) / T::kBM) * ((p.N + T::kBN - 1) / T::kBN);
  hipLaunchKernelGGL((gemm_dense_tile<T16, FA, FB, WM, WN, WK, NBUF>), dim3((unsigned)tiles), dim3(T::kThreads), 0, s, p);
  return launch_status("tgm_gemm_dense");
}

// The tile shape for a product, and the tile itself in *tile.  cus: compute units of the stream's device (0 if
// unknown).
int dense_tile_shape(int64_t m, int64_t n, int64_t k, int cus, TileChoice* tile = nullptr);
int launch_gemm_dense_tile(int shape, int dtype, const DenseTileArgs& p, hipStream_t s);

}  // namespace tgm
