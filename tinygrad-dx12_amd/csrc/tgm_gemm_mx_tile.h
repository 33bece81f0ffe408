// Scaled-MFMA GEMM over an FP4 / FP6 operand pair, one output tile per workgroup, for products whose 256-row
// tiles leave compute units idle.
//
//   C[m, n] = sum_k deq(A)[m, k] * deq(B)[n, k]      A [M, K], B [N, K], K contiguous
//
// What bounds it.  At 1001 x 4096 x 4096 the operands take 3 us of HBM time and the MFMAs 7 us.  On 256 x 128 tiles
// that product has 128 workgroups, each a serial chain of 32 K steps whose loads are one step ahead and whose fragments
// are read from LDS right before their MFMAs: 1.1 us a step.  Here
//
//  * a workgroup is WM x WN x WK waves: wave tiles of 32 FA x 32 FB, and the WK groups take every WK-th K step, so
//    small tiles still put waves on every SIMD; their partial tiles meet in LDS in group order (deterministic);
//  * NBUF stages of WK steps are in LDS or on their way there (buffer_load ... lds); a wave waits only for its share
//    of the next stage (vmcnt counts down in issue order) and one barrier per stage publishes it;
//  * behind that barrier the next stage's fragments are read into registers while the current one's, read a stage
//    earlier, are multiplied; the refill of the buffer just freed is issued between the MFMAs;
//  * E8M0 scales come four steps at a time (16 bytes per row) into a ring of their own, a few rows per wave with each
//    stage, so that every wave issues the same number of loads per stage.
//
// Measured against the 256-row kernels that took these products before (us, K = 4096 unless noted):
//
//   E2M3 x FP4   1001 x 4096: 37.8 -> 25.1   333 x 4096: 31.9 -> 16.6   17 x 4096: 30.7 -> 8.1   2048 x 14336: 149 -> 129
//   E2M3 x E2M3  1001 x 4096: 46.8 -> 29.6   64 x 4096: 41.9 -> 9.9     4096 x 14336: 320 -> 292
//   FP4 x FP4    1001 x 4096: 27.1 -> 18.1   256 x 14336: 28.4 -> 18.9  17 x 2048 x 1280: 10.2 -> 5.1
//
// A stage (two K steps) of the 128 x 128 shape takes 0.7 us for FP4 x FP4 and 1.0 us for E2M3 x FP4; launch, prologue
// and epilogue are 7 us.  At 1001 x 4096 x 4096 the latter keeps the LDS active for 29 % of the cycles, almost half of
// that in bank conflicts of the 24-byte FP6 fragments, and the MFMA pipe busy for 10 % (profiles/one_tile_products.txt):
// what is left is the chain of barrier, fragment reads and MFMAs of a stage, with one workgroup on a compute unit.
#pragma once

#include "tgm_gemm_w_tile.h"
#include "tgm_mx_operand.h"

namespace tgm {

struct MxTileArgs {
  const uint8_t *a, *sa, *b, *sb;  // codes and E8M0 bytes [rows, K / 32] (null: unscaled)
  void* c;
  int64_t ldc;
  unsigned lda, ldb;  // bytes between rows
  int M, N, K, cdt;
};

// lds_dma16 by the first N lanes of a wave whose lanes are all active; no branch, which would let the compiler
// move the MFMAs around it together.
template <int N>
__device__ __forceinline__ void lds_dma16_lanes(i32x4v rsrc, unsigned lds_addr, unsigned voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n\ts_mov_b64 exec, -1"
               : : "s"(lds_addr), "v"(voff), "s"(rsrc), "n"((1 << N) - 1) : "memory");
}

template <int TA, int TB, int FA, int FB, int WM, int WN, int WK, int NBUF>
struct MxTile {
  using OA = F8F6F4<TA>;
  using OB = F8F6F4<TB>;
  static constexpr int kW = WM * WN, kWaves = kW * WK, kThreads = 64 * kWaves;
  static constexpr int kBM = 32 * FA * WM, kBN = 32 * FB * WN;
  static constexpr int kPA = kBM * OA::RB, kPB = kBN * OB::RB;  // panel bytes of one K step
  static constexpr int kStep = kPA + kPB, kStage = WK * kStep;
  static constexpr int kNA = kPA / 1024, kNB = kPB / 1024;      // 1 KB load instructions per panel
  static constexpr int kQA = (kNA + kW - 1) / kW, kQB = (kNB + kW - 1) / kW;
  static constexpr int kLoads = kQA + kQB + 2;                  // per wave and stage, two of them scales
  static constexpr int kSpb = 4 / WK;                           // stages per batch of scales (four steps)
  static constexpr int kRA = 8 * FA / WN, kRB = 8 * FB / WM;    // scale rows per wave and stage
  static constexpr int kBatch = (kBM + kBN) * 16;
  static constexpr int kNsb = 4;  // ring of scale batches: those being read, waited for and filled
  static constexpr int kEpi = (WK - 1) * kW * FA * FB * 4096 + kW * 32 * 36 * 4;
  static constexpr int kMain = NBUF * kStage + kNsb * kBatch;
  static constexpr int kLds = kMain > kEpi ? kMain : kEpi;
  // waves per SIMD, by LDS and by the registers of a wave tile's sums and two stages of fragments
  static constexpr int kByLds = kWaves * (160 * 1024 / kLds) / 4, kByRegs = FA * FB == 1 ? 4 : 2;
  static constexpr int kOccupancy = kByLds < kByRegs ? kByLds : kByRegs;
  static constexpr bool kFits = kLds <= 160 * 1024 && kLoads * (NBUF - 1) < 64 && (NBUF - 1 + kSpb - 1) / kSpb + 2 <= kNsb && 4 % WK == 0 && 8 * FA % WN == 0 &&
                                8 * FB % WM == 0 && kRA < 32 && kRB < 32;
};

template <int TA, int TB, int FA, int FB, int WM, int WN, int WK, int NBUF>
__global__ void __launch_bounds__(64 * WM * WN * WK)
__attribute__((amdgpu_waves_per_eu(MxTile<TA, TB, FA, FB, WM, WN, WK, NBUF>::kOccupancy,
                                   MxTile<TA, TB, FA, FB, WM, WN, WK, NBUF>::kOccupancy)))
gemm_mx_tile(MxTileArgs p) {
  using T = MxTile<TA, TB, FA, FB, WM, WN, WK, NBUF>;
  using OA = F8F6F4<TA>;
  using OB = F8F6F4<TB>;
  __shared__ __attribute__((aligned(16))) unsigned char lds[T::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / T::kW, w = wave % T::kW, wm = w / WN, wn = w % WN;
  const int tiles_m = (p.M + T::kBM - 1) / T::kBM, tiles_n = (p.N + T::kBN - 1) / T::kBN;
  int tm, tn;
  tile_of_ranges(blockIdx.x, p.K, tiles_m, tiles_n, 8, tm, tn);
  const int m0 = tm * T::kBM, n0 = tn * T::kBN;
  const int nsteps = p.K / kMxK, nstages = (nsteps + WK - 1) / WK;
  const unsigned kblk = (unsigned)(p.K / 32);
  const i32x4v ra = buffer_rsrc(p.a, (unsigned)(p.M - 1) * p.lda + (unsigned)p.K * OA::bits / 8);
  const i32x4v rb = buffer_rsrc(p.b, (unsigned)(p.N - 1) * p.ldb + (unsigned)p.K * OB::bits / 8);
  const i32x4v rsa = buffer_rsrc(p.sa, p.sa ? (unsigned)p.M * kblk : 0u);
  const i32x4v rsb = buffer_rsrc(p.sb, p.sb ? (unsigned)p.N * kblk : 0u);
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  const unsigned scale_base = (unsigned)(NBUF * T::kStage);

  auto dma = [](i32x4v rsrc, unsigned at, unsigned off) __attribute__((always_inline)) {
    lds_dma16(rsrc, (unsigned)__builtin_amdgcn_readfirstlane((int)at), off);
  };
  // Load instruction i of a panel fills its LDS bytes [1024 i, + 1024): lane l writes 16-byte slot 64 i + l,
  // physical column slot % C of row slot / C.  Wave w of a K group issues instructions w, w + kW, ...; where
  // they don't divide, the last one is issued again, so that every wave counts the same number.
  unsigned voa[T::kQA], vob[T::kQB];
#pragma unroll
  for (int q = 0; q < T::kQA; ++q) {
    const int s = 64 * min(w + T::kW * q, T::kNA - 1) + lane, r = s / OA::C;
    voa[q] = (unsigned)(m0 + r) * p.lda + 16u * (unsigned)col_logical<OA::C>(r, s % OA::C) + (unsigned)(wk * OA::RB);
  }
#pragma unroll
  for (int q = 0; q < T::kQB; ++q) {
    const int s = 64 * min(w + T::kW * q, T::kNB - 1) + lane, r = s / OB::C;
    vob[q] = (unsigned)(n0 + r) * p.ldb + 16u * (unsigned)col_logical<OB::C>(r, s % OB::C) + (unsigned)(wk * OB::RB);
  }
  // Scales of batch bt (steps 4 bt .. 4 bt + 3): 16 bytes per row at 16 r (A's rows, then B's).  Part pt (of
  // kSpb) of a batch is kRA rows of A and kRB of B per wave, one lane each.
  auto load_scales = [&](int bt, int pt, int which) __attribute__((always_inline)) {
    const unsigned dst = lds_base + scale_base + (unsigned)(((unsigned)bt % T::kNsb) * T::kBatch);
    const int chunk = pt * T::kWaves + wave;
    if (which == 0)
      lds_dma16_lanes<T::kRA>(rsa, (unsigned)__builtin_amdgcn_readfirstlane((int)(dst + (unsigned)(16 * T::kRA * chunk))),
                              (unsigned)(m0 + T::kRA * chunk + lane) * kblk + 16u * (unsigned)bt);
    else
      lds_dma16_lanes<T::kRB>(
          rsb, (unsigned)__builtin_amdgcn_readfirstlane((int)(dst + (unsigned)(16 * (T::kBM + T::kRB * chunk)))),
          (unsigned)(n0 + T::kRB * chunk + lane) * kblk + 16u * (unsigned)bt);
  };
  // Load piece q (< kLoads) of stage st into buffer buf; with its panels come a part of the next scale batch.
  auto load_piece = [&](int st, int buf, int q) __attribute__((always_inline)) {
    const unsigned base = lds_base + (unsigned)(buf * T::kStage + wk * T::kStep);
    const int sc = st < nstages ? st : nstages - 1;  // past the end: the last stage again, into a free buffer
    const unsigned s0 = (unsigned)(sc * WK);
    const bool inside = WK == 1 || (int)s0 + wk < nsteps;  // a step past K loads zeros
    if (q < T::kQA)
      dma(ra, base + (unsigned)min(w + T::kW * q, T::kNA - 1) * 1024u,
                inside ? voa[q < T::kQA ? q : 0] + s0 * (unsigned)OA::RB : 0xFFFFFFF0u);
    else if (q < T::kQA + T::kQB) {
      const int i = q - T::kQA;
      dma(rb, base + (unsigned)T::kPA + (unsigned)min(w + T::kW * i, T::kNB - 1) * 1024u,
                inside ? vob[i >= 0 && i < T::kQB ? i : 0] + s0 * (unsigned)OB::RB : 0xFFFFFFF0u);
    } else {
      load_scales((int)((unsigned)st / T::kSpb) + 1, (int)((unsigned)st % T::kSpb), q - T::kQA - T::kQB);
    }
  };

  const int half = lane >> 5;
  const int ar = wm * FA * 32 + (lane & 31), br = wn * FB * 32 + (lane & 31);  // + 32 t
  struct Frags {
    i32x8 a[2][FA], b[2][FB];
    unsigned sa[FA], sb[FB];
  };
  auto read = [&](Frags& f, int st, int buf) __attribute__((always_inline)) {
    const unsigned char* pa = lds + buf * T::kStage + wk * T::kStep;
    const unsigned char* pb = pa + T::kPA;
    const int step = st * WK + wk;
    const unsigned* bat = (const unsigned*)(lds + scale_base + (((unsigned)step / 4) % T::kNsb) * T::kBatch) + (step & 3);
#pragma unroll
    for (int t = 0; t < FA; ++t) f.sa[t] = bat[4 * (ar + 32 * t)];
#pragma unroll
    for (int t = 0; t < FB; ++t) f.sb[t] = bat[4 * (T::kBM + br + 32 * t)];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int t = 0; t < FA; ++t) f.a[u][t] = read_block<TA>(pa, ar + 32 * t, 2 * u + half);
#pragma unroll
      for (int t = 0; t < FB; ++t) f.b[u][t] = read_block<TB>(pb, br + 32 * t, 2 * u + half);
    }
  };
  f32x16 acc[FA][FB];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) acc[i][j] = f32x16{};

#pragma unroll
  for (int pt = 0; pt < T::kSpb; ++pt) {
    load_scales(0, pt, 0);
    load_scales(0, pt, 1);
  }
#pragma unroll
  for (int s = 0; s < NBUF; ++s)
#pragma unroll
    for (int q = 0; q < T::kLoads; ++q) load_piece(s, s, q);
  wait_loads<(NBUF - 1) * T::kLoads>();
  lds_barrier();
  // Stage st, its fragments in f: wait for this wave's loads of the next stage; behind the barrier that stage
  // is complete and this stage's buffer free; the next fragments are read and the buffer's refill is issued
  // between the MFMAs.
  int cur = 0;
  auto stage = [&](const Frags& f, Frags& g, int st) __attribute__((always_inline)) {
    const int nxt = cur + 1 < NBUF ? cur + 1 : 0;
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // f is read: its buffer may be overwritten
    wait_loads<(NBUF - 2) * T::kLoads>();
    lds_barrier();
    read(g, st + 1, nxt);
    __builtin_amdgcn_sched_barrier(0);
    // a step past K multiplies zeros, by 1.0: the bytes behind a row's scales could be a NaN's
    const bool inside = WK == 1 || st * WK + wk < nsteps;
    const unsigned keep_a = p.sa && inside ? ~0u : 0u, one_a = ~keep_a & 0x7F7F7F7Fu;
    const unsigned keep_b = p.sb && inside ? ~0u : 0u, one_b = ~keep_b & 0x7F7F7F7Fu;
    constexpr int kMfmas = 2 * FA * FB;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j) {
          const int kb = 8 * (2 * u + half), idx = (u * FA + i) * FB + j;
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f.a[u][i], f.b[u][j], acc[i][j], TA, TB, 0,
                                                                      (int)((f.sa[i] & keep_a | one_a) >> kb), 0,
                                                                      (int)((f.sb[j] & keep_b | one_b) >> kb));
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < T::kLoads; ++q)
            if (q * kMfmas / T::kLoads == idx) load_piece(st + NBUF, cur, q);
          __builtin_amdgcn_sched_barrier(0);
        }
    cur = nxt;
  };
  Frags f0, f1;
  read(f0, 0, 0);
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

template <int TA, int TB, int FA, int FB, int WM, int WN, int WK, int NBUF>
int launch_mx_tile(const MxTileArgs& p, hipStream_t s, const char* who) {
  using T = MxTile<TA, TB, FA, FB, WM, WN, WK, NBUF>;
  static_assert(T::kFits, "tile shape");
  const int64_t tiles = (int64_t)((p.M + T::kBM - 1) / T::kBM) * ((p.N + T::kBN - 1) / T::kBN);
  hipLaunchKernelGGL((gemm_mx_tile<TA, TB, FA, FB, WM, WN, WK, NBUF>), dim3((unsigned)tiles), dim3(T::kThreads), 0, s, p);
  return launch_status(who);
}

// The tile shape for a product, -1 for the large-tile kernels.  fp4_big: the 256 x 256 FP4 kernels take the
// operands (else gemm_f8f6f4 does).  cus: compute units of the stream's device (0 if unknown).  The tile that
// runs goes to *tile.
int mx_tile_shape(int ta, int tb, int64_t m, int64_t n, int64_t k, bool fp4_big, int cus, TileChoice* tile = nullptr);
int launch_gemm_mx_tile(int shape, int ta, int tb, const MxTileArgs& p, hipStream_t s, const char* who);

}  // namespace tgm
