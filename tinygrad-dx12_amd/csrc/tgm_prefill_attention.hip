// Causal prompt attention in one kernel (flash-attention form) on bf16 MFMA, with the accuracy
// of fp32 arithmetic.
//
// For every (sequence, q head) and prompt token t at position p = pos[b] + t:
//
//   out[t] = sum_{k <= p} softmax_k(q_t . K_k / sqrt(hd)) V_k        (K, V: the bf16 cache)
//
// The scores and probabilities never leave the chip.  A workgroup takes 128 prompt tokens of
// one (sequence, head), 32 per wave, and walks the cache in blocks of 64 keys up to its last
// token's position.  The products are computed transposed, so that everything a query owns
// sits in one lane (the 32x32 MFMA D layout gives lane l column l % 32):
//
//   S^T[key, query]  = K . Q^T       A = the K block (LDS),     B = q (registers)
//   O^T[dim, query] += V^T . P^T     A = the V^T block (LDS),   B = p (registers)
//
// Accuracy: q (scaled by log2(e) / sqrt(hd), so that the softmax runs on exp2) and each
// probability are split into three bf16 terms
// x = t0 + t1 + t2 (t0 = bf16(x), each later term the bf16 of what the earlier ones leave;
// three terms hold the 24 bits of an fp32 value) and every term meets the bf16 K or V
// operand in its own MFMA.  Products of bf16 values are exact in fp32, so S and O carry only
// fp32 accumulation error, like an fp32 kernel.  The softmax is online per lane in fp32.
//
// D layout and the probability operand: lane (query, half h) holds S^T rows (keys)
// 8 (v / 4) + 4 h + v % 4 of each 32-key tile, v = 0 .. 15.  The P . V MFMA u of a tile
// (16 keys) takes the lane's values v = 8 u .. 8 u + 7 as its B operand, i.e. keys
// 16 u + 4 h + {0..3} and 16 u + 8 + 4 h + {0..3}; the V^T operand reads the same keys (two
// 8-byte pieces of a V^T row), so both sides agree on which key each product belongs to.
//
// LDS (double buffered, one barrier per key block): K and V blocks as 64 rows of hd bf16, as the cache
// holds them, loaded straight to LDS (buffer_load ... lds) while the previous block is computed.  16-byte
// chunks are XOR-swizzled by the row so that neither operand's reads conflict: K's are 16-byte reads of 32
// rows, V's are transposing reads (ds_read_b64_tr_b16: a 16-lane group reads 4 keys x 16 dims and each
// lane gets one dim's 4 keys).
//
// What bounds it: the chain from scores to probabilities to sums within a wave, with two waves per SIMD to
// overlap.  The MFMAs, 96 per wave and block (three terms each way), would take 28 us of the 87 at 8 x 512
// tokens, 32 heads of 128; they keep their pipe busy for 25 % of the cycles, and the LDS is active for 5 % of
// them, without bank conflicts (profiles/prefill_attention.txt).  V was transposed by 2-byte LDS stores from registers before (32 conflicting stores
// per thread and block), and with them the kernel held 404 registers, one wave per SIMD, so nothing ran
// beside the softmax: 208 us there and 348 us for one 2048-token prompt, 87 and 146 us now, at the same
// error (2.2e-7 against 64 bits).
#include <math.h>

#include "../../include/tgm_decoder.h"
#include "tgm_mfma_common.h"

namespace tgm {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 pa_bf16x8;
typedef _Float16 pa_f16x4 __attribute__((ext_vector_type(4)));
typedef short pa_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) pa_s16x4 pa_lds_s16x4;

constexpr int kPaKeys = 64;      // keys per block
constexpr int kPaQueries = 128;  // prompt tokens per workgroup (32 per wave)
constexpr int kPaTerms = 3;      // bf16 terms per fp32 operand value

// The three bf16 terms of 8 fp32 values.
__device__ __forceinline__ void pa_split(float (&r)[8], pa_bf16x8 (&t)[kPaTerms]) {
#pragma unroll
  for (int s = 0; s < kPaTerms; ++s) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const __bf16 v = (__bf16)r[i];  // round to nearest even
      t[s][i] = v;
      r[i] -= (float)v;  // exact: the residual has at most 16 significant bits
    }
  }
}

// Grid (ceil(T / 128), heads, batch), 256 threads.
template <int HD>
__global__ void __launch_bounds__(256, 2) dec_prefill_attention(const float* __restrict__ qkv, int T, int H, int HK,
                                                                const int32_t* __restrict__ pos,
                                                                const uint16_t* __restrict__ kc,
                                                                const uint16_t* __restrict__ vc, int max_seq, float scale,
                                                                void* __restrict__ out, int odt) {
  constexpr int NJ = HD / 16;                         // 16-wide steps of q . k
  constexpr int ND = HD / 32;                         // 32-row tiles of O^T
  constexpr int ROW = HD * 2, CH = ROW / 16;          // a key's row of K or V: CH 16-byte chunks
  constexpr int BLOCK = kPaKeys * ROW, STAGE = 2 * BLOCK;
  constexpr int RPI = 1024 / ROW;                     // rows per load instruction
  constexpr int NLD = kPaKeys / RPI / 4;              // load instructions per wave and block, for K and for V
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * STAGE];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.y, b = blockIdx.z, j = h / (H / HK);
  const int p0 = pos[b];
  const int64_t ld = (int64_t)(H + 2 * HK) * HD;
  // the longest query blocks (the last tokens, which see the most keys) are launched first
  const int qblk = (int)(gridDim.x - 1 - blockIdx.x);
  const int tq = qblk * kPaQueries + wave * 32 + l32;  // this lane's prompt token
  const bool qvalid = tq < T;
  const int tqc = qvalid ? tq : T - 1;
  const int qpos = p0 + tqc;
  const int t_end = min(qblk * kPaQueries + kPaQueries, T);
  const int nkeys = min(p0 + t_end, max_seq);                 // keys 0 .. nkeys - 1 serve the workgroup
  const int nblocks = nkeys > 0 ? (nkeys + kPaKeys - 1) / kPaKeys : 0;
  const int wave_end = min(qblk * kPaQueries + wave * 32 + 32, T);
  const int wave_maxpos = p0 + wave_end - 1;                  // blocks past it are masked for every lane
  const int wave_minpos = p0 + min(qblk * kPaQueries + wave * 32, T - 1);  // blocks up to it need no mask
  const uint16_t* kbase = kc + ((int64_t)b * HK + j) * max_seq * HD;
  const uint16_t* vbase = vc + ((int64_t)b * HK + j) * max_seq * HD;
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;

  // Swizzle of a row's chunks.  K: 32 rows at one logical chunk must differ in chunk (or row parity where
  // two rows share the 64 banks); V: four consecutive rows of 64 consecutive bytes must.
  auto swz_k = [](int key) { return CH == 16 ? key & 15 : (key >> 1) & 7; };
  auto swz_v = [](int key) { return CH == 16 ? (key & 3) << 2 : ((key >> 1) & 1) << 2; };
  // Load offsets: instruction i = wave + 4 q covers rows RPI i ..; lane l fills chunk l % CH of its row.
  unsigned vok[NLD], vov[NLD];
#pragma unroll
  for (int q = 0; q < NLD; ++q) {
    const int key = RPI * (wave + 4 * q) + lane / CH, ch = lane % CH;
    vok[q] = (unsigned)(key * ROW + (ch ^ swz_k(key)) * 16);
    vov[q] = (unsigned)(key * ROW + (ch ^ swz_v(key)) * 16);
  }
  auto load_block = [&](int kb) __attribute__((always_inline)) {
    const int64_t first = (int64_t)kb * kPaKeys;
    const unsigned bytes = (unsigned)min(kPaKeys, max_seq - (int)first) * ROW;  // keys past the cache read zeros
    const i32x4v rk = buffer_rsrc(kbase + first * HD, bytes), rv = buffer_rsrc(vbase + first * HD, bytes);
    const unsigned st = lds_base + (unsigned)((kb & 1) * STAGE + wave * 1024);
#pragma unroll
    for (int q = 0; q < NLD; ++q) lds_dma16(rk, st + q * 4096u, vok[q]);
#pragma unroll
    for (int q = 0; q < NLD; ++q) lds_dma16(rv, st + (unsigned)BLOCK + q * 4096u, vov[q]);
  };
  if (nblocks > 0) load_block(0);

  // q terms as the B operand of S^T: lane (query, half) holds q[16 s + 8 half + i] * scale.
  pa_bf16x8 qt[NJ][kPaTerms];
  {
    const float* qrow = qkv + ((int64_t)b * T + tqc) * ld + (int64_t)h * HD;
#pragma unroll
    for (int s = 0; s < NJ; ++s) {
      const f32x4 x0 = *(const f32x4*)(qrow + 16 * s + 8 * half);
      const f32x4 x1 = *(const f32x4*)(qrow + 16 * s + 8 * half + 4);
      const float sl = scale * 1.4426950408889634f;  // log2(e): the softmax runs on exp2
      float r[8] = {x0[0] * sl, x0[1] * sl, x0[2] * sl, x0[3] * sl, x1[0] * sl, x1[1] * sl, x1[2] * sl, x1[3] * sl};
      pa_split(r, qt[s]);
    }
  }

  // Per-lane LDS offsets.  V: lane i of 16-lane group g reads key + i / 4, dims 16 (g % 2) + 4 (i % 4) .. + 4
  // of an O^T tile (groups 2 and 3 the keys of lane half 1), and receives dim 16 (g % 2) + i of four keys.
  const int vi = lane & 15, vg = lane >> 4;
  const int vkey = 4 * half + (vi >> 2);
  unsigned voff[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
    voff[dt] = (unsigned)(BLOCK + vkey * ROW + ((4 * dt + 2 * (vg & 1) + ((vi & 3) >> 1)) ^ swz_v(vkey)) * 16 + (vi & 1) * 8);

  f32x16 O[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt) O[dt] = f32x16{};
  float m = -INFINITY, l = 0.f;
#pragma unroll 1
  for (int kb = 0; kb < nblocks; ++kb) {
    wait_lds_dma();   // this wave's loads of block kb
    __syncthreads();  // everybody's; and everybody is done with block kb - 1
    if (kb + 1 < nblocks) load_block(kb + 1);
    if (kb * kPaKeys > wave_maxpos) continue;  // uniform over the wave
    const unsigned char* st = lds + (kb & 1) * STAGE;
    f32x16 S[2] = {f32x16{}, f32x16{}};
#pragma unroll
    for (int s = 0; s < NJ; ++s)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const pa_bf16x8 a = *(const pa_bf16x8*)(st + (kt * 32 + l32) * ROW + (((2 * s + half) ^ swz_k(l32)) * 16));
#pragma unroll
        for (int t = 0; t < kPaTerms; ++t) S[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qt[s][t], S[kt], 0, 0, 0);
      }
    // online softmax of this lane's query over the block (the lane pair l, l ^ 32 holds it)
    // (scores are in log2 units: q carries scale * log2(e))
    if (kb * kPaKeys + kPaKeys - 1 > wave_minpos) {  // the block reaches past some query: mask (uniform)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = kb * kPaKeys + kt * 32 + 8 * (v >> 2) + 4 * half + (v & 3);
          if (key > qpos) S[kt][v] = -INFINITY;
        }
    }
    float bm = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v) bm = fmaxf(bm, S[kt][v]);
    bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
    const float mn = fmaxf(m, bm);  // finite: block 0 holds key 0 <= qpos
    if (__any(mn != m)) {  // some lane's maximum moved: rescale (a wave-uniform branch)
      const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) O[dt][v] *= alpha;
    }
    m = mn;
    float ls = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float r[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          // v_exp_f32: within one unit in the last place; results below 2^-126 become 0, far below the
          // last place of a sum that holds exp2(0) = 1.  0 for masked keys.
          r[i] = __builtin_amdgcn_exp2f(S[kt][8 * u + i] - mn);
          ls += r[i];
        }
        pa_bf16x8 pb[kPaTerms];
        pa_split(r, pb);
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {  // keys 16 u + 4 h .. + 4 of tile kt, then the ones 8 on
          const unsigned char* row = st + voff[dt] + (kt * 32 + u * 16) * ROW;
          const pa_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_s16x4*)row);
          const pa_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_s16x4*)(row + 8 * ROW));
          const pa_bf16x8 a = __builtin_bit_cast(pa_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
          for (int t = 0; t < kPaTerms; ++t) O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pb[t], O[dt], 0, 0, 0);
        }
      }
    l += ls;
  }
  l += __shfl_xor(l, 32, 64);
  if (!qvalid) return;
  const float inv = 1.0f / l;
  const int64_t o = ((int64_t)b * T + tq) * H * HD + (int64_t)h * HD;
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int64_t e = o + dt * 32 + 8 * g + 4 * half;  // dims 8 g + 4 h .. + 4 of tile dt
      if (odt == TGM_F16) {
        *(pa_f16x4*)((_Float16*)out + e) = pa_f16x4{(_Float16)(O[dt][4 * g] * inv), (_Float16)(O[dt][4 * g + 1] * inv),
                                                    (_Float16)(O[dt][4 * g + 2] * inv), (_Float16)(O[dt][4 * g + 3] * inv)};
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) store_c(out, odt, e + i, O[dt][4 * g + i] * inv);
      }
    }
}

}  // namespace tgm

using namespace tgm;

extern "C" int tgm_dec_prefill_attention(const float* qkv, int64_t rows, int64_t seq_rows, int64_t heads,
                                         int64_t kv_heads, int64_t head_dim, const int32_t* pos, const void* k_cache,
                                         const void* v_cache, int64_t max_seq, void* out, int out_dtype, void* stream) {
  clear_error();
  TGM_CHECK_ARG(qkv && pos && k_cache && v_cache && out, "null operand");
  TGM_CHECK_ARG(rows >= 0 && seq_rows > 0 && rows % seq_rows == 0, "rows must be a multiple of seq_rows");
  TGM_CHECK_ARG(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "heads must be a multiple of kv_heads");
  TGM_CHECK_ARG(out_dtype == TGM_F16 || out_dtype == TGM_BF16 || out_dtype == TGM_F32, "output must be f16, bf16 or f32");
  TGM_CHECK_ARG(max_seq > 0 && max_seq < (1 << 30) && rows < (1ll << 31), "invalid sizes");
  TGM_CHECK_ARG(heads <= 65535 && rows / seq_rows <= 65535, "at most 65535 heads and sequences");
  if (head_dim != 64 && head_dim != 128) TGM_UNSUPPORTED("tgm_dec_prefill_attention: head_dim must be 64 or 128");
  if ((uintptr_t)qkv % 16 || (uintptr_t)k_cache % 16 || (uintptr_t)v_cache % 16 ||
      (out_dtype == TGM_F16 && (uintptr_t)out % 8))
    TGM_UNSUPPORTED("tgm_dec_prefill_attention: qkv and the caches must be 16-byte aligned, f16 output 8-byte");
  if (rows == 0) return TGM_OK;
  const dim3 grid((unsigned)((seq_rows + kPaQueries - 1) / kPaQueries), (unsigned)heads, (unsigned)(rows / seq_rows));
  const float scale = (float)(1.0 / sqrt((double)head_dim));
  const hipStream_t st = (hipStream_t)stream;
  if (head_dim == 64)
    hipLaunchKernelGGL(dec_prefill_attention<64>, grid, dim3(256), 0, st, qkv, (int)seq_rows, (int)heads,
                       (int)kv_heads, pos, (const uint16_t*)k_cache, (const uint16_t*)v_cache, (int)max_seq, scale, out,
                       out_dtype);
  else
    hipLaunchKernelGGL(dec_prefill_attention<128>, grid, dim3(256), 0, st, qkv, (int)seq_rows, (int)heads,
                       (int)kv_heads, pos, (const uint16_t*)k_cache, (const uint16_t*)v_cache, (int)max_seq, scale, out,
                       out_dtype);
  return launch_status("tgm_dec_prefill_attention");
}
