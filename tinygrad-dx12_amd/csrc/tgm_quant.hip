// Tensor-level pack: MX block quantisation and the LSB-first code packer.
//
// The reference accepts only pre-packed bytes (alexandreteles/tinygrad-dx12
// src/tinygrad_dx12/codegen/decomp/dx12.py:26-30); its only packers live in the
// harness and tests (scripts/benchmark_dtypes.py:129-152, test/backend/test_packed.py:81-84)
// and pack payload codes least-significant bit first.  tgm_pack_codes produces that
// byte stream; tgm_quantize_mx adds the OCP MX quantiser that the reference lacks.
#include "tgm_common.h"
#include "tgm_lanes.h"

namespace tgm {

// Largest-normal exponent of each MX element format.
__device__ __forceinline__ int emax_elem(int fmt) { return fmt == TGM_FMT_FP6_E3M2 ? 4 : 2; }

// One thread per (row, block): amax -> shared exponent -> RNE codes -> packed bytes.
// Requires rows and blocks to start on byte boundaries (checked on the host).
__global__ void __launch_bounds__(256) quantize_mx_kernel(const void* __restrict__ x, int xdt, int64_t rows, int64_t k,
                                                          int fmt, int64_t bs, int64_t nblk,
                                                          uint8_t* __restrict__ data, uint8_t* __restrict__ scales) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= rows * nblk) return;
  const int64_t row = id / nblk, blk = id - row * nblk;
  const int64_t c0 = blk * bs;
  const int64_t c1 = c0 + bs < k ? c0 + bs : k;
  const FormatInfo f = format_info(fmt);
  const int64_t base = row * k;
  float amax = 0.f;
  for (int64_t c = c0; c < c1; ++c) amax = fmaxf(amax, fabsf(load_f32(x, xdt, base + c)));
  int shared = 0;
  if (amax > 0.f) {
    int e;
    frexpf(amax, &e);  // amax = m * 2^e, m in [0.5, 1)
    shared = (e - 1) - emax_elem(fmt);
    shared = shared < -127 ? -127 : (shared > 127 ? 127 : shared);
  }
  scales[id] = (uint8_t)(shared + 127);
  // ascending magnitudes of the positive payloads and their midpoints
  const int npos = 1 << (f.bits - 1);
  float mids[31];
  float prev = decode_float(0, f);
  for (int j = 1; j < npos; ++j) {
    const float cur = decode_float((uint32_t)j, f);
    mids[j - 1] = 0.5f * (prev + cur);
    prev = cur;
  }
  uint64_t acc = 0;
  int nbits = 0;
  int64_t out = (base + c0) * f.bits / 8;
  for (int64_t c = c0; c < c1; ++c) {
    const float v = ldexpf(load_f32(x, xdt, base + c), -shared);
    const float a = fabsf(v);
    uint32_t idx = 0;
    for (int j = 0; j < npos - 1; ++j)
      if (a > mids[j] || (a == mids[j] && (j & 1))) idx = (uint32_t)j + 1;
    const uint32_t sign = (v < 0.f && idx > 0) ? 1u : 0u;
    const uint32_t code = (sign << (f.bits - 1)) | idx;
    acc |= (uint64_t)code << nbits;
    nbits += f.bits;
    while (nbits >= 8) {
      data[out++] = (uint8_t)(acc & 0xFF);
      acc >>= 8;
      nbits -= 8;
    }
  }
  if (nbits > 0) data[out] = (uint8_t)(acc & 0xFF);
}

// ---- Whole 32-element blocks (the OCP MX block) of 16-byte aligned input: quantize_mx32.
//
// Bound by HBM.  quantize_mx_kernel reads each element twice with scalar loads, searches a table of
// midpoints that lives in scratch memory and stores single bytes: 237 us for bf16 4096 x 4096 to FP4
// (42 MB: 0.18 TB/s).  Here every element is read once with 16-byte loads and stays in registers, the
// block maximum is an integer maximum of the magnitude bits, and gfx950's scaled conversions round the
// codes (to nearest even, like the midpoint search; the payloads ascend with the magnitude, so an even
// mantissa is an even payload).  Measured on that shape: 9.0 us (4.7 TB/s).
//
//  * FP4: a lane takes 8 elements (one 16-byte load of 16-bit input, one 4-byte store), four lanes a
//    block; the maximum crosses them by two DPP exchanges.  Loads and stores are contiguous over the wave.
//  * FP6: a lane takes a whole block, the operand of the 32-wide conversion, and stores its 24 bytes.
//
// The conversions differ from the midpoint search in what they do with values outside its normal range,
// so a block goes to a per-element path when its maximum is infinite or NaN (the search ignores NaN in
// the maximum and gives it code 0) or below 2^-100 (zero blocks, and exponents near the clamp at -127).
// A value that rounds to zero gets the positive zero code: negative zeros are cleared afterwards.
typedef __bf16 q_bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 q_bf16x32 __attribute__((ext_vector_type(32)));
typedef _Float16 q_f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 q_f16x32 __attribute__((ext_vector_type(32)));
typedef float q_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned q_u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned q_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned q_u32x6 __attribute__((ext_vector_type(6)));
typedef unsigned short q_u16x2 __attribute__((ext_vector_type(2)));

constexpr int kQBlock = 32;          // elements per scale
constexpr int kQMinExp = 127 - 100;  // biased exponent of the smallest block maximum on the fast path

// Shared exponent of a block with the positive finite maximum amax.
__device__ __forceinline__ int shared_exponent(float amax, int fmt) {
  if (!(amax > 0.f)) return 0;
  int e;
  frexpf(amax, &e);  // amax = m * 2^e, m in [0.5, 1)
  const int shared = (e - 1) - emax_elem(fmt);
  return shared < -127 ? -127 : (shared > 127 ? 127 : shared);
}

// Code of one value: the midpoint search over the format's ascending magnitudes.
__device__ __forceinline__ uint32_t nearest_code(float x, int shared, const FormatInfo f) {
  const float v = ldexpf(x, -shared), a = fabsf(v);
  uint32_t idx = 0;
  float prev = decode_float(0, f);
  for (uint32_t j = 1; j < (1u << (f.bits - 1)); ++j) {
    const float cur = decode_float(j, f), mid = 0.5f * (prev + cur);
    if (a > mid || (a == mid && !(j & 1))) idx = j;
    prev = cur;
  }
  return (v < 0.f && idx > 0 ? 1u << (f.bits - 1) : 0u) | idx;
}

// N elements of a lane as 32-bit words (two 16-bit elements or one float each).
template <int XDT, int N>
struct QLane {
  static constexpr int kWords = XDT == TGM_F32 ? N : N / 2;
  unsigned w[kWords];

  __device__ __forceinline__ void load(const void* x, int64_t first) {
    const q_u32x4* p = (const q_u32x4*)((const uint8_t*)x + first * (XDT == TGM_F32 ? 4 : 2));
#pragma unroll
    for (int i = 0; i < kWords / 4; ++i) {
      const q_u32x4 v = __builtin_nontemporal_load(p + i);
#pragma unroll
      for (int e = 0; e < 4; ++e) w[4 * i + e] = v[e];
    }
  }
  // Largest magnitude as the bits of an fp32 value of the same exponent class: NaN > infinity > all others.
  __device__ __forceinline__ unsigned max_bits() const {
    if constexpr (XDT == TGM_F32) {
      unsigned m = 0;
#pragma unroll
      for (int i = 0; i < kWords; ++i) m = max(m, w[i] & 0x7FFFFFFFu);
      return m;
    } else {
      q_u16x2 m = {0, 0};
#pragma unroll
      for (int i = 0; i < kWords; ++i)
        m = __builtin_elementwise_max(m, __builtin_bit_cast(q_u16x2, w[i] & 0x7FFF7FFFu));
      const unsigned h = max((unsigned)m[0], (unsigned)m[1]);
      if constexpr (XDT == TGM_BF16) return h << 16;
      else return f32_bits((float)__builtin_bit_cast(_Float16, (unsigned short)h));
    }
  }
  __device__ __forceinline__ float value(int i) const {
    if constexpr (XDT == TGM_F32) return bits_f32(w[i]);
    else if constexpr (XDT == TGM_BF16) return bits_f32(i & 1 ? w[i / 2] & 0xFFFF0000u : w[i / 2] << 16);
    else return (float)__builtin_bit_cast(_Float16, (unsigned short)(w[i / 2] >> (16 * (i & 1))));
  }
};

// Largest magnitude of N values, NaN ignored.
template <int XDT, int N>
__device__ __forceinline__ float amax_of(const QLane<XDT, N>& q) {
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float a = fabsf(q.value(i));
    m = a > m ? a : m;  // not fmaxf: a signalling NaN would come through it
  }
  return m;
}

__device__ __forceinline__ float quad_max(float v) { return fmaxf(fmaxf(v, xor1(v)), fmaxf(xor2(v), xor2(xor1(v)))); }
__device__ __forceinline__ unsigned quad_max(unsigned v) {
  v = max(v, f32_bits(xor1(bits_f32(v))));
  return max(v, f32_bits(xor2(bits_f32(v))));
}

// Eight elements per lane to FP4; the scale byte is stored by the first lane of each block.
template <int XDT>
__global__ void __launch_bounds__(256) quantize_mx32_fp4(const void* __restrict__ x, int64_t chunks,
                                                         uint32_t* __restrict__ data, uint8_t* __restrict__ scales) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;  // chunks is a multiple of 4: quads are whole
  if (c >= chunks) return;
  QLane<XDT, 8> q;
  q.load(x, c * 8);
  const unsigned mb = quad_max(q.max_bits());
  const int e = (int)(mb >> 23);
  unsigned codes = 0;
  int shared;
  if (e >= kQMinExp && e < 255) {
    shared = e - 127 - 2;
    const float s = bits_f32((unsigned)(shared + 127) << 23);
    if constexpr (XDT == TGM_F32) {
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bits_f32(q.w[0]), bits_f32(q.w[1]), s, 0);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bits_f32(q.w[2]), bits_f32(q.w[3]), s, 1);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bits_f32(q.w[4]), bits_f32(q.w[5]), s, 2);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bits_f32(q.w[6]), bits_f32(q.w[7]), s, 3);
    } else if constexpr (XDT == TGM_BF16) {
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(codes, __builtin_bit_cast(q_bf16x2, q.w[0]), s, 0);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(codes, __builtin_bit_cast(q_bf16x2, q.w[1]), s, 1);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(codes, __builtin_bit_cast(q_bf16x2, q.w[2]), s, 2);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(codes, __builtin_bit_cast(q_bf16x2, q.w[3]), s, 3);
    } else {
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(codes, __builtin_bit_cast(q_f16x2, q.w[0]), s, 0);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(codes, __builtin_bit_cast(q_f16x2, q.w[1]), s, 1);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(codes, __builtin_bit_cast(q_f16x2, q.w[2]), s, 2);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(codes, __builtin_bit_cast(q_f16x2, q.w[3]), s, 3);
    }
    // clear the sign of zero codes: (magnitude + 7) carries into bit 3 of its nibble unless it is 0
    codes &= 0x77777777u | (((codes & 0x77777777u) + 0x77777777u) & 0x88888888u);
  } else {  // the four lanes of a block take this branch together
    shared = shared_exponent(quad_max(amax_of(q)), TGM_FMT_FP4_E2M1);
    const FormatInfo f = format_info(TGM_FMT_FP4_E2M1);
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
      float v = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) v = i == j ? q.value(j) : v;
      codes |= nearest_code(v, shared, f) << (4 * i);
    }
  }
  data[c] = codes;
  if ((threadIdx.x & 3) == 0) scales[c >> 2] = (uint8_t)(shared + 127);
}

// A whole block per lane to FP6 (24 bytes, little-endian 6-bit fields).
template <int FMT, int XDT>
__global__ void __launch_bounds__(256) quantize_mx32_fp6(const void* __restrict__ x, int64_t blocks,
                                                         q_u32x2* __restrict__ data, uint8_t* __restrict__ scales) {
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= blocks) return;
  QLane<XDT, 32> q;
  q.load(x, b * kQBlock);
  const int e = (int)(q.max_bits() >> 23);
  unsigned out[6];
  int shared;
  if (e >= kQMinExp && e < 255) {
    shared = e - 127 - (FMT == TGM_FMT_FP6_E3M2 ? 4 : 2);
    const float s = bits_f32((unsigned)(shared + 127) << 23);
    q_u32x6 r;
    if constexpr (XDT == TGM_F32) {
      // the conversion interleaves its two operands: result element 2 i is lo[i], 2 i + 1 is hi[i]
      q_f32x16 lo, hi;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        lo[i] = bits_f32(q.w[2 * i]);
        hi[i] = bits_f32(q.w[2 * i + 1]);
      }
      if constexpr (FMT == TGM_FMT_FP6_E2M3) r = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(lo, hi, s);
      else r = __builtin_amdgcn_cvt_scalef32_2xpk16_bf6_f32(lo, hi, s);
    } else if constexpr (XDT == TGM_BF16) {
      q_bf16x32 v;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const q_bf16x2 p = __builtin_bit_cast(q_bf16x2, q.w[i]);
        v[2 * i] = p[0];
        v[2 * i + 1] = p[1];
      }
      if constexpr (FMT == TGM_FMT_FP6_E2M3) r = __builtin_amdgcn_cvt_scalef32_pk32_fp6_bf16(v, s);
      else r = __builtin_amdgcn_cvt_scalef32_pk32_bf6_bf16(v, s);
    } else {
      q_f16x32 v;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const q_f16x2 p = __builtin_bit_cast(q_f16x2, q.w[i]);
        v[2 * i] = p[0];
        v[2 * i + 1] = p[1];
      }
      if constexpr (FMT == TGM_FMT_FP6_E2M3) r = __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(v, s);
      else r = __builtin_amdgcn_cvt_scalef32_pk32_bf6_f16(v, s);
    }
    // clear the sign of zero codes, 16 codes (three words) at a time as even and odd 12-bit halves:
    // (magnitude + 31) carries into bit 5 of its field unless it is 0
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      unsigned w0 = r[3 * h], w1 = r[3 * h + 1], w2 = r[3 * h + 2];
      // four words of four 6-bit codes each, so that every field lies inside one word
      unsigned f[4] = {w0 & 0xFFFFFFu, (w0 >> 24) | ((w1 & 0xFFFFu) << 8), (w1 >> 16) | ((w2 & 0xFFu) << 16), w2 >> 8};
#pragma unroll
      for (int i = 0; i < 4; ++i) f[i] &= 0x7DF7DFu | (((f[i] & 0x7DF7DFu) + 0x7DF7DFu) & 0x820820u);
      out[3 * h] = f[0] | (f[1] << 24);
      out[3 * h + 1] = (f[1] >> 8) | (f[2] << 16);
      out[3 * h + 2] = (f[2] >> 16) | (f[3] << 8);
    }
  } else {
    shared = shared_exponent(amax_of(q), FMT);
    const FormatInfo f = format_info(FMT);
    uint64_t acc[3] = {0, 0, 0};
#pragma unroll 1
    for (int i = 0; i < kQBlock; ++i) {
      float v = 0.f;
#pragma unroll
      for (int j = 0; j < kQBlock; ++j) v = i == j ? q.value(j) : v;
      const uint64_t code = nearest_code(v, shared, f);
      const int bit = 6 * i, w = bit >> 6, sh = bit & 63;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        if (j == w) acc[j] |= code << sh;
        if (j == w + 1 && sh > 58) acc[j] |= code >> (64 - sh);
      }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      out[2 * j] = (unsigned)acc[j];
      out[2 * j + 1] = (unsigned)(acc[j] >> 32);
    }
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) data[b * 3 + j] = q_u32x2{out[2 * j], out[2 * j + 1]};
  scales[b] = (uint8_t)(shared + 127);
}

template <int XDT>
void launch_quantize_mx32(hipStream_t s, const void* x, int64_t blocks, int fmt, void* data, void* scales) {
  const int64_t lanes = fmt == TGM_FMT_FP4_E2M1 ? blocks * 4 : blocks;
  const dim3 grid((unsigned)((lanes + 255) / 256));
  if (fmt == TGM_FMT_FP4_E2M1)
    hipLaunchKernelGGL(quantize_mx32_fp4<XDT>, grid, dim3(256), 0, s, x, lanes, (uint32_t*)data, (uint8_t*)scales);
  else if (fmt == TGM_FMT_FP6_E2M3)
    hipLaunchKernelGGL((quantize_mx32_fp6<TGM_FMT_FP6_E2M3, XDT>), grid, dim3(256), 0, s, x, lanes, (q_u32x2*)data,
                       (uint8_t*)scales);
  else
    hipLaunchKernelGGL((quantize_mx32_fp6<TGM_FMT_FP6_E3M2, XDT>), grid, dim3(256), 0, s, x, lanes, (q_u32x2*)data,
                       (uint8_t*)scales);
}

// Eight codes per thread: 4 bytes (4-bit) or 6 bytes (6-bit) at byte offset t*bits.
__global__ void __launch_bounds__(256) pack_codes_kernel(const uint8_t* __restrict__ codes, int64_t count, int bits,
                                                         uint8_t* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t first = t * 8;
  if (first >= count) return;
  uint64_t acc = 0;
  const uint32_t mask = (1u << bits) - 1u;
  for (int j = 0; j < 8; ++j) {
    const int64_t i = first + j;
    const uint64_t c = i < count ? (uint64_t)(codes[i] & mask) : 0ull;
    acc |= c << (j * bits);
  }
  const int64_t nbytes_total = (count * bits + 7) / 8;
  const int64_t o = t * bits;
  for (int b = 0; b < bits; ++b)
    if (o + b < nbytes_total) out[o + b] = (uint8_t)((acc >> (8 * b)) & 0xFF);
}

}  // namespace tgm

using namespace tgm;

extern "C" int tgm_quantize_mx(const void* x, int x_dtype, int64_t rows, int64_t k, int fmt, int64_t block_size,
                               void* data, void* scales, void* stream) {
  clear_error();
  TGM_CHECK_ARG(fmt == TGM_FMT_FP4_E2M1 || fmt == TGM_FMT_FP6_E2M3 || fmt == TGM_FMT_FP6_E3M2,
                "MX quantisation needs an FP4/FP6 format");
  TGM_CHECK_ARG(x_dtype == TGM_BF16 || x_dtype == TGM_F16 || x_dtype == TGM_F32, "quantiser input must be bf16/f16/f32");
  TGM_CHECK_ARG(rows >= 0 && k >= 1 && block_size >= 1, "invalid quantiser sizes");
  const int bits = format_info(fmt).bits;
  TGM_CHECK_ARG((k * bits) % 8 == 0 && (block_size * bits) % 8 == 0,
                "rows and blocks must start on byte boundaries (K*bits and block*bits multiples of 8)");
  if (rows == 0) return TGM_OK;
  const int64_t nblk = (k + block_size - 1) / block_size;
  const int64_t total = rows * nblk;
  // Whole 32-element blocks of aligned operands (every contiguous tensor with K a multiple of 32): the
  // vector kernels.  Other block sizes, ragged last blocks and odd addresses keep the scalar kernel, and so
  // do arrays whose lanes (four a block for FP4, one for FP6) would not fit a launch of 2^32 work items.
  const int64_t lanes = total * (fmt == TGM_FMT_FP4_E2M1 ? 4 : 1);
  if (block_size == kQBlock && k % kQBlock == 0 && (uintptr_t)x % 16 == 0 &&
      (uintptr_t)data % (fmt == TGM_FMT_FP4_E2M1 ? 4 : 8) == 0 && lanes <= (1ll << 32) - 256) {
    const hipStream_t s = (hipStream_t)stream;
    if (x_dtype == TGM_F32) launch_quantize_mx32<TGM_F32>(s, x, total, fmt, data, scales);
    else if (x_dtype == TGM_BF16) launch_quantize_mx32<TGM_BF16>(s, x, total, fmt, data, scales);
    else launch_quantize_mx32<TGM_F16>(s, x, total, fmt, data, scales);
    return launch_status("tgm_quantize_mx");
  }
  hipLaunchKernelGGL(quantize_mx_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x,
                     x_dtype, rows, k, fmt, block_size, nblk, (uint8_t*)data, (uint8_t*)scales);
  return launch_status("tgm_quantize_mx");
}

extern "C" int tgm_pack_codes(const void* codes, int64_t count, int bits, void* out, void* stream) {
  clear_error();
  TGM_CHECK_ARG(bits == 4 || bits == 6, "pack width must be 4 or 6 bits");
  TGM_CHECK_ARG(count >= 0, "invalid code count");
  if (count == 0) return TGM_OK;
  const int64_t threads = (count + 7) / 8;
  hipLaunchKernelGGL(pack_codes_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const uint8_t*)codes, count, bits, (uint8_t*)out);
  return launch_status("tgm_pack_codes");
}
