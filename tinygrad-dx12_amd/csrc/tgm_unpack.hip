// Packed decode (PackedTensor.unpack, alexandreteles/tinygrad-dx12
// src/tinygrad_dx12/codegen/decomp/dx12.py:49-106) and the library's error plumbing.
//
// One thread decodes eight consecutive logical elements of the flattened array.  The
// payload of element i is read straight from the bit stream (two bytes cover any
// 4- or 6-bit payload), so rows that do not start on a byte boundary (odd K for
// 4-bit, K % 4 != 0 for 6-bit) decode exactly like the reference's flat word view.
#include <atomic>

#include "tgm_common.h"

namespace tgm {

static thread_local char g_last_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
}

void clear_error() { g_last_error[0] = 0; }

int launch_status(const char* what) {
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    set_error("%s launch failed: %s (%d)", what, hipGetErrorString(err), (int)err);
    return (int)err;
  }
  return TGM_OK;
}

int stream_cu_count(hipStream_t stream) {
  static std::atomic<int> counts[64];  // per device, 0 = not looked up yet
  int device = -1;
  if (stream != nullptr && stream != hipStreamLegacy && stream != hipStreamPerThread) {
    hipDevice_t d = -1;
    if (hipStreamGetDevice(stream, &d) != hipSuccess) return 0;
    device = (int)d;
  } else if (hipGetDevice(&device) != hipSuccess) {
    return 0;
  }
  if (device < 0 || device >= 64) return 0;
  int n = counts[device].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n < 0) return 0;
    counts[device].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Keeps a product and its narrowing to f16 apart: merged into one v_fma_mixlo_f16 with a +0 addend
// the compiler's code turns -0 into +0.
__device__ __forceinline__ void keep_product(float& v) { asm("" : "+v"(v)); }
__device__ __forceinline__ void keep_product(double&) {}

// Value of one element in the multiplication type of dx12.py:103 and its final cast.
template <typename MT>
__device__ __forceinline__ void decode_store(uint32_t p, int fmt, FormatInfo f, bool has_scale, MT scale,
                                             void* out, int odt, int64_t i) {
  if (is_int_format(fmt)) {
    const int32_t v = decode_int(p, fmt);
    if (has_scale) {
      store_from_f64(out, odt, i, (double)((MT)v * scale));
    } else if (odt == TGM_F32 || odt == TGM_F16 || odt == TGM_BF16) {
      store_from_f32(out, odt, i, (float)v);
    } else {
      store_from_i64(out, odt, i, (int64_t)v);
    }
  } else {
    const float v = decode_float(p, f);
    if (has_scale) {
      MT prod = (MT)v * scale;
      keep_product(prod);
      if (sizeof(MT) == 4) store_from_f32(out, odt, i, (float)prod);
      else store_from_f64(out, odt, i, (double)prod);
    } else {
      store_from_f32(out, odt, i, v);
    }
  }
}

template <typename MT>
__global__ void __launch_bounds__(256) unpack_kernel(const uint8_t* __restrict__ data, int64_t nbytes, int fmt,
                                                     int64_t count, int64_t k, const void* __restrict__ scales,
                                                     int sdt, int64_t nblk, int64_t bs, void* __restrict__ out,
                                                     int odt, int fp8_target) {
  const FormatInfo f = format_info(fmt);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x * 8;
  for (int64_t base = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8; base < count; base += stride) {
    int64_t row = base / k, col = base - row * k;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t i = base + j;
      if (i >= count) break;
      const uint32_t p = payload_at(data, nbytes, i, f.bits);
      if (fp8_target) {
        ((uint8_t*)out)[i] = fp8_target == 1 ? fp8_direct(p, f, 3, 7) : fp8_direct(p, f, 2, 15);
      } else if (scales) {
        const int64_t si = row * nblk + col / bs;
        MT s;
        if (sizeof(MT) == 8) s = (MT)load_f64(scales, sdt, si);
        else s = (MT)load_f32(scales, sdt, si);
        decode_store<MT>(p, fmt, f, true, s, out, odt, i);
      } else {
        decode_store<MT>(p, fmt, f, false, (MT)1, out, odt, i);
      }
      if (++col == k) { col = 0; ++row; }
    }
  }
}

// ---- bf16 / f16 / f32 output: unpack_vec.
//
// Bound by HBM.  unpack_kernel reads each payload with two byte loads, forms every product through the
// all-types helpers and stores element by element: 202 us for FP4 14336 x 4096 with E8M0 scales to bf16
// (149 MB: 0.74 TB/s).  Here a lane decodes the consecutive elements of one 16-byte store (8 of a 16-bit
// type, 4 fp32) from the one or two aligned dwords that hold their payloads, so every store instruction
// of a wave writes 1 KB in a row.  Measured on that shape: 25 us (6.0 TB/s).
// The stores are non-temporal: the results are several times the size of the L2s and would displace what
// the loads share there (with ordinary stores 40 us; two 16-byte stores per lane, 32 bytes apart, cost
// FP6 8000 x 4096 to bf16 51 us against 16.6).
//
// Values are exact (the same fp32 code values, the same single fp32 product with the scale and the same
// rounding), so the results are bit-identical.  A lane reads one scale; where a row or a scale block ends
// among its elements it reads one per element (the next block's, of this row or the next, follows in
// memory).  Integer formats with a scale that is not finite go element by element through decode_store,
// which gives NaN results their canonical bits, and so do the last elements, whose dwords would reach
// past the storage.
typedef unsigned un_u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned un_u32x4 __attribute__((ext_vector_type(4)));

// fp32 value of a payload in the low bits of p (upper bits ignored).
template <int FMT>
__device__ __forceinline__ float payload_value(uint32_t p) {
  if constexpr (FMT == TGM_FMT_INT4) return (float)((int32_t)(p << 28) >> 28);
  else if constexpr (FMT == TGM_FMT_UINT4) return (float)(p & 15u);
  else {
    // the magnitude bits under an fp32 exponent field that is too small by 127 - bias: one exact
    // multiplication by a power of two puts normal and subnormal payloads in place
    constexpr int M = FMT == TGM_FMT_FP4_E2M1 ? 1 : FMT == TGM_FMT_FP6_E2M3 ? 3 : 2;
    constexpr int B = FMT == TGM_FMT_FP4_E2M1 ? 4 : 6, BIAS = FMT == TGM_FMT_FP6_E3M2 ? 3 : 1;
    const float mag = bits_f32((p & ((1u << (B - 1)) - 1u)) << (23 - M)) * bits_f32((unsigned)(254 - BIAS) << 23);
    return bits_f32(f32_bits(mag) | ((p << (32 - B)) & 0x80000000u));
  }
}

template <int FMT, int ODT>
struct UnpackChunk {
  static constexpr int kBits = FMT == TGM_FMT_FP6_E2M3 || FMT == TGM_FMT_FP6_E3M2 ? 6 : 4;
  static constexpr int kElems = ODT == TGM_F32 ? 4 : 8;  // elements of a lane: one 16-byte store
  static constexpr int kWords = kBits == 6 ? 2 : 1;      // dwords that hold them, wherever they start
};

// U: chunks of a thread, 256 apart.
template <int FMT, int ODT, int U>
__global__ void __launch_bounds__(256) unpack_vec(const uint8_t* __restrict__ data, int64_t nbytes, int64_t count,
                                                  uint32_t chunks, uint32_t k, const void* __restrict__ scales, int sdt,
                                                  uint32_t nblk, uint32_t bs, void* __restrict__ out) {
  using C = UnpackChunk<FMT, ODT>;
  constexpr bool INT = FMT == TGM_FMT_INT4 || FMT == TGM_FMT_UINT4;
  constexpr int B = C::kBits, E = C::kElems, W = C::kWords;
  const uint32_t c0 = blockIdx.x * (256u * U) + threadIdx.x;
  const FormatInfo f = format_info(FMT);
  uint32_t raw[U][W];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t c = c0 + 256u * u;
    if (c < chunks) {
      const uint32_t* p = (const uint32_t*)data + (((uint64_t)c * (E * B)) >> 5);
#pragma unroll
      for (int w = 0; w < W; ++w) raw[u][w] = p[w];
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t c = c0 + 256u * u;
    if (c >= chunks) break;
    const uint32_t i0 = c * E;  // count < 2^32
    float sc[E];
    uint32_t row = 0, col = 0;
    bool finite = true;
    if (scales) {
      row = i0 / k;
      col = i0 - row * k;
      const uint32_t blk = col / bs;
      uint32_t left = bs - (col - blk * bs);  // elements to the end of the scale block
      int64_t si = (int64_t)row * nblk + blk;
      const float s0 = load_f32(scales, sdt, si);
#pragma unroll
      for (int j = 0; j < E; ++j) sc[j] = s0;
      if (left < E || k - col < E) {
        uint32_t cj = col;
#pragma unroll
        for (int j = 1; j < E; ++j) {
          const bool wrap = ++cj == k;
          if (--left == 0 || wrap) {
            left = bs;
            ++si;
          }
          if (wrap) cj = 0;
          sc[j] = load_f32(scales, sdt, si);
        }
      }
      if (INT)
#pragma unroll
        for (int j = 0; j < E; ++j) finite = finite && fabsf(sc[j]) < __builtin_inff();
    }
    const int sh = (int)((c * (uint32_t)(E * B)) & 31u);
    uint32_t pay[E];
    const uint64_t v64 = ((W == 2 ? (uint64_t)raw[u][W - 1] << 32 : 0ull) | raw[u][0]) >> sh;
#pragma unroll
    for (int j = 0; j < E; ++j) pay[j] = (uint32_t)(v64 >> (j * B));
    if (finite) {
      float v[E];
#pragma unroll
      for (int j = 0; j < E; ++j) {
        v[j] = payload_value<FMT>(pay[j]);
        if (scales) v[j] *= sc[j];
        if constexpr (ODT == TGM_F16) keep_product(v[j]);
      }
      un_u32x4 o;
      if constexpr (ODT == TGM_F32) {
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = f32_bits(v[j]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (ODT == TGM_BF16) o[j] = bf16x2_bits(v[2 * j], v[2 * j + 1]);
          else
            o[j] = __builtin_bit_cast(unsigned short, (_Float16)v[2 * j]) |
                   ((unsigned)__builtin_bit_cast(unsigned short, (_Float16)v[2 * j + 1]) << 16);
        }
      }
      __builtin_nontemporal_store(o, (un_u32x4*)out + c);
    } else {
#pragma unroll 1
      for (int j = 0; j < E; ++j) {
        decode_store<float>((uint32_t)(v64 >> (j * B)) & ((1u << B) - 1u), FMT, f, true,
                            load_f32(scales, sdt, (int64_t)row * nblk + col / bs), out, ODT, (int64_t)i0 + j);
        if (++col == k) { col = 0; ++row; }
      }
    }
  }
  // the last elements (fewer than 256), by the last block
  const int64_t i = (int64_t)chunks * E + threadIdx.x;
  if (blockIdx.x == gridDim.x - 1 && i < count) {
    const uint32_t p = payload_at(data, nbytes, i, B), row = (uint32_t)i / k, col = (uint32_t)i - row * k;
    decode_store<float>(p, FMT, f, scales != nullptr,
                        scales ? load_f32(scales, sdt, (int64_t)row * nblk + col / bs) : 1.f, out, ODT, i);
  }
}

template <int FMT, int ODT>
void launch_unpack_vec(hipStream_t s, const void* data, int64_t nbytes, int64_t count, int64_t k, const void* scales,
                       int sdt, int64_t nblk, int64_t bs, void* out) {
  using C = UnpackChunk<FMT, ODT>;
  // chunk c reads kWords dwords from the dword that holds its first payload: at most bytes
  // c * elems * bits / 8 .. + 4 * kWords, which must lie inside the storage
  const int64_t bits = C::kElems * C::kBits, spare = nbytes - 4 * C::kWords;
  const int64_t inside = spare < 0 ? 0 : spare * 8 / bits + 1;
  const int64_t chunks = count / C::kElems < inside ? count / C::kElems : inside;
  // four chunks per thread keep four loads in flight; one where that would leave the chip's 1024 SIMDs
  // without two waves each (51,600 elements of FP4, rows ending inside chunks: 10.7 against 4.2 us)
  const int per = chunks >= 256 * 4 * 512 ? 4 : 1;
  const dim3 grid((unsigned)(chunks > 0 ? (chunks + 256 * per - 1) / (256 * per) : 1));
#define TGM_UNPACK_VEC(U)                                                                                         \
  hipLaunchKernelGGL((unpack_vec<FMT, ODT, U>), grid, dim3(256), 0, s, (const uint8_t*)data, nbytes, count,        \
                     (uint32_t)chunks, (uint32_t)k, scales, sdt, (uint32_t)nblk, (uint32_t)bs, out)
  if (per == 4) TGM_UNPACK_VEC(4);
  else TGM_UNPACK_VEC(1);
#undef TGM_UNPACK_VEC
}

template <int FMT>
void launch_unpack_vec(hipStream_t s, const void* data, int64_t nbytes, int64_t count, int64_t k, const void* scales,
                       int sdt, int64_t nblk, int64_t bs, void* out, int odt) {
  if (odt == TGM_BF16) launch_unpack_vec<FMT, TGM_BF16>(s, data, nbytes, count, k, scales, sdt, nblk, bs, out);
  else if (odt == TGM_F16) launch_unpack_vec<FMT, TGM_F16>(s, data, nbytes, count, k, scales, sdt, nblk, bs, out);
  else launch_unpack_vec<FMT, TGM_F32>(s, data, nbytes, count, k, scales, sdt, nblk, bs, out);
}

}  // namespace tgm

using namespace tgm;

extern "C" int tgm_abi_version(void) { return TGM_ABI_VERSION; }

extern "C" const char* tgm_last_error(void) { return g_last_error; }

extern "C" int tgm_device_arch(int ordinal, char* out, int64_t len) {
  clear_error();
  TGM_CHECK_ARG(out && len > 0, "null output");
  hipDeviceProp_t prop;
  const hipError_t e = hipGetDeviceProperties(&prop, ordinal);
  if (e != hipSuccess) {
    set_error("hipGetDeviceProperties(%d) failed: %s", ordinal, hipGetErrorString(e));
    return (int)e;
  }
  snprintf(out, (size_t)len, "%s", prop.gcnArchName);
  return TGM_OK;
}

extern "C" int tgm_unpack(const void* data, int64_t nbytes, int fmt, int64_t count, int64_t k, const void* scales,
                          int scale_dtype, int64_t block_size, void* out, int out_dtype, void* stream) {
  clear_error();
  TGM_CHECK_ARG(valid_format(fmt), "unknown packed format %d", fmt);
  TGM_CHECK_ARG(count >= 0 && k >= 1 && block_size >= 1 && nbytes >= 0, "invalid unpack sizes");
  const int bits = format_info(fmt).bits;
  TGM_CHECK_ARG(nbytes >= (count * bits + 7) / 8, "packed storage is smaller than the declared shape");
  TGM_CHECK_ARG(dtype_size(out_dtype) > 0 && out_dtype != TGM_E8M0, "invalid output dtype %d", out_dtype);
  TGM_CHECK_ARG(!scales || (dtype_size(scale_dtype) > 0), "invalid scale dtype %d", scale_dtype);
  if (count == 0) return TGM_OK;
  int fp8_target = 0;
  if (!scales && !is_int_format(fmt)) {
    // FP8_CANDIDATES (dx12.py:11): fp4 -> {e4m3, e5m2}; e2m3 -> {e4m3}; e3m2 -> {e4m3, e5m2}
    if (out_dtype == TGM_FP8E4M3) fp8_target = 1;
    if (out_dtype == TGM_FP8E5M2 && fmt != TGM_FMT_FP6_E2M3) fp8_target = 2;
  }
  const int64_t nblk = (k + block_size - 1) / block_size;
  const bool wide = scales && (scale_dtype == TGM_F64 || out_dtype == TGM_F64);
  const int64_t threads = (count + 7) / 8;
  int64_t blocks = (threads + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipStream_t s = (hipStream_t)stream;
  // Floating outputs of up to 32 bits from aligned storage: the vector kernel (32-bit element indices).
  // fp64 scales or results, integer and FP8 results, odd addresses and larger arrays keep the scalar one.
  if (!wide && (out_dtype == TGM_BF16 || out_dtype == TGM_F16 || out_dtype == TGM_F32) && count < (1ll << 32) - 65536 &&
      k < (1ll << 32) && block_size < (1ll << 31) && (uintptr_t)data % 4 == 0 && (uintptr_t)out % 16 == 0) {
#define TGM_UNPACK_FMT(F) \
  case F: launch_unpack_vec<F>(s, data, nbytes, count, k, scales, scale_dtype, nblk, block_size, out, out_dtype); break
    switch (fmt) {
      TGM_UNPACK_FMT(TGM_FMT_INT4);
      TGM_UNPACK_FMT(TGM_FMT_UINT4);
      TGM_UNPACK_FMT(TGM_FMT_FP4_E2M1);
      TGM_UNPACK_FMT(TGM_FMT_FP6_E2M3);
      default: launch_unpack_vec<TGM_FMT_FP6_E3M2>(s, data, nbytes, count, k, scales, scale_dtype, nblk, block_size, out, out_dtype);
    }
#undef TGM_UNPACK_FMT
    return launch_status("tgm_unpack");
  }
  if (wide)
    hipLaunchKernelGGL(unpack_kernel<double>, dim3((unsigned)blocks), dim3(256), 0, s, (const uint8_t*)data, nbytes,
                       fmt, count, k, scales, scale_dtype, nblk, block_size, out, out_dtype, fp8_target);
  else
    hipLaunchKernelGGL(unpack_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, s, (const uint8_t*)data, nbytes,
                       fmt, count, k, scales, scale_dtype, nblk, block_size, out, out_dtype, fp8_target);
  return launch_status("tgm_unpack");
}
