// Rowwise quantization codecs for gfx950: the formats the nbit lookup reads.
//
// Semantics: fbgemm_gpu FloatToFused8BitRowwiseQuantized /
// Fused8BitRowwiseQuantizedToFloat and FloatToFusedNBitRowwiseQuantizedSBHalf
// / FusedNBitRowwiseQuantizedSBHalfToFloat (upstream src/quantize_ops/,
// recalled), i.e. FBGEMM's FloatOrHalfToFused8BitRowwiseQuantizedSBFloat and
// FloatOrHalfToFusedNBitRowwiseQuantizedSBHalf (torch/include/fbgemm/
// QuantUtils.h declares them; torch's quantized::embedding_bag_{byte,4bit,
// 2bit}_prepack call them):
//   8-bit:  per row min m, max M; scale = (M - m) / 255, bias = m,
//           q = rint((x - m) * (255 / (M - m + 1e-8))); row = codes, fp32
//           scale, fp32 bias (D + 8 bytes).
//   N-bit:  bias = half(m); scale = half((M - bias) / (2^b - 1)) (1 if the
//           range is 0 or the scale underflows); q = clamp(rint((x - bias) *
//           (1 / scale)), 0, 2^b - 1), packed low bits first; row = codes,
//           fp16 scale, fp16 bias (ceil(D*b/8) + 4 bytes).
//   dequantize: x = q * scale + bias (one fma).
//
// Bound: one read and one write of every row; nothing else is large.  A group
// of G lanes takes a row, each lane a whole 32-bit word of its codes: the row's
// elements arrive with 16-byte loads, stay in registers between the min/max
// and the codes (one read), and the codes leave as words.  A group keeps
// several rows in flight.  Rows of any byte size start at any byte, so the
// word stores and code loads are unaligned ones; only a row's last, partial
// word is written by bytes.  Measured, encode + decode to fp32, against one
// wave per row with element loads and byte stores: 4-bit 500,000 x 120 308 ->
// 118 us (4.6 TB/s of rows read and written), x 37 240 -> 58; 8-bit x 128
// 368 -> 142; 2-bit x 64 279 -> 59; fused 8-bit x 128 284 -> 136.
#include <type_traits>

#include "mx_common.h"

namespace mx {
namespace {

template <typename T>
__device__ __forceinline__ float to_f32(T v);
template <>
__device__ __forceinline__ float to_f32<float>(float v) {
  return v;
}
template <>
__device__ __forceinline__ float to_f32<__half>(__half v) {
  return __half2float(v);
}

template <int G>
__device__ __forceinline__ float group_min(float v) {
#pragma unroll
  for (int m = G / 2; m >= 1; m >>= 1) v = fminf(v, __shfl_xor(v, m, 64));
  return v;
}
template <int G>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
  for (int m = G / 2; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
  return v;
}

__device__ __forceinline__ float round_to_half(float v) { return __half2float(__float2half_rn(v)); }

// A row's codec: scale and bias from its range, one element's code, and the
// scale and bias as the row ends with them.  BITS 8 with FUSED8: the 8-bit
// format (fp32 scale and bias); else the N-bit format (fp16).
template <int BITS, bool FUSED8>
struct RowCodec {
  static constexpr int kTail = FUSED8 ? 8 : 4;  // bytes after the codes
  static constexpr int kMax = (1 << BITS) - 1;
  float scale, bias, inv;
  __device__ __forceinline__ void set(float mn, float mx) {
    if constexpr (FUSED8) {
      const float range = mx - mn;
      scale = range / 255.0f;
      inv = 255.0f / (range + 1e-8f);
      bias = mn;
    } else {
      bias = round_to_half(mn);
      const float range = mx - bias;
      scale = range == 0.0f ? 1.0f : range / static_cast<float>(kMax);
      scale = round_to_half(scale);
      if (scale == 0.0f) scale = 1.0f;  // underflow in fp16
      inv = 1.0f / scale;
      if (__builtin_isinf(inv)) {
        scale = 1.0f;
        inv = 1.0f;
      }
    }
  }
  __device__ __forceinline__ uint32_t code(float x) const {
    float q = __builtin_rintf(__fmul_rn(x - bias, inv));
    if constexpr (FUSED8) return static_cast<uint8_t>(q);
    q = q < 0.0f ? 0.0f : (q > static_cast<float>(kMax) ? static_cast<float>(kMax) : q);
    return static_cast<uint32_t>(q);
  }
  __device__ __forceinline__ void store(uint8_t* o) const {
    if constexpr (FUSED8) {
      __builtin_memcpy(o, &scale, 4);
      __builtin_memcpy(o + 4, &bias, 4);
    } else {
      const __half hs = __float2half_rn(scale), hb = __float2half_rn(bias);
      const uint32_t w = static_cast<uint32_t>(__half_as_ushort(hs)) |
                         (static_cast<uint32_t>(__half_as_ushort(hb)) << 16);
      __builtin_memcpy(o, &w, 4);
    }
  }
  __device__ __forceinline__ void load(const uint8_t* x) {
    if constexpr (FUSED8) {
      __builtin_memcpy(&scale, x, 4);
      __builtin_memcpy(&bias, x + 4, 4);
    } else {
      uint32_t w;
      __builtin_memcpy(&w, x, 4);
      scale = __half2float(__ushort_as_half(static_cast<uint16_t>(w & 0xffffu)));
      bias = __half2float(__ushort_as_half(static_cast<uint16_t>(w >> 16)));
    }
  }
};

// N elements (4, 8 or 16) from p, at the element type's own alignment.
template <int N>
__device__ __forceinline__ void load_elems(const float* p, float (&x)[N]) {
  typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(p + i);
    x[i] = v.x;
    x[i + 1] = v.y;
    x[i + 2] = v.z;
    x[i + 3] = v.w;
  }
}
template <int N>
__device__ __forceinline__ void load_elems(const __half* p, float (&x)[N]) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2), aligned(2)));
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    const u32x2 v = *reinterpret_cast<const u32x2*>(p + i);
    x[i] = __half2float(__ushort_as_half(static_cast<uint16_t>(v.x & 0xffffu)));
    x[i + 1] = __half2float(__ushort_as_half(static_cast<uint16_t>(v.x >> 16)));
    x[i + 2] = __half2float(__ushort_as_half(static_cast<uint16_t>(v.y & 0xffffu)));
    x[i + 3] = __half2float(__ushort_as_half(static_cast<uint16_t>(v.y >> 16)));
  }
}

// Encodes R consecutive rows per G-lane group; lane k owns code words
// k + q*G (q < Q), E elements each; D <= G*Q*E.
template <typename T, int BITS, bool FUSED8, int G, int Q, int R>
__global__ void __launch_bounds__(256)
    quantize_rows_kernel(const T* __restrict__ in, int64_t rows, int32_t D,
                         uint8_t* __restrict__ out) {
  using C = RowCodec<BITS, FUSED8>;
  constexpr int E = 32 / BITS;
  const int k = threadIdx.x % G;
  const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * (256 / G) + threadIdx.x / G) * R;
  const int32_t nbytes = (D * BITS + 7) / 8;
  float x[R][Q][E];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int32_t c = (k + q * G) * E;
      if (r0 + i >= rows || c >= D) continue;
      const T* p = in + (r0 + i) * D + c;
      if (c + E <= D) {
        load_elems<E>(p, x[i][q]);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) x[i][q][e] = c + e < D ? to_f32(p[e]) : 0.0f;
      }
    }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (r0 + i >= rows) break;  // whole group
    float lo = INFINITY, hi = -INFINITY;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((k + q * G) * E + e < D) {
          lo = fminf(lo, x[i][q][e]);
          hi = fmaxf(hi, x[i][q][e]);
        }
    C codec;
    codec.set(group_min<G>(lo), group_max<G>(hi));
    uint8_t* o = out + (r0 + i) * (nbytes + C::kTail);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int32_t c = (k + q * G) * E, at = (k + q * G) * 4;
      if (c >= D) continue;
      uint32_t w = 0u;
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (c + e < D) w |= codec.code(x[i][q][e]) << (e * BITS);
      if (at + 4 <= nbytes) {
        __builtin_memcpy(o + at, &w, 4);
      } else {
        for (int b = 0; at + b < nbytes; ++b) o[at + b] = static_cast<uint8_t>(w >> (8 * b));
      }
    }
    if (k == 0) codec.store(o + nbytes);
  }
}

// Rows wider than the lanes hold: one wave per row, which reads it twice
// (min/max, then codes; the second read hits L2).
template <typename T, int BITS, bool FUSED8>
__global__ void __launch_bounds__(256)
    quantize_wide_kernel(const T* __restrict__ in, int64_t rows, int64_t D,
                         uint8_t* __restrict__ out) {
  using C = RowCodec<BITS, FUSED8>;
  constexpr int kPerByte = 8 / BITS;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int lane = threadIdx.x & 63;
  const int64_t nbytes = (D + kPerByte - 1) / kPerByte;
  const T* x = in + r * D;
  uint8_t* o = out + r * (nbytes + C::kTail);
  float lo = INFINITY, hi = -INFINITY;
  for (int64_t j = lane; j < D; j += 64) {
    const float v = to_f32(x[j]);
    lo = fminf(lo, v);
    hi = fmaxf(hi, v);
  }
  C codec;
  codec.set(group_min<64>(lo), group_max<64>(hi));
  for (int64_t p = lane; p < nbytes; p += 64) {
    uint32_t byte = 0;
    for (int e = 0; e < kPerByte; ++e) {
      const int64_t j = p * kPerByte + e;
      if (j >= D) break;
      byte |= codec.code(to_f32(x[j])) << (e * BITS);
    }
    o[p] = static_cast<uint8_t>(byte);
  }
  if (lane == 0) codec.store(o + nbytes);
}

// Decodes R consecutive rows per G-lane group, four elements per lane and
// step, so that consecutive lanes store consecutive 16 (fp16: 8) bytes.  The
// codes of a row's last, partial step are read past its end into its own
// scale and bias, never past the row.
template <int BITS, bool FUSED8, bool F16, int G, int R>
__global__ void __launch_bounds__(256)
    dequantize_rows_kernel(const uint8_t* __restrict__ in, int64_t rows, int64_t D,
                           void* __restrict__ out) {
  using C = RowCodec<BITS, FUSED8>;
  constexpr int kStep = 4 * BITS / 8;  // bytes of four codes
  const int k = threadIdx.x % G;
  const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * (256 / G) + threadIdx.x / G) * R;
  const int64_t nbytes = (D * BITS + 7) / 8, stride = nbytes + C::kTail;
  C codec[R];
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (r0 + i < rows) codec[i].load(in + (r0 + i) * stride + nbytes);
  for (int64_t c = 4 * k; c < D; c += 4 * G) {
    uint32_t w[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      w[i] = 0u;
      if (r0 + i < rows) __builtin_memcpy(&w[i], in + (r0 + i) * stride + c * BITS / 8, kStep);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (r0 + i >= rows) break;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = __builtin_fmaf(static_cast<float>((w[i] >> (e * BITS)) & ((1u << BITS) - 1u)),
                              codec[i].scale, codec[i].bias);
      const int64_t o = (r0 + i) * D + c;
      if (c + 4 <= D) {
        if constexpr (F16) {
          typedef uint32_t u32x2 __attribute__((ext_vector_type(2), aligned(2)));
          const __half2 a = __floats2half2_rn(fp32_value(v[0]), fp32_value(v[1]));
          const __half2 b = __floats2half2_rn(fp32_value(v[2]), fp32_value(v[3]));
          *reinterpret_cast<u32x2*>(reinterpret_cast<__half*>(out) + o) =
              u32x2{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
        } else {
          typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + o) =
              f32x4{v[0], v[1], v[2], v[3]};
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (c + e >= D) break;
          if constexpr (F16)
            reinterpret_cast<__half*>(out)[o + e] = __float2half_rn(fp32_value(v[e]));
          else
            reinterpret_cast<float*>(out)[o + e] = v[e];
        }
      }
    }
  }
}

template <int V>
using Int = std::integral_constant<int, V>;

// Rows per group: several in flight pay where the grid fills the chip anyway, in
// a small batch they only follow each other in time (1000 rows of 64, 4 bits,
// encoded and decoded twice: 9.7 us with four per group, 6.3 with one; 16,000
// rows 10.8 and 7.9; 64,000 of 128 columns, past the line: 26).
bool few_rows(int64_t rows, int g, int r) {
  return ceil_div(rows, 256 / g * r) < 2 * static_cast<int64_t>(num_cus());
}

template <typename T, int BITS, bool FUSED8>
void launch_quantize(const void* in, int64_t rows, int64_t D, uint8_t* out, hipStream_t s) {
  constexpr int E = 32 / BITS, R = E == 16 ? 2 : 4;
  const auto* x = static_cast<const T*>(in);
  const int64_t words = ceil_div(D, E);
  auto launch = [&](auto kernel, int per_block) {
    kernel<<<dim3(static_cast<uint32_t>(ceil_div(rows, per_block))), 256, 0, s>>>(
        x, rows, static_cast<int32_t>(D), out);
  };
  auto go = [&](auto g, auto q, auto r) {
    constexpr int G = decltype(g)::value, Q = decltype(q)::value, RR = decltype(r)::value;
    if (RR > 1 && few_rows(rows, G, RR))
      launch(quantize_rows_kernel<T, BITS, FUSED8, G, Q, 1>, 256 / G);
    else
      launch(quantize_rows_kernel<T, BITS, FUSED8, G, Q, RR>, 256 / G * RR);
  };
  if (words <= 8)
    go(Int<8>{}, Int<1>{}, Int<R>{});
  else if (words <= 16)
    go(Int<16>{}, Int<1>{}, Int<R>{});
  else if (words <= 32)
    go(Int<32>{}, Int<1>{}, Int<R>{});
  else if (words <= 64)
    go(Int<64>{}, Int<1>{}, Int<R>{});
  else if (words <= 128)
    go(Int<64>{}, Int<2>{}, Int<R / 2>{});
  else if (words <= 256)
    go(Int<64>{}, Int<4>{}, Int<1>{});
  else
    quantize_wide_kernel<T, BITS, FUSED8>
        <<<dim3(static_cast<uint32_t>(ceil_div(rows, 4))), 256, 0, s>>>(x, rows, D, out);
}

template <int BITS, bool FUSED8, bool F16>
void launch_dequantize(const uint8_t* in, int64_t rows, int64_t D, void* out, hipStream_t s) {
  constexpr int R = 4;
  auto launch = [&](auto kernel, int per_block) {
    kernel<<<dim3(static_cast<uint32_t>(ceil_div(rows, per_block))), 256, 0, s>>>(in, rows, D,
                                                                                  out);
  };
  auto go = [&](auto g) {
    constexpr int G = decltype(g)::value;
    if (few_rows(rows, G, R))
      launch(dequantize_rows_kernel<BITS, FUSED8, F16, G, 1>, 256 / G);
    else
      launch(dequantize_rows_kernel<BITS, FUSED8, F16, G, R>, 256 / G * R);
  };
  if (D <= 32)
    go(Int<8>{});
  else if (D <= 64)
    go(Int<16>{});
  else if (D <= 128)
    go(Int<32>{});
  else
    go(Int<64>{});
}

// hfp8 codecs: elementwise, grid-stride.
__global__ void __launch_bounds__(256)
    float_to_hfp8_kernel(const float* __restrict__ in, int64_t n, Hfp8 f, float clamp,
                         uint8_t* __restrict__ out) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * 256)
    out[i] = static_cast<uint8_t>(f.encode(in[i], clamp));
}

__global__ void __launch_bounds__(256)
    hfp8_to_float_kernel(const uint8_t* __restrict__ in, int64_t n, Hfp8 f,
                         float* __restrict__ out) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * 256)
    out[i] = f.decode(in[i]);
}

dim3 elementwise_grid(int64_t n) {
  const int64_t b = ceil_div(n, 256);
  return dim3(static_cast<uint32_t>(b < 8192 ? b : 8192));
}

}  // namespace
}  // namespace mx

using namespace mx;

extern "C" int mx_float_to_hfp8(const float* in, int64_t n, int32_t ebits, int32_t exponent_bias,
                                float max_pos, uint8_t* out, void* stream) {
  clear_error();
  MX_REQUIRE(n >= 0, "negative size");
  MX_REQUIRE(hfp8_format_ok(ebits, exponent_bias),
             "hfp8 needs 1 <= ebits <= 7 and 0 <= exponent_bias <= 120 (got %d, %d)", ebits,
             exponent_bias);
  MX_REQUIRE(max_pos > 0.0f, "max_pos must be positive");
  if (n == 0) return MX_OK;
  MX_REQUIRE(in && out, "null pointer argument");
  const Hfp8 f = Hfp8::make(ebits, exponent_bias);
  float_to_hfp8_kernel<<<elementwise_grid(n), 256, 0, as_stream(stream)>>>(
      in, n, f, max_pos < f.max_code ? max_pos : f.max_code, out);
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_hfp8_to_float(const uint8_t* in, int64_t n, int32_t ebits,
                                int32_t exponent_bias, float* out, void* stream) {
  clear_error();
  MX_REQUIRE(n >= 0, "negative size");
  MX_REQUIRE(hfp8_format_ok(ebits, exponent_bias),
             "hfp8 needs 1 <= ebits <= 7 and 0 <= exponent_bias <= 120 (got %d, %d)", ebits,
             exponent_bias);
  if (n == 0) return MX_OK;
  MX_REQUIRE(in && out, "null pointer argument");
  hfp8_to_float_kernel<<<elementwise_grid(n), 256, 0, as_stream(stream)>>>(
      in, n, Hfp8::make(ebits, exponent_bias), out);
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_quantize_fused8bit_rowwise(const void* in, int32_t in_dtype, int64_t rows,
                                             int64_t D, uint8_t* out, void* stream) {
  clear_error();
  MX_REQUIRE(rows >= 0 && D >= 0, "negative size");
  MX_REQUIRE(in_dtype == MX_DTYPE_F32 || in_dtype == MX_DTYPE_F16, "input must be fp32 or fp16");
  MX_REQUIRE(ceil_div(rows, 4) <= 0x7fffffffll, "too many rows");
  if (rows == 0) return MX_OK;
  MX_REQUIRE(in && out, "null pointer argument");
  auto* s = as_stream(stream);
  if (in_dtype == MX_DTYPE_F32)
    launch_quantize<float, 8, true>(in, rows, D, out, s);
  else
    launch_quantize<__half, 8, true>(in, rows, D, out, s);
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_dequantize_fused8bit_rowwise(const uint8_t* in, int64_t rows, int64_t D,
                                               void* out, int32_t out_dtype, void* stream) {
  clear_error();
  MX_REQUIRE(rows >= 0 && D >= 0, "negative size");
  MX_REQUIRE(out_dtype == MX_DTYPE_F32 || out_dtype == MX_DTYPE_F16, "output must be fp32 or fp16");
  MX_REQUIRE(ceil_div(rows, 4) <= 0x7fffffffll, "too many rows");
  if (rows == 0 || D == 0) return MX_OK;
  MX_REQUIRE(in && out, "null pointer argument");
  if (out_dtype == MX_DTYPE_F16)
    launch_dequantize<8, true, true>(in, rows, D, out, as_stream(stream));
  else
    launch_dequantize<8, true, false>(in, rows, D, out, as_stream(stream));
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_quantize_fused_nbit_rowwise(const void* in, int32_t in_dtype, int64_t rows,
                                              int64_t D, int32_t bit_rate, uint8_t* out,
                                              void* stream) {
  clear_error();
  MX_REQUIRE(rows >= 0 && D >= 0, "negative size");
  MX_REQUIRE(bit_rate == 2 || bit_rate == 4 || bit_rate == 8, "bit_rate must be 2, 4 or 8");
  MX_REQUIRE(in_dtype == MX_DTYPE_F32 || in_dtype == MX_DTYPE_F16, "input must be fp32 or fp16");
  MX_REQUIRE(ceil_div(rows, 4) <= 0x7fffffffll, "too many rows");
  if (rows == 0) return MX_OK;
  MX_REQUIRE(in && out, "null pointer argument");
  auto* s = as_stream(stream);
  auto go = [&](auto bits) {
    constexpr int kBits = decltype(bits)::value;
    if (in_dtype == MX_DTYPE_F32)
      launch_quantize<float, kBits, false>(in, rows, D, out, s);
    else
      launch_quantize<__half, kBits, false>(in, rows, D, out, s);
  };
  if (bit_rate == 2)
    go(std::integral_constant<int, 2>{});
  else if (bit_rate == 4)
    go(std::integral_constant<int, 4>{});
  else
    go(std::integral_constant<int, 8>{});
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_dequantize_fused_nbit_rowwise(const uint8_t* in, int64_t rows, int64_t D,
                                                int32_t bit_rate, void* out, int32_t out_dtype,
                                                void* stream) {
  clear_error();
  MX_REQUIRE(rows >= 0 && D >= 0, "negative size");
  MX_REQUIRE(bit_rate == 2 || bit_rate == 4 || bit_rate == 8, "bit_rate must be 2, 4 or 8");
  MX_REQUIRE(out_dtype == MX_DTYPE_F32 || out_dtype == MX_DTYPE_F16, "output must be fp32 or fp16");
  MX_REQUIRE(ceil_div(rows, 4) <= 0x7fffffffll, "too many rows");
  if (rows == 0 || D == 0) return MX_OK;
  MX_REQUIRE(in && out, "null pointer argument");
  auto go = [&](auto bits) {
    constexpr int kBits = decltype(bits)::value;
    if (out_dtype == MX_DTYPE_F16)
      launch_dequantize<kBits, false, true>(in, rows, D, out, as_stream(stream));
    else
      launch_dequantize<kBits, false, false>(in, rows, D, out, as_stream(stream));
  };
  if (bit_rate == 2)
    go(std::integral_constant<int, 2>{});
  else if (bit_rate == 4)
    go(std::integral_constant<int, 4>{});
  else
    go(std::integral_constant<int, 8>{});
  MX_LAUNCH_CHECK();
  return MX_OK;
}
