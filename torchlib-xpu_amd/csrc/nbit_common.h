// Shared by the pooled and the sequence nbit lookups: the call's arguments, the
// TBE row layout, code loads and the output conversions.
#pragma once

#include "mx_common.h"

namespace mx {
namespace {

struct NbitArgs {
  const uint8_t* W;
  const int64_t* w_off;
  const uint8_t* tys;
  const int32_t* D_off;
  const void* idx;
  const void* off;
  const float* iw;
  void* out;
  int64_t B;
  int64_t Bp;  // B rounded up to bags-per-block
  int64_t total_D;
  int64_t nwaves;
  int32_t T;
  int32_t pooling;
  int32_t row_align;
  int32_t out_kind;        // output element: 0 fp32, 1 fp16, 2 bf16
  int32_t served;          // bit ty set: the call launches type ty
  Hfp8 fp8;                // FP8 tables' format (when served)
  uint32_t nchk;           // trailing blocks that check the tables (T in the first launch, else 0)
  unsigned int* mailbox;   // host-visible status words of the device, may be null
};

// A table the call can serve: its type has a launch, its D is not negative,
// and its codes fill whole bytes (INT4: D even, INT2: D a multiple of 4; the
// row holds D*bits/8 code bytes, rounded down).
template <int TY>
__device__ __forceinline__ bool whole_bytes(int32_t D) {
  if constexpr (TY == MX_SPARSE_INT4) return (D & 1) == 0;
  if constexpr (TY == MX_SPARSE_INT2) return (D & 3) == 0;
  return true;
}

__device__ __host__ __forceinline__ int64_t row_bytes_of(int32_t ty, int32_t D, int32_t align) {
  int64_t u;
  switch (ty) {
    case MX_SPARSE_FP32: u = 4ll * D; break;
    case MX_SPARSE_FP16: u = 2ll * D; break;
    case MX_SPARSE_INT8: u = D + 4ll; break;
    case MX_SPARSE_INT4: u = D / 2 + 4ll; break;
    case MX_SPARSE_INT2: u = D / 4 + 4ll; break;
    case MX_SPARSE_FP8: u = D; break;
    default: return -1;
  }
  if (align > 1) u = (u + align - 1) / align * align;
  return u;
}

// Rows start at 4-byte boundaries (the kernels read codes and qparams in
// 4-byte words): the table's first byte and its row stride are multiples of 4.
__device__ __host__ __forceinline__ bool rows_aligned(int64_t w_off, int64_t stride) {
  return ((w_off | stride) & 3) == 0;
}

__device__ __forceinline__ bool table_ok(int32_t ty, int32_t D, int32_t served, int64_t w_off,
                                         int32_t align) {
  if (ty < 0 || ty > MX_SPARSE_FP8 || ty == MX_SPARSE_BF16 || ((served >> ty) & 1) == 0 || D < 0)
    return false;
  if (!rows_aligned(w_off, row_bytes_of(ty, D, align))) return false;
  if (ty == MX_SPARSE_INT4) return whole_bytes<MX_SPARSE_INT4>(D);
  if (ty == MX_SPARSE_INT2) return whole_bytes<MX_SPARSE_INT2>(D);
  return true;
}

template <int TY>
struct TyInfo;
template <>
struct TyInfo<MX_SPARSE_FP32> {
  static constexpr int kBits = 32;
  static constexpr bool kQ = false;
};
template <>
struct TyInfo<MX_SPARSE_FP16> {
  static constexpr int kBits = 16;
  static constexpr bool kQ = false;
};
template <>
struct TyInfo<MX_SPARSE_INT8> {
  static constexpr int kBits = 8;
  static constexpr bool kQ = true;
};
template <>
struct TyInfo<MX_SPARSE_INT4> {
  static constexpr int kBits = 4;
  static constexpr bool kQ = true;
};
template <>
struct TyInfo<MX_SPARSE_INT2> {
  static constexpr int kBits = 2;
  static constexpr bool kQ = true;
};
template <>
struct TyInfo<MX_SPARSE_FP8> {
  static constexpr int kBits = 8;
  static constexpr bool kQ = false;
};

typedef uint32_t u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));

// Loads BPL bytes (a power of two) starting at p into 32-bit words.
template <int BPL>
__device__ __forceinline__ void load_codes(const uint8_t* p, uint32_t (&w)[BPL >= 4 ? BPL / 4 : 1]) {
  if constexpr (BPL == 1) {
    w[0] = *p;
  } else if constexpr (BPL == 2) {
    w[0] = *reinterpret_cast<const uint16_t*>(p);
  } else if constexpr (BPL == 4) {
    w[0] = *reinterpret_cast<const uint32_t*>(p);
  } else if constexpr (BPL == 8) {
    const u32x2a4 v = *reinterpret_cast<const u32x2a4*>(p);
    w[0] = v.x;
    w[1] = v.y;
  } else {
#pragma unroll
    for (int q = 0; q < BPL / 16; ++q) {
      const u32x4a4 v = *reinterpret_cast<const u32x4a4*>(p + 16 * q);
      w[4 * q + 0] = v.x;
      w[4 * q + 1] = v.y;
      w[4 * q + 2] = v.z;
      w[4 * q + 3] = v.w;
    }
  }
}

template <typename I>
__device__ __forceinline__ int64_t idx_at(const void* p, int64_t i) {
  return static_cast<int64_t>(reinterpret_cast<const I*>(p)[i]);
}

// A 16-bit output element: fp16 rounded to nearest even, or bf16 as FBGEMM's
// CPU kernels write it (the top half of the fp32 bits after adding 0x8000:
// to nearest, ties away from zero; NaN stays a quiet NaN).
__device__ __forceinline__ uint16_t out16(float v, int32_t kind) {
  if (kind == 1) return __half_as_ushort(__float2half_rn(v));
  const uint32_t x = __float_as_uint(v);
  if ((x & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((x >> 16) | 0x40u);
  return static_cast<uint16_t>((x + 0x8000u) >> 16);
}

__device__ __forceinline__ void store_out(const NbitArgs& a, int64_t col_base, int ncols,
                                          const float* v) {
  if (a.out_kind != 0) {
    uint16_t* o = reinterpret_cast<uint16_t*>(a.out) + col_base;
    for (int e = 0; e < ncols; ++e) o[e] = out16(v[e], a.out_kind);
  } else {
    float* o = reinterpret_cast<float*>(a.out) + col_base;
    for (int e = 0; e < ncols; ++e) o[e] = v[e];
  }
}

// Stores of 16 and 8 bytes at any 2- or 4-byte boundary: an output row starts
// at any element.
typedef uint32_t u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

}  // namespace
}  // namespace mx
