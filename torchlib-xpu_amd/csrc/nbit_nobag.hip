// PoolingMode NONE ("sequence") nbit lookups for gfx950, one launch per table
// type present.
//
// Semantics: fbgemm_gpu int_nbit_split_embedding_nobag_codegen_forward_
// unweighted_cuda (recalled): every table has the same D (the largest max_*_D)
// and position l writes its own dequantized row, out[l, :].  An INT8/INT4/INT2
// element is fma(scale, q, bias) in fp32 (one rounding, as FBGEMM's CPU kernels
// dequantize the first row of a bag); FP32, FP16 and FP8 elements are the row's
// values themselves.  Then the output rounding of the pooled lookup.
//
// Design: a gather over positions, one launch per type present, bound by the
// output writes and the rows' lines.  G lanes per position (the fewest whose
// 8-element blocks cover a row), lane k block k of the row: one vector load of
// codes, one 16-byte store of 16-bit output (two of fp32).  A group takes G
// consecutive positions (one coalesced index load), each lane finds its
// position's table by a binary search over the tables' first positions in LDS
// and its row from the table's base there; positions of another type's tables
// are left to that type's launch.  U rows are loaded before the first is
// stored.  The first launch ends with T + 1 blocks that zero and report the
// tables the call cannot serve (unlaunched type, partial code bytes, misaligned
// rows, D other than the call's) and zero the positions outside every bag.
// Four rows in flight (eight need 200 registers, two waves per SIMD).  409,600
// positions against 4-byte loads, element stores and a check launch, with the
// bounds check: INT8 D = 96 94 -> 30 us, INT4 D = 128 to bf16 104 -> 35, FP16
// D = 256 198 -> 75, 64 positions 25.5 -> 17.7.
#include <type_traits>

#include "nbit_common.h"

namespace mx {
namespace {

constexpr int kNobagMaxT = 1024;
constexpr int64_t kNotMine = -1;  // a table of another launch, or unservable

// A table's first byte in this launch, or kNotMine.
template <int TY>
__device__ __forceinline__ int64_t nobag_base(const NbitArgs& a, int32_t D, int64_t t) {
  const int32_t Dt = a.D_off[t + 1] - a.D_off[t];
  const int64_t wo = a.w_off[t];
  return static_cast<int32_t>(a.tys[t]) == TY && Dt == D &&
                 table_ok(TY, Dt, a.served, wo, a.row_align)
             ? wo
             : kNotMine;
}

// Element c of a row.
template <int TY>
__device__ __forceinline__ float row_elem(const NbitArgs& a, const uint8_t* row, int32_t c) {
  constexpr int bits = TyInfo<TY>::kBits;
  if constexpr (TY == MX_SPARSE_FP32) return reinterpret_cast<const float*>(row)[c];
  if constexpr (TY == MX_SPARSE_FP16)
    return __half2float(__ushort_as_half(reinterpret_cast<const uint16_t*>(row)[c]));
  if constexpr (TY == MX_SPARSE_FP8) return a.fp8.decode(row[c]);
  const uint32_t qp = *reinterpret_cast<const uint32_t*>(row);
  const uint32_t q = (row[4 + (c * bits >> 3)] >> (c * bits & 7)) & ((1u << bits) - 1u);
  return __builtin_fmaf(__half2float(__ushort_as_half(static_cast<uint16_t>(qp & 0xffffu))),
                        static_cast<float>(q),
                        __half2float(__ushort_as_half(static_cast<uint16_t>(qp >> 16))));
}

// The eight elements of a block of TY codes.
template <int TY>
__device__ __forceinline__ void block_elems(const NbitArgs& a, const uint32_t* w, uint32_t qp,
                                            float (&v)[8]) {
  constexpr int bits = TyInfo<TY>::kBits;
  const float scale = __half2float(__ushort_as_half(static_cast<uint16_t>(qp & 0xffffu)));
  const float bias = __half2float(__ushort_as_half(static_cast<uint16_t>(qp >> 16)));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t word = w[e * bits >> 5];
    const int sh = e * bits & 31;
    if constexpr (TY == MX_SPARSE_FP32)
      v[e] = __uint_as_float(word);
    else if constexpr (TY == MX_SPARSE_FP16)
      v[e] = __half2float(__ushort_as_half(static_cast<uint16_t>(word >> sh)));
    else if constexpr (TY == MX_SPARSE_FP8)
      v[e] = a.fp8.decode((word >> sh) & 0xffu);
    else
      v[e] = __builtin_fmaf(scale, static_cast<float>((word >> sh) & ((1u << bits) - 1u)), bias);
  }
}

// Eight elements at output element o (any element).
__device__ __forceinline__ void store_block(const NbitArgs& a, int64_t o, const float (&v)[8]) {
  if (a.out_kind == 0) {
    float* p = reinterpret_cast<float*>(a.out) + o;
    *reinterpret_cast<f32x4a4*>(p) = f32x4a4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4a4*>(p + 4) = f32x4a4{v[4], v[5], v[6], v[7]};
    return;
  }
  uint32_t h[4];
  if (a.out_kind == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      h[i] = __builtin_bit_cast(uint32_t, __floats2half2_rn(fp32_value(v[2 * i]), fp32_value(v[2 * i + 1])));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      h[i] = static_cast<uint32_t>(out16(v[2 * i], 2)) |
             (static_cast<uint32_t>(out16(v[2 * i + 1], 2)) << 16);
  }
  *reinterpret_cast<u32x4a2*>(reinterpret_cast<uint16_t*>(a.out) + o) =
      u32x4a2{h[0], h[1], h[2], h[3]};
}

// One block per table zeroes the positions of a table the call cannot serve
// and reports it; block T zeroes the positions outside every bag.
template <typename I>
__device__ __forceinline__ void nobag_check(const NbitArgs& a, int32_t D, int64_t N, int64_t t) {
  int64_t lo, hi, lo2 = 0, hi2 = 0;
  if (t < a.T) {
    const int32_t Dt = a.D_off[t + 1] - a.D_off[t];
    if (Dt == D && table_ok(a.tys[t], Dt, a.served, a.w_off[t], a.row_align)) return;
    lo = idx_at<I>(a.off, t * a.B);
    hi = idx_at<I>(a.off, (t + 1) * a.B);
    if (threadIdx.x == 0 && a.mailbox)
      __hip_atomic_store(a.mailbox + MX_STATUS_NBIT_TABLE, 1u, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  } else {
    lo = 0;
    hi = idx_at<I>(a.off, 0);
    lo2 = idx_at<I>(a.off, static_cast<int64_t>(a.T) * a.B);
    hi2 = N;
  }
  for (int r = 0; r < 2; ++r) {
    int64_t s0 = r == 0 ? lo : lo2, s1 = r == 0 ? hi : hi2;
    s0 = s0 < 0 ? 0 : s0;
    s1 = s1 > N ? N : s1;
    for (int64_t i = s0 * D + threadIdx.x; i < s1 * D; i += blockDim.x) {
      if (a.out_kind != 0)
        reinterpret_cast<uint16_t*>(a.out)[i] = 0u;
      else
        reinterpret_cast<float*>(a.out)[i] = 0.0f;
    }
  }
}

// nmain blocks walk the positions; the a.nchk blocks after them check tables.
template <typename I, int G, int TY>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
    nbit_nobag_kernel(NbitArgs a, int32_t D, int64_t N, uint32_t nmain) {
  constexpr int NG = 256 / G;
  constexpr int BITS = TyInfo<TY>::kBits;
  constexpr bool Q = TyInfo<TY>::kQ;
  constexpr int NB = BITS;                   // bytes of a full 8-element block
  constexpr int NW = NB >= 4 ? NB / 4 : 1;
  constexpr int U = 4;                       // rows in flight
  if (blockIdx.x >= nmain) {
    nobag_check<I>(a, D, N, blockIdx.x - nmain);
    return;
  }
  __shared__ int64_t s_pos[kNobagMaxT + 1], s_base[kNobagMaxT];
  const bool lds = a.T <= kNobagMaxT;
  if (lds)
    for (int t = threadIdx.x; t <= a.T; t += 256) {
      s_pos[t] = idx_at<I>(a.off, t * a.B);
      if (t < a.T) s_base[t] = nobag_base<TY>(a, D, t);
    }
  __syncthreads();
  auto pos = [&](int64_t t) { return lds ? s_pos[t] : idx_at<I>(a.off, t * a.B); };
  const int64_t p0 = pos(0), p1 = pos(a.T);
  const int64_t stride = row_bytes_of(TY, D, a.row_align);
  const int lane = threadIdx.x & 63;
  const int g = lane / G, k = lane % G;
  const int64_t lb = xcd_remap(blockIdx.x, nmain);
  const int64_t step = static_cast<int64_t>(nmain) * NG * G;
  for (int64_t base = (lb * NG + threadIdx.x / G) * G; base < N; base += step) {
    const int64_t l = base + k;
    int64_t my_row = kNotMine;  // byte offset of l's row in the weights
    if (l < N && l >= p0 && l < p1) {
      int32_t lo = 0, hi = a.T;  // the table: the last t with pos(t) <= l
      while (hi - lo > 1) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        if (pos(mid) <= l)
          lo = mid;
        else
          hi = mid;
      }
      const int64_t tb = lds ? s_base[lo] : nobag_base<TY>(a, D, lo);
      if (tb != kNotMine) my_row = tb + idx_at<I>(a.idx, l) * stride;
    }
    const int n = static_cast<int>(N - base < G ? N - base : G);
    for (int j = 0; j < n; j += U) {
      int64_t roff[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        roff[u] = __shfl(my_row, g * G + (j + u < n ? j + u : n - 1), 64);
      for (int cb = k * 8; cb + 8 <= D; cb += G * 8) {
        uint32_t w[U][NW];
        uint32_t qp[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          qp[u] = 0u;
          if (j + u < n && roff[u] >= 0) {
            const uint8_t* row = a.W + roff[u];
            load_codes<NB>(row + (Q ? 4 : 0) + cb * BITS / 8, w[u]);
            if constexpr (Q) qp[u] = *reinterpret_cast<const uint32_t*>(row);
          }
        }
        // Stores count as pending accesses too: said outright here, the rows'
        // arrival is not waited for again at each store, behind the store before
        // it (INT8 D = 96 32 -> 30 us, FP16 D = 256 110 -> 75).
        wait_loads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (j + u >= n || roff[u] < 0) continue;
          float v[8];
          block_elems<TY>(a, w[u], qp[u], v);
          store_block(a, (base + j + u) * D + cb, v);
        }
      }
    }
    if ((D & 7) != 0) {  // the rows' last, partial block: an element per lane (G >= 8)
      const int32_t c = (D & ~7) + k;
      for (int j = 0; j < n; ++j) {
        const int64_t ro = __shfl(my_row, g * G + j, 64);
        if (ro < 0 || c >= D) continue;
        const float v = row_elem<TY>(a, a.W + ro, c);
        store_out(a, (base + j) * D + c, 1, &v);
      }
    }
  }
}

template <int TY>
int launch_nobag_type(NbitArgs& a, int32_t max_D, int32_t D, int64_t N, int32_t index_bytes,
                      hipStream_t s) {
  if (max_D <= 0) return MX_OK;
  const int64_t want = ceil_div(N, 256);  // 256 positions per block and round
  const int64_t cap = static_cast<int64_t>(num_cus()) * 16;
  const uint32_t nmain = static_cast<uint32_t>(want < cap ? want : cap);
  const dim3 gd(nmain + a.nchk);
  auto go = [&](auto g) {
    constexpr int G = decltype(g)::value;
    if (index_bytes == 8)
      nbit_nobag_kernel<int64_t, G, TY><<<gd, 256, 0, s>>>(a, D, N, nmain);
    else
      nbit_nobag_kernel<int32_t, G, TY><<<gd, 256, 0, s>>>(a, D, N, nmain);
  };
  if (D <= 64)
    go(std::integral_constant<int, 8>{});
  else if (D <= 128)
    go(std::integral_constant<int, 16>{});
  else if (D <= 256)
    go(std::integral_constant<int, 32>{});
  else
    go(std::integral_constant<int, 64>{});
  MX_LAUNCH_CHECK();
  a.nchk = 0;
  return MX_OK;
}

}  // namespace
}  // namespace mx

using namespace mx;

extern "C" int mx_nbit_forward_nobag(const uint8_t* dev_weights, const int64_t* weights_offsets,
                                     const uint8_t* weights_tys, const int32_t* D_offsets,
                                     int32_t T, int64_t B, int32_t max_int2_D, int32_t max_int4_D,
                                     int32_t max_int8_D, int32_t max_float16_D,
                                     int32_t max_float32_D, const void* indices,
                                     const void* offsets, int32_t index_bytes, int64_t N,
                                     int32_t output_dtype, int32_t row_alignment,
                                     int32_t max_float8_D, int32_t fp8_exponent_bits,
                                     int32_t fp8_exponent_bias, void* out, void* stream) {
  clear_error();
  MX_REQUIRE(T >= 0 && B >= 0 && N >= 0, "negative T, B or N");
  MX_REQUIRE(index_bytes == 4 || index_bytes == 8, "indices must be int32 or int64");
  MX_REQUIRE(output_dtype == MX_SPARSE_FP32 || output_dtype == MX_SPARSE_FP16 ||
                 output_dtype == MX_SPARSE_BF16,
             "output_dtype %d not supported (FP32=0, FP16=1, BF16=5)", output_dtype);
  MX_REQUIRE(row_alignment >= 1, "row_alignment must be positive");
  int32_t D = 0;
  for (int32_t d :
       {max_int2_D, max_int4_D, max_int8_D, max_float16_D, max_float32_D, max_float8_D}) {
    MX_REQUIRE(d >= 0, "negative max_D");
    if (d > D) D = d;
  }
  MX_REQUIRE(D <= 1024, "max D %d above 1024", D);
  MX_REQUIRE(max_int4_D % 2 == 0 && max_int2_D % 4 == 0,
             "INT4 D must be even and INT2 D a multiple of 4 (max_int4_D %d, max_int2_D %d)",
             max_int4_D, max_int2_D);
  MX_REQUIRE(max_float8_D == 0 || hfp8_format_ok(fp8_exponent_bits, fp8_exponent_bias),
             "FP8 tables need 1 <= fp8_exponent_bits <= 7 and 0 <= fp8_exponent_bias <= 120 "
             "(got %d, %d)", fp8_exponent_bits, fp8_exponent_bias);
  if (N == 0 || D == 0) return MX_OK;
  MX_REQUIRE(T > 0 && B > 0, "%lld indices but no bags (T=%d, B=%lld)", (long long)N, T,
             (long long)B);
  MX_REQUIRE(dev_weights && weights_offsets && weights_tys && D_offsets && indices && offsets &&
                 out,
             "null pointer argument");
  NbitArgs a{};
  a.W = dev_weights;
  a.w_off = weights_offsets;
  a.tys = weights_tys;
  a.D_off = D_offsets;
  a.idx = indices;
  a.off = offsets;
  a.iw = nullptr;
  a.out = out;
  a.B = B;
  a.total_D = D;
  a.T = T;
  a.pooling = MX_POOL_NONE;
  a.row_align = row_alignment;
  a.out_kind = output_dtype == MX_SPARSE_FP16 ? 1 : (output_dtype == MX_SPARSE_BF16 ? 2 : 0);
  a.served = (max_int8_D > 0 ? 1 << MX_SPARSE_INT8 : 0) | (max_int4_D > 0 ? 1 << MX_SPARSE_INT4 : 0) |
             (max_int2_D > 0 ? 1 << MX_SPARSE_INT2 : 0) |
             (max_float16_D > 0 ? 1 << MX_SPARSE_FP16 : 0) |
             (max_float32_D > 0 ? 1 << MX_SPARSE_FP32 : 0) |
             (max_float8_D > 0 ? 1 << MX_SPARSE_FP8 : 0);
  a.fp8 = max_float8_D > 0 ? Hfp8::make(fp8_exponent_bits, fp8_exponent_bias) : Hfp8::make(4, 7);
  a.nchk = static_cast<uint32_t>(T) + 1;  // the first launch (D > 0: there is one) checks the tables
  a.mailbox = status_mailbox();
  auto* s = as_stream(stream);
  if (int rc = launch_nobag_type<MX_SPARSE_INT8>(a, max_int8_D, D, N, index_bytes, s)) return rc;
  if (int rc = launch_nobag_type<MX_SPARSE_INT4>(a, max_int4_D, D, N, index_bytes, s)) return rc;
  if (int rc = launch_nobag_type<MX_SPARSE_INT2>(a, max_int2_D, D, N, index_bytes, s)) return rc;
  if (int rc = launch_nobag_type<MX_SPARSE_FP16>(a, max_float16_D, D, N, index_bytes, s)) return rc;
  if (int rc = launch_nobag_type<MX_SPARSE_FP8>(a, max_float8_D, D, N, index_bytes, s)) return rc;
  return launch_nobag_type<MX_SPARSE_FP32>(a, max_float32_D, D, N, index_bytes, s);
}
