// Jagged <-> padded-dense kernels for gfx950.
//
// Semantics follow fbgemm_gpu's jagged_to_padded_dense_forward,
// dense_to_jagged_forward, jagged_dense_elementwise_add_jagged_output and
// jagged_dense_elementwise_mul (upstream src/jagged_tensor_ops/, recalled;
// outside the dense the add gives x + 0 and the mul x * 0), restated from torch's own
// port of the same ops: torch/_inductor/jagged_lowerings.py:161-177 (masked
// load, else padding value) and :231-249 (jagged rows past max length become
// 0).
//
// Design: the ops are pure HBM streams.  One work item moves VEC bytes
// (16 when the row size and pointers allow it), consecutive work items walk
// a row, so every wave issues fully coalesced transactions.  The rows of one
// innermost list (a "bag": with one jagged dim a batch element) lie together
// on both sides, so a group of threads moves a whole bag with no per-item
// index arithmetic; with more jagged dims the bag's place on the other side is
// found once per bag, by walking the offsets levels (padded dense -> list) or
// by a binary search per outer level (list -> padded dense).  A group is 16,
// 64 or 256 threads by the bag's size.  (Two jagged dims, 256 x 20 x 50 x 64
// bf16, against coordinates per chunk: padding 26.6 -> 11.3 us, back 14.3 ->
// 11.0 by trace; the fp32 add 21.2 -> 15.6 us per call.)
#include "mx_common.h"

namespace mx {
namespace {

struct JaggedMeta {
  const void* off[MX_MAX_JAGGED_DIM];
  int64_t off_len[MX_MAX_JAGGED_DIM];  // entries in each offsets array
  int64_t max_len[MX_MAX_JAGGED_DIM];
  int32_t ndim;
};

template <int VEC>
struct alignas(VEC) Chunk {
  uint8_t b[VEC];
};

template <typename I>
__device__ __forceinline__ int64_t off_at(const JaggedMeta& m, int k, int64_t i) {
  return static_cast<int64_t>(reinterpret_cast<const I*>(m.off[k])[i]);
}

// Innermost list of dense bag r (over B * prod(max_len of the outer dims)):
// its first values row and its length, 0 for a list that is not there.
template <typename I>
__device__ __forceinline__ void dense_bag(int64_t r, const JaggedMeta& m, int64_t& begin,
                                          int64_t& len) {
  const int last = m.ndim - 1;
  int64_t idx = r;
  if (last > 0) {
    int64_t coord[MX_MAX_JAGGED_DIM - 1];
    for (int k = last - 1; k >= 0; --k) {
      const int64_t q = idx / m.max_len[k];
      coord[k] = idx - q * m.max_len[k];
      idx = q;
    }
    for (int k = 0; k < last; ++k) {
      const int64_t b = off_at<I>(m, k, idx);
      const int64_t e = off_at<I>(m, k, idx + 1);
      if (coord[k] >= e - b) {
        begin = len = 0;
        return;
      }
      idx = b + coord[k];
    }
  }
  begin = off_at<I>(m, last, idx);
  len = off_at<I>(m, last, idx + 1) - begin;
}

// Last p in [0, n-1) with off[p] <= x, or -1 when x is past the last offset.
template <typename I>
__device__ int64_t owner_of(const JaggedMeta& m, int k, int64_t x) {
  const int64_t n = m.off_len[k];
  if (n < 2 || x < off_at<I>(m, k, 0) || x >= off_at<I>(m, k, n - 1)) return -1;
  int64_t lo = 0, hi = n - 1;  // off[lo] <= x < off[hi]
  while (hi - lo > 1) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (off_at<I>(m, k, mid) <= x)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Innermost list p -> its dense bag, or -1 if it has no dense position.
template <typename I>
__device__ __forceinline__ int64_t list_dense_bag(int64_t p, const JaggedMeta& m) {
  const int last = m.ndim - 1;
  if (last == 0) return p;
  int64_t coord[MX_MAX_JAGGED_DIM - 1];
  int64_t idx = p;
  for (int k = last - 1; k >= 0; --k) {
    const int64_t q = owner_of<I>(m, k, idx);
    if (q < 0) return -1;
    coord[k] = idx - off_at<I>(m, k, q);
    if (coord[k] >= m.max_len[k]) return -1;
    idx = q;
  }
  for (int k = 0; k < last; ++k) idx = idx * m.max_len[k] + coord[k];
  return idx;
}

// ---- element arithmetic for the jagged + dense add ------------------------

__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __uint_as_float(static_cast<uint32_t>(h) << 16);
}
// Round to nearest even, NaN kept quiet (same rule as c10::BFloat16).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}

// x (op) y per element in the element type's arithmetic: f32/f64 natively,
// f16/bf16 computed in fp32 (sums and products of two such values are then
// rounded once to the element type, to nearest even).
template <int DT, bool MUL>
struct BinOp;

template <bool MUL>
struct BinOp<MX_DTYPE_F32, MUL> {
  static constexpr int kBytes = 4;
  __device__ static void apply(const uint8_t* x, const uint8_t* y, uint8_t* o) {
    const float a = *reinterpret_cast<const float*>(x), b = *reinterpret_cast<const float*>(y);
    *reinterpret_cast<float*>(o) = MUL ? a * b : a + b;
  }
};
template <bool MUL>
struct BinOp<MX_DTYPE_F64, MUL> {
  static constexpr int kBytes = 8;
  __device__ static void apply(const uint8_t* x, const uint8_t* y, uint8_t* o) {
    const double a = *reinterpret_cast<const double*>(x), b = *reinterpret_cast<const double*>(y);
    *reinterpret_cast<double*>(o) = MUL ? a * b : a + b;
  }
};
template <bool MUL>
struct BinOp<MX_DTYPE_F16, MUL> {
  static constexpr int kBytes = 2;
  __device__ static void apply(const uint8_t* x, const uint8_t* y, uint8_t* o) {
    const float a = __half2float(*reinterpret_cast<const __half*>(x));
    const float b = __half2float(*reinterpret_cast<const __half*>(y));
    *reinterpret_cast<__half*>(o) = __float2half_rn(MUL ? a * b : a + b);
  }
};
template <bool MUL>
struct BinOp<MX_DTYPE_BF16, MUL> {
  static constexpr int kBytes = 2;
  __device__ static void apply(const uint8_t* x, const uint8_t* y, uint8_t* o) {
    const float a = bf16_to_f32(*reinterpret_cast<const uint16_t*>(x));
    const float b = bf16_to_f32(*reinterpret_cast<const uint16_t*>(y));
    *reinterpret_cast<uint16_t*>(o) = f32_to_bf16(MUL ? a * b : a + b);
  }
};

// ---- a bag is a contiguous copy ---------------------------------------------
//
// Dense bag r's rows [r*max_L, (r+1)*max_L) and its list's values rows are both
// contiguous, so each bag is one straight copy plus padding.  2^lg threads per
// bag (x), parts of a bag in y; every thread keeps kJagItems chunks in flight.
// ONE: one jagged dim and a block per bag, as constants (a large bf16 round
// trip 103.6 -> 101.5 us, a small add 6.8 -> 6.1 us against run-time values).

constexpr int kJagItems = 4;

template <int VEC, typename I, bool ONE>
__global__ void __launch_bounds__(256)
    j2pd_kernel(const uint8_t* __restrict__ values, uint8_t* __restrict__ out, JaggedMeta m,
                int64_t nbags, int32_t lg, int64_t vpr, Chunk<VEC> pad) {
  if constexpr (ONE) {
    lg = 8;
    m.ndim = 1;
  }
  const int32_t tpb = 1 << lg, t = threadIdx.x & (tpb - 1);
  const int64_t max_L = m.max_len[m.ndim - 1];
  const int64_t span = static_cast<int64_t>(tpb) * kJagItems;
  const int64_t step = static_cast<int64_t>(gridDim.x) << (8 - lg);
  for (int64_t b = (static_cast<int64_t>(blockIdx.x) << (8 - lg)) + (threadIdx.x >> lg); b < nbags;
       b += step) {
    int64_t begin, len;
    dense_bag<I>(b, m, begin, len);
    len = len < 0 ? 0 : (len > max_L ? max_L : len);
    const int64_t n_copy = len * vpr, n_all = max_L * vpr;
    const Chunk<VEC>* __restrict__ src =
        reinterpret_cast<const Chunk<VEC>*>(values) + begin * vpr;
    Chunk<VEC>* __restrict__ dst = reinterpret_cast<Chunk<VEC>*>(out) + b * n_all;
    for (int64_t base = blockIdx.y * span; base < n_all; base += gridDim.y * span) {
      Chunk<VEC> c[kJagItems];
#pragma unroll
      for (int it = 0; it < kJagItems; ++it) {
        const int64_t i = base + it * tpb + t;
        if (i < n_copy) c[it] = src[i];
      }
      // Stores count as pending accesses too: said outright here, the loads are not
      // waited for again before each store, behind the store before it (a large
      // bf16 round trip 102.1 -> 101.3 us).
      wait_loads();
#pragma unroll
      for (int it = 0; it < kJagItems; ++it) {
        const int64_t i = base + it * tpb + t;
        if (i >= n_copy) c[it] = pad;
        if (i < n_all) {
          // The dense output streams past the caches (config 1 cold round trip
          // 12.4 -> 11.8 us; the same for dense_to_jagged's output gained nothing).
          if constexpr (VEC == 16) {
            typedef unsigned int u4nt __attribute__((ext_vector_type(4)));
            __builtin_nontemporal_store(*reinterpret_cast<const u4nt*>(&c[it]),
                                        reinterpret_cast<u4nt*>(&dst[i]));
          } else {
            dst[i] = c[it];
          }
        }
      }
    }
  }
}

// Values rows [r0, r1) whose first `copy_rows` rows take dense rows from
// `dense_row0` on and the rest 0; ADD combines x with them (x + y, or x * y
// with MUL), else the dense value is copied (dense -> jagged).
template <int VEC, bool ADD, int DT, bool MUL>
__device__ __forceinline__ void emit_rows(const uint8_t* __restrict__ dense,
                                          const uint8_t* __restrict__ x,
                                          uint8_t* __restrict__ out, int64_t r0, int64_t r1,
                                          int64_t copy_rows, int64_t dense_row0, int64_t vpr,
                                          int32_t tpb) {
  const int32_t t = threadIdx.x & (tpb - 1);
  const int64_t span = static_cast<int64_t>(tpb) * kJagItems;
  const int64_t n_all = (r1 - r0) * vpr, n_copy = copy_rows * vpr;
  const Chunk<VEC>* __restrict__ src = reinterpret_cast<const Chunk<VEC>*>(dense) + dense_row0 * vpr;
  Chunk<VEC>* __restrict__ dst = reinterpret_cast<Chunk<VEC>*>(out) + r0 * vpr;
  const Chunk<VEC>* __restrict__ xs = reinterpret_cast<const Chunk<VEC>*>(x) + r0 * vpr;
  for (int64_t base = blockIdx.y * span; base < n_all; base += gridDim.y * span) {
    Chunk<VEC> y[kJagItems];
#pragma unroll
    for (int it = 0; it < kJagItems; ++it) {
      const int64_t i = base + it * tpb + t;
      if (i < n_copy) {
        y[it] = src[i];
      } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) y[it].b[e] = 0;  // +0 in every element type
      }
    }
    if constexpr (!ADD) wait_loads();
#pragma unroll
    for (int it = 0; it < kJagItems; ++it) {
      const int64_t i = base + it * tpb + t;
      if (i >= n_all) continue;
      if constexpr (ADD) {
        const Chunk<VEC> cx = xs[i];
        Chunk<VEC> co;
#pragma unroll
        for (int e = 0; e < VEC; e += BinOp<DT, MUL>::kBytes)
          BinOp<DT, MUL>::apply(cx.b + e, y[it].b + e, co.b + e);
        dst[i] = co;
      } else {
        dst[i] = y[it];
      }
    }
  }
}

// Group x < nlists: innermost list x.  Group x == nlists: the values rows no
// list covers (before the first offset, from the last on), which have no dense
// position.  Row ranges are clamped to [0, total_L], so malformed offsets never
// write out of bounds.
template <int VEC, typename I, bool ADD, int DT, bool MUL, bool ONE>
__global__ void __launch_bounds__(256)
    jagged_out_kernel(const uint8_t* __restrict__ dense, const uint8_t* __restrict__ x,
                      uint8_t* __restrict__ out, JaggedMeta m, int64_t nlists, int32_t lg,
                      int64_t total_L, int64_t vpr) {
  if constexpr (ONE) {
    lg = 8;
    m.ndim = 1;
  }
  auto clamp = [&](int64_t v, int64_t lo) { return v < lo ? lo : (v > total_L ? total_L : v); };
  const int last = m.ndim - 1;
  const int64_t max_L = m.max_len[last];
  const int32_t tpb = 1 << lg;
  const int64_t step = static_cast<int64_t>(gridDim.x) << (8 - lg);
  for (int64_t p = (static_cast<int64_t>(blockIdx.x) << (8 - lg)) + (threadIdx.x >> lg);
       p <= nlists; p += step) {
    if (p < nlists) {
      const int64_t r0 = clamp(off_at<I>(m, last, p), 0);
      const int64_t r1 = clamp(off_at<I>(m, last, p + 1), r0);
      if (r1 == r0) continue;
      const int64_t bag = list_dense_bag<I>(p, m);
      const int64_t copy = bag < 0 ? 0 : (r1 - r0 < max_L ? r1 - r0 : max_L);
      emit_rows<VEC, ADD, DT, MUL>(dense, x, out, r0, r1, copy, bag < 0 ? 0 : bag * max_L, vpr,
                                   tpb);
    } else {
      const int64_t head = clamp(off_at<I>(m, last, 0), 0);
      const int64_t tail = clamp(off_at<I>(m, last, nlists), head);
      emit_rows<VEC, ADD, DT, MUL>(dense, x, out, 0, head, 0, 0, vpr, tpb);
      emit_rows<VEC, ADD, DT, MUL>(dense, x, out, tail, total_L, 0, 0, vpr, tpb);
    }
  }
}

// ---- host side ------------------------------------------------------------

// Threads per bag (2^lg) and grid: the smallest group that holds a full bag's
// chunks in one round, kJagItems per thread, up to a block; bags in x, parts of
// a bag in y (the kernels loop over what the grid leaves).
struct BagGrid {
  dim3 grid;
  int32_t lg;
};

BagGrid bag_grid(int64_t bags, int64_t chunks_per_bag) {
  const int64_t chunks = chunks_per_bag > 0 ? chunks_per_bag : 1;
  BagGrid g;
  g.lg = chunks <= 16 * kJagItems ? 4 : (chunks <= 64 * kJagItems ? 6 : 8);
  int64_t parts = ceil_div(chunks, static_cast<int64_t>(kJagItems) << g.lg);
  if (parts > 64) parts = 64;
  int64_t x = ceil_div(bags, int64_t(1) << (8 - g.lg));
  if (x > (int64_t(1) << 30)) x = int64_t(1) << 30;
  g.grid = dim3(static_cast<uint32_t>(x), static_cast<uint32_t>(parts));
  return g;
}

int pick_vec(int64_t row_bytes, std::initializer_list<const void*> ptrs) {
  for (int vec : {16, 8, 4, 2, 1}) {
    if (row_bytes % vec) continue;
    bool ok = true;
    for (const void* p : ptrs)
      if (reinterpret_cast<uintptr_t>(p) % vec) ok = false;
    if (ok) return vec;
  }
  return 1;
}

int build_meta(JaggedMeta& m, int32_t ndim, const void* const* offsets, int32_t offset_bytes,
               const int64_t* offsets_numel, const int64_t* max_lengths) {
  MX_REQUIRE(ndim >= 1 && ndim <= MX_MAX_JAGGED_DIM, "num_jagged_dim %d not in [1, %d]", ndim,
             MX_MAX_JAGGED_DIM);
  MX_REQUIRE(offset_bytes == 4 || offset_bytes == 8, "offsets must be int32 or int64");
  MX_REQUIRE(offsets != nullptr && offsets_numel != nullptr && max_lengths != nullptr,
             "null offsets/offsets_numel/max_lengths");
  m.ndim = ndim;
  for (int k = 0; k < ndim; ++k) {
    MX_REQUIRE(offsets_numel[k] >= 1, "offsets[%d] must have at least one entry", k);
    MX_REQUIRE(offsets[k] != nullptr, "null offsets[%d]", k);
    MX_REQUIRE(max_lengths[k] >= 0, "negative max_length[%d]", k);
    m.off[k] = offsets[k];
    m.off_len[k] = offsets_numel[k];
    m.max_len[k] = max_lengths[k];
  }
  for (int k = ndim; k < MX_MAX_JAGGED_DIM; ++k) {
    m.off[k] = nullptr;
    m.off_len[k] = 0;
    m.max_len[k] = 1;
  }
  return MX_OK;
}

bool valid_elem(int64_t eb) { return eb == 1 || eb == 2 || eb == 4 || eb == 8; }

int64_t dtype_bytes(int32_t dt) {
  switch (dt) {
    case MX_DTYPE_F32: return 4;
    case MX_DTYPE_F64: return 8;
    case MX_DTYPE_F16:
    case MX_DTYPE_BF16: return 2;
    default: return -1;
  }
}

}  // namespace
}  // namespace mx

using namespace mx;

#define MX_VEC_SWITCH(vec, ...)                             \
  switch (vec) {                                            \
    case 16: { constexpr int V = 16; __VA_ARGS__; break; } \
    case 8: { constexpr int V = 8; __VA_ARGS__; break; }   \
    case 4: { constexpr int V = 4; __VA_ARGS__; break; }   \
    case 2: { constexpr int V = 2; __VA_ARGS__; break; }   \
    default: { constexpr int V = 1; __VA_ARGS__; break; }  \
  }

extern "C" int mx_jagged_to_padded_dense(const void* values, int64_t elem_bytes, int64_t inner,
                                         int32_t num_jagged_dim, const void* const* offsets,
                                         int32_t offset_bytes, const int64_t* offsets_numel,
                                         const int64_t* max_lengths, uint64_t pad_bits,
                                         void* out, void* stream) {
  clear_error();
  JaggedMeta m;
  if (int rc = build_meta(m, num_jagged_dim, offsets, offset_bytes, offsets_numel, max_lengths))
    return rc;
  MX_REQUIRE(valid_elem(elem_bytes), "element size %lld not supported", (long long)elem_bytes);
  MX_REQUIRE(inner >= 0, "negative inner size");
  int64_t rows = offsets_numel[0] - 1;
  for (int k = 0; k < num_jagged_dim; ++k) rows *= max_lengths[k];
  const int64_t row_bytes = inner * elem_bytes;
  if (rows == 0 || row_bytes == 0) return MX_OK;
  MX_REQUIRE(out != nullptr, "null out");  // values may be empty (every row padding)
  int vec = pick_vec(row_bytes, {values, out});
  if (vec < elem_bytes) vec = static_cast<int>(elem_bytes);  // keep elements whole
  MX_REQUIRE(row_bytes % vec == 0, "misaligned tensors");
  uint8_t pat[16];  // padding pattern replicated over a 16-byte chunk
  for (int i = 0; i < 16; ++i) pat[i] = static_cast<uint8_t>(pad_bits >> (8 * (i % elem_bytes)));
  const int64_t vpr = row_bytes / vec;
  auto* s = as_stream(stream);
  const auto* v = static_cast<const uint8_t*>(values);
  auto* o = static_cast<uint8_t*>(out);
  const int64_t max_L = max_lengths[num_jagged_dim - 1];
  const int64_t nbags = rows / max_L;  // rows > 0: max_L > 0
  const BagGrid g = bag_grid(nbags, max_L * vpr);
  const bool one = num_jagged_dim == 1 && g.lg == 8;
  MX_VEC_SWITCH(vec, {
    Chunk<V> pad;
    for (int i = 0; i < V; ++i) pad.b[i] = pat[i];
    const auto kernel = one ? (offset_bytes == 8 ? j2pd_kernel<V, int64_t, true>
                                                 : j2pd_kernel<V, int32_t, true>)
                            : (offset_bytes == 8 ? j2pd_kernel<V, int64_t, false>
                                                 : j2pd_kernel<V, int32_t, false>);
    kernel<<<g.grid, 256, 0, s>>>(v, o, m, nbags, g.lg, vpr, pad);
  });
  MX_LAUNCH_CHECK();
  return MX_OK;
}

// Shared host path of dense_to_jagged (x_values == NULL) and of the
// jagged (op) dense elementwise ops (x_values != NULL; mul: x * y, else x + y).
static int jagged_output_op(const void* dense, int64_t elem_bytes, int64_t inner,
                            int32_t num_jagged_dim, const void* const* offsets,
                            int32_t offset_bytes, const int64_t* offsets_numel,
                            const int64_t* max_lengths, int64_t total_L, const void* x_values,
                            int32_t add_dtype, bool mul, void* out, void* stream) {
  JaggedMeta m;
  if (int rc = build_meta(m, num_jagged_dim, offsets, offset_bytes, offsets_numel, max_lengths))
    return rc;
  MX_REQUIRE(valid_elem(elem_bytes), "element size %lld not supported", (long long)elem_bytes);
  MX_REQUIRE(inner >= 0 && total_L >= 0, "negative size");
  const int64_t row_bytes = inner * elem_bytes;
  if (total_L == 0 || row_bytes == 0) return MX_OK;
  MX_REQUIRE(out != nullptr, "null out");
  int64_t dense_rows = offsets_numel[0] - 1;
  for (int k = 0; k < num_jagged_dim; ++k) dense_rows *= max_lengths[k];
  MX_REQUIRE(dense != nullptr || dense_rows == 0, "null dense");
  const int vec0 = x_values ? pick_vec(row_bytes, {dense, out, x_values})
                            : pick_vec(row_bytes, {dense, out});
  const int vec = vec0 < elem_bytes ? static_cast<int>(elem_bytes) : vec0;
  MX_REQUIRE(row_bytes % vec == 0, "misaligned tensors");
  const int64_t vpr = row_bytes / vec;
  auto* s = as_stream(stream);
  const auto* d = static_cast<const uint8_t*>(dense);
  auto* o = static_cast<uint8_t*>(out);
  const int last = num_jagged_dim - 1;
  const int64_t nlists = offsets_numel[last] - 1;
  const BagGrid g = bag_grid(nlists + 1, max_lengths[last] * vpr);
  const bool one = num_jagged_dim == 1 && g.lg == 8;
  if (x_values == nullptr) {
    MX_VEC_SWITCH(vec, {
      constexpr int F = MX_DTYPE_F32;  // a copy: no element type
      const auto kernel = one ? (offset_bytes == 8 ? jagged_out_kernel<V, int64_t, false, F, false, true>
                                                   : jagged_out_kernel<V, int32_t, false, F, false, true>)
                              : (offset_bytes == 8 ? jagged_out_kernel<V, int64_t, false, F, false, false>
                                                   : jagged_out_kernel<V, int32_t, false, F, false, false>);
      kernel<<<g.grid, 256, 0, s>>>(d, nullptr, o, m, nlists, g.lg, total_L, vpr);
    });
    MX_LAUNCH_CHECK();
    return MX_OK;
  }
  MX_REQUIRE(dtype_bytes(add_dtype) == elem_bytes, "dtype %d does not match element size %lld",
             add_dtype, (long long)elem_bytes);
  const auto* x = static_cast<const uint8_t*>(x_values);
#define MX_OP_LAUNCH(DTC, MULC)                                                                 \
  MX_VEC_SWITCH(vec, {                                                                          \
    if constexpr (V >= BinOp<DTC, MULC>::kBytes) {                                              \
      const auto kernel =                                                                       \
          one ? (offset_bytes == 8 ? jagged_out_kernel<V, int64_t, true, DTC, MULC, true>       \
                                   : jagged_out_kernel<V, int32_t, true, DTC, MULC, true>)      \
              : (offset_bytes == 8 ? jagged_out_kernel<V, int64_t, true, DTC, MULC, false>      \
                                   : jagged_out_kernel<V, int32_t, true, DTC, MULC, false>);    \
      kernel<<<g.grid, 256, 0, s>>>(d, x, o, m, nlists, g.lg, total_L, vpr);                    \
    }                                                                                           \
  })
#define MX_ADD_LAUNCH(DTC)    \
  if (mul) {                  \
    MX_OP_LAUNCH(DTC, true);  \
  } else {                    \
    MX_OP_LAUNCH(DTC, false); \
  }
  switch (add_dtype) {
    case MX_DTYPE_F32: MX_ADD_LAUNCH(MX_DTYPE_F32); break;
    case MX_DTYPE_F64: MX_ADD_LAUNCH(MX_DTYPE_F64); break;
    case MX_DTYPE_F16: MX_ADD_LAUNCH(MX_DTYPE_F16); break;
    case MX_DTYPE_BF16: MX_ADD_LAUNCH(MX_DTYPE_BF16); break;
    default: return set_error(MX_EUNSUPPORTED, "dtype %d not supported", add_dtype);
  }
#undef MX_ADD_LAUNCH
#undef MX_OP_LAUNCH
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_dense_to_jagged(const void* dense, int64_t elem_bytes, int64_t inner,
                                  int32_t num_jagged_dim, const void* const* offsets,
                                  int32_t offset_bytes, const int64_t* offsets_numel,
                                  const int64_t* max_lengths, int64_t total_L, void* out,
                                  void* stream) {
  clear_error();
  return jagged_output_op(dense, elem_bytes, inner, num_jagged_dim, offsets, offset_bytes,
                          offsets_numel, max_lengths, total_L, nullptr, 0, false, out, stream);
}

extern "C" int mx_jagged_dense_elementwise_add(const void* x_values, const void* y_dense,
                                               int32_t dtype, int64_t inner,
                                               int32_t num_jagged_dim, const void* const* offsets,
                                               int32_t offset_bytes, const int64_t* offsets_numel,
                                               const int64_t* max_lengths, int64_t total_L,
                                               void* out, void* stream) {
  clear_error();
  const int64_t eb = dtype_bytes(dtype);
  if (eb < 0) return set_error(MX_EUNSUPPORTED, "dtype %d not supported", dtype);
  MX_REQUIRE(x_values != nullptr || total_L == 0, "null x_values");
  if (total_L == 0 || inner == 0) return MX_OK;
  return jagged_output_op(y_dense, eb, inner, num_jagged_dim, offsets, offset_bytes,
                          offsets_numel, max_lengths, total_L, x_values, dtype, false, out, stream);
}

extern "C" int mx_jagged_dense_elementwise_mul(const void* x_values, const void* y_dense,
                                               int32_t dtype, int64_t inner,
                                               int32_t num_jagged_dim, const void* const* offsets,
                                               int32_t offset_bytes, const int64_t* offsets_numel,
                                               const int64_t* max_lengths, int64_t total_L,
                                               void* out, void* stream) {
  clear_error();
  const int64_t eb = dtype_bytes(dtype);
  if (eb < 0) return set_error(MX_EUNSUPPORTED, "dtype %d not supported", dtype);
  MX_REQUIRE(x_values != nullptr || total_L == 0, "null x_values");
  if (total_L == 0 || inner == 0) return MX_OK;
  return jagged_output_op(y_dense, eb, inner, num_jagged_dim, offsets, offset_bytes,
                          offsets_numel, max_lengths, total_L, x_values, dtype, true, out, stream);
}
