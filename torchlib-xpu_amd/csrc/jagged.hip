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
#include <type_traits>

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

// In whole words: cleared byte by byte, a chunk that may also be loaded lives in a
// register per byte, and its load is waited for at once.
template <int VEC>
__device__ __forceinline__ void clear(Chunk<VEC>& c) {
  using W = std::conditional_t<(VEC >= 4), uint32_t, std::conditional_t<VEC == 2, uint16_t, uint8_t>>;
#pragma unroll
  for (int e = 0; e < VEC; e += static_cast<int>(sizeof(W))) *reinterpret_cast<W*>(c.b + e) = W(0);
}

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
  const uint32_t u = __float_as_uint(f);
  const uint32_t r = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16, nan = (u >> 16) | 0x40u;
  return static_cast<uint16_t>((u & 0x7fffffffu) > 0x7f800000u ? nan : r);
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
  // Two elements of one 32-bit word.  The asm holds the unpacking back to here:
  // else the compiler unpacks every word as it is loaded, into twice the
  // registers (150 in all, three waves per SIMD).
  __device__ static void apply_word(const uint8_t* x, const uint8_t* y, uint8_t* o) {
    uint32_t a = *reinterpret_cast<const uint32_t*>(x), b = *reinterpret_cast<const uint32_t*>(y);
    asm("" : "+v"(a), "+v"(b));
    const float a0 = __uint_as_float(a << 16), a1 = __uint_as_float(a & 0xffff0000u);
    const float b0 = __uint_as_float(b << 16), b1 = __uint_as_float(b & 0xffff0000u);
    *reinterpret_cast<uint32_t*>(o) = f32_to_bf16(MUL ? a0 * b0 : a0 + b0) |
                                      (static_cast<uint32_t>(f32_to_bf16(MUL ? a1 * b1 : a1 + b1)) << 16);
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

// Part `part` of `parts` of values rows [r0, r1), whose first `copy_rows` rows
// take dense rows from `dense_row0` on and the rest 0; ADD combines x with them
// (x + y, or x * y with MUL), else the dense value is copied (dense -> jagged).
template <int VEC, bool ADD, int DT, bool MUL>
__device__ __forceinline__ void emit_rows(const uint8_t* __restrict__ dense,
                                          const uint8_t* __restrict__ x,
                                          uint8_t* __restrict__ out, int64_t r0, int64_t r1,
                                          int64_t copy_rows, int64_t dense_row0, int64_t vpr,
                                          int32_t tpb, int64_t part, int64_t parts) {
  const int32_t t = threadIdx.x & (tpb - 1);
  const int64_t span = static_cast<int64_t>(tpb) * kJagItems;
  const int64_t n_all = (r1 - r0) * vpr, n_copy = copy_rows * vpr;
  const Chunk<VEC>* __restrict__ src = reinterpret_cast<const Chunk<VEC>*>(dense) + dense_row0 * vpr;
  Chunk<VEC>* __restrict__ dst = reinterpret_cast<Chunk<VEC>*>(out) + r0 * vpr;
  const Chunk<VEC>* __restrict__ xs = reinterpret_cast<const Chunk<VEC>*>(x) + r0 * vpr;
  for (int64_t base = part * span; base < n_all; base += parts * span) {
    Chunk<VEC> y[kJagItems];
    [[maybe_unused]] Chunk<VEC> cx[kJagItems];
#pragma unroll
    for (int it = 0; it < kJagItems; ++it) {
      const int64_t i = base + it * tpb + t;
      if constexpr (ADD)
        if (i < n_all) cx[it] = xs[i];
      if (i < n_copy) y[it] = src[i];
    }
    wait_loads();
#pragma unroll
    for (int it = 0; it < kJagItems; ++it) {
      const int64_t i = base + it * tpb + t;
      if (i >= n_all) continue;
      if (i >= n_copy) clear(y[it]);  // +0 in every element type
      if constexpr (ADD) {
        using Op = BinOp<DT, MUL>;
        Chunk<VEC> co;
        if constexpr (DT == MX_DTYPE_BF16 && VEC >= 4) {
#pragma unroll
          for (int e = 0; e < VEC; e += 4) Op::apply_word(cx[it].b + e, y[it].b + e, co.b + e);
        } else {
#pragma unroll
          for (int e = 0; e < VEC; e += Op::kBytes) Op::apply(cx[it].b + e, y[it].b + e, co.b + e);
        }
        dst[i] = co;
      } else {
        dst[i] = y[it];
      }
    }
  }
}

// How the values rows are dealt out.  The groups of the first list_blocks
// columns of the grid take the innermost lists, each its first cap rows; what a
// longer list holds past them, and the rows that no list covers, fall to windows
// of `window` rows (at most cap), a block each, in the columns after.  So a list
// far longer than the others -- or than max_length, past which rows are only
// cleared -- is spread over the grid.  (512 lists of 8 rows but one of 200,000, 16
// fp32 columns, max_length 16: 2,950 us with each list to one group, 7.4; the add
// 18,200 and 8.7; 500,000 rows past the last list, two jagged dims, 64 columns:
// 1,776 and 32.  A batch without either pays for windows that find nothing: 300
// lists of 20 rows 2.6 us, 2.7.)
struct ListGrid {
  int64_t list_blocks;
  int64_t cap;
  int64_t window;
  int64_t windows;
};

// The list that row x lies in: the last p in [0, n) with off[p] <= x (0 if none).
// A wave's lanes probe 64 offsets per round.
template <typename I>
__device__ __forceinline__ int64_t wave_owner(const JaggedMeta& m, int k, int64_t n, int64_t x) {
  const int lane = threadIdx.x & 63;
  int64_t lo = 0, hi = n;
  while (hi - lo > 1) {  // wave-uniform; the range shrinks whatever the offsets hold
    const int64_t stride = (hi - lo + 63) >> 6, pos = lo + lane * stride;
    const int c = __popcll(__ballot(off_at<I>(m, k, pos < hi ? pos : lo) <= x && pos < hi));
    lo += (c > 0 ? c - 1 : 0) * stride;
    hi = lo + stride < hi ? lo + stride : hi;
  }
  return lo;
}

// Row ranges are clamped to [0, total_L], so malformed offsets never write out
// of bounds.
template <int VEC, typename I, bool ADD, int DT, bool MUL, bool ONE>
__global__ void __launch_bounds__(256)
    jagged_out_kernel(const uint8_t* __restrict__ dense, const uint8_t* __restrict__ x,
                      uint8_t* __restrict__ out, const JaggedMeta m, int64_t nlists,
                      int32_t group_lg, int64_t total_L, int64_t vpr, const ListGrid g) {
  const int32_t lg = ONE ? 8 : group_lg;
  auto clamp = [&](int64_t v, int64_t lo) { return v < lo ? lo : (v > total_L ? total_L : v); };
  const int last = ONE ? 0 : m.ndim - 1;
  const int64_t max_L = m.max_len[last];
  // Of rows [s, e) of list p, whose rows are [r0, r1): how many have a dense row,
  // and the first one's.
  auto place = [&](int64_t p, int64_t r0, int64_t r1, int64_t s, int64_t e, int64_t& row) {
    const int64_t bag = ONE ? p : list_dense_bag<I>(p, m);
    const int64_t left = bag < 0 ? 0 : r0 + (r1 - r0 < max_L ? r1 - r0 : max_L) - s;
    const int64_t copy = left < 0 ? 0 : (left < e - s ? left : e - s);
    row = copy > 0 ? bag * max_L + (s - r0) : 0;
    return copy;
  };
  if (static_cast<int64_t>(blockIdx.x) < g.list_blocks) {  // block-uniform
    const int64_t step = g.list_blocks << (8 - lg);
    for (int64_t p = (static_cast<int64_t>(blockIdx.x) << (8 - lg)) + (threadIdx.x >> lg);
         p < nlists; p += step) {
      const int64_t r0 = clamp(off_at<I>(m, last, p), 0);
      const int64_t r1 = clamp(off_at<I>(m, last, p + 1), r0);
      if (r1 == r0) continue;
      const int64_t e = r1 - r0 < g.cap ? r1 : r0 + g.cap;
      int64_t row;
      const int64_t copy = place(p, r0, r1, r0, e, row);
      emit_rows<VEC, ADD, DT, MUL>(dense, x, out, r0, e, copy, row, vpr, 1 << lg, blockIdx.y,
                                   gridDim.y);
    }
    return;
  }
  const int64_t w = (blockIdx.x - g.list_blocks) * gridDim.y + blockIdx.y;
  if (w >= g.windows) return;
  const int64_t a = w * g.window, b = a + g.window < total_L ? a + g.window : total_L;
  const int64_t head = clamp(off_at<I>(m, last, 0), 0);
  const int64_t tail = clamp(off_at<I>(m, last, nlists), head);
  // The list that row a lies in: only it can reach past its cap here, as one that
  // starts later in the window has its first cap rows in it and beyond.
  int64_t p = 0, r0 = 0, past = b, r1 = 0;
  if (g.cap < total_L && a >= head && a < tail) {
    p = wave_owner<I>(m, last, nlists, a);
    r0 = clamp(off_at<I>(m, last, p), 0);
    r1 = clamp(off_at<I>(m, last, p + 1), r0);
    past = a > r0 + g.cap ? a : r0 + g.cap;
    r1 = r1 < b ? r1 : b;
  }
  if (a >= head && b <= tail && past >= r1) return;  // the usual end
#pragma unroll 1
  for (int i = 0; i < 3; ++i) {  // rows before the first list, past the last, past a cap
    const int64_t s = i == 0 ? a : (i == 2 ? past : (a > tail ? a : tail));
    const int64_t e = i == 0 ? (b < head ? b : head) : (i == 1 ? b : r1);
    int64_t copy = 0, row = 0;
    if (s >= e) continue;
    if (i == 2) copy = place(p, r0, clamp(off_at<I>(m, last, p + 1), r0), s, e, row);
    emit_rows<VEC, ADD, DT, MUL>(dense, x, out, s, e, copy, row, vpr, 256, 0, 1);
  }
}

// ---- host side ------------------------------------------------------------

// Threads per bag (2^lg) and grid: the smallest group that holds a usual bag's
// chunks in one round, kJagItems per thread, up to a block; or one chunk per
// thread, while all bags' threads are on the chip at once (a small call waits for
// its slowest thread).  Bags in x, parts of a large bag in y (the kernels loop
// over what the grid leaves).
struct BagGrid {
  dim3 grid;
  int32_t lg;
};

BagGrid bag_grid(int64_t bags, int64_t usual_chunks, int64_t large_chunks) {
  const int64_t resident = static_cast<int64_t>(num_cus()) * 2048;
  BagGrid g;
  g.lg = 4;
  while (g.lg < 8 && (usual_chunks > (int64_t(kJagItems) << g.lg) ||
                      (usual_chunks > (int64_t(1) << g.lg) && bags << (g.lg + 2) <= resident)))
    g.lg += 2;
  int64_t parts = ceil_div(large_chunks, static_cast<int64_t>(kJagItems) << g.lg);
  parts = parts < 1 ? 1 : (parts > 64 ? 64 : parts);
  int64_t x = ceil_div(bags, int64_t(1) << (8 - g.lg));
  if (x > (int64_t(1) << 30)) x = int64_t(1) << 30;
  g.grid = dim3(static_cast<uint32_t>(x), static_cast<uint32_t>(parts));
  return g;
}

// Jagged outputs: groups by the mean list, parts by max_length within one and two
// means (lists that max_length truncates are cleared whole; a padded dense far
// longer than its lists would launch mostly blocks without rows).  A group takes
// a list of up to eight times that (so that the windows of an ordinary batch, few
// then, find nothing), or an even share of 1024 windows, or any list where all of
// them together are 32 rounds of a group at most.  (2,560 lists of 5 rows of 64
// columns under a max_length of 1000, copied back: 62 us with groups and parts by
// max_length, 5.5; of 25 rows under 50, added in bf16: 17.0 and 10.5.)
BagGrid list_grid(int64_t nlists, int64_t max_L, int64_t total_L, int64_t vpr, ListGrid& lg) {
  const int64_t mean = ceil_div(total_L, nlists > 0 ? nlists : 1);
  int64_t rows = max_L < mean ? mean : (max_L < 2 * mean ? max_L : 2 * mean);
  if (rows * vpr < 16 * kJagItems) rows = ceil_div(16 * kJagItems, vpr);
  BagGrid g = bag_grid(nlists, mean * vpr, rows * vpr);
  const int64_t share = ceil_div(total_L, 1024);
  const int64_t block_rows = ceil_div(8 * 256 * kJagItems, vpr);
  lg.list_blocks = g.grid.x;
  lg.cap = 8 * rows > share ? 8 * rows : share;
  if (total_L * vpr <= (int64_t(32 * kJagItems) << g.lg)) lg.cap = total_L;
  lg.window = share > block_rows ? share : block_rows;
  if (lg.window > lg.cap) lg.window = lg.cap;
  lg.windows = ceil_div(total_L, lg.window);
  g.grid.x += static_cast<uint32_t>(ceil_div(lg.windows, static_cast<int64_t>(g.grid.y)));
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
  const BagGrid g = bag_grid(nbags, max_L * vpr, max_L * vpr);
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
  ListGrid lists;
  const BagGrid g = list_grid(nlists, max_lengths[last], total_L, vpr, lists);
  const bool one = num_jagged_dim == 1 && g.lg == 8;
  if (x_values == nullptr) {
    MX_VEC_SWITCH(vec, {
      constexpr int F = MX_DTYPE_F32;  // a copy: no element type
      const auto kernel = one ? (offset_bytes == 8 ? jagged_out_kernel<V, int64_t, false, F, false, true>
                                                   : jagged_out_kernel<V, int32_t, false, F, false, true>)
                              : (offset_bytes == 8 ? jagged_out_kernel<V, int64_t, false, F, false, false>
                                                   : jagged_out_kernel<V, int32_t, false, F, false, false>);
      kernel<<<g.grid, 256, 0, s>>>(d, nullptr, o, m, nlists, g.lg, total_L, vpr, lists);
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
      kernel<<<g.grid, 256, 0, s>>>(d, x, o, m, nlists, g.lg, total_L, vpr, lists);                    \
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
