// Sparse-feature helpers either side of the TBE lookup, for gfx950: the
// prefix sums that turn lengths into offsets, and the feature permute of a
// [T, B] batch of lengths and indices.
//
// Semantics (fbgemm_gpu sparse ops, recalled):
//  * asynchronous_exclusive_cumsum(x)[i] = x[0] + ... + x[i-1];
//    asynchronous_inclusive_cumsum(x)[i] = x[0] + ... + x[i];
//    asynchronous_complete_cumsum(x) = [0, inclusive...] (n + 1 entries; a
//    2-D input is summed per row).  int32 or int64, in the input's type (two's
//    complement wrap-around, as the integer adds of the GPU op).
//  * permute_2D_sparse_data(permute, lengths [T, B], indices, weights): output
//    feature f is input feature permute[f]: permuted_lengths[f, :] =
//    lengths[permute[f], :], and the indices (and weights) of each bag (f, b)
//    are the input's bag (permute[f], b), in order.  permute may repeat or
//    drop features.  permute_1D_sparse_data is the same with one bag per
//    feature (lengths [T]).
//  * offsets_range(offsets [N], range_size): out[j] = j - offsets[i] for j in
//    segment i = [offsets[i], offsets[i + 1]) (the last ends at range_size).
//  * expand_into_jagged_permute(permute [T], input_offsets, output_offsets,
//    output_size): out[output_offsets[t] + j] = input_offsets[permute[t]] + j
//    for j below output feature t's length.
//
// Design: integer work, HBM-bound.  The scans are reduce-then-scan with no
// waits between blocks: a block sums its 8192-element tile, then every block
// scans its tile from its prefix, the sum of the tiles before it (added up by
// the block itself up to 1024 tiles, beyond that scanned first by one block;
// a batch of one tile takes only the last launch).  A 2-D complete cumsum gives each
// row to one block.  A permute keeps the order of a feature's bags, so each
// output feature is one contiguous copy of an input feature, and only the
// features' sums and their prefixes are needed: one launch sums each feature's
// lengths and copies the permuted lengths, a second copies the data, each of
// its blocks building the prefixes in LDS.  (40 features x 4096 bags, 1.6M
// int64 indices with weights, the new offsets' cumsum included: 50 us with a
// permute launch, two cumsums and a copy per bag, 27 this way; 3 x 16 bags 28.5
// -> 18.3, 800 x 16 bags 37 -> 31.)  Batches of more than kPermMaxT features take that longer
// way: one 16-lane group per output bag, from the two complete cumsums.
#include <type_traits>

#include "mx_common.h"

namespace mx {
namespace {

constexpr int kCsThreads = 1024;
constexpr int kCsItems = 8;
constexpr int64_t kCsTile = static_cast<int64_t>(kCsThreads) * kCsItems;

// Sums in the type's own wrap-around arithmetic (signed overflow is not
// defined in C++: add as unsigned).
template <typename T>
__device__ __forceinline__ T wadd(T a, T b) {
  using U = std::make_unsigned_t<T>;
  return static_cast<T>(static_cast<U>(a) + static_cast<U>(b));
}

template <typename T>
__device__ __forceinline__ T wsub(T a, T b) {
  using U = std::make_unsigned_t<T>;
  return static_cast<T>(static_cast<U>(a) - static_cast<U>(b));
}

// Exclusive scan of one value per thread over a block of kCsThreads; the
// block's total in *total.
template <typename T>
__device__ __forceinline__ T block_excl(T v, T* total) {
  __shared__ T wsum[kCsThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  T incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T o = __shfl_up(incl, d, 64);
    if (lane >= d) incl = wadd(incl, o);
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  T before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < kCsThreads / 64; ++i) {
    if (i < w) before = wadd(before, wsum[i]);
    all = wadd(all, wsum[i]);
  }
  __syncthreads();  // wsum is reused by the next call
  *total = all;
  return wsub(wadd(before, incl), v);
}

// A tile's sum: wrap-around integer sums do not depend on the order, so each
// thread adds a strided slice and every load instruction is coalesced.
template <typename T>
__global__ void __launch_bounds__(kCsThreads)
    cumsum_tile_kernel(const T* __restrict__ x, int64_t n, T* __restrict__ partial) {
  const int64_t tile0 = static_cast<int64_t>(blockIdx.x) * kCsTile;
  T s = 0;
#pragma unroll
  for (int it = 0; it < kCsItems; ++it) {
    const int64_t i = tile0 + it * kCsThreads + threadIdx.x;
    if (i < n) s = wadd(s, x[i]);
  }
  T total;
  (void)block_excl<T>(s, &total);
  if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// One block: the tile sums into their exclusive prefixes, in place.
template <typename T>
__global__ void __launch_bounds__(kCsThreads) cumsum_spine_kernel(T* __restrict__ partial,
                                                                   int64_t ntiles) {
  T carry = 0;
  for (int64_t c = 0; c < ntiles; c += kCsThreads) {
    const int64_t i = c + threadIdx.x;
    const T v = i < ntiles ? partial[i] : T(0);
    T total;
    const T ex = block_excl<T>(v, &total);
    if (i < ntiles) partial[i] = wadd(carry, ex);
    carry = wadd(carry, total);
  }
}

// KIND 0 exclusive, 1 inclusive, 2 complete (out[0] = 0, out[i + 1] = inclusive[i]).
// The tile passes through LDS both ways, so that the global loads and stores
// are coalesced while each thread scans kCsItems consecutive elements; a row
// of kCsItems elements takes kCsPad slots (fewer bank conflicts).
constexpr int kCsPad = kCsItems + 1;
__device__ __forceinline__ int cs_slot(int j) { return (j / kCsItems) * kCsPad + j % kCsItems; }

// prefix: null (one tile), the tiles' exclusive prefixes, or with `raw` the
// tiles' sums (at most kCsThreads tiles), which each block adds up to its own.
template <typename T, int KIND>
__global__ void __launch_bounds__(kCsThreads)
    cumsum_scan_kernel(const T* __restrict__ x, int64_t n, const T* __restrict__ prefix,
                       bool raw, T* __restrict__ out) {
  __shared__ T s_buf[kCsThreads * kCsPad];
  const int64_t tile0 = static_cast<int64_t>(blockIdx.x) * kCsTile;
  T pre = 0;
  if (raw) {  // block-uniform
    (void)block_excl<T>(threadIdx.x < blockIdx.x ? prefix[threadIdx.x] : T(0), &pre);
  } else if (prefix) {
    pre = prefix[blockIdx.x];
  }
#pragma unroll
  for (int it = 0; it < kCsItems; ++it) {
    const int j = it * kCsThreads + threadIdx.x;
    s_buf[cs_slot(j)] = tile0 + j < n ? x[tile0 + j] : T(0);
  }
  __syncthreads();
  T v[kCsItems];
  T s = 0;
#pragma unroll
  for (int it = 0; it < kCsItems; ++it) {
    v[it] = s_buf[threadIdx.x * kCsPad + it];
    s = wadd(s, v[it]);
  }
  T total;
  // block_excl's barriers also order every thread's reads above before the
  // writes below.
  T run = wadd(block_excl<T>(s, &total), pre);
#pragma unroll
  for (int it = 0; it < kCsItems; ++it) {
    const T before = run;
    run = wadd(run, v[it]);
    s_buf[threadIdx.x * kCsPad + it] = KIND == 0 ? before : run;
  }
  __syncthreads();
  if (KIND == 2 && blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0;
#pragma unroll
  for (int it = 0; it < kCsItems; ++it) {
    const int j = it * kCsThreads + threadIdx.x;
    if (tile0 + j < n) out[tile0 + j + (KIND == 2 ? 1 : 0)] = s_buf[cs_slot(j)];
  }
}

// 2-D complete cumsum: block r scans row r of x [rows, n] into out [rows, n + 1].
template <typename T>
__global__ void __launch_bounds__(kCsThreads)
    cumsum_rows_kernel(const T* __restrict__ x, int64_t n, T* __restrict__ out) {
  const T* xr = x + static_cast<int64_t>(blockIdx.x) * n;
  T* orow = out + static_cast<int64_t>(blockIdx.x) * (n + 1);
  if (threadIdx.x == 0) orow[0] = 0;
  T carry = 0;
  for (int64_t c = 0; c < n; c += kCsTile) {
    const int64_t base = c + threadIdx.x * kCsItems;
    T v[kCsItems];
    T s = 0;
#pragma unroll
    for (int it = 0; it < kCsItems; ++it) {
      v[it] = base + it < n ? xr[base + it] : T(0);
      s = wadd(s, v[it]);
    }
    T total;
    T run = wadd(block_excl<T>(s, &total), carry);
#pragma unroll
    for (int it = 0; it < kCsItems; ++it) {
      if (base + it >= n) break;
      run = wadd(run, v[it]);
      orow[base + it + 1] = run;
    }
    carry = wadd(carry, total);
  }
}

template <typename T>
int cumsum_t(const T* x, int64_t n, int32_t kind, T* out, T* partial, hipStream_t s) {
  const int64_t nt = ceil_div(n > 0 ? n : 1, kCsTile);  // n = 0: one block writes out[0]
  MX_REQUIRE(nt <= 0x7fffffffll, "cumsum of %lld elements too long", (long long)n);
  const dim3 gd(static_cast<uint32_t>(nt));
  const T* prefix = nullptr;
  // Up to kCsThreads tiles each scan block adds the tile sums before its own
  // (one launch fewer than the spine kernel, which scans them beyond that).
  const bool raw = nt > 1 && nt <= kCsThreads;
  if (nt > 1) {
    cumsum_tile_kernel<T><<<gd, kCsThreads, 0, s>>>(x, n, partial);
    if (!raw) cumsum_spine_kernel<T><<<1, kCsThreads, 0, s>>>(partial, nt);
    prefix = partial;
  }
  if (kind == 0)
    cumsum_scan_kernel<T, 0><<<gd, kCsThreads, 0, s>>>(x, n, prefix, raw, out);
  else if (kind == 1)
    cumsum_scan_kernel<T, 1><<<gd, kCsThreads, 0, s>>>(x, n, prefix, raw, out);
  else
    cumsum_scan_kernel<T, 2><<<gd, kCsThreads, 0, s>>>(x, n, prefix, raw, out);
  MX_LAUNCH_CHECK();
  return MX_OK;
}

// ---- permute_2D_sparse_data --------------------------------------------------

template <typename L>
__global__ void __launch_bounds__(256)
    permute_lengths_kernel(const int32_t* __restrict__ permute, const L* __restrict__ lengths,
                           int32_t T, int64_t B, int64_t Tp, L* __restrict__ out) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < Tp * B;
       i += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t f = i / B, b = i - f * B;
    const int32_t src = permute[f];
    out[i] = src >= 0 && src < T ? lengths[static_cast<int64_t>(src) * B + b] : L(0);
  }
}

// A 16-lane group per output bag (f, b): copies the input bag (permute[f], b).
template <typename L, typename I, typename W>
__global__ void __launch_bounds__(256)
    permute_data_kernel(const int32_t* __restrict__ permute, const L* __restrict__ in_off,
                        const L* __restrict__ out_off, int32_t T, int64_t B, int64_t Tp,
                        const I* __restrict__ indices, const W* __restrict__ weights,
                        int64_t in_len, I* __restrict__ out_indices, W* __restrict__ out_weights,
                        int64_t out_len) {
  constexpr int G = 16;
  const int k = threadIdx.x % G;
  const int64_t ngrp = static_cast<int64_t>(gridDim.x) * (256 / G);
  for (int64_t bag = static_cast<int64_t>(blockIdx.x) * (256 / G) + threadIdx.x / G;
       bag < Tp * B; bag += ngrp) {
    const int64_t f = bag / B, b = bag - f * B;
    const int32_t src = permute[f];
    if (src < 0 || src >= T) continue;  // its length is 0
    const int64_t s0 = static_cast<int64_t>(in_off[static_cast<int64_t>(src) * B + b]);
    const int64_t d0 = static_cast<int64_t>(out_off[bag]);
    const int64_t len = static_cast<int64_t>(out_off[bag + 1]) - d0;
    if (s0 < 0 || d0 < 0) continue;  // negative lengths upstream: nothing in bounds to copy
    for (int64_t j = k; j < len; j += G) {
      // Lengths that disagree with the index count or the given output size
      // stop the copy instead of reading or writing past either array.
      if (d0 + j >= out_len || s0 + j >= in_len) break;
      out_indices[d0 + j] = indices[s0 + j];
      if (weights) out_weights[d0 + j] = weights[s0 + j];
    }
  }
}

// Features whose sums fit a block's LDS, lengths summed per block, and the sums
// a block of the copy adds up itself.  Many features of a few bags each are
// cheaper by the cumsums, of one tile each then, than by every block's prefixes
// (1000 features of 4 bags 13.8 us, 16.7 by feature; of 16 bags 23.8 and 16.9).
constexpr int64_t kPermMaxT = 1024;
constexpr int64_t kPermPart = 8192;
constexpr int64_t kPermMaxSums = 8192;

int64_t perm_parts(int64_t B) { return ceil_div(B, kPermPart); }

bool perm_by_feature(int64_t T, int64_t Tp, int64_t B) {
  return T >= 1 && T <= kPermMaxT && Tp >= 1 && Tp <= kPermMaxT && B >= 1 &&
         (B >= 16 || (T <= kPermMaxT / 2 && Tp <= kPermMaxT / 2)) &&
         T * perm_parts(B) <= kPermMaxSums;
}

// Blocks [0, T * parts): the sum of part p of feature t's lengths.  The blocks
// after them: the permuted lengths, part p of output feature f.
template <typename L>
__global__ void __launch_bounds__(kCsThreads)
    permute_sums_kernel(const int32_t* __restrict__ permute, const L* __restrict__ lengths,
                        int32_t T, int64_t B, int32_t parts, L* __restrict__ out,
                        int64_t* __restrict__ sums) {
  const int64_t bid = blockIdx.x, nsum = static_cast<int64_t>(T) * parts;
  const bool sum = bid < nsum;  // block-uniform
  const int64_t x = sum ? bid : bid - nsum;
  const int64_t f = x / parts, b0 = (x - f * parts) * kPermPart;
  const int64_t b1 = b0 + kPermPart < B ? b0 + kPermPart : B;
  const int64_t src = sum ? f : static_cast<int64_t>(permute[f]);
  const bool valid = src >= 0 && src < T;
  L v[kPermPart / kCsThreads];
  int64_t s = 0;
#pragma unroll
  for (int it = 0; it < kPermPart / kCsThreads; ++it) {
    const int64_t b = b0 + it * kCsThreads + threadIdx.x;
    v[it] = valid && b < b1 ? lengths[src * B + b] : L(0);
    s += static_cast<int64_t>(v[it]);
  }
  if (sum) {
    int64_t total;
    (void)block_excl<int64_t>(s, &total);
    if (threadIdx.x == 0) sums[bid] = total;
    return;
  }
#pragma unroll
  for (int it = 0; it < kPermPart / kCsThreads; ++it) {
    const int64_t b = b0 + it * kCsThreads + threadIdx.x;
    if (b < b1) out[f * B + b] = v[it];
  }
}

constexpr int kPermThreads = 256;
constexpr int kPermOwn = kPermMaxT / kPermThreads;  // features per thread in the prefixes

// start[i] = val[0] + ... + val[i-1] for i <= n (n <= kPermMaxT), in LDS.
__device__ __forceinline__ void perm_starts(const int64_t* val, int32_t n, int64_t* start) {
  __shared__ int64_t wsum[kPermThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int32_t i0 = threadIdx.x * kPermOwn;
  int64_t own = 0;
#pragma unroll
  for (int i = 0; i < kPermOwn; ++i) own += i0 + i < n ? val[i0 + i] : 0;
  int64_t incl = own;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int64_t o = __shfl_up(incl, d, 64);
    if (lane >= d) incl += o;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int64_t at = incl - own;
  for (int i = 0; i < w; ++i) at += wsum[i];
#pragma unroll
  for (int i = 0; i < kPermOwn; ++i)
    if (i0 + i < n) {
      start[i0 + i] = at;
      at += val[i0 + i];
      if (i0 + i == n - 1) start[n] = at;
    }
  __syncthreads();
}

struct PermPrefixes {
  int64_t val[kPermMaxT];        // a feature's sum, input then output
  int64_t in[kPermMaxT + 1];     // first index of each input feature
  int64_t out[kPermMaxT + 1];    // first index of each output feature
};

__device__ __forceinline__ void perm_prefixes(const int32_t* __restrict__ permute, int32_t T,
                                              int32_t Tp, int32_t parts,
                                              const int64_t* __restrict__ sums, PermPrefixes& m) {
  for (int32_t t = threadIdx.x; t < T; t += kPermThreads) {
    int64_t s = 0;
    for (int32_t p = 0; p < parts; ++p) s += sums[static_cast<int64_t>(t) * parts + p];
    m.val[t] = s;
  }
  __syncthreads();
  perm_starts(m.val, T, m.in);
  int64_t mine[kPermOwn];
#pragma unroll
  for (int i = 0; i < kPermOwn; ++i) {
    const int32_t f = i * kPermThreads + static_cast<int32_t>(threadIdx.x);
    const int32_t src = f < Tp ? permute[f] : -1;
    mine[i] = src >= 0 && src < T ? m.val[src] : 0;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPermOwn; ++i) {
    const int32_t f = i * kPermThreads + static_cast<int32_t>(threadIdx.x);
    if (f < Tp) m.val[f] = mine[i];
  }
  __syncthreads();
  perm_starts(m.val, Tp, m.out);
}

// The permuted lengths' sum (the output's size).
__global__ void __launch_bounds__(kPermThreads)
    permute_total_kernel(const int32_t* __restrict__ permute, int32_t T, int32_t Tp, int32_t parts,
                         const int64_t* __restrict__ sums, int64_t* __restrict__ total) {
  __shared__ PermPrefixes m;
  perm_prefixes(permute, T, Tp, parts, sums, m);
  if (threadIdx.x == 0) *total = m.out[Tp];
}

// Copies out[o0, o1) from in + (s0 - o0): 16 bytes per thread and step, at the
// element type's own alignment.
template <typename E>
__device__ __forceinline__ void perm_copy(const E* __restrict__ in, E* __restrict__ out,
                                          int64_t o0, int64_t o1, int64_t shift) {
  constexpr int V = 16 / sizeof(E), K = 4;
  typedef E EV __attribute__((ext_vector_type(V), aligned(sizeof(E))));
  for (int64_t base = o0; base < o1; base += kPermThreads * V * K) {
    EV x[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t o = base + (k * kPermThreads + static_cast<int64_t>(threadIdx.x)) * V;
      if (o + V <= o1) {
        x[k] = *reinterpret_cast<const EV*>(in + o + shift);
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v) x[k][v] = o + v < o1 ? in[o + v + shift] : E(0);
      }
    }
    // Once, and not again before each store behind the store before it (100
    // features of 8192 bags 110.7 -> 101.0 us, 40 of 4096 26.9 -> 26.3).
    wait_loads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t o = base + (k * kPermThreads + static_cast<int64_t>(threadIdx.x)) * V;
      if (o + V <= o1) {
        *reinterpret_cast<EV*>(out + o) = x[k];
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v)
          if (o + v < o1) out[o + v] = x[k][v];
      }
    }
  }
}

// A block copies the output's indices [blockIdx * chunk, + chunk): the parts of
// the output features it meets, one contiguous copy each where they are long,
// else element by element, each finding its feature in the prefixes.  Lengths
// that disagree with the index count or the given output size stop the copy
// instead of reading or writing past either array.
template <typename I>
__global__ void __launch_bounds__(kPermThreads)
    permute_copy_kernel(const int32_t* __restrict__ permute, int32_t T, int32_t Tp, int32_t parts,
                        const int64_t* __restrict__ sums, const I* __restrict__ indices,
                        const float* __restrict__ weights, int64_t in_len, int64_t chunk,
                        I* __restrict__ out_indices, float* __restrict__ out_weights,
                        int64_t out_len) {
  __shared__ PermPrefixes m;
  perm_prefixes(permute, T, Tp, parts, sums, m);
  const int64_t total = m.out[Tp] < out_len ? m.out[Tp] : out_len;
  const int64_t c0 = blockIdx.x * chunk, c1 = c0 + chunk < total ? c0 + chunk : total;
  if (c0 >= c1) return;  // block-uniform
  auto feature = [&](int64_t o) {  // the last f with out[f] <= o
    int32_t lo = 0, hi = Tp;
    while (hi - lo > 1) {
      const int32_t mid = lo + ((hi - lo) >> 1);
      if (m.out[mid] <= o)
        lo = mid;
      else
        hi = mid;
    }
    return lo;
  };
  const int32_t f0 = feature(c0), f1 = feature(c1 - 1);
  // Block-uniform: a few features, each a round of a copy or more; fewer indices
  // than that find their features a thread each, all at once (3 features of one bag
  // 11.1 -> 6.7 us).
  if (f0 == f1 || (f1 - f0 < 4 && c1 - c0 > kPermThreads)) {
    for (int32_t f = f0; f <= f1; ++f) {
      const int32_t src = permute[f];
      if (src < 0 || src >= T) continue;  // its length is 0
      const int64_t s0 = m.in[src], d0 = m.out[f];
      if (s0 < 0 || d0 < 0) continue;  // negative lengths upstream: nothing in bounds to copy
      const int64_t shift = s0 - d0;
      const int64_t o0 = c0 > d0 ? c0 : d0;
      int64_t o1 = m.out[f + 1] < c1 ? m.out[f + 1] : c1;
      o1 = o1 < in_len - shift ? o1 : in_len - shift;
      if (o0 >= o1) continue;
      perm_copy<I>(indices, out_indices, o0, o1, shift);
      if (weights) perm_copy<float>(weights, out_weights, o0, o1, shift);
    }
    return;
  }
  for (int64_t o = c0 + threadIdx.x; o < c1; o += kPermThreads) {
    const int32_t f = feature(o), src = permute[f];
    if (src < 0 || src >= T || m.in[src] < 0 || m.out[f] < 0) continue;
    const int64_t i = m.in[src] + (o - m.out[f]);
    if (i < 0 || i >= in_len) continue;
    out_indices[o] = indices[i];
    if (weights) out_weights[o] = weights[i];
  }
}

// A 16-lane group per segment writes j - start over its range.
template <typename I>
__global__ void __launch_bounds__(256)
    offsets_range_kernel(const I* __restrict__ offsets, int64_t nseg, int64_t range_size,
                         I* __restrict__ out) {
  constexpr int G = 16;
  const int k = threadIdx.x % G;
  const int64_t ngrp = static_cast<int64_t>(gridDim.x) * (256 / G);
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * (256 / G) + threadIdx.x / G; i < nseg;
       i += ngrp) {
    int64_t s0 = static_cast<int64_t>(offsets[i]);
    int64_t s1 = i + 1 < nseg ? static_cast<int64_t>(offsets[i + 1]) : range_size;
    s0 = s0 < 0 ? 0 : s0;
    s1 = s1 > range_size ? range_size : s1;
    for (int64_t j = s0 + k; j < s1; j += G) out[j] = static_cast<I>(j - s0);
  }
}

// A 16-lane group per output feature t.
template <typename I>
__global__ void __launch_bounds__(256)
    expand_permute_kernel(const int32_t* __restrict__ permute, const I* __restrict__ in_off,
                          int64_t in_n, const I* __restrict__ out_off, int64_t T, bool out_has_end,
                          int64_t output_size, I* __restrict__ out) {
  constexpr int G = 16;
  const int k = threadIdx.x % G;
  const int64_t ngrp = static_cast<int64_t>(gridDim.x) * (256 / G);
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * (256 / G) + threadIdx.x / G; t < T;
       t += ngrp) {
    const int32_t src = permute[t];
    if (src < 0 || src >= in_n) continue;
    int64_t d0 = static_cast<int64_t>(out_off[t]);
    int64_t d1 = out_has_end || t + 1 < T ? static_cast<int64_t>(out_off[t + 1]) : output_size;
    d0 = d0 < 0 ? 0 : d0;
    d1 = d1 > output_size ? output_size : d1;
    const int64_t s0 = static_cast<int64_t>(in_off[src]);
    for (int64_t j = d0 + k; j < d1; j += G) out[j] = static_cast<I>(s0 + (j - d0));
  }
}

int grid_for(int64_t work, int64_t per_block) {
  const int64_t want = ceil_div(work > 0 ? work : 1, per_block);
  const int64_t cap = static_cast<int64_t>(num_cus()) * 16;
  return static_cast<int>(want < cap ? want : cap);
}

}  // namespace
}  // namespace mx

using namespace mx;

extern "C" size_t mx_cumsum_workspace_bytes(int64_t n, int32_t elem_bytes) {
  const int64_t nt = ceil_div(n > 0 ? n : 1, kCsTile);
  return static_cast<size_t>(nt) * static_cast<size_t>(elem_bytes > 0 ? elem_bytes : 8);
}

extern "C" int mx_cumsum(const void* in, int32_t elem_bytes, int64_t rows, int64_t n,
                         int32_t kind, void* out, void* workspace, size_t workspace_bytes,
                         void* stream) {
  clear_error();
  MX_REQUIRE(elem_bytes == 4 || elem_bytes == 8, "cumsum needs int32 or int64 elements");
  MX_REQUIRE(kind >= 0 && kind <= 2, "cumsum kind %d (0 exclusive, 1 inclusive, 2 complete)",
             kind);
  MX_REQUIRE(rows >= 1 && n >= 0, "cumsum of %lld rows of %lld", (long long)rows, (long long)n);
  MX_REQUIRE(rows == 1 || kind == 2, "a 2-D cumsum is complete only");
  auto* s = as_stream(stream);
  if (rows > 1) {
    MX_REQUIRE(rows <= 0x7fffffffll, "too many rows");
    MX_REQUIRE(out && (n == 0 || in), "null pointer argument");
    const dim3 gd(static_cast<uint32_t>(rows));
    if (elem_bytes == 8)
      cumsum_rows_kernel<int64_t><<<gd, kCsThreads, 0, s>>>(static_cast<const int64_t*>(in), n,
                                                            static_cast<int64_t*>(out));
    else
      cumsum_rows_kernel<int32_t><<<gd, kCsThreads, 0, s>>>(static_cast<const int32_t*>(in), n,
                                                            static_cast<int32_t*>(out));
    MX_LAUNCH_CHECK();
    return MX_OK;
  }
  if (n == 0) {
    if (kind != 2) return MX_OK;
    MX_REQUIRE(out, "null pointer argument");
    return elem_bytes == 8 ? cumsum_t<int64_t>(nullptr, 0, 2, static_cast<int64_t*>(out), nullptr, s)
                           : cumsum_t<int32_t>(nullptr, 0, 2, static_cast<int32_t*>(out), nullptr, s);
  }
  MX_REQUIRE(in && out, "null pointer argument");
  const int64_t nt = ceil_div(n, kCsTile);  // n > 0 here
  if (nt > 1 && (workspace == nullptr || workspace_bytes < mx_cumsum_workspace_bytes(n, elem_bytes)))
    return set_error(MX_EWORKSPACE, "workspace of %zu bytes needed",
                     mx_cumsum_workspace_bytes(n, elem_bytes));
  if (elem_bytes == 8)
    return cumsum_t<int64_t>(static_cast<const int64_t*>(in), n, kind, static_cast<int64_t*>(out),
                             static_cast<int64_t*>(workspace), s);
  return cumsum_t<int32_t>(static_cast<const int32_t*>(in), n, kind, static_cast<int32_t*>(out),
                           static_cast<int32_t*>(workspace), s);
}

extern "C" int mx_permute_2d_lengths(const int32_t* permute, int64_t T_out, const void* lengths,
                                     int32_t length_bytes, int32_t T, int64_t B,
                                     void* permuted_lengths, void* stream) {
  clear_error();
  MX_REQUIRE(length_bytes == 4 || length_bytes == 8, "lengths must be int32 or int64");
  MX_REQUIRE(T >= 0 && B >= 0 && T_out >= 0, "negative size");
  if (T_out * B == 0) return MX_OK;
  MX_REQUIRE(permute && permuted_lengths && (T == 0 || lengths), "null pointer argument");
  auto* s = as_stream(stream);
  const dim3 gd(static_cast<uint32_t>(grid_for(T_out * B, 256)));
  if (length_bytes == 8)
    permute_lengths_kernel<int64_t><<<gd, 256, 0, s>>>(permute, static_cast<const int64_t*>(lengths),
                                                       T, B, T_out,
                                                       static_cast<int64_t*>(permuted_lengths));
  else
    permute_lengths_kernel<int32_t><<<gd, 256, 0, s>>>(permute, static_cast<const int32_t*>(lengths),
                                                       T, B, T_out,
                                                       static_cast<int32_t*>(permuted_lengths));
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_permute_2d_data(const int32_t* permute, int64_t T_out, int32_t T, int64_t B,
                                  const void* input_offsets, const void* output_offsets,
                                  int32_t offset_bytes, const void* indices, int32_t index_bytes,
                                  int64_t in_len, const float* weights, int64_t out_len,
                                  void* permuted_indices, float* permuted_weights,
                                  void* stream) {
  clear_error();
  MX_REQUIRE(offset_bytes == 4 || offset_bytes == 8, "offsets must be int32 or int64");
  MX_REQUIRE(index_bytes == 4 || index_bytes == 8, "indices must be int32 or int64");
  MX_REQUIRE(T >= 0 && B >= 0 && T_out >= 0 && out_len >= 0 && in_len >= 0, "negative size");
  MX_REQUIRE(!weights == !permuted_weights, "weights and permuted_weights go together");
  if (T_out * B == 0 || out_len == 0) return MX_OK;
  MX_REQUIRE(permute && input_offsets && output_offsets && indices && permuted_indices,
             "null pointer argument");
  auto* s = as_stream(stream);
  const dim3 gd(static_cast<uint32_t>(grid_for(T_out * B, 256 / 16)));
#define MX_PERM(L, I)                                                                       \
  permute_data_kernel<L, I, float><<<gd, 256, 0, s>>>(                                      \
      permute, static_cast<const L*>(input_offsets), static_cast<const L*>(output_offsets), \
      T, B, T_out, static_cast<const I*>(indices), weights, in_len,                          \
      static_cast<I*>(permuted_indices), permuted_weights, out_len)
  if (offset_bytes == 8) {
    if (index_bytes == 8)
      MX_PERM(int64_t, int64_t);
    else
      MX_PERM(int64_t, int32_t);
  } else {
    if (index_bytes == 8)
      MX_PERM(int32_t, int64_t);
    else
      MX_PERM(int32_t, int32_t);
  }
#undef MX_PERM
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" size_t mx_permute_2d_workspace_bytes(int64_t T_out, int32_t T, int64_t B) {
  if (!perm_by_feature(T, T_out, B)) return 0;
  return static_cast<size_t>(T * perm_parts(B)) * sizeof(int64_t);
}

extern "C" int mx_permute_2d_sums(const int32_t* permute, int64_t T_out, const void* lengths,
                                  int32_t length_bytes, int32_t T, int64_t B,
                                  void* permuted_lengths, void* workspace,
                                  size_t workspace_bytes, int64_t* total, void* stream) {
  clear_error();
  MX_REQUIRE(length_bytes == 4 || length_bytes == 8, "lengths must be int32 or int64");
  MX_REQUIRE(T >= 0 && B >= 0 && T_out >= 0, "negative size");
  MX_REQUIRE(perm_by_feature(T, T_out, B), "too many features (or none) for sums per feature");
  MX_REQUIRE(permute && permuted_lengths && lengths, "null pointer argument");
  const size_t need = mx_permute_2d_workspace_bytes(T_out, T, B);
  if (workspace == nullptr || workspace_bytes < need)
    return set_error(MX_EWORKSPACE, "workspace of %zu bytes needed", need);
  auto* s = as_stream(stream);
  const int32_t parts = static_cast<int32_t>(perm_parts(B));
  const dim3 gd(static_cast<uint32_t>((T + T_out) * parts));
  auto* sums = static_cast<int64_t*>(workspace);
  if (length_bytes == 8)
    permute_sums_kernel<int64_t><<<gd, kCsThreads, 0, s>>>(
        permute, static_cast<const int64_t*>(lengths), T, B, parts,
        static_cast<int64_t*>(permuted_lengths), sums);
  else
    permute_sums_kernel<int32_t><<<gd, kCsThreads, 0, s>>>(
        permute, static_cast<const int32_t*>(lengths), T, B, parts,
        static_cast<int32_t*>(permuted_lengths), sums);
  MX_LAUNCH_CHECK();
  if (total) {
    permute_total_kernel<<<1, kPermThreads, 0, s>>>(permute, T, static_cast<int32_t>(T_out), parts,
                                                    sums, total);
    MX_LAUNCH_CHECK();
  }
  return MX_OK;
}

extern "C" int mx_permute_2d_copy(const int32_t* permute, int64_t T_out, int32_t T, int64_t B,
                                  const void* workspace, const void* indices, int32_t index_bytes,
                                  int64_t in_len, const float* weights, int64_t out_len,
                                  void* permuted_indices, float* permuted_weights,
                                  void* stream) {
  clear_error();
  MX_REQUIRE(index_bytes == 4 || index_bytes == 8, "indices must be int32 or int64");
  MX_REQUIRE(T >= 0 && B >= 0 && T_out >= 0 && out_len >= 0 && in_len >= 0, "negative size");
  MX_REQUIRE(perm_by_feature(T, T_out, B), "too many features (or none) for sums per feature");
  MX_REQUIRE(!weights == !permuted_weights, "weights and permuted_weights go together");
  if (out_len == 0) return MX_OK;
  MX_REQUIRE(permute && workspace && indices && permuted_indices, "null pointer argument");
  auto* s = as_stream(stream);
  // Per block one index per thread up to two blocks per CU (a block over many short
  // features searches for each of its indices in turn: 300 features of 4 bags 17.4
  // us with 2048 per block, 10.8), then up to 2048, then no more than eight blocks
  // per CU, whose prefixes cost more than a copy of that size.
  const int64_t cus = num_cus();
  const int64_t small = ceil_div(ceil_div(out_len, cus * 2), kPermThreads) * kPermThreads;
  const int64_t chunk =
      small < 2048 ? small : ceil_div(ceil_div(out_len, cus * 8), 2048) * 2048;
  const dim3 gd(static_cast<uint32_t>(ceil_div(out_len, chunk)));
  const int32_t parts = static_cast<int32_t>(perm_parts(B)), Tp = static_cast<int32_t>(T_out);
  const auto* sums = static_cast<const int64_t*>(workspace);
  if (index_bytes == 8)
    permute_copy_kernel<int64_t><<<gd, kPermThreads, 0, s>>>(
        permute, T, Tp, parts, sums, static_cast<const int64_t*>(indices), weights, in_len, chunk,
        static_cast<int64_t*>(permuted_indices), permuted_weights, out_len);
  else
    permute_copy_kernel<int32_t><<<gd, kPermThreads, 0, s>>>(
        permute, T, Tp, parts, sums, static_cast<const int32_t*>(indices), weights, in_len, chunk,
        static_cast<int32_t*>(permuted_indices), permuted_weights, out_len);
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_offsets_range(const void* offsets, int32_t index_bytes, int64_t nseg,
                                int64_t range_size, void* out, void* stream) {
  clear_error();
  MX_REQUIRE(index_bytes == 4 || index_bytes == 8, "offsets must be int32 or int64");
  MX_REQUIRE(nseg >= 0 && range_size >= 0, "negative size");
  if (nseg == 0 || range_size == 0) return MX_OK;
  MX_REQUIRE(offsets && out, "null pointer argument");
  auto* s = as_stream(stream);
  const dim3 gd(static_cast<uint32_t>(grid_for(nseg, 256 / 16)));
  if (index_bytes == 8)
    offsets_range_kernel<int64_t><<<gd, 256, 0, s>>>(static_cast<const int64_t*>(offsets), nseg,
                                                     range_size, static_cast<int64_t*>(out));
  else
    offsets_range_kernel<int32_t><<<gd, 256, 0, s>>>(static_cast<const int32_t*>(offsets), nseg,
                                                     range_size, static_cast<int32_t*>(out));
  MX_LAUNCH_CHECK();
  return MX_OK;
}

extern "C" int mx_expand_into_jagged_permute(const int32_t* permute, int64_t T,
                                             const void* input_offsets, int64_t input_numel,
                                             const void* output_offsets, int64_t output_numel,
                                             int32_t index_bytes, int64_t output_size, void* out,
                                             void* stream) {
  clear_error();
  MX_REQUIRE(index_bytes == 4 || index_bytes == 8, "offsets must be int32 or int64");
  MX_REQUIRE(T >= 0 && output_size >= 0, "negative size");
  MX_REQUIRE(output_numel == T || output_numel == T + 1,
             "output_offsets must have T or T+1 entries (T=%lld, got %lld)", (long long)T,
             (long long)output_numel);
  if (T == 0 || output_size == 0) return MX_OK;
  MX_REQUIRE(permute && input_offsets && output_offsets && out, "null pointer argument");
  auto* s = as_stream(stream);
  const dim3 gd(static_cast<uint32_t>(grid_for(T, 256 / 16)));
  const bool has_end = output_numel == T + 1;
  if (index_bytes == 8)
    expand_permute_kernel<int64_t><<<gd, 256, 0, s>>>(
        permute, static_cast<const int64_t*>(input_offsets), input_numel,
        static_cast<const int64_t*>(output_offsets), T, has_end, output_size,
        static_cast<int64_t*>(out));
  else
    expand_permute_kernel<int32_t><<<gd, 256, 0, s>>>(
        permute, static_cast<const int32_t*>(input_offsets), input_numel,
        static_cast<const int32_t*>(output_offsets), T, has_end, output_size,
        static_cast<int32_t*>(out));
  MX_LAUNCH_CHECK();
  return MX_OK;
}
