// Exact top-k (k <= 128) of short rows (at most 2048 elements; with many rows
// 8192 for k <= 16 and 4096 for k <= 32) for gfx950.
//
// A 1024-thread select workgroup per row (row_select.hip) spends its fixed
// latency on a few hundred elements ([65536, 128] f32, k = 8: 1444 us), so short
// rows are ordered whole, many to a workgroup.  The select key orders values as
// the reference's strict `>` admits them (tallax/_src/top_k.py:64: -0 == +0, NaN
// below -inf), ties by lowest column; values at or below finfo(dtype).min, and
// NaNs, come out as finfo.min.
//   * k <= 32 (topk_lanes_route): topk_lanes_kernel, 1 to 64 lanes per row, each keeping the
//     largest 8, 16 or 32 of its own elements, then merging them across the
//     row's lanes;
//   * other rows: block_bitonic_sort_c over P = 64 .. 2048 slots, E records
//     per thread (one wave up to P = 512, then 128 and 256 threads).
#include <stdint.h>

#include "tallax_hip.h"
#include "tx_block_sort.h"
#include "tx_common.h"
#include "tx_host.h"

namespace tx {

constexpr int kTopkShortCols = 2048;  // whole-row networks
constexpr int kLanesMaxCols = 8192;
constexpr int kLanesMaxK = 32;

// topk_lanes_kernel, against the select kernel (row_select.hip) and the whole-row
// networks: its fixed part grows with k (about 3, 4.5 and 7 us for lists of 8,
// 16 and 32), its cost per row is the lowest, so the line lies where the rows
// outweigh it (f32, others -> lanes, us).  k <= 8: [16, 256] 5.2 -> 3.4,
// [256, 2048] 6.8 -> 6.3, [1024, 4096] 24.6 -> 10.6, but [256, 4096] 7.1 -> 9.6;
// rows the one-wave networks of 64 and 128 slots take: [1, 64] 2.3 -> 3.4,
// [2000, 64] 3.1 -> 3.6, [3000, 64] 3.5 -> 3.6, [6000, 64] 4.3 -> 3.7, [1, 128]
// 3.0 -> 3.4, [512, 128] 3.6 -> 3.5, [2000, 128] 4.2 -> 3.7.
// k <= 16: [512, 128] 3.7 -> 5.4, [65536, 128] 43 -> 18, [16, 256] 5.3 -> 4.1,
// [256, 2048] 6.7 -> 7.1, [300, 2000] 11.6 -> 7.7.  k <= 32: [512, 128] 3.6 ->
// 8.2, [65536, 128] 42 -> 26, [512, 2048] 12.2 -> 11.5, [1000, 2048] 22 -> 13,
// [512, 4096] 12.7 -> 17.6, [1024, 4096] 24 -> 18, [1024, 8192] 24.6 -> 30.4.
// Rows of at most 32 have no other kernel made for many rows.
static bool topk_lanes_route(int64_t rows, int64_t cols, int k) {
  if (k > kLanesMaxK || cols > kLanesMaxCols) return false;
  if (cols <= 32) return true;
  if (k <= 8) {
    if (cols <= 64) return rows >= 3072;
    if (cols <= 128) return rows >= 512;
    return cols <= 2048 || rows >= 1024;
  }
  if (k <= 16) {
    if (cols <= 128) return rows * cols >= (int64_t)1 << 19;
    return cols <= 1024 || (cols <= 2048 ? rows > 256 : rows >= 1024);
  }
  return cols <= 4096 && rows * cols >= (int64_t)1 << 21 && (cols <= 2048 || rows >= 1024);
}

// Whole-row sorts pay off at any row count up to 256 elements; beyond that
// only with many rows, where the select kernel's per-row latency adds up
// (f32, k = 64, select -> sort: [65536, 512] 1711 -> 182 us, [32768, 1024]
// 1056 -> 223, [16384, 2048] 332 -> 271, [4096, 2048] 81 -> 80; few rows
// lose: [64, 1024] 10.3 -> 12.0, [256, 2048] 6.7 -> 14.8, [1024, 2048]
// 20.9 -> 28.9).
bool topk_short_route(int64_t rows, int64_t cols, int k) {
  return topk_lanes_route(rows, cols, k) || cols <= 256 || (cols <= 1024 && rows >= 512) ||
         (cols <= kTopkShortCols && rows >= 8192);
}

template <int DT>
__device__ __forceinline__ uint32_t topk_f32_bits(const void* x, int64_t i) {
  return DT == kBF16 ? (uint32_t)((const uint16_t*)x)[i] << 16 : ((const uint32_t*)x)[i];
}

// Output position i of a row, from float32 bits b with select key `key`.
template <int DT>
__device__ __forceinline__ void topk_short_store(uint32_t b, uint32_t key, uint32_t col, int64_t row, int i, int k,
                                                 const TopkShortOut& ot) {
  const int64_t o = row * k + i;
  if (key <= ineligible_key_max(DT)) b = DT == kBF16 ? 0xFF7F0000u : 0xFF7FFFFFu;
  if (ot.k_rows && i >= ot.k_rows[row]) b = ot.replace_bits;
  ot.idx[o] = (int32_t)col;
  if (DT == kBF16) ((uint16_t*)ot.vals)[o] = (uint16_t)(b >> 16);
  else ((uint32_t*)ot.vals)[o] = b;
}
template <int DT>
__device__ __forceinline__ void topk_short_out(uint64_t rec, const void* x, int64_t base, int64_t row, int i, int k,
                                               const TopkShortOut& ot) {
  const uint32_t col = (uint32_t)rec;
  topk_short_store<DT>(topk_f32_bits<DT>(x, base + col), ~(uint32_t)(rec >> 32), col, row, i, k, ot);
}

// ---------------------------------------------------------------------------
// k <= KK: a row on LPR lanes, E elements of it per lane at a time.
//
// A candidate is the double 1.mantissa with mantissa = select key << 20 |
// (0xFFFFF - column): all such doubles are normal, so their order as numbers is
// the order of the 52 bits (value descending, then column ascending), and a
// compare-exchange is v_max_f64 + v_min_f64, two full-rate instructions,
// against a 64-bit compare and four selects for integers.  Each lane sorts its
// elements KK at a time (Batcher's odd-even merge network) and keeps the KK
// largest; lanes then merge pairwise (max(a[i], b[KK - 1 - i]) is bitonic and
// holds the KK largest of both), so the work across lanes does not grow with
// the row.  f32, k = 8: [65536, 128] 43.4 -> 11.6 us (3.3 TB/s; one wave per row
// and a 128-record integer network before), [65536, 512] 177 -> 45, [16384, 2048]
// 269 -> 37 (3.7 TB/s); bf16 [22766, 614] 154 -> 33.  Bound by VALU issue: about
// 20 instructions per element and lane at KK = 8.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double cand_max(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double cand_min(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ void cand_cx(double& a, double& b) {  // a >= b
  const double hi = cand_max(a, b), lo = cand_min(a, b);
  a = hi;
  b = lo;
}
constexpr uint32_t kCandOne = 0x3FF00000u;  // high word of 1.0: the candidate below all others (no element)
__device__ __forceinline__ double make_cand(uint32_t key, uint32_t col) {
  const uint32_t hi = kCandOne | (key >> 12), lo = (key << 20) | (0xFFFFFu - col);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ uint32_t cand_key(double c) {
  return (uint32_t)((__builtin_bit_cast(uint64_t, c) & 0x000FFFFFFFFFFFFFull) >> 20);
}
__device__ __forceinline__ uint32_t cand_col(double c) {
  return 0xFFFFFu - ((uint32_t)__builtin_bit_cast(uint64_t, c) & 0xFFFFFu);
}

// One layer of Batcher's network: comparators (j, j + K) inside blocks of 2 P.
template <int N, int P, int K>
__device__ __forceinline__ void oddeven_layers(double (&v)[N]) {
#pragma unroll
  for (int a = 0; a < N; ++a) {
    const int j0 = K % P;
    if (a >= j0 && ((a - j0) & K) == 0 && a + K < N && a / (2 * P) == (a + K) / (2 * P)) cand_cx(v[a], v[a + K]);
  }
  if constexpr (K > 1) oddeven_layers<N, P, K / 2>(v);
  else if constexpr (2 * P < N) oddeven_layers<N, 2 * P, 2 * P>(v);
}
template <int N, int S>
__device__ __forceinline__ void bitonic_desc(double (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    if ((i & S) == 0) cand_cx(v[i], v[i + S]);
  if constexpr (S > 1) bitonic_desc<N, S / 2>(v);
}
// a <- the N largest of a u b (both descending), descending
template <int N>
__device__ __forceinline__ void merge_desc(double (&a)[N], const double (&b)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) a[i] = cand_max(a[i], b[N - 1 - i]);
  bitonic_desc<N, N / 2>(a);
}
template <int N, int D, int LPR>
__device__ __forceinline__ void merge_lanes(double (&a)[N]) {
  if constexpr (D < LPR) {
    double b[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
      b[i] = __builtin_bit_cast(double, shfl_xor_u64(__builtin_bit_cast(uint64_t, a[i]), D));
    merge_desc<N>(a, b);
    merge_lanes<N, 2 * D, LPR>(a);
  }
}

template <int DT, int KK, int LPR, int E>
__global__ __launch_bounds__(256) void topk_lanes_kernel(const void* __restrict__ x, int64_t rows, int cols, int k,
                                                         int vec, TopkShortOut ot) {
  static_assert(E % KK == 0, "whole runs of KK");
  constexpr int VEC = DT == kBF16 ? 8 : 4, RPB = 256 / LPR;
  const int q = threadIdx.x % LPR;  // lane of the row
  const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
  if (row >= rows) return;  // a row's lanes leave together
  const int64_t base = row * cols;
  double acc[KK];
#pragma unroll 1
  for (int c0 = 0; c0 < cols; c0 += LPR * E) {
    double v[E];
    if (vec) {  // rows of whole 16-byte vectors, 16-byte aligned
      const uint4* rv = (const uint4*)((const char*)x + base * (DT == kBF16 ? 2 : 4));
      uint4 raw[E / VEC];
#pragma unroll
      for (int j = 0; j < E / VEC; ++j) {
        const int c = c0 + (j * LPR + q) * VEC;
        raw[j] = c < cols ? load_once(rv + c / VEC) : make_uint4(0u, 0u, 0u, 0u);
      }
#pragma unroll
      for (int j = 0; j < E / VEC; ++j) {
        const int c = c0 + (j * LPR + q) * VEC;
        const uint32_t d[4] = {raw[j].x, raw[j].y, raw[j].z, raw[j].w};
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const uint32_t b = DT == kBF16 ? ((e & 1) ? d[e >> 1] & 0xFFFF0000u : d[e >> 1] << 16) : d[e];
          v[j * VEC + e] = c < cols ? make_cand(select_key(b), (uint32_t)(c + e)) : make_cand(0u, 0xFFFFFu);
        }
      }
    } else {
      uint32_t b[E];
#pragma unroll
      for (int j = 0; j < E; ++j) {
        const int c = c0 + j * LPR + q;
        b[j] = topk_f32_bits<DT>(x, base + (c < cols ? c : cols - 1));
      }
#pragma unroll
      for (int j = 0; j < E; ++j) {
        const int c = c0 + j * LPR + q;
        v[j] = c < cols ? make_cand(select_key(b[j]), (uint32_t)c) : make_cand(0u, 0xFFFFFu);
      }
    }
#pragma unroll
    for (int r = 0; r < E / KK; ++r) {
      double s[KK];
#pragma unroll
      for (int i = 0; i < KK; ++i) s[i] = v[r * KK + i];
      oddeven_layers<KK, 1, 1>(s);
      if (r == 0 && c0 == 0) {
#pragma unroll
        for (int i = 0; i < KK; ++i) acc[i] = s[i];
      } else {
        merge_desc<KK>(acc, s);
      }
    }
  }
  merge_lanes<KK, 1, LPR>(acc);  // every lane of the row ends with the same list
#pragma unroll
  for (int m = 0; m < KK; m += LPR) {
    constexpr int W = LPR < KK ? LPR : KK;
    double c = acc[m];
#pragma unroll
    for (int i = 1; i < W; ++i) c = q == i ? acc[m + i] : c;
    const int i = m + q;
    if (q < W && i < k) {
      const uint32_t key = cand_key(c), col = cand_col(c);
      // the key fixes the value except the sign of a zero
      const uint32_t b = key == 0x80000000u ? topk_f32_bits<DT>(x, base + col) : key_to_bits(key);
      topk_short_store<DT>(b, key, col, row, i, k, ot);
    }
  }
}

template <int DT, int P, int E>
__global__ __launch_bounds__(P / E) void topk_short_block_kernel(const void* __restrict__ x, int cols, int k,
                                                                 TopkShortOut ot) {
  __shared__ uint64_t lds[P];
  const int64_t row = blockIdx.x;
  const int64_t base = row * cols;
  const int t = threadIdx.x;
  uint64_t v[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int i = t * E + r;
    v[r] = i < cols ? ((uint64_t)~select_key(topk_f32_bits<DT>(x, base + i)) << 32) | (uint32_t)i : ~0ull;
  }
  block_bitonic_sort_c<uint64_t, E, P, false>(v, lds);
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int i = t * E + r;
    if (i < k) topk_short_out<DT>(v[r], x, base, row, i, k, ot);
  }
}

template <int DT, int KK, int LPR, int E>
static void launch_lanes_one(const void* x, int64_t rows, int cols, int k, const TopkShortOut& ot, hipStream_t s) {
  constexpr int RPB = 256 / LPR;
  const int vec = (uintptr_t)x % 16 == 0 && (size_t)cols * (DT == kBF16 ? 2 : 4) % 16 == 0;
  hipLaunchKernelGGL((topk_lanes_kernel<DT, KK, LPR, E>), dim3((unsigned)((rows + RPB - 1) / RPB)), dim3(256), 0, s, x,
                     rows, cols, k, vec, ot);
}

// Lanes per row: the fewest whose first pass (E elements per lane) holds the
// row, so that most of the work is inside lanes; 64 lanes take longer rows in
// several passes.
template <int DT, int KK>
static void launch_lanes(const void* x, int64_t rows, int cols, int k, const TopkShortOut& ot, hipStream_t s) {
  constexpr int E = KK < 16 ? 16 : KK;
  if (cols <= E) launch_lanes_one<DT, KK, 1, E>(x, rows, cols, k, ot, s);
  else if (cols <= 4 * E) launch_lanes_one<DT, KK, 4, E>(x, rows, cols, k, ot, s);
  else if (cols <= 8 * E) launch_lanes_one<DT, KK, 8, E>(x, rows, cols, k, ot, s);
  else if (cols <= 16 * E) launch_lanes_one<DT, KK, 16, E>(x, rows, cols, k, ot, s);
  else if (cols <= 32 * E) launch_lanes_one<DT, KK, 32, E>(x, rows, cols, k, ot, s);
  else launch_lanes_one<DT, KK, 64, E>(x, rows, cols, k, ot, s);
}

template <int DT>
static int launch_topk_short_dt(const void* x, int64_t rows, int64_t cols, int k, const TopkShortOut& ot,
                                hipStream_t s) {
  const int c = (int)cols;
  if (topk_lanes_route(rows, cols, k)) {
    if (k <= 8) launch_lanes<DT, 8>(x, rows, c, k, ot, s);
    else if (k <= 16) launch_lanes<DT, 16>(x, rows, c, k, ot, s);
    else launch_lanes<DT, 32>(x, rows, c, k, ot, s);
  } else if (cols <= 64) {
    hipLaunchKernelGGL((topk_short_block_kernel<DT, 64, 1>), dim3((unsigned)rows), dim3(64), 0, s, x, c, k, ot);
  } else if (cols <= 128) {
    hipLaunchKernelGGL((topk_short_block_kernel<DT, 128, 2>), dim3((unsigned)rows), dim3(64), 0, s, x, c, k, ot);
  } else if (cols <= 256) {
    hipLaunchKernelGGL((topk_short_block_kernel<DT, 256, 4>), dim3((unsigned)rows), dim3(64), 0, s, x, c, k, ot);
  } else if (cols <= 512) {
    hipLaunchKernelGGL((topk_short_block_kernel<DT, 512, 8>), dim3((unsigned)rows), dim3(64), 0, s, x, c, k, ot);
  } else if (cols <= 1024) {
    hipLaunchKernelGGL((topk_short_block_kernel<DT, 1024, 8>), dim3((unsigned)rows), dim3(128), 0, s, x, c, k, ot);
  } else {
    hipLaunchKernelGGL((topk_short_block_kernel<DT, 2048, 8>), dim3((unsigned)rows), dim3(256), 0, s, x, c, k, ot);
  }
  return launch_status("top-k (short rows)");
}

int launch_topk_short(const void* x, int dt, int64_t rows, int64_t cols, int k, const TopkShortOut& ot,
                      hipStream_t s) {
  return dt == kF32 ? launch_topk_short_dt<kF32>(x, rows, cols, k, ot, s)
                    : launch_topk_short_dt<kBF16>(x, rows, cols, k, ot, s);
}

}  // namespace tx
