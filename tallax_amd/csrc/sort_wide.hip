// Row sort for rows longer than one workgroup's LDS holds (> 16384
// elements): the wide-row route of tax.sort / tumpy.sort / tumpy.argsort.
//
// Reference: sort (tallax/_src/sort.py:768-929) sends such rows to its HBM
// substage engine (sort.py:574-758), a bitonic network whose large-stride
// substages each stream the whole array through HBM.  The results it defines
// are those of a stable sort by (standardised key, tie), S1-S2 in the key
// helpers' terms: ascending or descending key, ties by ascending original
// index (by descending index only on the packed bf16 non-stable descending
// route, utils.py:205-216).
//
// Here every element becomes a 64-bit record (order bits << 32 | tie), where
// the tie is the element's column (or 0x7FFFFFFF - column).  Records are
// unique, so any correct sort of them gives exactly that order, and two
// sorted runs merge without a stability rule.
//   1. sort_chunks_kernel: one 512-thread workgroup sorts each 16384- or
//      8192-record chunk of a row in LDS (a stable LSD radix sort on the key,
//      8-bit digits) and writes the sorted run to the workspace.
//   2. Rows of 3 to kBucketMaxRuns chunks: bucket_split_kernel cuts the key
//      range into buckets by samples of the runs, and bucket_sort_kernel orders
//      each bucket in LDS and writes the outputs.  One pass over the records.
//   3. Rows of two chunks, or more than that: merge_runs_kernel,
//      ceil(log2(chunks)) passes.  Runs of length L are
//      merged pairwise into runs of 2L, ping-ponging between two workspace
//      buffers.  A workgroup produces 4096 consecutive outputs of one pair:
//      two waves find the tile's start and end on the merge path with a
//      64-way search (one ballot per step, so about three dependent global
//      round trips for a 2^18 run), the tile's inputs are staged in LDS,
//      each thread finds its own 16-output diagonal by binary search in LDS
//      and merges sequentially, and the tile leaves through LDS as coalesced
//      stores.  The last pass writes the permutation, the decoded keys and
//      the gathered second key instead of records.
// Every merge pass reads and writes each record once (16 bytes per element per
// pass), the buckets read it once; no kernel waits on another workgroup.
#include <stdint.h>

#include "tallax_hip.h"
#include "tx_block_sort.h"
#include "tx_common.h"
#include "tx_host.h"
#include "tx_scan.h"
#include "tx_sort_keys.h"

namespace tx {

constexpr int kWideChunk = 16384;  // records per chunk sorted in LDS
constexpr int kChunkNT = 512;
constexpr int kChunkE = kWideChunk / kChunkNT;
constexpr int kMergeNT = 256;
constexpr int kMergeItems = 16;                      // outputs per thread
constexpr int kMergeTile = kMergeNT * kMergeItems;   // outputs per workgroup
constexpr uint32_t kTieMask = 0x7FFFFFFFu;
static_assert((2 * kWideChunk) % kMergeTile == 0, "a merge tile never straddles two pairs of runs");
static_assert(kChunkE * kChunkNT == kWideChunk, "whole chunks per workgroup");

// Stable LSD radix sort by the key (the records' high 32 bits) of the per x NT
// records (per <= E) a workgroup holds in registers in slot order, slot
// (per * 64) w + 64 r + l being record r of lane l of wave w; 8-bit digits, the
// digits in which no key varies skipped.  Slots n and above hold all-ones
// records, which stay last: waves wholly past n neither count nor move theirs.
// buf holds E * NT records, hist 256 * (NT / 64 + 1) counters.  Every thread
// of the workgroup calls it.
//   * each wave counts its digits in its own 256 LDS counters (digit-major,
//     NW + 1 words apart) with one atomic per record, r = 0..E-1 in turn; the
//     atomics of one instruction on one address return in ascending lane order
//     (gfx950; tallax_testing_lds_atomic_order checks it), so the value before
//     a record's increment is its stable rank among the wave's earlier slots
//     of that digit;
//   * an exclusive scan over (digit, wave) in digit-major order gives each
//     pair its start, records move to start + rank through LDS, and the next
//     pass reads them back in slot order.
template <int E, int NT>
__device__ __forceinline__ void radix_sort_slots(uint64_t (&v)[E], uint64_t* buf, uint32_t* hist, uint32_t* wsum,
                                                 uint32_t varying, int n, int per = E) {
  constexpr int NW = NT / kWave;
  constexpr int HS = NW + 1;  // counter stride per digit
  static_assert(256 * NW == 4 * NT, "four counters per thread in the scan");
  const int t = threadIdx.x, l = lane_id(), w = t / kWave;
  const bool live = w * (per * kWave) < n;  // wave-uniform: the wave holds a slot below n
#pragma unroll 1
  for (int sh = 0; sh < 32; sh += 8) {
    if (((varying >> sh) & 0xFFu) == 0u) continue;  // every key has this digit: the pass is the identity
#pragma unroll
    for (int d = l; d < 256; d += kWave) hist[d * HS + w] = 0u;  // this wave's counters
    uint32_t rk[E];
    if (live) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        if (r < per) {
          const uint32_t d = (uint32_t)(v[r] >> (32 + sh)) & 0xFFu;
          rk[r] = atomicAdd(&hist[d * HS + w], 1u);
        }
      }
    }
    __syncthreads();  // every count is in
    // exclusive scan over i = digit * NW + wave: thread t takes i = 4t .. 4t + 3
    const int d0 = (4 * t) / NW, w0 = (4 * t) % NW;
    uint32_t cq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) cq[q] = hist[d0 * HS + w0 + q];
    const uint32_t run = cq[0] + cq[1] + cq[2] + cq[3];
    const uint32_t incl = wave_incl_scan(run);
    if (l == kWave - 1) wsum[w] = incl;
    __syncthreads();
    uint32_t pre = incl - run;
#pragma unroll
    for (int i = 0; i < NW; ++i) pre += i < w ? wsum[i] : 0u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      hist[d0 * HS + w0 + q] = pre;
      pre += cq[q];
    }
    __syncthreads();
    if (live) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        if (r < per) {
          const uint32_t d = (uint32_t)(v[r] >> (32 + sh)) & 0xFFu;
          buf[hist[d * HS + w] + rk[r]] = v[r];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (per * kWave) + r * kWave + l;
      v[r] = r < per && L < n ? buf[L] : ~0ull;
    }
  }
}

// Pass 1: sorted runs of CH = E * kChunkNT records, by a stable LSD radix sort on
// the 32-bit key in 8-bit digits (radix_sort_slots: at most four passes; a
// digit that every key of the chunk shares is skipped).  Slot p of the chunk
// holds record (order bits << 32 | tie) of linear index p (column c0 + p, or
// its reverse for descending ties), so the stable sort by key alone is the
// order of the full records; slots past the row hold all-ones records, which
// stay last.  (Eight passes of 4-bit digits with per-thread packed counters
// took 2.93 ms at [1024, 201088]; these four, 1.60 ms.)
template <int DT, bool PERM, int E>
__global__ __launch_bounds__(kChunkNT) void sort_chunks_kernel(SortArgs a, int nchunks, uint64_t* out) {
  constexpr int NW = kChunkNT / kWave;
  constexpr int CH = E * kChunkNT;                     // records of a chunk
  extern __shared__ __align__(16) unsigned char smem[];
  uint64_t* buf = (uint64_t*)smem;                     // CH records
  uint32_t* hist = (uint32_t*)(buf + CH);              // 256 * (NW + 1) counters
  __shared__ uint32_t wsum[NW];
  __shared__ uint32_t red[2][NW];
  const int t = threadIdx.x, l = lane_id(), w = t / kWave;
  const int64_t row = blockIdx.x / (unsigned)nchunks;
  const int c = (int)(blockIdx.x - row * nchunks);
  const int64_t base = row * a.cols;
  const int64_t c0 = (int64_t)c * CH;
  const int n = (int)min((int64_t)CH, a.cols - c0);
  // records in slot order (coalesced reads, every load of the chunk in
  // flight at once), and which key bits vary
  uint32_t kand = ~0u, kor = 0u;
  uint64_t v[E];
  {
    uint32_t raw[E];
    int32_t src[E];
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (E * kWave) + r * kWave + l;
      src[r] = (int32_t)(c0 + (a.ties_desc ? n - 1 - L : L));
      if (PERM && L < n) src[r] = a.perm_in[base + src[r]];
    }
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (E * kWave) + r * kWave + l;
      raw[r] = L < n ? key_bits_at<DT>(a.key, base + src[r]) : 0u;
    }
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (E * kWave) + r * kWave + l;
      v[r] = ~0ull;
      if (L < n) {
        uint32_t k = order_from_bits(raw[r], DT);
        if (a.descending) k = ~k;
        const uint32_t p = (uint32_t)(c0 + (a.ties_desc ? n - 1 - L : L));
        const uint32_t tie = a.ties_desc ? kTieMask - p : p;
        v[r] = ((uint64_t)k << 32) | tie;
        kand &= k;
        kor |= k;
      }
    }
  }
  kand = wave_and_u32(kand);
  kor = wave_or_u32(kor);
  if (l == 0) {
    red[0][w] = kand;
    red[1][w] = kor;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    kand &= red[0][i];
    kor |= red[1][i];
  }
  // bfloat16 keys: the low 16 order bits follow from the high 16 (as in
  // sort_row_radix_kernel), so only the high digits are sorted
  const uint32_t varying = (kand ^ kor) & (DT == kBF16 ? 0xFFFF0000u : ~0u);
  radix_sort_slots<E, kChunkNT>(v, buf, hist, wsum, varying, n);
  uint64_t* dst = out + base + c0;
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int L = w * (E * kWave) + r * kWave + l;
    if (L < n) dst[L] = v[r];
  }
}

// Merge path: the number of A records among the first d records of the
// merge of sorted A[0, la) and B[0, lb), i.e. the first i in
// [max(0, d - lb), min(d, la)) with A[i] > B[d - 1 - i], or min(d, la) when
// there is none.  One wave; every lane returns the same value.  Each step
// probes 64 positions (at most n / 64 apart) and keeps the interval between
// the last false and the first true probe.
__device__ int merge_split_wave(const uint64_t* A, int la, const uint64_t* B, int lb, int d) {
  const int l = lane_id();
  int lo = max(0, d - lb), hi = min(d, la);
  while (hi > lo) {
    const int n = hi - lo;
    const bool small = n <= kWave;
    const int q = small ? lo + l : lo + (int)(((int64_t)(l + 1) * n) / kWave) - 1;
    const bool f = (!small || l < n) && A[q] > B[d - 1 - q];
    const uint64_t b = __ballot(f);
    if (!b) return hi;
    const int l0 = __ffsll((unsigned long long)b) - 1;
    if (small) return lo + l0;
    const int qprev = lo + (int)(((int64_t)l0 * n) / kWave) - 1;  // lo - 1 for l0 = 0
    hi = lo + (int)(((int64_t)(l0 + 1) * n) / kWave) - 1;         // a true probe
    lo = qprev + 1;
  }
  return lo;
}

// One merge pass over runs of length `run`: the pair of runs starting at
// column s = 2 run j merges into columns [s, s + 2 run) of dst.  A run with
// no partner (the row's last) is copied.  FINAL writes the outputs instead.
// LDS slot of merge-tile record j: one spare slot per 16 records, so that
// the 64 lanes of a wave, each merging its own run of 16 outputs (records 16
// apart), spread over the banks instead of all hitting one.
__device__ __forceinline__ int ms(int j) { return j + (j >> 4); }

template <bool FINAL>
__global__ __launch_bounds__(kMergeNT) void merge_runs_kernel(SortArgs a, const uint64_t* src, uint64_t* dst,
                                                              int64_t run, int tiles) {
  __shared__ uint64_t lds[kMergeTile + kMergeTile / 16];  // record j at ms(j)
  __shared__ int split[2];
  const int t = threadIdx.x, w = t / kWave;
  // Workgroups go to the 8 XCDs round-robin, each with its own L2: the tile
  // order is remapped so that every XCD takes a contiguous range of tiles, and
  // neighbouring tiles, whose merge-path searches probe the same lines of the
  // same runs, share an L2.
  const unsigned nwg = gridDim.x;
  const unsigned vb = nwg % 8u == 0u ? (blockIdx.x % 8u) * (nwg / 8u) + blockIdx.x / 8u : blockIdx.x;
  const int64_t row = vb / (unsigned)tiles;
  const int ti = (int)(vb - row * tiles);
  const int64_t base = row * a.cols;
  const int64_t o0 = (int64_t)ti * kMergeTile;  // first output column of the tile
  const int64_t s = o0 / (2 * run) * (2 * run);
  const int la = (int)min(run, a.cols - s);
  const int lb = (int)max((int64_t)0, min(run, a.cols - s - run));
  const int d0 = (int)(o0 - s);
  const int count = min(kMergeTile, la + lb - d0);
  const uint64_t* A = src + base + s;
  const uint64_t* B = A + run;  // read only where lb > 0
  if (w < 2) {
    const int sp = merge_split_wave(A, la, B, lb, d0 + w * count);
    if (lane_id() == 0) split[w] = sp;
  }
  __syncthreads();
  const int a0 = split[0];
  const int na = split[1] - a0;
  const int b0 = d0 - a0;
  const int nb = count - na;
  {
    uint64_t st[kMergeItems];  // every load of the tile in flight at once
#pragma unroll
    for (int k = 0; k < kMergeItems; ++k) {
      const int j = k * kMergeNT + t;
      st[k] = j < count ? (j < na ? A[a0 + j] : B[b0 + (j - na)]) : 0ull;
    }
#pragma unroll
    for (int k = 0; k < kMergeItems; ++k) {
      const int j = k * kMergeNT + t;
      if (j < count) lds[ms(j)] = st[k];
    }
  }
  __syncthreads();
  uint64_t out[kMergeItems];
  const int dt = t * kMergeItems;
  if (dt < count) {
    int lo = max(0, dt - nb), hi = min(dt, na);
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (lds[ms(mid)] > lds[ms(na + dt - 1 - mid)]) hi = mid;
      else lo = mid + 1;
    }
    int ia = lo, ib = dt - lo;
    uint64_t x = ia < na ? lds[ms(ia)] : ~0ull;
    uint64_t y = ib < nb ? lds[ms(na + ib)] : ~0ull;
#pragma unroll
    for (int r = 0; r < kMergeItems; ++r) {
      const bool take_a = x < y;
      out[r] = take_a ? x : y;
      if (take_a) {
        ++ia;
        x = ia < na ? lds[ms(ia)] : ~0ull;
      } else {
        ++ib;
        y = ib < nb ? lds[ms(na + ib)] : ~0ull;
      }
    }
  }
  __syncthreads();
  if (dt < count) {
#pragma unroll
    for (int r = 0; r < kMergeItems; ++r)
      if (dt + r < count) lds[ms(dt + r)] = out[r];
  }
  __syncthreads();
  if (!FINAL) {
    for (int j = t; j < count; j += kMergeNT) dst[base + o0 + j] = lds[ms(j)];
    return;
  }
  // outputs: source columns, then the gathered second key, each batch of
  // dependent loads in flight at once
  int32_t col[kMergeItems];  // columns are < 2^31
#pragma unroll
  for (int k = 0; k < kMergeItems; ++k) {
    const int j = k * kMergeNT + t;
    col[k] = 0;
    if (j < count) {
      const uint32_t tie = (uint32_t)lds[ms(j)];
      const int32_t pos = (int32_t)(a.ties_desc ? kTieMask - tie : tie);
      col[k] = a.perm_in ? a.perm_in[base + pos] : pos;
    }
  }
#pragma unroll
  for (int k = 0; k < kMergeItems; ++k) {
    const int j = k * kMergeNT + t;
    if (j >= count) continue;
    a.perm_out[base + o0 + j] = col[k];
    if (a.key_out) {
      uint32_t key = (uint32_t)(lds[ms(j)] >> 32);
      if (a.descending) key = ~key;
      store_sorted(a.key_out, a.key_out_dtype, a.key_dtype, base + o0 + j, key);
    }
  }
  if (a.aux_out) {
    uint32_t u[kMergeItems];
    if (a.aux_dtype == kBF16) {
#pragma unroll
      for (int k = 0; k < kMergeItems; ++k)
        u[k] = k * kMergeNT + t < count ? key_bits_at<kBF16>(a.aux, base + col[k]) : 0u;
    } else {
#pragma unroll
      for (int k = 0; k < kMergeItems; ++k)
        u[k] = k * kMergeNT + t < count ? key_bits_at<kF32>(a.aux, base + col[k]) : 0u;
    }
#pragma unroll
    for (int k = 0; k < kMergeItems; ++k) {
      const int j = k * kMergeNT + t;
      if (j < count)
        store_sorted(a.aux_out, a.aux_out_dtype, a.aux_dtype, base + o0 + j, order_from_bits(u[k], a.aux_dtype));
    }
  }
}

// ---------------------------------------------------------------------------
// Multiway merge by splitters (rows of 3 to kBucketMaxRuns chunks): one pass
// instead of ceil(log2 chunks) pairwise merge passes.
//   * bucket_split_kernel, one workgroup per row: every G-th record of every
//     sorted run is a sample (record (a + 1) G - 1 of a run); the samples (at
//     most 4096) are sorted by a block bitonic network, and every m-th one of
//     them in that order is a splitter s_k.
//     For every splitter and run, the run's first position p_kj with a record
//     >= s_k: the run's samples below s_k, c, put it in [c G, (c + 1) G), so a
//     binary search of G records finds it.  Bucket k holds the records in
//     [s_k, s_k+1).  From run j it takes at most (q_j + 1) G records, q_j its
//     samples in the bucket, and the bucket's samples number at most m, so a
//     bucket never exceeds (m + runs) G records: m is chosen so that this is
//     the bucket kernel's capacity.  The table holds every p_kj and each
//     bucket's first output rank, sum_j p_kj.
//     G is 64 where the samples fit: the finer they are, the more runs a bucket
//     of 4096 records takes (m = 64 - runs samples: at 25 runs 39, buckets 61 %
//     full on average; with 13 whole chunks and buckets of 8192, G = 64 fills 79 %
//     and G = 256 58 %).  Few rows take smaller buckets, so that they fill the chip.
//   * bucket_sort_kernel, one workgroup per (row, bucket): the bucket's part of
//     every run, in tie order, sorted in LDS; the outputs (permutation, keys,
//     gathered second key) are written from the bucket's first output rank.
// Traffic: the chunk pass (4 bytes in, 8 out per element), then 8 in and the
// outputs out: 28 bytes per element with keys and indices out, against 76 for
// four pairwise merge passes at [1024, 201088].  There the three kernels take
// 991 + 271 + 983 us: chunks bound by LDS (bank conflicts of the scattered
// records), buckets by the latency of their loads and LDS steps.
// ---------------------------------------------------------------------------
constexpr int kBucketStride = 256;       // G: records between samples ...
constexpr int kBucketStrideFine = 64;    // ... of rows of at most kSplitSamples * 64 elements
constexpr int64_t kHalfChunkCols = 229376;  // longest rows sorted in half chunks
constexpr int kBucketMaxRuns = 56;       // (m >= 8) + runs <= 64: buckets of at most 64 G = 16384 records
constexpr int kSplitNT = 1024;
constexpr int kSplitSamples = 4096;      // >= kBucketMaxRuns * kWideChunk / kBucketStride
constexpr int kBucketPad = 4;            // records read at a time in a bin
constexpr uint32_t kBinMost = 24;        // records in one bin past which the radix sort takes over
static_assert(kBucketMaxRuns * (kWideChunk / kBucketStride) <= kSplitSamples, "every sample fits the sort");

struct BucketPlan {
  int runs;     // chunks of a row
  int chunk;    // records of a run (the row's last one may be shorter)
  int G;        // records between samples of a run
  int samples;  // S: samples of a row
  int m;        // samples per bucket
  int K;        // buckets of a row
  int cap;      // records a bucket may hold: 4096, 8192 or 16384
};

__host__ __device__ inline int run_len(int64_t cols, int chunk, int j) {
  const int64_t left = cols - (int64_t)j * chunk;
  return (int)(left < chunk ? left : chunk);
}

__global__ __launch_bounds__(kSplitNT) void bucket_split_kernel(SortArgs a, BucketPlan bp, const uint64_t* runs,
                                                                int32_t* table) {
  __shared__ uint64_t srt[kSplitSamples];   // samples, sorted
  __shared__ uint64_t per[kSplitSamples];   // samples in run order (each run's ascending)
  __shared__ int sp[kBucketMaxRuns + 1];    // first sample of each run
  __shared__ int soff[kSplitSamples / 8 + 2];
  const int t = threadIdx.x;
  const int64_t row = blockIdx.x;
  const int64_t base = row * a.cols;
  const int R = bp.runs, G = bp.G;
  if (t <= R) sp[t] = t < R ? t * (bp.chunk / G) : bp.samples;
  for (int k = t; k <= bp.K; k += kSplitNT) soff[k] = 0;
  __syncthreads();
  // sample i = 4t + r: run j with sp[j] <= i < sp[j + 1], record (i - sp[j] + 1) G - 1 of it
  uint64_t v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 4 * t + r;
    v[r] = ~0ull;
    if (i < bp.samples) {
      const int j = i / (bp.chunk / G);  // every run but the last has chunk / G samples
      v[r] = runs[base + (int64_t)j * bp.chunk + (int64_t)(i - sp[j] + 1) * G - 1];
      per[i] = v[r];
    }
  }
  block_bitonic_sort_c<uint64_t, 4, kSplitSamples, false>(v, srt);
#pragma unroll
  for (int r = 0; r < 4; ++r) srt[4 * t + r] = v[r];
  __syncthreads();
  // p_kj for k = 0..K (k = 0: 0; k = K: the run's length), one (k, j) per thread in turn
  int32_t* tp = table + row * (int64_t)(bp.K + 1) * (R + 1);  // [(K + 1) R] positions, then [K + 1] offsets
  for (int q = t; q < (bp.K + 1) * R; q += kSplitNT) {
    const int k = q / R, j = q - k * R;
    const int len = run_len(a.cols, bp.chunk, j);
    int pos;
    if (k == 0) {
      pos = 0;
    } else if (k == bp.K) {
      pos = len;
    } else {
      const uint64_t sk = srt[k * bp.m];
      // samples of run j below sk (each run's samples ascend)
      int lo = sp[j], hi = sp[j + 1];
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (per[mid] < sk) lo = mid + 1;
        else hi = mid;
      }
      const int c = lo - sp[j];
      // first record >= sk in [c G, min((c + 1) G - 1, len)]
      int l0 = c * G, h0 = c < sp[j + 1] - sp[j] ? (c + 1) * G - 1 : len;
      const uint64_t* rj = runs + base + (int64_t)j * bp.chunk;
      while (l0 < h0) {
        const int mid = (l0 + h0) >> 1;
        if (rj[mid] < sk) l0 = mid + 1;
        else h0 = mid;
      }
      pos = l0;
    }
    tp[q] = pos;
    atomicAdd(&soff[k], pos);
  }
  __syncthreads();
  for (int k = t; k <= bp.K; k += kSplitNT) tp[(bp.K + 1) * R + k] = soff[k];
}

// Bins of a bucket of E * NT records: half as many, which fit the radix sort's
// counters (16-bit, and the end of the last one).  Larger buckets (E = 32, rows
// of more than 24 runs) take the radix sort: the bins' registers would spill.
constexpr int bucket_bins(int nt, int e) { return e <= 16 ? 8 * nt : 0; }
static_assert(bucket_bins(256, 16) * 2 + 4 <= 256 * 5 * 4 && bucket_bins(512, 16) * 2 + 4 <= 256 * 9 * 4, "bins fit");

// Multiplier that spreads key offsets 0 .. range over the bins: offset * scale >> 32
// is below BINS and ascends with the offset.
template <int BINS>
__device__ __forceinline__ uint32_t bin_scale(uint32_t range) {
  if (range < (uint32_t)BINS) return ~0u;
  return (uint32_t)(((uint64_t)BINS << 32) / ((uint64_t)range + 1u));
}

// One workgroup per (row, bucket).  Slot L of the bucket is record L - s_off[i] of
// its part of the i-th run in tie order: chunk j holds columns [j, j + 1) * chunk,
// so with descending ties (tie = kTieMask - column) the last run comes first.
//
// A bucket's keys lie in a narrow range of the row's, so they spread nearly
// evenly over bins of equal key ranges: one atomic per record gives it a place
// in its bin, a scan the bins' starts, and after one move through LDS a
// record's rank is its bin's start + the smaller records of its bin.  That is
// one pass and five barriers, against three to four radix passes of five
// ([1024, 201088] f32 in whole chunks, buckets of 8192: 1792 -> 1210 us; of 4096,
// four workgroups to a CU: 994; in half chunks 1185, 1138 with one order of slots
// throughout, which left no register spilled, 983 with the slots shared out
// evenly).  bf16 keys, key ranges of few values and bunched keys pile up in the
// bins and take the stable radix sort on the key; the records are held in its
// slot order from the start.  f32 rows of few values pay the counting pass for
// nothing: whole sort [64, 50257] of ten values 148 us without bins and in whole
// chunks, 158 now ([64, 201088] 356 / 297), of bf16 values held in f32 122 / 125
// (329 / 276).
template <int NT, int E, int DT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(E <= 16 ? 4 : 2, 8)))
void bucket_sort_kernel(SortArgs a, BucketPlan bp, const uint64_t* runs, const int32_t* table) {
  constexpr int NW = NT / kWave;
  constexpr int BINS = bucket_bins(NT, E);  // 0: the radix sort only
  constexpr int CAP = E * NT;
  extern __shared__ __align__(16) unsigned char smem[];
  uint64_t* buf = (uint64_t*)smem;                        // CAP records + kBucketPad
  uint32_t* hist = (uint32_t*)(buf + CAP + kBucketPad);   // 256 * (NW + 1) counters, or the bins
  __shared__ uint32_t wsum[NW];
  __shared__ uint32_t red[2][NW];
  __shared__ int s_off[kBucketMaxRuns + 1];
  __shared__ uint32_t s_src[kBucketMaxRuns];  // slot L of run i is the row's record s_src[i] + L
  const int t = threadIdx.x, l = lane_id(), w = t / kWave;
  const int R = bp.runs;
  const int64_t row = blockIdx.x / (unsigned)bp.K;
  const int k = (int)(blockIdx.x - row * bp.K);
  const int64_t base = row * a.cols;
  const int32_t* tp = table + row * (int64_t)(bp.K + 1) * (R + 1);
  if (w == 0) {  // the bucket's range in each run and its slots, by a wave scan
    const int j = a.ties_desc ? R - 1 - l : l;
    int lo = 0, sz = 0;
    if (l < R) {
      lo = tp[k * R + j];
      sz = tp[(k + 1) * R + j] - lo;
    }
    int tot;
    const int pre = wave_exscan_i32(sz, tot);
    if (l < R) {
      s_off[l] = pre;
      s_src[l] = (uint32_t)(j * bp.chunk + lo - pre);
    }
    if (l == 0) s_off[R] = tot;
  }
  uint32_t* bins = hist;  // BINS 16-bit counters, two to a word
  if (DT != kBF16)
    for (int q = t; q < BINS / 2; q += NT) bins[q] = 0u;
  __syncthreads();
  const int n = s_off[R];  // at most CAP (the split's bound)
  if (n > CAP) return;     // never taken; keeps a broken table from writing past the LDS buffer
  const int64_t o0 = tp[(bp.K + 1) * R + k];
  // A thread's slots, as the radix sort numbers them: ascending, and shared out
  // evenly where the bucket is not full (with 16 per thread, a bucket of a quarter
  // lay in one wave: f32 [21, 40622] 61.0 -> 54.8 us, [1024, 201088] 2338 -> 2191).
  const int per = (n + NT - 1) / NT;
  auto slot_of = [&](int r) -> int { return r < per ? w * (per * kWave) + r * kWave + l : CAP; };
  uint64_t v[E];
  {
    // a row's records span less than 2^32 bytes: 32-bit offsets from its start
    const char* rr = (const char*)(runs + base);
    int i = 0;
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = slot_of(r);
      v[r] = ~0ull;
      if (L < n) {
        while (s_off[i + 1] <= L) ++i;
        v[r] = *(const uint64_t*)(rr + (s_src[i] + (uint32_t)L) * 8u);
      }
    }
  }
  bool spread = false;  // block-uniform: the bins order the bucket
  uint32_t kmin = ~0u, scale = 0u;
  auto bin_of = [&](uint64_t x) -> uint32_t { return __umulhi((uint32_t)(x >> 32) - kmin, scale); };
  const uint16_t* start = (const uint16_t*)bins;
  if constexpr (DT != kBF16 && BINS > 0) {
    uint32_t kmax = 0u;
#pragma unroll
    for (int r = 0; r < E; ++r) {
      if (slot_of(r) < n) {
        const uint32_t key = (uint32_t)(v[r] >> 32);
        kmin = key < kmin ? key : kmin;
        kmax = key > kmax ? key : kmax;
      }
    }
    kmin = wave_min_u32(kmin);
    kmax = wave_max_u32(kmax);
    if (l == 0) {
      red[0][w] = kmin;
      red[1][w] = kmax;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      kmin = red[0][i] < kmin ? red[0][i] : kmin;
      kmax = red[1][i] > kmax ? red[1][i] : kmax;
    }
    kmin = __builtin_amdgcn_readfirstlane(kmin);
    kmax = __builtin_amdgcn_readfirstlane(kmax);
    scale = bin_scale<BINS>(kmax - kmin);
    if (kmax - kmin >= (uint32_t)n / 4u) {  // block-uniform: else few values
      uint32_t pb[E];  // place in the bin << 16 | bin
#pragma unroll
      for (int r = 0; r < E; ++r) {
        pb[r] = 0u;
        if (slot_of(r) < n) {
          const uint32_t b = bin_of(v[r]), sh = (b & 1u) * 16u;
          pb[r] = ((atomicAdd(&bins[b >> 1], 1u << sh) >> sh) << 16) | b;
        }
      }
      __syncthreads();
      constexpr int PW = BINS / 2 / NT;  // words per thread
      uint32_t cw[PW], most = 0u;
      int sum = 0;
#pragma unroll
      for (int q = 0; q < PW; ++q) {
        cw[q] = bins[t * PW + q];
        const uint32_t lo = cw[q] & 0xFFFFu, hi = cw[q] >> 16;
        sum += (int)(lo + hi);
        most = max(most, max(lo, hi));
      }
      int tot;
      const int pre = wave_exscan_i32(sum, tot);
      most = wave_max_u32(most);
      if (l == 0) {
        wsum[w] = (uint32_t)tot;
        red[0][w] = most;
      }
      __syncthreads();
      uint32_t run = (uint32_t)pre;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        run += i < w ? wsum[i] : 0u;
        most = max(most, red[0][i]);
      }
      spread = __builtin_amdgcn_readfirstlane(most) <= kBinMost;
      if (spread) {
#pragma unroll
        for (int q = 0; q < PW; ++q) {
          const uint32_t lo = cw[q] & 0xFFFFu, hi = cw[q] >> 16;
          bins[t * PW + q] = run | ((run + lo) << 16);  // the bins' starts, below 2^16
          run += lo + hi;
        }
        if (t == 0) bins[BINS / 2] = (uint32_t)n;  // the end of the last bin
        __syncthreads();
#pragma unroll
        for (int r = 0; r < E; ++r)
          if (slot_of(r) < n) buf[start[pb[r] & 0xFFFFu] + (pb[r] >> 16)] = v[r];
        if (t < kBucketPad) buf[n + t] = ~0ull;  // read past the last bin: larger than any record
        __syncthreads();
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = slot_of(r) < n ? buf[slot_of(r)] : ~0ull;
      }
    }
    __syncthreads();  // red is read, and the radix sort clears its counters over the bins
  }
  if (!spread) {
    // the digits in which no key varies are skipped: all but two or three of a
    // tied bucket's, the low two of bf16 values held in f32.  (From the smallest
    // and largest key alone, every digit below their first difference was
    // sorted: [64, 201088] f32 holding bf16 values 328 -> 412 us.)
    uint32_t kand = ~0u, kor = 0u;
#pragma unroll
    for (int r = 0; r < E; ++r) {
      if (slot_of(r) < n) {
        kand &= (uint32_t)(v[r] >> 32);
        kor |= (uint32_t)(v[r] >> 32);
      }
    }
    kand = wave_and_u32(kand);
    kor = wave_or_u32(kor);
    if (l == 0) {
      red[0][w] = kand;
      red[1][w] = kor;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      kand &= red[0][i];
      kor |= red[1][i];
    }
    // the low order bits of a bf16 key follow from the high
    radix_sort_slots<E, NT>(v, buf, hist, wsum, (kand ^ kor) & (DT == kBF16 ? 0xFFFF0000u : ~0u), n, per);
  }
  // outputs at o0 + rank: the source column, the sorted key and the gathered
  // second key (32-bit offsets from the bucket's first output)
  const int64_t ob = base + o0;
  int32_t* po = a.perm_out + ob;
  const uint32_t tmask = a.ties_desc ? kTieMask : 0u, dmask = a.descending ? ~0u : 0u;
  char* ko = (char*)a.key_out + ob * (DT == kBF16 && a.key_out_dtype == kBF16 ? 2 : 4);
  auto rank_of = [&](uint64_t x, int L) -> uint32_t {
    if (!spread) return (uint32_t)L;
    const uint32_t b = bin_of(x);
    uint32_t k0 = start[b];
    const uint32_t s1 = start[b + 1];
    // records past the bin's end are larger: only the loop's end needs it
    for (uint32_t i = k0; i < s1; i += kBucketPad) {
      uint64_t m[kBucketPad];
#pragma unroll
      for (int u = 0; u < kBucketPad; ++u) m[u] = buf[i + u];
#pragma unroll
      for (int u = 0; u < kBucketPad; ++u) k0 += m[u] < x ? 1u : 0u;
    }
    return k0;
  };
  if (!a.perm_in && !a.aux_out) {
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = slot_of(r);
      if (L >= n) continue;
      const uint64_t x = v[r];
      const uint32_t k0 = rank_of(x, L);
      po[k0] = (int32_t)((uint32_t)x ^ tmask);
      if (a.key_out) store_sorted(ko, a.key_out_dtype, DT, k0, (uint32_t)(x >> 32) ^ dmask);
    }
    return;
  }
  // composed with an incoming permutation, or a second key to gather: each
  // batch of dependent loads in flight at once
  uint32_t rank[E], col[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int L = slot_of(r);
    rank[r] = 0u;
    col[r] = 0u;
    if (L >= n) continue;
    const uint64_t x = v[r];
    rank[r] = rank_of(x, L);
    const uint32_t pos = (uint32_t)x ^ tmask;
    col[r] = a.perm_in ? (uint32_t)a.perm_in[base + pos] : pos;
    if (a.key_out) store_sorted(ko, a.key_out_dtype, DT, rank[r], (uint32_t)(x >> 32) ^ dmask);
  }
#pragma unroll
  for (int r = 0; r < E; ++r)
    if (slot_of(r) < n) po[rank[r]] = (int32_t)col[r];
  if (a.aux_out) {
    uint32_t u[E];
    if (a.aux_dtype == kBF16) {
#pragma unroll
      for (int r = 0; r < E; ++r)
        u[r] = slot_of(r) < n ? key_bits_at<kBF16>(a.aux, base + col[r]) : 0u;
    } else {
#pragma unroll
      for (int r = 0; r < E; ++r)
        u[r] = slot_of(r) < n ? key_bits_at<kF32>(a.aux, base + col[r]) : 0u;
    }
#pragma unroll
    for (int r = 0; r < E; ++r)
      if (slot_of(r) < n)
        store_sorted(a.aux_out, a.aux_out_dtype, a.aux_dtype, ob + rank[r], order_from_bits(u[r], a.aux_dtype));
  }
}

// Rows of at most E * kChunkNT (<= kWideChunk) elements sorted whole by one
// workgroup: the chunk pass's records and radix sort, then the outputs
// straight from the sorted records (the bucket pass's output step at rank 0).
// An LDS bitonic network moves O(n log^2 n) records per row; this sort moves
// each record once per varying digit ([256, 16384] f32: 32.4 us against
// 190.8 us for the network).  For bfloat16 keys the low 16 order bits follow
// from the high 16 (they are zero or the sign's complement, and every NaN
// has one order), so only the high two digits are sorted.
template <int DT, bool PERM, int E>
__global__ __launch_bounds__(kChunkNT) void sort_row_radix_kernel(SortArgs a) {
  constexpr int NW = kChunkNT / kWave;
  extern __shared__ __align__(16) unsigned char smem[];
  uint64_t* buf = (uint64_t*)smem;                 // E * kChunkNT records
  uint32_t* hist = (uint32_t*)(buf + E * kChunkNT);  // 256 * (NW + 1) counters
  __shared__ uint32_t wsum[NW];
  __shared__ uint32_t red[2][NW];
  const int t = threadIdx.x, l = lane_id(), w = t / kWave;
  const int64_t row = blockIdx.x;
  const int64_t base = row * a.cols;
  const int n = (int)a.cols;  // 1 <= n <= E * kChunkNT (host routing)
  uint32_t kand = ~0u, kor = 0u;
  uint64_t v[E];
  {
    uint32_t raw[E];
    int32_t src[E];
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (E * kWave) + r * kWave + l;
      src[r] = a.ties_desc ? n - 1 - L : L;
      if (PERM && L < n) src[r] = a.perm_in[base + src[r]];
    }
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (E * kWave) + r * kWave + l;
      raw[r] = L < n ? key_bits_at<DT>(a.key, base + src[r]) : 0u;
    }
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (E * kWave) + r * kWave + l;
      v[r] = ~0ull;
      if (L < n) {
        uint32_t k = order_from_bits(raw[r], DT);
        if (a.descending) k = ~k;
        const uint32_t p = (uint32_t)(a.ties_desc ? n - 1 - L : L);
        const uint32_t tie = a.ties_desc ? kTieMask - p : p;
        v[r] = ((uint64_t)k << 32) | tie;
        kand &= k;
        kor |= k;
      }
    }
  }
  kand = wave_and_u32(kand);
  kor = wave_or_u32(kor);
  if (l == 0) {
    red[0][w] = kand;
    red[1][w] = kor;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    kand &= red[0][i];
    kor |= red[1][i];
  }
  const uint32_t varying = (kand ^ kor) & (DT == kBF16 ? 0xFFFF0000u : ~0u);
  radix_sort_slots<E, kChunkNT>(v, buf, hist, wsum, varying, n);
  int32_t col[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int L = w * (E * kWave) + r * kWave + l;
    col[r] = 0;
    if (L < n) {
      const uint32_t tie = (uint32_t)v[r];
      const int32_t pos = (int32_t)(a.ties_desc ? kTieMask - tie : tie);
      col[r] = PERM ? a.perm_in[base + pos] : pos;
    }
  }
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int L = w * (E * kWave) + r * kWave + l;
    if (L >= n) continue;
    a.perm_out[base + L] = col[r];
    if (a.key_out) {
      uint32_t key = (uint32_t)(v[r] >> 32);
      if (a.descending) key = ~key;
      store_sorted(a.key_out, a.key_out_dtype, a.key_dtype, base + L, key);
    }
  }
  if (a.aux_out) {
    uint32_t u[E];
    if (a.aux_dtype == kBF16) {
#pragma unroll
      for (int r = 0; r < E; ++r)
        u[r] = w * (E * kWave) + r * kWave + l < n ? key_bits_at<kBF16>(a.aux, base + col[r]) : 0u;
    } else {
#pragma unroll
      for (int r = 0; r < E; ++r)
        u[r] = w * (E * kWave) + r * kWave + l < n ? key_bits_at<kF32>(a.aux, base + col[r]) : 0u;
    }
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const int L = w * (E * kWave) + r * kWave + l;
      if (L < n)
        store_sorted(a.aux_out, a.aux_out_dtype, a.aux_dtype, base + L, order_from_bits(u[r], a.aux_dtype));
    }
  }
}

template <int DT, bool PERM, int E>
static int launch_row_radix_e(const SortArgs& a, int64_t rows, hipStream_t s) {
  const int lds = E * kChunkNT * 8 + 256 * (kChunkNT / kWave + 1) * 4;
  const hipError_t attr = set_dynamic_lds_limit((const void*)sort_row_radix_kernel<DT, PERM, E>, lds, s);
  if (attr != hipSuccess) {
    set_error("hipFuncSetAttribute: %s", hipGetErrorString(attr));
    return kHipError;
  }
  hipLaunchKernelGGL((sort_row_radix_kernel<DT, PERM, E>), dim3((unsigned)rows), dim3(kChunkNT), lds, s, a);
  return kOk;
}

template <int DT, bool PERM>
static int launch_row_radix_dt(const SortArgs& a, int64_t rows, hipStream_t s) {
  if (a.cols <= 4 * kChunkNT) return launch_row_radix_e<DT, PERM, 4>(a, rows, s);
  if (a.cols <= 8 * kChunkNT) return launch_row_radix_e<DT, PERM, 8>(a, rows, s);
  if (a.cols <= 16 * kChunkNT) return launch_row_radix_e<DT, PERM, 16>(a, rows, s);
  return launch_row_radix_e<DT, PERM, 32>(a, rows, s);
}

template <int DT, bool PERM, int E>
static int launch_chunks_one(const SortArgs& a, int64_t rows, int64_t nchunks, uint64_t* out, hipStream_t s) {
  const int lds = E * kChunkNT * 8 + 256 * (kChunkNT / kWave + 1) * 4;  // records + digit counters
  const hipError_t attr = set_dynamic_lds_limit((const void*)sort_chunks_kernel<DT, PERM, E>, lds, s);
  if (attr != hipSuccess) {
    set_error("hipFuncSetAttribute: %s", hipGetErrorString(attr));
    return kHipError;
  }
  hipLaunchKernelGGL((sort_chunks_kernel<DT, PERM, E>), dim3((unsigned)(rows * nchunks)), dim3(kChunkNT), lds, s, a,
                     (int)nchunks, out);
  return kOk;
}
template <int DT, bool PERM>
static int launch_chunks(const SortArgs& a, int64_t rows, int64_t nchunks, int chunk, uint64_t* out, hipStream_t s) {
  return chunk == kWideChunk ? launch_chunks_one<DT, PERM, kChunkE>(a, rows, nchunks, out, s)
                             : launch_chunks_one<DT, PERM, kChunkE / 2>(a, rows, nchunks, out, s);
}

template <int NT, int E, int DT>
static int launch_buckets_one(const SortArgs& a, int64_t rows, const BucketPlan& bp, const uint64_t* runs,
                              const int32_t* table, hipStream_t s) {
  const int lds = (E * NT + kBucketPad) * 8 + 256 * (NT / kWave + 1) * 4;
  const hipError_t attr = set_dynamic_lds_limit((const void*)bucket_sort_kernel<NT, E, DT>, lds, s);
  if (attr != hipSuccess) {
    set_error("hipFuncSetAttribute: %s", hipGetErrorString(attr));
    return kHipError;
  }
  hipLaunchKernelGGL((bucket_sort_kernel<NT, E, DT>), dim3((unsigned)(rows * bp.K)), dim3(NT), lds, s, a, bp, runs,
                     table);
  return kOk;
}
template <int DT>
static int launch_buckets(const SortArgs& a, int64_t rows, const BucketPlan& bp, const uint64_t* runs,
                          const int32_t* table, hipStream_t s) {
  if (bp.cap == 4096) return launch_buckets_one<256, 16, DT>(a, rows, bp, runs, table, s);
  if (bp.cap == 8192) return launch_buckets_one<512, 16, DT>(a, rows, bp, runs, table, s);
  return launch_buckets_one<512, 32, DT>(a, rows, bp, runs, table, s);
}

static int wide_passes(int64_t cols) {
  const int64_t nchunks = (cols + kWideChunk - 1) / kWideChunk;
  int passes = 0;
  while (((int64_t)1 << passes) < nchunks) ++passes;
  return passes;
}

size_t sort_wide_workspace_bytes(int64_t rows, int64_t cols) {
  if (cols <= kWideChunk || rows <= 0) return 0;
  return (size_t)(wide_passes(cols) > 1 ? 2 : 1) * (size_t)rows * (size_t)cols * sizeof(uint64_t);
}

int launch_sort_wide(const SortArgs& a, int64_t rows, void* ws, size_t ws_bytes, hipStream_t s) {
  const int64_t cols = a.cols;
  if (cols > (int64_t)kTieMask) {
    set_error("rows of %lld elements exceed the wide sort's limit of 2^31 - 1", (long long)cols);
    return kUnsupported;
  }
  // Rows whose samples fit at a stride of 64 take half chunks, two workgroups to a
  // CU: one's LDS work covers the other's barriers (f32 [1024, 201088], whole / half
  // chunks: 2510 / 2405 us, chunks 1340 / 1000, splitters 177 / 272, buckets
  // 994 / 1197; [300, 50257] i32 282 / 225, [14, 60833] 60 / 55, bf16 [64, 131072]
  // 140 / 123).  Past kHalfChunkCols twice the runs cost the splitters and the
  // buckets more than the chunks gain (f32, [16, 229377] 98 / 109, [50, 262144]
  // 228 / 245, [4, 262144] 89 / 96; [4, 201088] 83 / 73).  Rows of two whole chunks
  // stay on the merge pass: their workspace holds no splitter table.
  const bool fine = cols > 2 * kWideChunk && cols <= (int64_t)kSplitSamples * kBucketStrideFine;
  const bool half = fine && cols <= kHalfChunkCols;
  const int chunk = half ? kWideChunk / 2 : kWideChunk;
  const int64_t nchunks = (cols + chunk - 1) / chunk;
  const int64_t tiles = (cols + kMergeTile - 1) / kMergeTile;
  if (rows * tiles > 2147483647 || rows * nchunks > 2147483647) {
    set_error("sort of %lld x %lld elements needs more than 2^31 - 1 workgroups", (long long)rows, (long long)cols);
    return kUnsupported;
  }
  const size_t need = sort_wide_workspace_bytes(rows, cols);
  if (!ws || ws_bytes < need) {
    set_error("rows of %lld elements need a workspace of %zu bytes, got %zu", (long long)cols, need,
              ws ? ws_bytes : (size_t)0);
    return kWorkspaceTooSmall;
  }
  uint64_t* buf[2] = {(uint64_t*)ws, (uint64_t*)ws + (size_t)rows * (size_t)cols};
  int st = a.key_dtype == kBF16 ? (a.perm_in ? launch_chunks<kBF16, true>(a, rows, nchunks, chunk, buf[0], s)
                                              : launch_chunks<kBF16, false>(a, rows, nchunks, chunk, buf[0], s))
         : a.key_dtype == kI32  ? (a.perm_in ? launch_chunks<kI32, true>(a, rows, nchunks, chunk, buf[0], s)
                                              : launch_chunks<kI32, false>(a, rows, nchunks, chunk, buf[0], s))
                                : (a.perm_in ? launch_chunks<kF32, true>(a, rows, nchunks, chunk, buf[0], s)
                                              : launch_chunks<kF32, false>(a, rows, nchunks, chunk, buf[0], s));
  if (!st) st = launch_status("tallax_sort_rows (chunks)");
  if (st) return st;
  // rows of 3 .. kBucketMaxRuns chunks: the multiway merge by splitters
  // (the table lives in the second workspace buffer, which exists whenever
  // there are two or more pairwise passes)
  if (nchunks >= 3 && nchunks <= kBucketMaxRuns) {
    BucketPlan bp;
    bp.runs = (int)nchunks;
    bp.chunk = chunk;
    bp.G = fine ? kBucketStrideFine : kBucketStride;
    bp.cap = fine ? 4096 : bp.runs <= 24 ? 8192 : 16384;
    bp.samples = 0;
    for (int j = 0; j < bp.runs; ++j) bp.samples += run_len(cols, bp.chunk, j) / bp.G;
    bp.m = bp.cap / bp.G - bp.runs;  // (m + runs) G = capacity
    // few rows: smaller buckets, so that they fill the chip once
    const int64_t want = ((int64_t)256 * (16384 / bp.cap) + rows - 1) / rows;
    int64_t fine = (bp.samples + want - 1) / want;
    // ... but at most about two searches per thread of the splitter kernel
    const int64_t least = ((int64_t)bp.samples * bp.runs + 2 * kSplitNT - 1) / (2 * kSplitNT);
    fine = fine < least ? least : fine;
    if (fine < bp.m) bp.m = fine < 8 ? 8 : (int)fine;
    bp.K = (bp.samples + bp.m - 1) / bp.m;
    if (bp.K < 1) bp.K = 1;
    if (rows * bp.K > 2147483647) {
      set_error("sort of %lld rows needs more than 2^31 - 1 workgroups", (long long)rows);
      return kUnsupported;
    }
    int32_t* table = (int32_t*)buf[1];
    hipLaunchKernelGGL(bucket_split_kernel, dim3((unsigned)rows), dim3(kSplitNT), 0, s, a, bp, buf[0], table);
    st = launch_status("tallax_sort_rows (splitters)");
    if (st) return st;
    const int st2 = a.key_dtype == kBF16 ? launch_buckets<kBF16>(a, rows, bp, buf[0], table, s)
                    : a.key_dtype == kI32 ? launch_buckets<kI32>(a, rows, bp, buf[0], table, s)
                                          : launch_buckets<kF32>(a, rows, bp, buf[0], table, s);
    if (st2) return st2;
    return launch_status("tallax_sort_rows (buckets)");
  }
  const int passes = wide_passes(cols);
  for (int p = 0; p < passes && !st; ++p) {
    const int64_t run = (int64_t)kWideChunk << p;
    const dim3 grid((unsigned)(rows * tiles));
    if (p + 1 == passes)
      hipLaunchKernelGGL(merge_runs_kernel<true>, grid, dim3(kMergeNT), 0, s, a, buf[p & 1], nullptr, run,
                         (int)tiles);
    else
      hipLaunchKernelGGL(merge_runs_kernel<false>, grid, dim3(kMergeNT), 0, s, a, buf[p & 1], buf[(p + 1) & 1],
                         run, (int)tiles);
    st = launch_status("tallax_sort_rows (merge)");
  }
  return st;
}

int launch_sort_row_radix(const SortArgs& a, int64_t rows, hipStream_t s) {
  if (a.cols < 1 || a.cols > kWideChunk) {
    set_error("row radix sort: %lld columns outside [1, %d]", (long long)a.cols, kWideChunk);
    return kInvalidArgument;
  }
  if (a.key_dtype == kBF16)
    return a.perm_in ? launch_row_radix_dt<kBF16, true>(a, rows, s) : launch_row_radix_dt<kBF16, false>(a, rows, s);
  if (a.key_dtype == kI32)
    return a.perm_in ? launch_row_radix_dt<kI32, true>(a, rows, s) : launch_row_radix_dt<kI32, false>(a, rows, s);
  return a.perm_in ? launch_row_radix_dt<kF32, true>(a, rows, s) : launch_row_radix_dt<kF32, false>(a, rows, s);
}

}  // namespace tx
