// Device-wide radix sorts used by kernel-map construction (output-coordinate
// ordering and the row permutation of the sorted implicit-GEMM map).  The sort
// itself is rocPRIM's; scratch comes from the caller.
#include <algorithm>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include "common.h"

using namespace tsmi;

namespace {
constexpr int64_t kAlign = 256;
}

extern "C" int64_t tsmi_sort_temp_bytes(int64_t n) {
  if (n < 0) return -1;
  if (n == 0) n = 1;
  size_t a = 0, b = 0;
  hipError_t e1 = rocprim::radix_sort_keys(nullptr, a, (const unsigned long long *)nullptr,
                                           (unsigned long long *)nullptr, (size_t)n, 0, 64,
                                           (hipStream_t)0);
  hipError_t e2 = rocprim::radix_sort_pairs_desc(
      nullptr, b, (const int32_t *)nullptr, (int32_t *)nullptr,
      rocprim::counting_iterator<int32_t>(0), (int32_t *)nullptr, (size_t)n, 0, 32, (hipStream_t)0);
  if (e1 != hipSuccess || e2 != hipSuccess) {
    fail(TSMI_ERR_HIP, "sort_temp_bytes: size query failed");
    return -1;
  }
  int64_t m = (int64_t)(a > b ? a : b);
  return (m + kAlign - 1) / kAlign * kAlign + kAlign;
}

extern "C" int tsmi_sort_keys(tsmi_stream_t s, const int64_t *keys_in, int64_t *keys_out, int64_t n,
                              int end_bit, void *temp, int64_t temp_bytes) {
  TSMI_REQUIRE(n >= 0 && end_bit >= 1 && end_bit <= 64, "sort_keys: bad arguments");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(keys_in && keys_out && temp, "sort_keys: null pointer");
  size_t need = 0;
  (void)rocprim::radix_sort_keys(nullptr, need, (const unsigned long long *)keys_in,
                                 (unsigned long long *)keys_out, (size_t)n, 0, end_bit,
                                 (hipStream_t)s);
  TSMI_REQUIRE((int64_t)need <= temp_bytes, "sort_keys: scratch too small (%lld < %lld)",
               (long long)temp_bytes, (long long)need);
  hipError_t e = rocprim::radix_sort_keys(temp, need, (const unsigned long long *)keys_in,
                                          (unsigned long long *)keys_out, (size_t)n, 0, end_bit,
                                          (hipStream_t)s);
  if (e != hipSuccess) return fail(TSMI_ERR_HIP, "sort_keys: %s", hipGetErrorString(e));
  return check_launch("tsmi_sort_keys");
}

extern "C" int tsmi_argsort_desc(tsmi_stream_t s, const int32_t *keys_in, int32_t *keys_out,
                                 int32_t *idx_out, int rows, int64_t n, void *temp,
                                 int64_t temp_bytes) {
  TSMI_REQUIRE(rows >= 1 && n >= 0 && n < (int64_t(1) << 31), "argsort_desc: bad sizes");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(keys_in && keys_out && idx_out && temp, "argsort_desc: null pointer");
  size_t need = 0;
  (void)rocprim::radix_sort_pairs_desc(nullptr, need, keys_in, keys_out,
                                       rocprim::counting_iterator<int32_t>(0), idx_out, (size_t)n,
                                       0, 32, (hipStream_t)s);
  TSMI_REQUIRE((int64_t)need <= temp_bytes, "argsort_desc: scratch too small (%lld < %lld)",
               (long long)temp_bytes, (long long)need);
  for (int r = 0; r < rows; ++r) {
    hipError_t e = rocprim::radix_sort_pairs_desc(
        temp, need, keys_in + (int64_t)r * n, keys_out + (int64_t)r * n,
        rocprim::counting_iterator<int32_t>(0), idx_out + (int64_t)r * n, (size_t)n, 0, 32,
        (hipStream_t)s);
    if (e != hipSuccess) return fail(TSMI_ERR_HIP, "argsort_desc: %s", hipGetErrorString(e));
  }
  return check_launch("tsmi_argsort_desc");
}

// ---------------------------------------------------------------- grouping by index
// order = the entries of idx with a value in [0, n_groups), sorted by (value, position);
// starts[v] = first position of value v in `order`.  Row sums over the entries of a group
// (voxelize, the gradient of devoxelize) then run without atomics and in a fixed order.
//
// Two levels, four launches.  The high bits of a value name a bucket of at most 2048 neighbouring
// groups: group_count_kernel counts every tile's entries per bucket, group_scan_kernel turns a
// bucket's counts into positions, group_scatter_kernel moves (value, position) pairs to their bucket,
// and group_bucket_kernel - a workgroup per bucket - sorts its pairs by the low bits and writes
// `order` and `starts`.  Every step keeps entries of one value in the order of their positions: a
// wavefront ranks its 64 entries by ballots over the digit's bits, wavefronts and tiles follow each
// other in order.  What bounds it are the dependent round trips of four short launches.  The library
// sort it replaces made 13 and more (merge sort of 32-bit keys with block merges): 104k and 832k entries in
// 52k groups took 211 us together, 70 in this form.

namespace {

constexpr int kTileThreads = 512;                    // eight wavefronts
constexpr int kTileWaves = kTileThreads / 64;
constexpr int kPerLane = 8;                          // entries per lane: a tile is 4096 entries
constexpr int kTile = kTileThreads * kPerLane;
constexpr int kMaxBuckets = 1024, kMaxLow = 2048;    // digits the two levels take
constexpr int kMaxBits = 21;

struct Split {
  int low_bits, buckets;  // value = bucket << low_bits | low
};

// Low digits as small as the buckets allow: many buckets keep many workgroups busy, but no fewer
// than 64 groups to a bucket, whose starts a workgroup writes together.
inline Split split_for(int64_t n_groups) {
  int bits = 1;
  while ((int64_t(1) << bits) < n_groups) ++bits;
  Split s;
  s.low_bits = bits - 10 > 6 ? bits - 10 : 6;
  s.buckets = (int)((n_groups + (int64_t(1) << s.low_bits) - 1) >> s.low_bits);
  return s;
}

// Lanes of the wavefront with the same `digit` among those that are `in`.
__device__ __forceinline__ unsigned long long same_digit(uint32_t digit, int bits, bool in) {
  unsigned long long peers = __ballot(in);
  for (int b = 0; b < bits; ++b) {
    const bool one = (digit >> b) & 1;
    const unsigned long long m = __ballot(in && one);
    peers &= one ? m : ~m;
  }
  return peers;
}

__global__ __launch_bounds__(kTileThreads) void group_count_kernel(const int32_t *idx, int64_t m, uint32_t n_groups,
                                                                   int low_bits, int buckets, int64_t n_tiles,
                                                                   int32_t *counts) {
  __shared__ int32_t hist[kMaxBuckets];
  for (int b = threadIdx.x; b < buckets; b += kTileThreads) hist[b] = 0;
  __syncthreads();
  const int64_t first = (int64_t)blockIdx.x * kTile;
  uint32_t v[kPerLane];
#pragma unroll
  for (int r = 0; r < kPerLane; ++r) {
    const int64_t i = first + r * kTileThreads + threadIdx.x;
    v[r] = i < m ? (uint32_t)idx[i] : 0xFFFFFFFFu;
  }
#pragma unroll
  for (int r = 0; r < kPerLane; ++r)
    if (v[r] < n_groups) atomicAdd(&hist[v[r] >> low_bits], 1);
  __syncthreads();
  for (int b = threadIdx.x; b < buckets; b += kTileThreads) counts[(int64_t)b * n_tiles + blockIdx.x] = hist[b];
}

// counts[b][t] -> entries of bucket b in the tiles before t; totals[b] = entries of bucket b.
__global__ __launch_bounds__(256) void group_scan_kernel(int32_t *counts, int64_t n_tiles, int32_t *totals) {
  __shared__ int32_t wave_sum[4];
  int32_t *row = counts + (int64_t)blockIdx.x * n_tiles;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int32_t carry = 0;
  for (int64_t t0 = 0; t0 < n_tiles; t0 += 256) {
    const int64_t t = t0 + threadIdx.x;
    const int32_t c = t < n_tiles ? row[t] : 0;
    int32_t incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t up = __shfl_up(incl, d);
      if (lane >= d) incl += up;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    int32_t before = carry;
    for (int w = 0; w < wave; ++w) before += wave_sum[w];
    if (t < n_tiles) row[t] = before + incl - c;
    carry += wave_sum[0] + wave_sum[1] + wave_sum[2] + wave_sum[3];
    __syncthreads();
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// out[b] = sum of totals[0..b), b < n <= 2048, by a whole workgroup of kTileThreads threads.
__device__ __forceinline__ void exclusive_sums(const int32_t *totals, int n, int32_t *out, int32_t *wave_sum) {
  constexpr int kPer = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int32_t c[kPer], sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int b = threadIdx.x * kPer + j;
    c[j] = b < n ? totals[b] : 0;
    sum += c[j];
  }
  int32_t incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t up = __shfl_up(incl, d);
    if (lane >= d) incl += up;
  }
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  int32_t before = incl - sum;
  for (int w = 0; w < wave; ++w) before += wave_sum[w];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int b = threadIdx.x * kPer + j;
    if (b < n) out[b] = before;
    before += c[j];
  }
  __syncthreads();
}

__global__ __launch_bounds__(kTileThreads) void group_scatter_kernel(const int32_t *idx, int64_t m, uint32_t n_groups,
                                                                     int low_bits, int buckets, int bucket_bits,
                                                                     int64_t n_tiles, const int32_t *offsets,
                                                                     const int32_t *totals, int2 *pairs) {
  extern __shared__ int32_t lds[];
  int32_t *base = lds;             // [buckets] first position of every bucket
  int32_t *hist = lds + buckets;   // [wavefront][buckets]
  __shared__ int32_t wave_sum[kTileWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int32_t *mine = hist + wave * buckets;
  for (int b = threadIdx.x; b < kTileWaves * buckets; b += kTileThreads) hist[b] = 0;
  exclusive_sums(totals, buckets, base, wave_sum);
  const int64_t first = (int64_t)blockIdx.x * kTile + wave * (64 * kPerLane) + lane;
  uint32_t v[kPerLane];
  int32_t rank[kPerLane];
#pragma unroll
  for (int r = 0; r < kPerLane; ++r) {
    const int64_t i = first + r * 64;
    v[r] = i < m ? (uint32_t)idx[i] : 0xFFFFFFFFu;
  }
#pragma unroll
  for (int r = 0; r < kPerLane; ++r) {
    const bool in = v[r] < n_groups;
    const uint32_t b = in ? v[r] >> low_bits : 0;
    const unsigned long long peers = same_digit(b, bucket_bits, in);
    if (in) {
      const int32_t seen = mine[b];
      rank[r] = seen + __popcll(peers & ((1ULL << lane) - 1ULL));
      if (lane == __ffsll(peers) - 1) mine[b] = seen + __popcll(peers);
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < buckets; b += kTileThreads) {
    int32_t at = base[b] + offsets[(int64_t)b * n_tiles + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) {
      const int32_t c = hist[w * buckets + b];
      hist[w * buckets + b] = at;
      at += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPerLane; ++r)
    if (v[r] < n_groups)
      pairs[mine[v[r] >> low_bits] + rank[r]] = make_int2((int)v[r], (int)(first + r * 64));
}

__global__ __launch_bounds__(kTileThreads) void group_bucket_kernel(const int2 *pairs, const int32_t *totals,
                                                                    int buckets, int low_bits, int64_t n_groups,
                                                                    int32_t *order, int32_t *starts) {
  extern __shared__ int32_t lds[];
  const int lows = 1 << low_bits;
  int32_t *base = lds;            // [buckets] first position of every bucket, then [lows] of every group
  int32_t *hist = lds + (buckets > lows ? buckets : lows);  // [wavefront][lows]
  __shared__ int32_t wave_sum[kTileWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int bucket = blockIdx.x;
  exclusive_sums(totals, buckets, base, wave_sum);
  const int32_t first = base[bucket], count = totals[bucket];
  const int64_t group0 = (int64_t)bucket << low_bits;
  for (int d = threadIdx.x; d < lows; d += kTileThreads) hist[d] = 0;
  __syncthreads();
  const int2 *in = pairs + first;
  for (int32_t i = threadIdx.x; i < count; i += kTileThreads) atomicAdd(&hist[in[i].x & (lows - 1)], 1);
  __syncthreads();
  exclusive_sums(hist, lows, base, wave_sum);
  for (int d = threadIdx.x; d < lows; d += kTileThreads)
    if (group0 + d < n_groups) starts[group0 + d] = first + base[d];
  if (bucket == buckets - 1 && threadIdx.x == 0) starts[n_groups] = first + count;
  int32_t *mine = hist + wave * lows;
  for (int32_t i0 = 0; i0 < count; i0 += kTile) {
    __syncthreads();  // (hist and base of the tile before are no longer read)
    for (int d = threadIdx.x; d < kTileWaves * lows; d += kTileThreads) hist[d] = 0;
    __syncthreads();
    int2 e[kPerLane];
    int32_t rank[kPerLane];
    const int32_t at0 = i0 + wave * (64 * kPerLane) + lane;
#pragma unroll
    for (int r = 0; r < kPerLane; ++r)
      if (at0 + r * 64 < count) e[r] = in[at0 + r * 64];
#pragma unroll
    for (int r = 0; r < kPerLane; ++r) {
      const bool ok = at0 + r * 64 < count;
      const uint32_t d = ok ? (uint32_t)e[r].x & (lows - 1) : 0;
      const unsigned long long peers = same_digit(d, low_bits, ok);
      if (ok) {
        const int32_t seen = mine[d];
        rank[r] = seen + __popcll(peers & ((1ULL << lane) - 1ULL));
        if (lane == __ffsll(peers) - 1) mine[d] = seen + __popcll(peers);
      }
    }
    __syncthreads();
    for (int d = threadIdx.x; d < lows; d += kTileThreads) {
      int32_t at = base[d];
#pragma unroll
      for (int w = 0; w < kTileWaves; ++w) {
        const int32_t c = hist[w * lows + d];
        hist[w * lows + d] = at;
        at += c;
      }
      base[d] = at;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPerLane; ++r)
      if (at0 + r * 64 < count) order[first + mine[(uint32_t)e[r].x & (lows - 1)] + rank[r]] = e[r].y;
  }
}

// More groups than the two levels take (2^21): the library sort.

struct GroupKey {
  uint32_t n_groups;
  __device__ uint32_t operator()(int32_t v) const {
    return (v < 0 || (uint32_t)v >= n_groups) ? n_groups : (uint32_t)v;  // sentinel sorts last
  }
};

using GroupKeyIter = rocprim::transform_iterator<const int32_t *, GroupKey, uint32_t>;

__global__ void group_starts_kernel(const uint32_t *sorted, int64_t m, int64_t n_groups,
                                    int32_t *starts) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v > n_groups) return;
  int64_t lo = 0, hi = m;  // first position with sorted[pos] >= v
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)sorted[mid] < v) lo = mid + 1; else hi = mid;
  }
  starts[v] = (int32_t)lo;
}

inline int64_t align_up(int64_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

}  // namespace

static int64_t two_level_bytes(int64_t m) {
  return align_up(m * 8) + align_up(4 * kMaxBuckets) + align_up(4 * kMaxBuckets * ceil_div(m, kTile));
}

extern "C" int64_t tsmi_group_temp_bytes(int64_t m) {
  if (m < 0) return -1;
  if (m == 0) m = 1;
  size_t need = 0;
  hipError_t e = rocprim::radix_sort_pairs(nullptr, need, GroupKeyIter((const int32_t *)nullptr, GroupKey{1}),
                                           (uint32_t *)nullptr, rocprim::counting_iterator<int32_t>(0),
                                           (int32_t *)nullptr, (size_t)m, 0, 32, (hipStream_t)0);
  if (e != hipSuccess) {
    fail(TSMI_ERR_HIP, "group_temp_bytes: size query failed");
    return -1;
  }
  return std::max(align_up(m * 4) + align_up((int64_t)need), two_level_bytes(m));
}

extern "C" int tsmi_group_by_index(tsmi_stream_t s, const int32_t *idx, int64_t m, int64_t n_groups,
                                   void *temp, int64_t temp_bytes, int32_t *order, int32_t *starts) {
  TSMI_REQUIRE(m >= 0 && m < (int64_t(1) << 31) && n_groups >= 0 && n_groups < (int64_t(1) << 31),
               "group_by_index: bad sizes");
  TSMI_REQUIRE(starts, "group_by_index: null starts");
  if (m == 0 || n_groups == 0) {
    const int64_t blocks0 = ceil_div(n_groups + 1, 256);
    TSMI_REQUIRE(grid_fits(blocks0), "group_by_index: too many groups");
    hipLaunchKernelGGL(group_starts_kernel, dim3((unsigned)blocks0), dim3(256), 0, (hipStream_t)s,
                       (const uint32_t *)nullptr, (int64_t)0, n_groups, starts);
    return check_launch("tsmi_group_by_index");
  }
  TSMI_REQUIRE(idx && order && temp, "group_by_index: null pointer");
  if (n_groups <= (int64_t(1) << kMaxBits)) {
    TSMI_REQUIRE(temp_bytes >= two_level_bytes(m), "group_by_index: scratch too small (%lld < %lld)",
                 (long long)temp_bytes, (long long)two_level_bytes(m));
    const Split sp = split_for(n_groups);
    int bucket_bits = 0;
    while ((1 << bucket_bits) < sp.buckets) ++bucket_bits;
    const int64_t n_tiles = ceil_div(m, kTile);
    int2 *pairs = (int2 *)temp;
    int32_t *totals = (int32_t *)((char *)temp + align_up(m * 8));
    int32_t *counts = totals + align_up(4 * kMaxBuckets) / 4;
    const int lows = 1 << sp.low_bits;
    hipLaunchKernelGGL(group_count_kernel, dim3((unsigned)n_tiles), dim3(kTileThreads), 0, (hipStream_t)s, idx, m,
                       (uint32_t)n_groups, sp.low_bits, sp.buckets, n_tiles, counts);
    hipLaunchKernelGGL(group_scan_kernel, dim3((unsigned)sp.buckets), dim3(256), 0, (hipStream_t)s, counts, n_tiles,
                       totals);
    hipLaunchKernelGGL(group_scatter_kernel, dim3((unsigned)n_tiles), dim3(kTileThreads),
                       (size_t)sp.buckets * (1 + kTileWaves) * 4, (hipStream_t)s, idx, m, (uint32_t)n_groups,
                       sp.low_bits, sp.buckets, bucket_bits, n_tiles, counts, totals, pairs);
    static std::atomic<uint64_t> configured{0};
    const size_t lds = ((size_t)std::max(sp.buckets, lows) + (size_t)kTileWaves * lows) * 4;
    if (int e = raise_dynamic_lds((const void *)group_bucket_kernel, (kMaxLow + kTileWaves * kMaxLow) * 4, configured,
                                  "group_bucket_kernel"))
      return e;
    hipLaunchKernelGGL(group_bucket_kernel, dim3((unsigned)sp.buckets), dim3(kTileThreads), lds, (hipStream_t)s, pairs,
                       totals, sp.buckets, sp.low_bits, n_groups, order, starts);
    return check_launch("tsmi_group_by_index");
  }
  int bits = 1;
  while (bits < 32 && (int64_t(1) << bits) <= n_groups) ++bits;  // values 0..n_groups inclusive
  uint32_t *sorted = (uint32_t *)temp;
  void *sort_temp = (char *)temp + align_up(m * 4);
  GroupKeyIter keys(idx, GroupKey{(uint32_t)n_groups});
  size_t need = 0;
  (void)rocprim::radix_sort_pairs(nullptr, need, keys, sorted, rocprim::counting_iterator<int32_t>(0),
                                  order, (size_t)m, 0, bits, (hipStream_t)s);
  TSMI_REQUIRE(align_up(m * 4) + (int64_t)need <= temp_bytes,
               "group_by_index: scratch too small (%lld < %lld)", (long long)temp_bytes,
               (long long)(align_up(m * 4) + (int64_t)need));
  hipError_t e = rocprim::radix_sort_pairs(sort_temp, need, keys, sorted,
                                           rocprim::counting_iterator<int32_t>(0), order, (size_t)m, 0,
                                           bits, (hipStream_t)s);
  if (e != hipSuccess) return fail(TSMI_ERR_HIP, "group_by_index: %s", hipGetErrorString(e));
  const int64_t blocks = ceil_div(n_groups + 1, 256);
  TSMI_REQUIRE(grid_fits(blocks), "group_by_index: too many groups");
  hipLaunchKernelGGL(group_starts_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)s,
                     (const uint32_t *)sorted, m, n_groups, starts);
  return check_launch("tsmi_group_by_index");
}
