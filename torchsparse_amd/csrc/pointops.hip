// Point-voxel operators for gfx950 and their C entry points: coordinate hashing, per-voxel
// counts, voxelize (mean of the points of a voxel), devoxelize (trilinear interpolation
// from 8 corner voxels), dense <-> sparse copies.
//
// All of them are HBM-bound row copies or row sums.  A thread owns V consecutive channels
// of one row (16 bytes when the channel count allows it, one element otherwise), so a row
// is read and written in whole 16-byte pieces and neighbouring lanes touch neighbouring
// addresses.  Sums over several rows run in fp32.  The two scatter-shaped sums (voxelize
// forward, devoxelize backward) are turned into gathers: the caller groups the indices once
// (tsmi_group_by_index: entries sorted by (voxel, position) + the start of every voxel's
// run), and a thread then adds the rows of its voxel in that fixed order — no atomics, the
// result is the same bit pattern on every run.  (fp32 atomic adds into the output, the
// reference's way, ran at ~40 G adds/s here: 1.8 ms / 12.6 ms for the 1M-point cases
// against a fraction of a millisecond for the gathers.)
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <initializer_list>

#include "common.h"

namespace tsmi {
namespace {

constexpr int kBlock = 256;

inline dim3 grid_for(int64_t n) { return dim3((unsigned)ceil_div(n > 0 ? n : 1, kBlock)); }

#define TSMI_GRID_CHECK(n) \
  TSMI_REQUIRE(grid_fits(ceil_div((n), kBlock)), "%s: problem too large for one launch", __func__)

template <typename T>
struct Elem;
template <>
struct Elem<float> {
  static __device__ __forceinline__ float load(const float *p) { return *p; }
  static __device__ __forceinline__ void store(float *p, float v) { *p = v; }
};
template <>
struct Elem<_Float16> {
  static __device__ __forceinline__ float load(const _Float16 *p) { return (float)*p; }
  static __device__ __forceinline__ void store(_Float16 *p, float v) { *p = (_Float16)v; }
};
template <>
struct Elem<__bf16> {
  static __device__ __forceinline__ float load(const __bf16 *p) { return (float)*p; }
  static __device__ __forceinline__ void store(__bf16 *p, float v) { *p = (__bf16)v; }
};

// V elements of type T as one vector access (V * sizeof(T) is 16 bytes or one element).
template <typename T, int V>
struct alignas(sizeof(T) * V) Pack {
  T v[V];
};

template <typename T, int V>
__device__ __forceinline__ void load_row(const T *p, float *out) {
  const Pack<T, V> q = *(const Pack<T, V> *)p;
#pragma unroll
  for (int e = 0; e < V; ++e) out[e] = Elem<T>::load(&q.v[e]);
}
template <typename T, int V>
__device__ __forceinline__ void store_row(T *p, const float *in) {
  Pack<T, V> q;
#pragma unroll
  for (int e = 0; e < V; ++e) Elem<T>::store(&q.v[e], in[e]);
  *(Pack<T, V> *)p = q;
}

template <typename T>
__global__ void fill_kernel(T *p, int64_t n, T v) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = v;
}

__device__ __forceinline__ unsigned long long fnv4(int a, int b, int c, int d) {
  unsigned long long h = 14695981039346656037ULL;
  h = (h ^ (unsigned int)a) * 1099511628211ULL;
  h = (h ^ (unsigned int)b) * 1099511628211ULL;
  h = (h ^ (unsigned int)c) * 1099511628211ULL;
  h = (h ^ (unsigned int)d) * 1099511628211ULL;
  return h;
}

__global__ void hash_kernel(const int4 *coords, int64_t n, long long *out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int4 c = coords[i];
  out[i] = (long long)fnv4(c.x, c.y, c.z, c.w);
}

// out[k*n + i]: thread per output element, i fastest (coalesced 8-byte stores; the row is
// re-read from cache for every offset).
__global__ void kernel_hash_kernel(const int4 *coords, int64_t n, const int *offsets, int kvol,
                                   long long *out) {
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * kvol) return;
  const int64_t k = t / n, i = t - k * n;
  const int4 c = coords[i];
  const int *o = offsets + 3 * k;
  out[t] = (long long)fnv4(c.x, c.y + o[0], c.z + o[1], c.w + o[2]);
}

__global__ void count_kernel(const int *idx, int64_t n, int s, int *out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int v = idx[i];
  if (v >= 0 && v < s) atomicAdd(out + v, 1);
}

// ---- an index over 64-bit keys
//
// An open-addressing table of 32-bit slots, four per key: row + 1 in the low bits and, where 20 bits
// hold every row, 12 bits of the hash above them, so that a look-up reads another row's key in one of 4096
// cases only; 0: empty.  What an insertion costs is its chain of compare-and-swaps, one memory round trip
// each: at a quarter full nearly every key is done after the first (52k keys 9 us with the
// launch that empties the table; 18 us half full, with 32-bit or 64-bit slots alike; 350k keys 25 against 37).
// Building it without device-wide atomics - workgroups that own a part of the table in LDS and read
// all keys - took 27 to 31 us for 52k keys, bound by the instructions that look at every key.
constexpr int kTagBits = 12;
constexpr int64_t kMaxTagged = (int64_t(1) << (32 - kTagBits)) - 1;

struct KeySlot {
  uint32_t slot, tag;  // tag: in place above the row bits
};
__device__ __forceinline__ KeySlot slot_of(unsigned long long k, uint32_t cap, uint32_t tag_mask) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdULL;
  k ^= k >> 29;
  return {(uint32_t)(((k >> 20 & 0xFFFFFFFFULL) * cap) >> 32), ((uint32_t)k * 0x9E3779B1u) & tag_mask};
}

__global__ void index_clear_kernel(uint4 *slots, int64_t n4) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n4) slots[i] = make_uint4(0u, 0u, 0u, 0u);
}

__global__ void index_insert_kernel(const unsigned long long *keys, int64_t n, uint32_t cap, uint32_t tag_mask,
                                    uint32_t *slots) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const unsigned long long k = keys[i];
  const KeySlot at = slot_of(k, cap, tag_mask);
  const uint32_t stored = at.tag | (uint32_t)(i + 1);
  uint32_t slot = at.slot;
  for (;;) {  // (three slots in four stay empty: the chain ends)
    const uint32_t prev = atomicCAS(&slots[slot], 0u, stored);
    if (prev == 0u) return;
    if (((prev ^ at.tag) & tag_mask) == 0u && keys[(prev & ~tag_mask) - 1u] == k) return;
    slot = slot + 1 == cap ? 0 : slot + 1;
  }
}

__global__ void index_find_kernel(const unsigned long long *keys, uint32_t cap, uint32_t tag_mask,
                                  const uint32_t *slots, const unsigned long long *queries, int64_t m, int32_t *out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= m) return;
  const unsigned long long k = queries[i];
  const KeySlot at = slot_of(k, cap, tag_mask);
  uint32_t slot = at.slot;
  int32_t found = -1;
  for (;;) {
    const uint32_t held = slots[slot];
    if (held == 0u) break;
    if (((held ^ at.tag) & tag_mask) == 0u && keys[(held & ~tag_mask) - 1u] == k) {
      found = (int32_t)(held & ~tag_mask) - 1;
      break;
    }
    slot = slot + 1 == cap ? 0 : slot + 1;
  }
  out[i] = found;
}

// Trilinear weights, a thread per point: what twelve element-wise operations per corner and axis
// computed one launch at a time (55 launches, 110 us of kernels for 104k points; 5.8 here), in the order they did.
template <typename I>
__global__ void ti_weights_kernel(const float *points, int64_t n, int64_t rs, int64_t cs, const I *index, int64_t irs,
                                  int64_t ics, float scale, float inv, float inv3, float4 *weights) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float hi[3], lo[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float p = points[i * rs + a * cs];
    const float low = scale != 1.f ? __fmul_rn(floorf(__fmul_rn(p, inv)), scale) : floorf(p);
    hi[a] = __fsub_rn(p, low);
    lo[a] = __fsub_rn(__fadd_rn(low, scale), p);
  }
  float w[8], sum = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    float v = __fmul_rn(__fmul_rn((k & 4) ? hi[0] : lo[0], (k & 2) ? hi[1] : lo[1]), (k & 1) ? hi[2] : lo[2]);
    if (scale != 1.f) v = __fmul_rn(v, inv3);
    w[k] = index[i * irs + k * ics] == (I)-1 ? 0.f : v;
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) sum = __fadd_rn(sum, w[k]);
  sum = __fadd_rn(sum, 1e-8f);
#pragma unroll
  for (int k = 0; k < 8; ++k) w[k] = w[k] / sum;
  weights[2 * i] = make_float4(w[0], w[1], w[2], w[3]);
  weights[2 * i + 1] = make_float4(w[4], w[5], w[6], w[7]);
}

// Rows a thread has on their way at once in the two sums below: a voxel's rows are a chain
// of two dependent reads each (its place in `order`, then the row), which one at a time leave the
// memory system idle (64 fp16 channels, 104k points in 52k voxels: 20 us against 16; 832k corner entries: 61 us
// against 45, of it 7 through the order of the blocks, xcd_band_block).  The sums still run in the order of the entries.
constexpr int kInFlight = 4;

// out[v, :] = (sum of feats[order[p], :] for p in [starts[v], starts[v+1])) / counts[v]
template <typename T, int V>
__global__ void voxelize_forward_kernel(const T *feats, const int *order, const int *starts,
                                        const int *counts, int c, int64_t n1, T *out) {
  const int chunks = c / V;
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= n1 * chunks) return;
  const int64_t v = t / chunks;
  const int j = (int)(t - v * chunks) * V;
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = 0.f;
  const int cnt = counts[v];
  if (cnt != 0) {
    const int p1 = starts[v + 1];
    for (int p = starts[v]; p < p1; p += kInFlight) {
      int row[kInFlight];
      float x[kInFlight][V];
#pragma unroll
      for (int q = 0; q < kInFlight; ++q) row[q] = p + q < p1 ? order[p + q] : -1;
#pragma unroll
      for (int q = 0; q < kInFlight; ++q)
        if (row[q] >= 0) load_row<T, V>(feats + (int64_t)row[q] * c + j, x[q]);
#pragma unroll
      for (int q = 0; q < kInFlight; ++q)
        if (row[q] >= 0)
#pragma unroll
          for (int e = 0; e < V; ++e) acc[e] += x[q][e];
    }
    const float inv = 1.0f / (float)cnt;
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] *= inv;
  }
  store_row<T, V>(out + v * c + j, acc);
}

// bottom[i, :] = top[idx[i], :] / counts[idx[i]]
template <typename T, int V>
__global__ void voxelize_backward_kernel(const T *top, const int *idx, const int *counts, int64_t n,
                                         int c, int64_t n1, T *bottom) {
  const int chunks = c / V;
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * chunks) return;
  const int64_t i = t / chunks;
  const int j = (int)(t - i * chunks) * V;
  const int pos = idx[i];
  float v[V];
#pragma unroll
  for (int e = 0; e < V; ++e) v[e] = 0.f;
  if (pos >= 0 && pos < n1) {
    const int cnt = counts[pos];
    if (cnt != 0) {
      load_row<T, V>(top + (int64_t)pos * c + j, v);
      const float inv = 1.0f / (float)cnt;
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] *= inv;
    }
  }
  store_row<T, V>(bottom + i * c + j, v);
}

// out[i, :] = sum_k weight[i,k] * feat[indices[i,k], :]
template <typename T, int V>
__global__ void devoxelize_forward_kernel(const T *feat, const int *indices, const float *weight,
                                          int64_t n, int64_t n_vox, int c, T *out) {
  const int chunks = c / V;
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * chunks) return;
  const int64_t i = t / chunks;
  const int j = (int)(t - i * chunks) * V;
  const int4 ia = *(const int4 *)(indices + 8 * i), ib = *(const int4 *)(indices + 8 * i + 4);
  const float4 wa = *(const float4 *)(weight + 8 * i), wb = *(const float4 *)(weight + 8 * i + 4);
  const int id[8] = {ia.x, ia.y, ia.z, ia.w, ib.x, ib.y, ib.z, ib.w};
  const float w[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (id[k] < 0 || id[k] >= n_vox) continue;
    float v[V];
    load_row<T, V>(feat + (int64_t)id[k] * c + j, v);
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] += w[k] * v[e];
  }
  store_row<T, V>(out + i * c + j, acc);
}

// Workgroups go to the 8 XCDs round-robin, each with an L2 of its own.  Block b of n such that an XCD works
// on runs of 64 consecutive blocks: voxels that are neighbours read the same points (a point's row
// is needed by eight voxels), and ascending rows keep most of those within a run or the next.  A
// bijection on [0, n): the last, incomplete group of 512 blocks keeps the launch order.
__device__ __forceinline__ unsigned xcd_band_block(unsigned b, unsigned n) {
  if (b >= (n & ~511u)) return b;
  return (b & ~511u) + ((b & 7) << 6) + ((b >> 3) & 63);
}

// bottom[v, :] = sum over the entries e = order[p] (e = 8*i + k) of voxel v of weight[e] * top[i, :]
template <typename T, int V>
__global__ void devoxelize_backward_kernel(const T *top, const float *weight, const int *order,
                                           const int *starts, int64_t n_vox, int c, T *bottom) {
  const int chunks = c / V;
  const int64_t t = (int64_t)xcd_band_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (t >= n_vox * chunks) return;
  const int64_t v = t / chunks;
  const int j = (int)(t - v * chunks) * V;
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) acc[e] = 0.f;
  const int p1 = starts[v + 1];
  for (int p = starts[v]; p < p1; p += kInFlight) {
    int entry[kInFlight];
    float w[kInFlight], g[kInFlight][V];
#pragma unroll
    for (int q = 0; q < kInFlight; ++q) entry[q] = p + q < p1 ? order[p + q] : -1;
#pragma unroll
    for (int q = 0; q < kInFlight; ++q)
      if (entry[q] >= 0) {
        w[q] = weight[entry[q]];
        load_row<T, V>(top + (int64_t)(entry[q] >> 3) * c + j, g[q]);
      }
#pragma unroll
    for (int q = 0; q < kInFlight; ++q)
      if (entry[q] >= 0)
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] += w[q] * g[q][e];
  }
  store_row<T, V>(bottom + v * c + j, acc);
}

struct Range4 {
  int r[4];
};

__device__ __forceinline__ int64_t dense_cell(const int4 q, const Range4 &rg) {
  return (((int64_t)q.x * rg.r[1] + q.y) * rg.r[2] + q.z) * rg.r[3] + q.w;
}
__device__ __forceinline__ bool in_range(const int4 q, const Range4 &rg) {
  return q.x >= 0 && q.x < rg.r[0] && q.y >= 0 && q.y < rg.r[1] && q.z >= 0 && q.z < rg.r[2] &&
         q.w >= 0 && q.w < rg.r[3];
}

// dense[cell(coords[i]), :] = feats[i, :]  (TO_DENSE) or  feats[i, :] = dense[cell, :]
template <typename T, int V, bool TO_DENSE>
__global__ void dense_copy_kernel(T *feats, const int4 *coords, int64_t n, int c, Range4 rg, T *dense) {
  const int chunks = c / V;
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (t >= n * chunks) return;
  const int64_t i = t / chunks;
  const int j = (int)(t - i * chunks) * V;
  const int4 q = coords[i];
  const bool ok = in_range(q, rg);
  T *cell = dense + dense_cell(q, rg) * c + j;
  if (TO_DENSE) {
    if (ok) *(Pack<T, V> *)cell = *(const Pack<T, V> *)(feats + i * c + j);
  } else {
    Pack<T, V> v;
#pragma unroll
    for (int e = 0; e < V; ++e) v.v[e] = (T)0.f;
    if (ok) v = *(const Pack<T, V> *)cell;
    *(Pack<T, V> *)(feats + i * c + j) = v;
  }
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// Elements per thread: a 16-byte piece when the rows are made of whole, aligned pieces.
template <typename T>
inline int vec_width(int c, std::initializer_list<const void *> ptrs) {
  const int v = 16 / (int)sizeof(T);
  if (c % v != 0) return 1;
  for (const void *p : ptrs)
    if (!aligned16(p)) return 1;
  return v;
}

// Rows of c elements laid out in whole 16-byte pieces: a thread makes one piece.
template <typename T>
__global__ __launch_bounds__(256) void pad_columns_kernel(const T *x, int64_t n, int c, int pieces, uint4 *y) {
  constexpr int kPer = 16 / (int)sizeof(T);
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n * pieces) return;
  const int64_t r = i / pieces;
  const int first = (int)(i - r * pieces) * kPer;
  alignas(16) T v[kPer];
#pragma unroll
  for (int e = 0; e < kPer; ++e) v[e] = first + e < c ? x[r * c + first + e] : T{0};
  y[i] = *(const uint4 *)v;
}

}  // namespace
}  // namespace tsmi

using namespace tsmi;

#define TSMI_BY_DTYPE(dtype, CALL)                                   \
  switch (dtype) {                                                    \
    case TSMI_F32: { using T = float; CALL; break; }                  \
    case TSMI_F16: { using T = _Float16; CALL; break; }               \
    case TSMI_BF16: { using T = __bf16; CALL; break; }                \
    default: return fail(TSMI_ERR_INVALID_ARGUMENT, "%s: unknown dtype %d", __func__, dtype); \
  }

extern "C" int tsmi_hash_coords(tsmi_stream_t s, const int32_t *coords, int64_t n, int64_t *out) {
  TSMI_REQUIRE(n >= 0 && (n == 0 || (coords && out)), "hash_coords: bad arguments");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(aligned16(coords), "hash_coords: coords must be 16-byte aligned");
  TSMI_GRID_CHECK(n);
  hipLaunchKernelGGL(hash_kernel, grid_for(n), dim3(kBlock), 0, (hipStream_t)s, (const int4 *)coords, n,
                     (long long *)out);
  return check_launch("tsmi_hash_coords");
}

extern "C" int tsmi_kernel_hash(tsmi_stream_t s, const int32_t *coords, int64_t n,
                                const int32_t *offsets, int kvol, int64_t *out) {
  TSMI_REQUIRE(n >= 0 && kvol >= 0, "kernel_hash: bad sizes");
  if (n == 0 || kvol == 0) return TSMI_OK;
  TSMI_REQUIRE(coords && offsets && out, "kernel_hash: null pointer");
  TSMI_REQUIRE(aligned16(coords), "kernel_hash: coords must be 16-byte aligned");
  TSMI_GRID_CHECK(n * kvol);
  hipLaunchKernelGGL(kernel_hash_kernel, grid_for(n * kvol), dim3(kBlock), 0, (hipStream_t)s,
                     (const int4 *)coords, n, offsets, kvol, (long long *)out);
  return check_launch("tsmi_kernel_hash");
}

static inline uint32_t index_tag_mask(int64_t n) { return n <= kMaxTagged ? ~0u << (32 - kTagBits) : 0u; }

extern "C" int64_t tsmi_hash_index_words(int64_t n) {
  if (n < 0 || n >= (int64_t(1) << 29)) return -1;
  return 4 * (n > 16 ? n : 16);
}

extern "C" int tsmi_hash_index_build(tsmi_stream_t s, const int64_t *keys, int64_t n, int32_t *index) {
  const int64_t cap = tsmi_hash_index_words(n);
  TSMI_REQUIRE(cap > 0, "hash_index_build: %lld keys", (long long)n);
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(keys && index && aligned16(index), "hash_index_build: null or misaligned pointer");
  hipLaunchKernelGGL(index_clear_kernel, grid_for(cap / 4), dim3(kBlock), 0, (hipStream_t)s, (uint4 *)index, cap / 4);
  hipLaunchKernelGGL(index_insert_kernel, grid_for(n), dim3(kBlock), 0, (hipStream_t)s,
                     (const unsigned long long *)keys, n, (uint32_t)cap, index_tag_mask(n), (uint32_t *)index);
  return check_launch("tsmi_hash_index_build");
}

extern "C" int tsmi_hash_index_find(tsmi_stream_t s, const int64_t *keys, int64_t n, const int32_t *index,
                                    const int64_t *queries, int64_t m, int32_t *out) {
  const int64_t cap = tsmi_hash_index_words(n);
  TSMI_REQUIRE(cap > 0 && m >= 0, "hash_index_find: bad sizes");
  if (m == 0) return TSMI_OK;
  TSMI_REQUIRE(queries && out && (n == 0 || (keys && index)), "hash_index_find: null pointer");
  TSMI_GRID_CHECK(m);
  if (n == 0) {
    hipLaunchKernelGGL(fill_kernel<int32_t>, grid_for(m), dim3(kBlock), 0, (hipStream_t)s, out, m, -1);
    return check_launch("tsmi_hash_index_find");
  }
  hipLaunchKernelGGL(index_find_kernel, grid_for(m), dim3(kBlock), 0, (hipStream_t)s,
                     (const unsigned long long *)keys, (uint32_t)cap, index_tag_mask(n), (const uint32_t *)index,
                     (const unsigned long long *)queries, m, out);
  return check_launch("tsmi_hash_index_find");
}

extern "C" int tsmi_ti_weights(tsmi_stream_t s, const float *points, int64_t n, int64_t row_stride,
                               int64_t col_stride, const void *index, int index64, int64_t index_row_stride,
                               int64_t index_col_stride, float scale, float *weights) {
  TSMI_REQUIRE(n >= 0, "ti_weights: bad size");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(points && index && weights && aligned16(weights), "ti_weights: null or misaligned pointer");
  TSMI_GRID_CHECK(n);
  // (a division by a host value is a multiplication by its reciprocal, as torch has it)
  const float inv = 1.0f / scale, inv3 = 1.0f / (float)((double)scale * scale * scale);
  if (index64)
    hipLaunchKernelGGL(ti_weights_kernel<int64_t>, grid_for(n), dim3(kBlock), 0, (hipStream_t)s, points, n,
                       row_stride, col_stride, (const int64_t *)index, index_row_stride, index_col_stride, scale,
                       inv, inv3, (float4 *)weights);
  else
    hipLaunchKernelGGL(ti_weights_kernel<int32_t>, grid_for(n), dim3(kBlock), 0, (hipStream_t)s, points, n,
                       row_stride, col_stride, (const int32_t *)index, index_row_stride, index_col_stride, scale,
                       inv, inv3, (float4 *)weights);
  return check_launch("tsmi_ti_weights");
}

extern "C" int tsmi_count(tsmi_stream_t s, const int32_t *idx, int64_t n, int32_t *out, int num) {
  TSMI_REQUIRE(n >= 0 && num >= 0 && (num == 0 || out) && (n == 0 || idx), "count: bad arguments");
  if (num > 0)
    hipLaunchKernelGGL(fill_kernel<int32_t>, grid_for(num), dim3(kBlock), 0, (hipStream_t)s, out,
                       (int64_t)num, 0);
  if (n > 0 && num > 0) {
    TSMI_GRID_CHECK(n);
    hipLaunchKernelGGL(count_kernel, grid_for(n), dim3(kBlock), 0, (hipStream_t)s, idx, n, num, out);
  }
  return check_launch("tsmi_count");
}

namespace {

template <typename T>
int voxelize_forward_t(hipStream_t s, const void *feats, const int32_t *counts, const int32_t *order,
                       const int32_t *starts, int c, int64_t n1, void *out) {
  if (vec_width<T>(c, {feats, out}) > 1) {
    constexpr int V = 16 / (int)sizeof(T);
    hipLaunchKernelGGL((voxelize_forward_kernel<T, V>), grid_for(n1 * (c / V)), dim3(kBlock), 0, s,
                       (const T *)feats, order, starts, counts, c, n1, (T *)out);
  } else {
    hipLaunchKernelGGL((voxelize_forward_kernel<T, 1>), grid_for(n1 * c), dim3(kBlock), 0, s,
                       (const T *)feats, order, starts, counts, c, n1, (T *)out);
  }
  return check_launch("tsmi_voxelize_forward");
}

template <typename T>
int voxelize_backward_t(hipStream_t s, const void *top, const int32_t *idx, const int32_t *counts,
                        int64_t n, int c, int64_t n1, void *bottom) {
  if (vec_width<T>(c, {top, bottom}) > 1) {
    constexpr int V = 16 / (int)sizeof(T);
    hipLaunchKernelGGL((voxelize_backward_kernel<T, V>), grid_for(n * (c / V)), dim3(kBlock), 0, s,
                       (const T *)top, idx, counts, n, c, n1, (T *)bottom);
  } else {
    hipLaunchKernelGGL((voxelize_backward_kernel<T, 1>), grid_for(n * c), dim3(kBlock), 0, s,
                       (const T *)top, idx, counts, n, c, n1, (T *)bottom);
  }
  return check_launch("tsmi_voxelize_backward");
}

template <typename T>
int devoxelize_forward_t(hipStream_t s, const void *feat, const int32_t *indices, const float *weight,
                         int64_t n, int64_t n_vox, int c, void *out) {
  if (vec_width<T>(c, {feat, out}) > 1) {
    constexpr int V = 16 / (int)sizeof(T);
    hipLaunchKernelGGL((devoxelize_forward_kernel<T, V>), grid_for(n * (c / V)), dim3(kBlock), 0, s,
                       (const T *)feat, indices, weight, n, n_vox, c, (T *)out);
  } else {
    hipLaunchKernelGGL((devoxelize_forward_kernel<T, 1>), grid_for(n * c), dim3(kBlock), 0, s,
                       (const T *)feat, indices, weight, n, n_vox, c, (T *)out);
  }
  return check_launch("tsmi_devoxelize_forward");
}

template <typename T>
int devoxelize_backward_t(hipStream_t s, const void *top, const float *weight, const int32_t *order,
                          const int32_t *starts, int64_t n_vox, int c, void *bottom) {
  if (vec_width<T>(c, {top, bottom}) > 1) {
    constexpr int V = 16 / (int)sizeof(T);
    hipLaunchKernelGGL((devoxelize_backward_kernel<T, V>), grid_for(n_vox * (c / V)), dim3(kBlock), 0, s,
                       (const T *)top, weight, order, starts, n_vox, c, (T *)bottom);
  } else {
    hipLaunchKernelGGL((devoxelize_backward_kernel<T, 1>), grid_for(n_vox * c), dim3(kBlock), 0, s,
                       (const T *)top, weight, order, starts, n_vox, c, (T *)bottom);
  }
  return check_launch("tsmi_devoxelize_backward");
}

template <typename T, bool TO_DENSE>
int dense_copy_t(hipStream_t s, void *feats, const int32_t *coords, int64_t n, int c, const int *range,
                 void *dense) {
  Range4 rg{{range[0], range[1], range[2], range[3]}};
  if (vec_width<T>(c, {feats, dense}) > 1) {
    constexpr int V = 16 / (int)sizeof(T);
    hipLaunchKernelGGL((dense_copy_kernel<T, V, TO_DENSE>), grid_for(n * (c / V)), dim3(kBlock), 0, s,
                       (T *)feats, (const int4 *)coords, n, c, rg, (T *)dense);
  } else {
    hipLaunchKernelGGL((dense_copy_kernel<T, 1, TO_DENSE>), grid_for(n * c), dim3(kBlock), 0, s,
                       (T *)feats, (const int4 *)coords, n, c, rg, (T *)dense);
  }
  return check_launch("tsmi_to_dense");
}

}  // namespace

extern "C" int tsmi_voxelize_forward(tsmi_stream_t s, const void *feats, const int32_t *counts,
                                     const int32_t *order, const int32_t *starts, int64_t n, int c,
                                     int64_t n1, int dtype, void *out) {
  TSMI_REQUIRE(n >= 0 && n1 >= 0 && c >= 1, "voxelize_forward: bad sizes");
  if (n1 == 0) return TSMI_OK;
  TSMI_REQUIRE(out && counts && starts && (n == 0 || (feats && order)), "voxelize_forward: null pointer");
  TSMI_GRID_CHECK(n1 * c);
  TSMI_BY_DTYPE(dtype, return voxelize_forward_t<T>((hipStream_t)s, feats, counts, order, starts, c, n1,
                                                    out));
  return TSMI_OK;
}

extern "C" int tsmi_voxelize_backward(tsmi_stream_t s, const void *top_grad, const int32_t *idx,
                                      const int32_t *counts, int64_t n, int c, int64_t n1, int dtype,
                                      void *bottom_grad) {
  TSMI_REQUIRE(n >= 0 && n1 >= 0 && c >= 1, "voxelize_backward: bad sizes");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(bottom_grad && idx && (n1 == 0 || (top_grad && counts)), "voxelize_backward: null pointer");
  TSMI_GRID_CHECK(n * c);
  TSMI_BY_DTYPE(dtype, return voxelize_backward_t<T>((hipStream_t)s, top_grad, idx, counts, n, c, n1,
                                                     bottom_grad));
  return TSMI_OK;
}

extern "C" int tsmi_devoxelize_forward(tsmi_stream_t s, const void *feat, const int32_t *indices,
                                       const float *weight, int64_t n, int64_t n_vox, int c, int dtype,
                                       void *out) {
  TSMI_REQUIRE(n >= 0 && n_vox >= 0 && c >= 1, "devoxelize_forward: bad sizes");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(out && indices && weight && (n_vox == 0 || feat), "devoxelize_forward: null pointer");
  TSMI_REQUIRE(aligned16(indices) && aligned16(weight),
               "devoxelize_forward: indices and weight must be 16-byte aligned");
  TSMI_GRID_CHECK(n * c);
  TSMI_BY_DTYPE(dtype, return devoxelize_forward_t<T>((hipStream_t)s, feat, indices, weight, n, n_vox, c,
                                                      out));
  return TSMI_OK;
}

extern "C" int tsmi_devoxelize_backward(tsmi_stream_t s, const void *top_grad, const float *weight,
                                        const int32_t *order, const int32_t *starts, int64_t n,
                                        int64_t n_vox, int c, int dtype, void *bottom_grad) {
  TSMI_REQUIRE(n >= 0 && n_vox >= 0 && c >= 1, "devoxelize_backward: bad sizes");
  if (n_vox == 0) return TSMI_OK;
  TSMI_REQUIRE(bottom_grad && starts && (n == 0 || (top_grad && weight && order)),
               "devoxelize_backward: null pointer");
  TSMI_GRID_CHECK(n_vox * c);
  TSMI_BY_DTYPE(dtype, return devoxelize_backward_t<T>((hipStream_t)s, top_grad, weight, order, starts,
                                                       n_vox, c, bottom_grad));
  return TSMI_OK;
}

extern "C" int tsmi_to_dense_forward(tsmi_stream_t s, const void *feats, const int32_t *coords,
                                     int64_t n, int c, const int32_t *spatial_range, int dtype,
                                     void *dense) {
  TSMI_REQUIRE(n >= 0 && c >= 1 && spatial_range, "to_dense_forward: bad arguments");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(feats && coords && dense && aligned16(coords), "to_dense_forward: null or misaligned pointer");
  TSMI_GRID_CHECK(n * c);
  TSMI_BY_DTYPE(dtype, return (dense_copy_t<T, true>((hipStream_t)s, (void *)feats, coords, n, c,
                                                     spatial_range, dense)));
  return TSMI_OK;
}

extern "C" int tsmi_to_dense_backward(tsmi_stream_t s, const void *top_grad, const int32_t *coords,
                                      int64_t n, int c, const int32_t *spatial_range, int dtype,
                                      void *bottom_grad) {
  TSMI_REQUIRE(n >= 0 && c >= 1 && spatial_range, "to_dense_backward: bad arguments");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(top_grad && coords && bottom_grad && aligned16(coords),
               "to_dense_backward: null or misaligned pointer");
  TSMI_GRID_CHECK(n * c);
  TSMI_BY_DTYPE(dtype, return (dense_copy_t<T, false>((hipStream_t)s, bottom_grad, coords, n, c,
                                                      spatial_range, (void *)top_grad)));
  return TSMI_OK;
}

extern "C" int tsmi_pad_columns(tsmi_stream_t s, const void *x, int64_t n, int c, int dtype, void *y) {
  TSMI_REQUIRE(n >= 0 && c >= 1, "pad_columns: bad arguments");
  if (n == 0) return TSMI_OK;
  TSMI_REQUIRE(x && y && aligned16(y), "pad_columns: null or misaligned pointer");
  const int per = dtype == TSMI_F32 ? 4 : 8, pieces = (c + per - 1) / per;
  TSMI_GRID_CHECK(n * pieces);
  const dim3 grid((unsigned)ceil_div(n * pieces, 256));
  if (dtype == TSMI_F32)
    hipLaunchKernelGGL(pad_columns_kernel<uint32_t>, grid, dim3(256), 0, (hipStream_t)s, (const uint32_t *)x, n, c,
                       pieces, (uint4 *)y);
  else  // (bits are moved, whatever the 16-bit type)
    hipLaunchKernelGGL(pad_columns_kernel<uint16_t>, grid, dim3(256), 0, (hipStream_t)s, (const uint16_t *)x, n, c,
                       pieces, (uint4 *)y);
  return check_launch("pad_columns_kernel");
}
