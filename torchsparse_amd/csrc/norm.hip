// Batch normalisation of a row-major feature matrix [N, C] in training mode for gfx950:
// per-channel statistics over the N rows, the normalised output, and the backward.
//
// What follows the normalisation in a network runs with it: the output is
// y = act((x - mean) * scale + bias + residual), and the backward takes the gradient through the
// activation on its way into the sums (and hands it on to the residual).
//
// Every pass is HBM-bound: a thread owns one 16-byte piece of a row (8 half / bf16 or 4 float
// channels), neighbouring lanes read neighbouring addresses, and column sums are kept in fp32
// registers while a block strides over its rows.  Blocks leave their partial sums in a
// [blocks, 2, C] fp32 array; the last block of every group of 16 to arrive adds its group's, and the
// last group to arrive adds the groups', both in a fixed order: no floating-point atomics, the same bits
// on every run.  (A second launch over 256 partial sums took 7.7 us behind reductions of 4 to 6; one
// block that adds all 256 by itself reads for longer than that.)  Matrices of at most 4096 rows take one launch
// (bn_small_kernel).  The variance comes from sums of (x - x[0, c]) and its square: the
// shift by the column's first row keeps E[d^2] - E[d]^2 away from cancellation when a column's
// mean is large next to its spread.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <initializer_list>

#include "common.h"

namespace tsmi {
namespace {

constexpr int kBlock = 256;
constexpr int kGroup = 16;                   // partial sums one block adds
constexpr int kMaxBlocks = kGroup * kGroup;  // partial sums per column

template <typename T>
struct Vec;
template <>
struct Vec<float> {
  static constexpr int V = 4;
};
template <>
struct Vec<_Float16> {
  static constexpr int V = 8;
};
template <>
struct Vec<__bf16> {
  static constexpr int V = 8;
};

template <typename T, int V>
struct alignas(sizeof(T) * V) Pack {
  T v[V];
};

template <typename T, int V>
__device__ __forceinline__ void load_piece(const T *p, float *out) {
  const Pack<T, V> q = *(const Pack<T, V> *)p;
#pragma unroll
  for (int e = 0; e < V; ++e) out[e] = (float)q.v[e];
}

template <typename T, int V>
__device__ __forceinline__ void store_piece(T *p, const float *in) {
  Pack<T, V> q;
#pragma unroll
  for (int e = 0; e < V; ++e) q.v[e] = (T)in[e];
  *(Pack<T, V> *)p = q;
}

// Parameters and running statistics come in the module's own type.
__device__ __forceinline__ float load_param(const void *p, int i, int code, float missing) {
  if (!p) return missing;
  if (code == TSMI_F32) return ((const float *)p)[i];
  if (code == TSMI_F16) return (float)((const _Float16 *)p)[i];
  return (float)((const __bf16 *)p)[i];
}

__device__ __forceinline__ void store_param(void *p, int i, int code, float v) {
  if (code == TSMI_F32)
    ((float *)p)[i] = v;
  else if (code == TSMI_F16)
    ((_Float16 *)p)[i] = (_Float16)v;
  else
    ((__bf16 *)p)[i] = (__bf16)v;
}

// What one call works on.  Forward: stats [4 C] receives mean, 1/sqrt(var + eps), scale = weight / std,
// bias.  Backward: stats as the forward left them, sums [5 C] = sum g, sum g * xhat and the constants of the
// element-wise pass dx = g * sums[2C:] + (x - mean) * sums[3C:] + sums[4C:], where g is dy taken through
// the activation.
template <typename T>
struct Bn {
  const T *x, *dy;
  const T *y_saved;   // backward of a layer with an activation and a residual: its output
  const T *residual;  // forward
  T *out, *dz;        // y or dx; the gradient of the residual (null: not wanted)
  int64_t n;
  int c, relu;
  float *partial;
  int32_t *counters;  // zero, and left zero: one per group of blocks and one for the groups
  float *stats, *sums;
  const void *weight, *bias;
  void *running_mean, *running_var, *grads;
  int64_t *batches;   // counter of the batches seen, or null
  int param_code;
  float momentum, eps;
};

enum Mask { kNoMask, kMaskX, kMaskY };  // the activation's sign: none, from x again, from the saved output

// The gradient of one piece behind the activation.
template <typename T, int V, Mask kMask>
__device__ __forceinline__ void masked_grad(const Bn<T> &p, int64_t at, const float *xv, const float *mean,
                                            const float *scale, const float *bias, float *g) {
  load_piece<T, V>(p.dy + at, g);
  if (kMask == kMaskX) {
#pragma unroll
    for (int e = 0; e < V; ++e)  // (what the forward stored, rounded as it was stored)
      if (!((float)(T)((xv[e] - mean[e]) * scale[e] + bias[e]) > 0.f)) g[e] = 0.f;
  } else if (kMask == kMaskY) {
    float yv[V];
    load_piece<T, V>(p.y_saved + at, yv);
#pragma unroll
    for (int e = 0; e < V; ++e)
      if (!(yv[e] > 0.f)) g[e] = 0.f;
  }
}

// Everything derived from a column's two sums.
template <typename T, bool kBackward>
__device__ __forceinline__ void finish_column(const Bn<T> &p, int col, float t1, float t2) {
  const float inv_n = 1.f / (float)p.n;
  const int c = p.c;
  const float w = load_param(p.weight, col, p.param_code, 1.f);
  if (kBackward) {
    const float invstd = p.stats[c + col];
    const float s = w * invstd;
    p.sums[col] = t1;
    p.sums[c + col] = t2;
    p.sums[2 * c + col] = s;
    p.sums[3 * c + col] = -s * t2 * invstd * inv_n;
    p.sums[4 * c + col] = -s * t1 * inv_n;
    if (p.grads) {  // the two gradients once more, in the parameters' type
      store_param(p.grads, col, p.param_code, t1);
      store_param(p.grads, c + col, p.param_code, t2);
    }
    return;
  }
  const float shift = t1 * inv_n;
  const float mean = (float)p.x[col] + shift;
  const float var = fmaxf(t2 * inv_n - shift * shift, 0.f);  // biased, as used for normalising
  const float invstd = rsqrtf(var + p.eps);
  p.stats[col] = mean;
  p.stats[c + col] = invstd;
  p.stats[2 * c + col] = invstd * w;
  p.stats[3 * c + col] = load_param(p.bias, col, p.param_code, 0.f);
  if (p.running_mean) {
    const float rm = load_param(p.running_mean, col, p.param_code, 0.f);
    store_param(p.running_mean, col, p.param_code, (1.f - p.momentum) * rm + p.momentum * mean);
  }
  if (p.running_var) {
    const float unbiased = p.n > 1 ? var * ((float)p.n / (float)(p.n - 1)) : var;
    const float rv = load_param(p.running_var, col, p.param_code, 1.f);
    store_param(p.running_var, col, p.param_code, (1.f - p.momentum) * rv + p.momentum * unbiased);
  }
  if (col == 0 && p.batches) *p.batches += 1;
}

// Partial sums cross XCDs (an L2 each): device-scope stores and loads, ordered by waiting for the stores
// before the ticket.
__device__ __forceinline__ void share(float *p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float shared_value(const float *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// True, to every thread, in the block that takes the last of `parts` tickets; the counter is zero again.
__device__ __forceinline__ bool last_to_arrive(int32_t *counter, int parts) {
  __shared__ int last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (this thread's sums have landed)
  __syncthreads();
  if (threadIdx.x == 0) {
    const int old = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = old == parts - 1;
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  const bool mine = last != 0;
  __syncthreads();
  return mine;
}

// Column sums over the block's rows - forward: sum (x - k) and sum (x - k)^2 with k = x[0, c]; backward: sum g
// and sum g * xhat, xhat = (x - mean) * invstd - and, in the last block, everything that follows from them.
// Threads: piece q = tid % (C / V) of row tid / (C / V); 256 / (C / V) rows per sweep.
template <typename T, int V, bool kBackward, Mask kMask>
__global__ __launch_bounds__(kBlock) void bn_reduce_kernel(Bn<T> p) {
  extern __shared__ float red[];  // [rows per sweep][2 * C]
  const int c = p.c, cg = c / V;
  const int rows = kBlock / cg;
  const int r = threadIdx.x / cg, q = threadIdx.x - r * cg;
  if (r < rows) {
    float a1[V], a2[V], k[V], inv[V], scale[V], bias[V];
#pragma unroll
    for (int e = 0; e < V; ++e) a1[e] = a2[e] = k[e] = inv[e] = scale[e] = bias[e] = 0.f;
    if (kBackward) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        k[e] = p.stats[q * V + e];
        inv[e] = p.stats[c + q * V + e];
        if (kMask == kMaskX) {
          scale[e] = p.stats[2 * c + q * V + e];
          bias[e] = p.stats[3 * c + q * V + e];
        }
      }
    } else {
      load_piece<T, V>(p.x + q * V, k);
    }
#pragma unroll 2
    for (int64_t row = (int64_t)blockIdx.x * rows + r; row < p.n; row += (int64_t)gridDim.x * rows) {
      float xv[V];
      const int64_t at = row * c + q * V;
      load_piece<T, V>(p.x + at, xv);
      if (kBackward) {
        float g[V];
        masked_grad<T, V, kMask>(p, at, xv, k, scale, bias, g);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          a1[e] += g[e];
          a2[e] += g[e] * ((xv[e] - k[e]) * inv[e]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const float d = xv[e] - k[e];
          a1[e] += d;
          a2[e] += d * d;
        }
      }
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
      red[r * 2 * c + q * V + e] = a1[e];
      red[r * 2 * c + c + q * V + e] = a2[e];
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < 2 * c; t += kBlock) {
    float s = 0.f;
    for (int i = 0; i < rows; ++i) s += red[i * 2 * c + t];
    share(p.partial + (int64_t)blockIdx.x * 2 * c + t, s);
  }
  const int groups = (gridDim.x + kGroup - 1) / kGroup, group = blockIdx.x / kGroup;
  const int first = group * kGroup, members = min(kGroup, (int)gridDim.x - first);
  if (!last_to_arrive(p.counters + group, members)) return;
  float *group_sums = p.partial + (int64_t)kMaxBlocks * 2 * c;  // [groups][2 * C]
  for (int t = threadIdx.x; t < 2 * c; t += kBlock) {
    float v[kGroup];
#pragma unroll
    for (int i = 0; i < kGroup; ++i)
      v[i] = i < members ? shared_value(p.partial + (int64_t)(first + i) * 2 * c + t) : 0.f;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kGroup; ++i) s += v[i];
    share(group_sums + (int64_t)group * 2 * c + t, s);
  }
  if (!last_to_arrive(p.counters + kGroup, groups)) return;
  for (int t = threadIdx.x; t < 2 * c; t += kBlock) {
    float v[kGroup];
#pragma unroll
    for (int i = 0; i < kGroup; ++i) v[i] = i < groups ? shared_value(group_sums + (int64_t)i * 2 * c + t) : 0.f;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kGroup; ++i) s += v[i];
    red[t] = s;
  }
  __syncthreads();
  for (int col = threadIdx.x; col < c; col += kBlock) finish_column<T, kBackward>(p, col, red[col], red[c + col]);
}

// The element-wise pass (the mean is subtracted before scaling, as torch does: x * scale + (bias - mean * scale)
// would lose the small difference of two large terms when a column's mean is large).  Thread layout as in the
// reduction; the column constants are read once per thread and serve kSweeps rows.
constexpr int kSweeps = 8;

template <typename T, int V, bool kBackward, Mask kMask>
__global__ __launch_bounds__(kBlock) void bn_apply_kernel(Bn<T> p) {
  const int c = p.c, cg = c / V;
  const int rows = kBlock / cg;
  const int r = threadIdx.x / cg, q = threadIdx.x - r * cg;
  if (r >= rows) return;
  float mean[V], ka[V], kb[V], kc[V], scale[V], bias[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    mean[e] = p.stats[q * V + e];
    scale[e] = !kBackward || kMask == kMaskX ? p.stats[2 * c + q * V + e] : 0.f;
    bias[e] = !kBackward || kMask == kMaskX ? p.stats[3 * c + q * V + e] : 0.f;
    ka[e] = kBackward ? p.sums[2 * c + q * V + e] : 0.f;
    kb[e] = kBackward ? p.sums[3 * c + q * V + e] : 0.f;
    kc[e] = kBackward ? p.sums[4 * c + q * V + e] : 0.f;
  }
  const int64_t row0 = (int64_t)blockIdx.x * rows * kSweeps + r;
#pragma unroll
  for (int sweep = 0; sweep < kSweeps; ++sweep) {
    const int64_t row = row0 + (int64_t)sweep * rows;
    if (row >= p.n) break;
    const int64_t at = row * c + q * V;
    float xv[V], g[V];
    load_piece<T, V>(p.x + at, xv);
    if (kBackward) {
      masked_grad<T, V, kMask>(p, at, xv, mean, scale, bias, g);
      if (p.dz) store_piece<T, V>(p.dz + at, g);
#pragma unroll
      for (int e = 0; e < V; ++e) g[e] = g[e] * ka[e] + (xv[e] - mean[e]) * kb[e] + kc[e];
    } else {
      float res[V];
      if (p.residual) load_piece<T, V>(p.residual + at, res);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        g[e] = (xv[e] - mean[e]) * scale[e] + bias[e];
        if (p.residual) g[e] += res[e];
        if (p.relu) g[e] = fmaxf(g[e], 0.f);
      }
    }
    store_piece<T, V>(p.out + at, g);
  }
}

// The whole call for a matrix of at most kSmallRows rows, in one launch: a block of 1024 threads owns one
// 16-byte piece of every row, keeps its rows in registers between the sums and the element-wise pass.  Its
// loads take 16 bytes of a row each, a quarter of what the caches move, which is why more rows go the other
// way; a few thousand rows are bound by launches, one here and two there.
constexpr int kSmallThreads = 1024, kSmallKeep = 4;
constexpr int kSmallRows = kSmallThreads * kSmallKeep;

template <typename T, int V, bool kBackward, Mask kMask>
__global__ __launch_bounds__(kSmallThreads) void bn_small_kernel(Bn<T> p) {
  __shared__ float red[kSmallThreads / 64][2 * V];
  __shared__ float total[2 * V];
  const int c = p.c, q = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float xv[kSmallKeep][V], g[kSmallKeep][V], k[V], inv[V], scale[V], bias[V], a[2 * V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    k[e] = inv[e] = scale[e] = bias[e] = a[e] = a[V + e] = 0.f;
    if (kBackward) {
      k[e] = p.stats[q * V + e];
      inv[e] = p.stats[c + q * V + e];
      if (kMask == kMaskX) {
        scale[e] = p.stats[2 * c + q * V + e];
        bias[e] = p.stats[3 * c + q * V + e];
      }
    }
  }
  if (!kBackward) load_piece<T, V>(p.x + q * V, k);
#pragma unroll
  for (int i = 0; i < kSmallKeep; ++i) {
    const int64_t row = threadIdx.x + i * kSmallThreads;
    if (row >= p.n) break;
    load_piece<T, V>(p.x + row * c + q * V, xv[i]);
  }
#pragma unroll
  for (int i = 0; i < kSmallKeep; ++i) {
    const int64_t row = threadIdx.x + i * kSmallThreads;
    if (row >= p.n) break;
    if (kBackward) masked_grad<T, V, kMask>(p, row * c + q * V, xv[i], k, scale, bias, g[i]);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float d = xv[i][e] - k[e];
      a[e] += kBackward ? g[i][e] : d;
      a[V + e] += kBackward ? g[i][e] * (d * inv[e]) : d * d;
    }
  }
#pragma unroll
  for (int e = 0; e < 2 * V; ++e) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) a[e] += __shfl_xor(a[e], d);
    if (lane == 0) red[wave][e] = a[e];
  }
  __syncthreads();
  if (threadIdx.x < 2 * V) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kSmallThreads / 64; ++w) s += red[w][threadIdx.x];
    total[threadIdx.x] = s;
  }
  __syncthreads();
  if (threadIdx.x < V) finish_column<T, kBackward>(p, q * V + threadIdx.x, total[threadIdx.x], total[V + threadIdx.x]);
  __threadfence_block();
  __syncthreads();
  float ka[V], kb[V], kc[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    if (kBackward) {
      ka[e] = p.sums[2 * c + q * V + e];
      kb[e] = p.sums[3 * c + q * V + e];
      kc[e] = p.sums[4 * c + q * V + e];
    } else {
      k[e] = p.stats[q * V + e];
      scale[e] = p.stats[2 * c + q * V + e];
      bias[e] = p.stats[3 * c + q * V + e];
    }
  }
#pragma unroll
  for (int i = 0; i < kSmallKeep; ++i) {
    const int64_t row = threadIdx.x + i * kSmallThreads;
    if (row >= p.n) break;
    const int64_t at = row * c + q * V;
    float res[V], o[V];
    if (!kBackward && p.residual) load_piece<T, V>(p.residual + at, res);
    if (kBackward && p.dz) store_piece<T, V>(p.dz + at, g[i]);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      if (kBackward) {
        o[e] = g[i][e] * ka[e] + (xv[i][e] - k[e]) * kb[e] + kc[e];
      } else {
        o[e] = (xv[i][e] - k[e]) * scale[e] + bias[e];
        if (p.residual) o[e] += res[e];
        if (p.relu) o[e] = fmaxf(o[e], 0.f);
      }
    }
    store_piece<T, V>(p.out + at, o);
  }
}

int check_shape(const char *what, int64_t n, int c, int dtype, int param_dtype, int *v) {
  TSMI_REQUIRE(dtype == TSMI_F32 || dtype == TSMI_F16 || dtype == TSMI_BF16, "%s: bad dtype %d", what, dtype);
  TSMI_REQUIRE(param_dtype == TSMI_F32 || param_dtype == TSMI_F16 || param_dtype == TSMI_BF16,
               "%s: bad parameter dtype %d", what, param_dtype);
  *v = dtype == TSMI_F32 ? 4 : 8;
  TSMI_REQUIRE(n >= 1, "%s: needs at least one row", what);
  TSMI_REQUIRE(c >= *v && c % *v == 0 && c / *v <= kBlock,
               "%s: the channel count must be a multiple of %d and at most %d (got %d)", what, *v,
               *v * kBlock, c);
  TSMI_REQUIRE(grid_fits(ceil_div(n * (c / *v), kBlock)), "%s: problem too large for one launch", what);
  return TSMI_OK;
}

int reduce_blocks(int64_t n, int c, int v) {
  const int rows = kBlock / (c / v);
  const int64_t b = ceil_div(n, rows);
  return (int)(b < kMaxBlocks ? b : kMaxBlocks);
}

template <typename T, bool kBackward, Mask kMask>
int launch(hipStream_t s, const Bn<T> &p) {
  constexpr int V = Vec<T>::V;
  if (p.n <= kSmallRows) {
    hipLaunchKernelGGL((bn_small_kernel<T, V, kBackward, kMask>), dim3(p.c / V), dim3(kSmallThreads), 0, s, p);
    return check_launch("bn_small_kernel");
  }
  const int rows = kBlock / (p.c / V);
  const size_t lds = (size_t)rows * 2 * p.c * sizeof(float);
  hipLaunchKernelGGL((bn_reduce_kernel<T, V, kBackward, kMask>), dim3(reduce_blocks(p.n, p.c, V)), dim3(kBlock), lds,
                     s, p);
  hipLaunchKernelGGL((bn_apply_kernel<T, V, kBackward, kMask>),
                     dim3((unsigned)ceil_div(p.n, (int64_t)rows * kSweeps)), dim3(kBlock), 0, s, p);
  return check_launch("bn_apply_kernel");
}

template <typename T>
Bn<T> bn_of(const void *x, int64_t n, int c, int relu, float *partial, int32_t *counters, float *stats,
            const void *weight, int param_dtype) {
  Bn<T> p{};
  p.x = (const T *)x;
  p.n = n;
  p.c = c;
  p.relu = relu;
  p.partial = partial;
  p.counters = counters;
  p.stats = stats;
  p.weight = weight;
  p.param_code = param_dtype;
  return p;
}

inline bool aligned(std::initializer_list<const void *> ptrs) {
  for (const void *p : ptrs)
    if ((uintptr_t)p % 16 != 0) return false;
  return true;
}

}  // namespace
}  // namespace tsmi

using namespace tsmi;

extern "C" int64_t tsmi_bn_partial_elems(int c) { return (int64_t)(kMaxBlocks + kGroup) * 2 * (c > 0 ? c : 0); }

#define TSMI_BN_BY_DTYPE(...)                           \
  do {                                                  \
    if (dtype == TSMI_F32) {                            \
      using T = float;                                  \
      __VA_ARGS__;                                      \
    } else if (dtype == TSMI_F16) {                     \
      using T = _Float16;                               \
      __VA_ARGS__;                                      \
    } else {                                            \
      using T = __bf16;                                 \
      __VA_ARGS__;                                      \
    }                                                   \
  } while (0)

extern "C" int tsmi_bn_forward_train(tsmi_stream_t s, const void *x, int64_t n, int c, int dtype,
                                     const void *weight, const void *bias, int param_dtype,
                                     void *running_mean, void *running_var, int64_t *batches, float momentum,
                                     float eps, const void *residual, int relu, float *partial, int32_t *counters,
                                     float *stats, void *y) {
  int v;
  if (int e = check_shape("bn_forward_train", n, c, dtype, param_dtype, &v)) return e;
  TSMI_REQUIRE(x && y && partial && counters && stats, "bn_forward_train: null pointer");
  TSMI_REQUIRE(aligned({x, y, residual}), "bn_forward_train: x, residual and y must be 16-byte aligned");
  TSMI_BN_BY_DTYPE({
    Bn<T> p = bn_of<T>(x, n, c, relu, partial, counters, stats, weight, param_dtype);
    p.bias = bias;
    p.running_mean = running_mean;
    p.running_var = running_var;
    p.batches = batches;
    p.momentum = momentum;
    p.eps = eps;
    p.residual = (const T *)residual;
    p.out = (T *)y;
    return launch<T, false, kNoMask>((hipStream_t)s, p);
  });
}

extern "C" int tsmi_bn_backward(tsmi_stream_t s, const void *dy, const void *x, const void *y, int64_t n, int c,
                                int dtype, int relu, const void *weight, int param_dtype, float *stats,
                                float *partial, int32_t *counters, float *sums, void *grads, void *dz,
                                void *dx) {
  int v;
  if (int e = check_shape("bn_backward", n, c, dtype, param_dtype, &v)) return e;
  TSMI_REQUIRE(dy && x && dx && partial && counters && stats && sums, "bn_backward: null pointer");
  TSMI_REQUIRE(aligned({dy, x, y, dz, dx}), "bn_backward: dy, x, y, dz and dx must be 16-byte aligned");
  TSMI_BN_BY_DTYPE({
    Bn<T> p = bn_of<T>(x, n, c, relu, partial, counters, stats, weight, param_dtype);
    p.dy = (const T *)dy;
    p.y_saved = (const T *)y;
    p.sums = sums;
    p.grads = grads;
    p.dz = (T *)dz;
    p.out = (T *)dx;
    if (!relu) return launch<T, true, kNoMask>((hipStream_t)s, p);
    if (y) return launch<T, true, kMaskY>((hipStream_t)s, p);
    return launch<T, true, kMaskX>((hipStream_t)s, p);
  });
}
