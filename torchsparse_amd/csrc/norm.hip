// Batch normalisation of a row-major feature matrix [N, C] in training mode for gfx950:
// per-channel statistics over the N rows, the normalised output, and the backward.
//
// What follows the normalisation in a network runs with it: the output is
// y = act((x - mean) * scale + bias + residual), and the backward takes the gradient through the
// activation on its way into the sums (and hands it on to the residual).
//
// Every pass is HBM-bound: a thread owns one 16-byte piece of a row (8 half / bf16 or 4 float
// channels), neighbouring lanes read neighbouring addresses, and column sums are kept in fp32
// registers while a block strides over its rows, with the loads of several rows in flight.  Blocks leave their
// partial sums in a [blocks, 2, C] fp32 array, which every block of the element-wise pass adds for itself
// before it starts, in a fixed order: no floating-point atomics, the same bits on every run.  (The sums of
// 80k x 96 half values took 13 us where the last blocks of a reduction to arrive added them up: what one block
// hands to another goes through memory, twice 4 us.  A launch between the two took 8 us.)  Matrices of at most
// 1024 rows take one launch (bn_small_kernel).  The variance comes from sums of (x - x[0, c]) and its square:
// the shift by the column's first row keeps E[d^2] - E[d]^2 away from cancellation when a column's
// mean is large next to its spread.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <initializer_list>

#include "common.h"

namespace tsmi {
namespace {

constexpr int kBlock = 512;
constexpr int kMaxPieces = 256;  // 16-byte pieces of a row
// Blocks of the reduction: enough to have the loads in flight that reading at full rate takes (128 x 512
// threads x 8 x 16 bytes), few enough that all of the next pass's blocks can read their sums.
constexpr int kMaxBlocks = 128;
constexpr int kApplyBlocks = 512;

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
__device__ __forceinline__ void unpack(const Pack<T, V> &q, float *out) {
#pragma unroll
  for (int e = 0; e < V; ++e) out[e] = (float)q.v[e];
}

template <typename T, int V>
__device__ __forceinline__ void load_piece(const T *p, float *out) {
  unpack<T, V>(*(const Pack<T, V> *)p, out);
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
// bias.  Backward: stats as the forward left them, sums [2 C] = sum g, sum g * xhat, where g is dy taken through
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
  int parts;  // blocks that left partial sums
  float *stats, *sums;
  const void *weight, *bias;
  void *running_mean, *running_var, *grads;
  int64_t *batches;   // counter of the batches seen, or null
  int param_code;
  float momentum, eps;
};

enum Mask { kNoMask, kMaskX, kMaskY };  // the activation's sign: none, from x again, from the saved output

// One piece of what the sums run over, loaded (to be used later) and converted.
template <typename T, int V, bool kBackward, Mask kMask>
struct Piece {
  Pack<T, V> x, g, y;
  __device__ __forceinline__ void load(const Bn<T> &p, int64_t at) {
    x = *(const Pack<T, V> *)(p.x + at);
    if (kBackward) g = *(const Pack<T, V> *)(p.dy + at);
    if (kBackward && kMask == kMaskY) y = *(const Pack<T, V> *)(p.y_saved + at);
  }
  // the gradient behind the activation
  __device__ __forceinline__ void grad(const float *xv, const float *mean, const float *scale, const float *bias,
                                       float *out) const {
    unpack<T, V>(g, out);
    if (kMask == kMaskX) {
#pragma unroll
      for (int e = 0; e < V; ++e)  // (what the forward stored, rounded as it was stored)
        if (!((float)(T)((xv[e] - mean[e]) * scale[e] + bias[e]) > 0.f)) out[e] = 0.f;
    } else if (kMask == kMaskY) {
#pragma unroll
      for (int e = 0; e < V; ++e)
        if (!((float)y.v[e] > 0.f)) out[e] = 0.f;
    }
  }
};

// What a column's results take besides its sums (loaded apart: early where there is something to wait for).
struct ColumnIn {
  float weight, bias, first, running_mean, running_var, invstd;
};
template <typename T, bool kBackward>
__device__ __forceinline__ ColumnIn load_column(const Bn<T> &p, int col) {
  ColumnIn in{};
  in.weight = load_param(p.weight, col, p.param_code, 1.f);
  if (kBackward) {
    in.invstd = p.stats[p.c + col];
  } else {
    in.first = (float)p.x[col];
    in.bias = load_param(p.bias, col, p.param_code, 0.f);
    in.running_mean = load_param(p.running_mean, col, p.param_code, 0.f);
    in.running_var = load_param(p.running_var, col, p.param_code, 1.f);
  }
  return in;
}

// Everything derived from a column's two sums.  Returns the constants of the element-wise pass: mean, scale, bias
// (forward) or the factors of g and x - mean and the addend (backward).
struct ColumnOut {
  float a, b, c;
};
// One block of a launch leaves the results (`keep`).
template <typename T, bool kBackward>
__device__ __forceinline__ ColumnOut finish_column(const Bn<T> &p, int col, const ColumnIn &in, float t1, float t2,
                                                   bool keep) {
  const float inv_n = 1.f / (float)p.n;
  const int c = p.c;
  const float w = in.weight;
  if (kBackward) {
    const float invstd = in.invstd;
    const float s = w * invstd;
    const ColumnOut out{s, -s * t2 * invstd * inv_n, -s * t1 * inv_n};
    if (!keep) return out;
    p.sums[col] = t1;
    p.sums[c + col] = t2;
    if (p.grads) {  // the two gradients once more, in the parameters' type
      store_param(p.grads, col, p.param_code, t1);
      store_param(p.grads, c + col, p.param_code, t2);
    }
    return out;
  }
  const float shift = t1 * inv_n;
  const float mean = in.first + shift;
  const float var = fmaxf(t2 * inv_n - shift * shift, 0.f);  // biased, as used for normalising
  const float invstd = rsqrtf(var + p.eps);
  const ColumnOut out{mean, invstd * w, in.bias};
  if (!keep) return out;
  p.stats[col] = mean;
  p.stats[c + col] = invstd;
  p.stats[2 * c + col] = out.b;
  p.stats[3 * c + col] = out.c;
  if (p.running_mean)
    store_param(p.running_mean, col, p.param_code, (1.f - p.momentum) * in.running_mean + p.momentum * mean);
  if (p.running_var) {
    const float unbiased = p.n > 1 ? var * ((float)p.n / (float)(p.n - 1)) : var;
    store_param(p.running_var, col, p.param_code, (1.f - p.momentum) * in.running_var + p.momentum * unbiased);
  }
  if (col == 0 && p.batches) *p.batches += 1;
  return out;
}

// Column sums over the block's rows - forward: sum (x - k) and sum (x - k)^2 with k = x[0, c]; backward: sum g
// and sum g * xhat, xhat = (x - mean) * invstd.
// Threads: piece q = tid % (C / V) of row tid / (C / V); kBlock / (C / V) rows per sweep.
template <typename T, int V, bool kBackward, Mask kMask>
__global__ __launch_bounds__(kBlock) void bn_reduce_kernel(Bn<T> p) {
  extern __shared__ float red[];  // [rows per sweep][2 * C]
  constexpr int kFlight = kBackward ? 4 : 8;  // rows whose loads a thread has in flight
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
    const int64_t step = (int64_t)gridDim.x * rows;
    for (int64_t row = (int64_t)blockIdx.x * rows + r; row < p.n; row += kFlight * step) {
      Piece<T, V, kBackward, kMask> piece[kFlight];
#pragma unroll
      for (int u = 0; u < kFlight; ++u)
        piece[u].load(p, min(row + u * step, p.n - 1) * c + q * V);
#pragma unroll
      for (int u = 0; u < kFlight; ++u) {
        if (row + u * step >= p.n) break;
        float xv[V];
        unpack<T, V>(piece[u].x, xv);
        if (kBackward) {
          float g[V];
          piece[u].grad(xv, k, scale, bias, g);
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
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
      red[r * 2 * c + q * V + e] = a1[e];
      red[r * 2 * c + c + q * V + e] = a2[e];
    }
  }
  __syncthreads();
  // The rows' sums of a column: kBlock / (2 C) threads take every so-many-th row each and leave their sum in the
  // place of their first one, which nobody else reads.
  const int parts = max(1, min(rows, kBlock / (2 * c)));
  for (int t = threadIdx.x; t < parts * 2 * c; t += kBlock) {
    float s = 0.f;
#pragma unroll 8
    for (int i = t / (2 * c); i < rows; i += parts) s += red[i * 2 * c + t % (2 * c)];
    red[t] = s;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < 2 * c; t += kBlock) {
    float s = red[t];
    for (int i = 1; i < parts; ++i) s += red[i * 2 * c + t];
    p.partial[(int64_t)blockIdx.x * 2 * c + t] = s;
  }
}

// The element-wise pass (the mean is subtracted before scaling, as torch does: x * scale + (bias - mean * scale)
// would lose the small difference of two large terms when a column's mean is large).  Thread layout as in the
// reduction; kSweeps rows' loads in flight, the first ones while the block adds up the partial sums.
constexpr int kSweeps = 4;

template <typename T, int V, bool kBackward, Mask kMask>
__global__ __launch_bounds__(kBlock) void bn_apply_kernel(Bn<T> p) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  extern __shared__ float sh[];  // sums: [parts][2 C], made: [3][C]
  const int c = p.c, cg = c / V;
  const int rows = kBlock / cg;
  const int r = threadIdx.x / cg, q = threadIdx.x - r * cg;
  const int64_t first = (int64_t)blockIdx.x * rows * kSweeps + min(r, rows - 1);
  Piece<T, V, kBackward, kMask> piece[kSweeps];
#pragma unroll
  for (int u = 0; u < kSweeps; ++u) piece[u].load(p, min(first + (int64_t)u * rows, p.n - 1) * c + q * V);

  const int quads = c / 2, parts = max(1, kBlock / quads);
  float *made = sh + parts * 2 * c;
  ColumnIn in{};
  if (threadIdx.x < c) in = load_column<T, kBackward>(p, threadIdx.x);
  for (int t = threadIdx.x; t < parts * quads; t += kBlock) {
    const int part = t / quads, quad = t - part * quads;
    f4 sum = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int i = part; i < p.parts; i += parts) sum += *(const f4 *)(p.partial + (int64_t)i * 2 * c + quad * 4);
    *(f4 *)(sh + part * 2 * c + quad * 4) = sum;
  }
  __syncthreads();
  for (int col = threadIdx.x; col < c; col += kBlock) {
    float t1 = 0.f, t2 = 0.f;
    for (int i = 0; i < parts; ++i) {
      t1 += sh[i * 2 * c + col];
      t2 += sh[i * 2 * c + c + col];
    }
    if (col >= kBlock) in = load_column<T, kBackward>(p, col);
    const ColumnOut out = finish_column<T, kBackward>(p, col, in, t1, t2, blockIdx.x == 0);
    made[col] = out.a;
    made[c + col] = out.b;
    made[2 * c + col] = out.c;
  }
  __syncthreads();
  if (r >= rows) return;
  float ka[V], kb[V], kc[V], mean[V], scale[V], bias[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    ka[e] = made[q * V + e];
    kb[e] = made[c + q * V + e];
    kc[e] = made[2 * c + q * V + e];
    mean[e] = kBackward ? p.stats[q * V + e] : 0.f;
    scale[e] = kBackward && kMask == kMaskX ? p.stats[2 * c + q * V + e] : 0.f;
    bias[e] = kBackward && kMask == kMaskX ? p.stats[3 * c + q * V + e] : 0.f;
  }
  const int64_t step = (int64_t)gridDim.x * rows * kSweeps;
  for (int64_t row0 = first; row0 < p.n; row0 += step) {
    if (row0 != first) {
#pragma unroll
      for (int u = 0; u < kSweeps; ++u) piece[u].load(p, min(row0 + (int64_t)u * rows, p.n - 1) * c + q * V);
    }
#pragma unroll
    for (int u = 0; u < kSweeps; ++u) {
      const int64_t row = row0 + (int64_t)u * rows;
      if (row >= p.n) break;
      const int64_t at = row * c + q * V;
      float xv[V], g[V];
      unpack<T, V>(piece[u].x, xv);
      if (kBackward) {
        piece[u].grad(xv, mean, scale, bias, g);
        if (p.dz) store_piece<T, V>(p.dz + at, g);
#pragma unroll
        for (int e = 0; e < V; ++e) g[e] = g[e] * ka[e] + (xv[e] - mean[e]) * kb[e] + kc[e];
      } else {
        float res[V];
        if (p.residual) load_piece<T, V>(p.residual + at, res);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          g[e] = (xv[e] - ka[e]) * kb[e] + kc[e];
          if (p.residual) g[e] += res[e];
          if (p.relu) g[e] = fmaxf(g[e], 0.f);
        }
      }
      store_piece<T, V>(p.out + at, g);
    }
  }
}

// The whole call for a matrix of at most kSmallRows rows, in one launch: a block of 1024 threads owns one
// 16-byte piece of every row, keeps its rows in registers between the sums and the element-wise pass.  Its
// loads take 16 bytes of a 128-byte line each, 3.4 us per 4096 rows and matrix, so that from there on
// (13 to 24 us) two launches are the faster ones.
constexpr int kSmallThreads = 1024, kSmallKeep = 1;
constexpr int kSmallRows = kSmallThreads * kSmallKeep;

template <typename T, int V, bool kBackward, Mask kMask>
__global__ __launch_bounds__(kSmallThreads) void bn_small_kernel(Bn<T> p) {
  __shared__ float red[kSmallThreads / 64][2 * V];
  __shared__ ColumnOut made[V];
  const int c = p.c, q = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  Piece<T, V, kBackward, kMask> piece[kSmallKeep];
#pragma unroll
  for (int i = 0; i < kSmallKeep; ++i)
    piece[i].load(p, min((int64_t)threadIdx.x + i * kSmallThreads, p.n - 1) * c + q * V);
  ColumnIn in{};
  if (threadIdx.x < V) in = load_column<T, kBackward>(p, q * V + threadIdx.x);
  float k[V], inv[V], scale[V], bias[V], a[2 * V];
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
    if ((int64_t)threadIdx.x + i * kSmallThreads >= p.n) break;
    float xv[V], g[V];
    unpack<T, V>(piece[i].x, xv);
    if (kBackward) piece[i].grad(xv, k, scale, bias, g);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float d = xv[e] - k[e];
      a[e] += kBackward ? g[e] : d;
      a[V + e] += kBackward ? g[e] * (d * inv[e]) : d * d;
    }
  }
  // 2 V sums over 64 lanes: in each of the first steps a lane hands on half of the sums it holds and keeps the other
  // half (17 exchanges for 16 sums instead of 96), so that a lane ends with the one of its upper lane bits
  int at = 0, width = 32;
#pragma unroll
  for (int m = V; m > 0; m /= 2) {
    const bool upper = lane & width;
#pragma unroll
    for (int e = 0; e < m; ++e) {
      const float keep = upper ? a[m + e] : a[e], give = upper ? a[e] : a[m + e];
      a[e] = keep + __shfl_xor(give, width);
    }
    at += upper ? m : 0;
    width /= 2;
  }
#pragma unroll
  for (int d = 16 / V; d > 0; d /= 2) a[0] += __shfl_xor(a[0], d);
  if ((lane & (32 / V - 1)) == 0) red[wave][at] = a[0];
  __syncthreads();
  if (threadIdx.x < V) {
    float t1 = 0.f, t2 = 0.f;
#pragma unroll
    for (int w = 0; w < kSmallThreads / 64; ++w) {
      t1 += red[w][threadIdx.x];
      t2 += red[w][V + threadIdx.x];
    }
    made[threadIdx.x] = finish_column<T, kBackward>(p, q * V + threadIdx.x, in, t1, t2, true);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSmallKeep; ++i) {
    const int64_t row = threadIdx.x + i * kSmallThreads;
    if (row >= p.n) break;
    const int64_t at = row * c + q * V;
    float xv[V], g[V], res[V], o[V];
    unpack<T, V>(piece[i].x, xv);
    if (kBackward) {
      piece[i].grad(xv, k, scale, bias, g);
      if (p.dz) store_piece<T, V>(p.dz + at, g);
    } else if (p.residual) {
      load_piece<T, V>(p.residual + at, res);
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const ColumnOut f = made[e];
      if (kBackward) {
        o[e] = g[e] * f.a + (xv[e] - k[e]) * f.b + f.c;
      } else {
        o[e] = (xv[e] - f.a) * f.b + f.c;
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
  TSMI_REQUIRE(c >= *v && c % *v == 0 && c / *v <= kMaxPieces,
               "%s: the channel count must be a multiple of %d and at most %d (got %d)", what, *v,
               *v * kMaxPieces, c);
  TSMI_REQUIRE(grid_fits(ceil_div(n * (c / *v), 256)), "%s: problem too large for one launch", what);
  return TSMI_OK;
}

template <typename T, bool kBackward, Mask kMask>
int launch(hipStream_t s, Bn<T> p) {
  constexpr int V = Vec<T>::V;
  if (p.n <= kSmallRows) {
    hipLaunchKernelGGL((bn_small_kernel<T, V, kBackward, kMask>), dim3(p.c / V), dim3(kSmallThreads), 0, s, p);
    return check_launch("bn_small_kernel");
  }
  const int rows = kBlock / (p.c / V), quads = p.c / 2;
  p.parts = (int)std::min<int64_t>(kMaxBlocks, ceil_div(p.n, (int64_t)rows * (kBackward ? 4 : 8)));
  hipLaunchKernelGGL((bn_reduce_kernel<T, V, kBackward, kMask>), dim3(p.parts), dim3(kBlock),
                     (size_t)rows * 2 * p.c * sizeof(float), s, p);
  const size_t lds = (size_t)(std::max(1, kBlock / quads) * 2 + 3) * p.c * sizeof(float);
  hipLaunchKernelGGL((bn_apply_kernel<T, V, kBackward, kMask>),
                     dim3((unsigned)std::min<int64_t>(kApplyBlocks, ceil_div(p.n, (int64_t)rows * kSweeps))),
                     dim3(kBlock), lds, s, p);
  return check_launch("bn_apply_kernel");
}

template <typename T>
Bn<T> bn_of(const void *x, int64_t n, int c, int relu, float *partial, float *stats,
            const void *weight, int param_dtype) {
  Bn<T> p{};
  p.x = (const T *)x;
  p.n = n;
  p.c = c;
  p.relu = relu;
  p.partial = partial;
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

extern "C" int64_t tsmi_bn_partial_elems(int c) { return (int64_t)kMaxBlocks * 2 * (c > 0 ? c : 0); }

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
                                     float eps, const void *residual, int relu, float *partial, float *stats,
                                     void *y) {
  int v;
  if (int e = check_shape("bn_forward_train", n, c, dtype, param_dtype, &v)) return e;
  TSMI_REQUIRE(x && y && partial && stats, "bn_forward_train: null pointer");
  TSMI_REQUIRE(aligned({x, y, residual}), "bn_forward_train: x, residual and y must be 16-byte aligned");
  TSMI_BN_BY_DTYPE({
    Bn<T> p = bn_of<T>(x, n, c, relu, partial, stats, weight, param_dtype);
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
                                float *partial, float *sums, void *grads, void *dz,
                                void *dx) {
  int v;
  if (int e = check_shape("bn_backward", n, c, dtype, param_dtype, &v)) return e;
  TSMI_REQUIRE(dy && x && dx && partial && stats && sums, "bn_backward: null pointer");
  TSMI_REQUIRE(aligned({dy, x, y, dz, dx}), "bn_backward: dy, x, y, dz and dx must be 16-byte aligned");
  TSMI_BN_BY_DTYPE({
    Bn<T> p = bn_of<T>(x, n, c, relu, partial, stats, weight, param_dtype);
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
