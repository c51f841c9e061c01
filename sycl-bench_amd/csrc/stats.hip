// Covariance and correlation of an n x m data matrix (n observations of m
// variables): the column statistics and the centring / normalising pass,
// then the m x m product dataᵀ·data on the triangle contraction kernels.
//
// Replaces the kernel sequences of polybench/covariance.cpp:76-128 (mean,
// centre, upper-triangle covariance + mirror) and
// polybench/correlation.cpp:92-158 (mean, standard deviation, centre and
// scale, upper-triangle correlation + mirror, unit diagonal).
//
// Column sums run as a two-level reduction: a grid of (64-column strip x row
// slab) blocks writes one partial sum per column and slab to the workspace,
// and the kernel that needs the finished statistic adds the slabs of its own
// 64 columns first (finish_columns), in a fixed order, so results do not
// depend on scheduling and no launch is spent on finishing.  Every sum is
// float, as in the reference, made compensated (Neumaier) so its error does
// not grow with the row count.  The arithmetic of each finished statistic
// follows the reference's types: the covariance mean divides a float sum by a
// float constant; the correlation standard deviation divides the float sum of
// float squares by the double constant FLOAT_N, takes a float square root and
// replaces values <= eps by 1; centring subtracts in float, and the
// correlation scaling divides by sqrt(FLOAT_N) in double and by the deviation
// in float.  Those two scalar divisions are the only double operations, and
// they are the reference's own.
#include <algorithm>
#include <cmath>

#include "mfx_internal.h"

namespace mfx {

mfx_status sym_common(Handle* h, mfx_precision prec, mfx_uplo uplo, int mirror, int64_t n, int64_t k, float alpha,
    const float* A, int64_t lda, const float* B, int64_t ldb, float beta, float* C, int64_t ldc, int nprod, bool trans,
    hipStream_t s);
mfx_status check_matrix(const char* name, const void* p, int64_t rows, int64_t cols, int64_t ld);

namespace {

// Compensated (Neumaier) float summation: `sum` plus the running rounding
// error `comp`, so a long column sum stays as accurate as a float can hold
// without widening the type the reference sums in.
struct FSum {
  float sum = 0.0f, comp = 0.0f;
  __device__ __forceinline__ void add(float x) {
    const float t = sum + x;
    comp += fabsf(sum) >= fabsf(x) ? (sum - t) + x : (x - t) + sum;
    sum = t;
  }
  __device__ __forceinline__ float value() const { return sum + comp; }
};

// Thread layout of every pass over the data: 64 columns per block, W of them
// (one 16-byte load for W = 4) per thread, the block's other threads on
// further rows.  Narrow data keeps its threads busy and a wave reads 256-byte
// row segments at least.
constexpr int STRIP = 64;
template <int W>
struct StripShape {
  static constexpr int TX = STRIP / W, TY = 256 / TX;
};

template <int W>
__device__ __forceinline__ void load_cols(const float* p, float (&x)[W]) {
  if constexpr(W == 4) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    x[0] = v.x;
    x[1] = v.y;
    x[2] = v.z;
    x[3] = v.w;
  } else {
    x[0] = p[0];
  }
}

// Sums the slab partials of the block's 64 columns [j0, j0 + 64) into
// total[0..63] (0 past m): four threads per column, each a quarter of the
// slabs (slab q to thread q % 4) with eight loads in flight, then the four in
// thread order.  Called by all 256 threads; ends with a barrier.
// One finishing kernel of ceil(m / 256) blocks walking up to 2048 slabs
// serially took 278 us for 500 columns (one load latency per slab).  With at
// most MAX_SLABS slabs, four ways and eight deep, inside the consumer, the
// statistics of a 20000 x 500 correlation (sums, deviations, centring) went
// from 591 us in five kernels to about 45 us in three.
constexpr int MAX_SLABS = 128;
__device__ __forceinline__ void finish_columns(int64_t m, int slabs, const float* partial, int64_t j0, float* total,
    float (*quarter)[STRIP]) {
  const int c = threadIdx.x & (STRIP - 1), g = threadIdx.x / STRIP;
  const int64_t j = j0 + c;
  FSum s;
  if(j < m) {
    int q = g;
    for(; q + 28 < slabs; q += 32) {
      float x[8];
#pragma unroll
      for(int u = 0; u < 8; ++u) x[u] = partial[(int64_t)(q + 4 * u) * m + j];
#pragma unroll
      for(int u = 0; u < 8; ++u) s.add(x[u]);
    }
    for(; q < slabs; q += 4) s.add(partial[(int64_t)q * m + j]);
  }
  quarter[g][c] = s.value();
  __syncthreads();
  if(g == 0) {
    FSum t;
#pragma unroll
    for(int u = 0; u < 4; ++u) t.add(quarter[u][c]);
    total[c] = t.value();
  }
  __syncthreads();
}

// Partial column sums of rows [slab * rows_per, ...): without `sums` the sum
// of x; with it (the slab partials of a finished column sum) the sum of
// (x - mean[j])^2, the difference and square in float, mean[j] being the
// float quotient total / n_const, which the blocks of slab 0 also write out.
// HBM-bound: 16 rows of 256 bytes per block and step, four steps in flight.
template <int W>
__global__ __launch_bounds__(256) void column_partial_kernel(int64_t m, int64_t n, const float* data, int64_t ld,
    int64_t rows_per, const float* sums, int slabs, float n_const, float* mean, float* partial) {
  constexpr int TX = StripShape<W>::TX, TY = StripShape<W>::TY;
  __shared__ float mu_s[STRIP];
  __shared__ float part[TY > 4 ? TY : 4][STRIP];
  const int64_t j0 = (int64_t)blockIdx.x * STRIP;
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int64_t j = j0 + tx * W;
  float mu[W] = {};
  if(sums) {
    finish_columns(m, slabs, sums, j0, mu_s, part);
    if(threadIdx.x < STRIP) {
      mu_s[threadIdx.x] /= n_const;
      if(blockIdx.y == 0 && j0 + threadIdx.x < m) mean[j0 + threadIdx.x] = mu_s[threadIdx.x];
    }
    __syncthreads();
#pragma unroll
    for(int w = 0; w < W; ++w) mu[w] = mu_s[tx * W + w];
  }
  const int64_t r1 = min(n, ((int64_t)blockIdx.y + 1) * rows_per);
  FSum acc[W];
  auto take = [&](const float(&x)[W]) __attribute__((always_inline)) {
#pragma unroll
    for(int w = 0; w < W; ++w) {
      const float d = x[w] - mu[w];  // mu is 0 without `sums`: x unchanged
      acc[w].add(sums ? d * d : x[w]);
    }
  };
  if(j < m) {
    int64_t r = (int64_t)blockIdx.y * rows_per + ty;
    for(; r + 3 * TY < r1; r += 4 * TY) {
      float x[4][W];
#pragma unroll
      for(int u = 0; u < 4; ++u) load_cols<W>(data + (r + u * TY) * ld + j, x[u]);
#pragma unroll
      for(int u = 0; u < 4; ++u) take(x[u]);
    }
    for(; r < r1; r += TY) {
      float x[W];
      load_cols<W>(data + r * ld + j, x);
      take(x);
    }
  }
#pragma unroll
  for(int w = 0; w < W; ++w) part[ty][tx * W + w] = acc[w].value();
  __syncthreads();
  if(threadIdx.x < STRIP && j0 + threadIdx.x < m) {
    FSum t;
#pragma unroll
    for(int u = 0; u < TY; ++u) t.add(part[u][threadIdx.x]);
    partial[(int64_t)blockIdx.y * m + j0 + threadIdx.x] = t.value();
  }
}

// What center_kernel subtracts and divides by.
struct CenterArgs {
  const float* sums;   // slab partials of the column sums (covariance) or squared deviations (correlation)
  int slabs;
  float* mean;         // covariance: written; correlation: read
  float* stddev;       // correlation: written; null for covariance
  float n_const;       // covariance: mean = total / n_const
  double n_const_d, eps, scale_d;  // correlation
};

// out[i][j] = data[i][j] - mean[j]; with a deviation, then divided in double
// by scale_d and in float by stddev[j].  Each block finishes its columns'
// statistic first: the mean, or stddev[j] = sqrtf(total / n_const) with the
// division in double (the reference's FLOAT_N is a double constant) and
// values <= eps replaced by 1; the blocks of row range 0 write it out.
template <int W>
__global__ __launch_bounds__(256) void center_kernel(int64_t m, int64_t n, const float* data, int64_t ld,
    const CenterArgs a, int64_t rows_per, float* out, int64_t ldo) {
  constexpr int TX = StripShape<W>::TX, TY = StripShape<W>::TY;
  __shared__ float stat[STRIP];
  __shared__ float quarter[4][STRIP];
  const int64_t j0 = (int64_t)blockIdx.x * STRIP;
  finish_columns(m, a.slabs, a.sums, j0, stat, quarter);
  if(threadIdx.x < STRIP) {
    const int64_t j = j0 + threadIdx.x;
    float v = stat[threadIdx.x];
    if(a.stddev) {
      v = sqrtf((float)((double)v / a.n_const_d));
      v = (double)v <= a.eps ? 1.0f : v;
    } else {
      v = v / a.n_const;
    }
    stat[threadIdx.x] = v;
    if(blockIdx.y == 0 && j < m) (a.stddev ? a.stddev : a.mean)[j] = v;
  }
  __syncthreads();
  const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  const int64_t j = j0 + tx * W;
  if(j >= m) return;
  float mu[W], sd[W];
#pragma unroll
  for(int w = 0; w < W; ++w) {
    mu[w] = a.stddev ? a.mean[j + w] : stat[tx * W + w];
    sd[w] = a.stddev ? stat[tx * W + w] : 1.0f;
  }
  const int64_t r1 = min(n, ((int64_t)blockIdx.y + 1) * rows_per);
  auto put = [&](int64_t i, float(&x)[W]) __attribute__((always_inline)) {
#pragma unroll
    for(int w = 0; w < W; ++w) {
      x[w] -= mu[w];
      if(a.stddev) x[w] = (float)((double)x[w] / a.scale_d) / sd[w];
    }
    float* o = out + i * ldo + j;
    if constexpr(W == 4) *reinterpret_cast<float4*>(o) = make_float4(x[0], x[1], x[2], x[3]);
    else o[0] = x[0];
  };
  int64_t i = (int64_t)blockIdx.y * rows_per + ty;
  for(; i + 3 * TY < r1; i += 4 * TY) {
    float x[4][W];
#pragma unroll
    for(int u = 0; u < 4; ++u) load_cols<W>(data + (i + u * TY) * ld + j, x[u]);
#pragma unroll
    for(int u = 0; u < 4; ++u) put(i + u * TY, x[u]);
  }
  for(; i < r1; i += TY) {
    float x[W];
    load_cols<W>(data + i * ld + j, x);
    put(i, x);
  }
}

__global__ void set_diagonal_kernel(int64_t m, float* C, int64_t ldc, float value) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(j < m) C[j * ldc + j] = value;
}

// Rows per block so that the grid has about `blocks` blocks of one strip
// each, at most `most` along the rows and at least 64 rows in each.
int64_t slab_rows(int64_t m, int64_t n, int64_t blocks, int64_t most) {
  const int64_t want = std::min(most, std::max<int64_t>(1, blocks / ceil_div(m, STRIP)));
  return std::max<int64_t>(64, ceil_div(n, want));
}

// 16-byte loads and stores of four columns: aligned rows and m % 4 == 0.
bool strip_vec_ok(const float* p, int64_t ld, int64_t m) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && ld % 4 == 0 && m % 4 == 0;
}

// Column partials of `data` (of squared deviations when `sums` is given).
mfx_status column_partials(Handle* h, int64_t m, int64_t n, const float* data, int64_t ld, int64_t rows_per,
    const float* sums, float n_const, float* mean, float* partial, hipStream_t s) {
  const int slabs = (int)ceil_div(n, rows_per);
  const dim3 grid((unsigned)ceil_div(m, STRIP), (unsigned)slabs);
  return timed_launch(h, sums ? "column_sqdev_partial" : "column_sum_partial", s, [&] {
    if(strip_vec_ok(data, ld, m))
      column_partial_kernel<4><<<grid, 256, 0, s>>>(m, n, data, ld, rows_per, sums, slabs, n_const, mean, partial);
    else
      column_partial_kernel<1><<<grid, 256, 0, s>>>(m, n, data, ld, rows_per, sums, slabs, n_const, mean, partial);
  });
}

mfx_status center(Handle* h, int64_t m, int64_t n, const float* data, int64_t ld, const CenterArgs& a, float* out,
    int64_t ldo, hipStream_t s) {
  const int64_t rows_per = slab_rows(m, n, 1024, 1024);
  const dim3 grid((unsigned)ceil_div(m, STRIP), (unsigned)ceil_div(n, rows_per));
  return timed_launch(h, a.stddev ? "center_scale_columns" : "center_columns", s, [&] {
    if(strip_vec_ok(data, ld, m) && strip_vec_ok(out, ldo, m))
      center_kernel<4><<<grid, 256, 0, s>>>(m, n, data, ld, a, rows_per, out, ldo);
    else
      center_kernel<1><<<grid, 256, 0, s>>>(m, n, data, ld, a, rows_per, out, ldo);
  });
}

mfx_status check_stats_args(mfx_precision prec, int64_t m, int64_t n, const float* data, int64_t ld,
    const float* centered, int64_t ldw, const float* symmat, int64_t lds) {
  if(prec < MFX_PREC_FP32 || prec > MFX_PREC_BF16) return unsupported("covariance / correlation: FP32, SPLIT_BF16 or BF16");
  if(m <= 0 || n <= 0) return invalid("covariance / correlation need m > 0 and n > 0");
  MFX_CHECK(check_matrix("data", data, n, m, ld));
  MFX_CHECK(check_matrix("centered", centered, n, m, ldw));
  MFX_CHECK(check_matrix("symmat", symmat, m, m, lds));
  return MFX_SUCCESS;
}

}  // namespace
}  // namespace mfx

using namespace mfx;

extern "C" {

mfx_status mfx_covariance(mfx_handle handle, mfx_precision prec, int64_t m, int64_t n, const float* data, int64_t ld,
    float n_const, float* mean, float* centered, int64_t ldw, float* symmat, int64_t lds, mfx_stream stream) {
  if(!handle) return invalid("null handle");
  Handle* h = &handle->h;
  MFX_HIP(hipSetDevice(h->device));
  MFX_CHECK(check_stats_args(prec, m, n, data, ld, centered, ldw, symmat, lds));
  if(!mean) return invalid("null mean");
  hipStream_t s = static_cast<hipStream_t>(stream);
  // one slab partial per column and row range
  const int64_t rows_per = slab_rows(m, n, 512, MAX_SLABS), slabs = ceil_div(n, rows_per);
  void* ws = nullptr;
  MFX_CHECK(workspace(h, (size_t)(slabs * m) * sizeof(float), &ws));
  float* sums = static_cast<float*>(ws);
  MFX_CHECK(column_partials(h, m, n, data, ld, rows_per, nullptr, 0.0f, nullptr, sums, s));
  CenterArgs a{};
  a.sums = sums;
  a.slabs = (int)slabs;
  a.mean = mean;
  a.n_const = n_const;
  MFX_CHECK(center(h, m, n, data, ld, a, centered, ldw, s));
  // symmat = centeredᵀ · centered: upper triangle, mirrored (covariance.cpp:114-126)
  return sym_common(h, prec, MFX_UPPER, 1, m, n, 1.0f, centered, ldw, nullptr, 0, 0.0f, symmat, lds, 1, true, s);
}

mfx_status mfx_correlation(mfx_handle handle, mfx_precision prec, int64_t m, int64_t n, const float* data,
    int64_t ld, double n_const, double eps, float* mean, float* stddev, float* centered, int64_t ldw, float* symmat,
    int64_t lds, mfx_stream stream) {
  if(!handle) return invalid("null handle");
  Handle* h = &handle->h;
  MFX_HIP(hipSetDevice(h->device));
  MFX_CHECK(check_stats_args(prec, m, n, data, ld, centered, ldw, symmat, lds));
  if(!mean || !stddev) return invalid("null mean or stddev");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t rows_per = slab_rows(m, n, 512, MAX_SLABS), slabs = ceil_div(n, rows_per);
  void* ws = nullptr;
  MFX_CHECK(workspace(h, (size_t)(2 * slabs * m) * sizeof(float), &ws));
  float* sums = static_cast<float*>(ws);
  float* sqdev = sums + slabs * m;
  MFX_CHECK(column_partials(h, m, n, data, ld, rows_per, nullptr, 0.0f, nullptr, sums, s));
  MFX_CHECK(column_partials(h, m, n, data, ld, rows_per, sums, (float)n_const, mean, sqdev, s));
  CenterArgs a{};
  a.sums = sqdev;
  a.slabs = (int)slabs;
  a.mean = mean;
  a.stddev = stddev;
  a.n_const_d = n_const;
  a.eps = eps;
  a.scale_d = std::sqrt(n_const);
  MFX_CHECK(center(h, m, n, data, ld, a, centered, ldw, s));
  // symmat = centeredᵀ · centered: upper triangle, mirrored, then a unit
  // diagonal (correlation.cpp:138-158)
  MFX_CHECK(sym_common(h, prec, MFX_UPPER, 1, m, n, 1.0f, centered, ldw, nullptr, 0, 0.0f, symmat, lds, 1, true, s));
  return timed_launch(h, "unit_diagonal", s, [&] {
    set_diagonal_kernel<<<(unsigned)ceil_div(m, 256), 256, 0, s>>>(m, symmat, lds, 1.0f);
  });
}

}  // extern "C"
