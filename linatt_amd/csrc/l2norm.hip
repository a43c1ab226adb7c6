// Row L2 normalisation y = x / sqrt(sum x^2 + eps) and its backward
// dx = rstd (dy - y <y, dy>), for the q/k normalisation fla applies inside
// its delta-rule kernels when use_qk_l2norm_in_kernel=True (third-party
// flash-linear-attention==0.5.0, scripts/setup.sh:27 of the reference;
// DeltaNet configs set qk_norm: l2, configs/model/200m/delta_net_200m.yaml:13).
// fp32 arithmetic.
//
// HBM-bound: one read and one write per element forward, two and one
// backward.  Rows of 64, 128 or 256 elements at 16-byte aligned pointers take
// the row-group kernels: eight lanes per row with 16-byte accesses (16-bit types),
// all loads of a lane's one to four rows issued before the first sum, DPP steps
// across the lanes.  Any other row length or alignment takes one wave per row
// with 2-byte (4-byte) accesses: at d = 64 that form leaves one element per lane
// and three quarters of each wave's time in the six shuffle steps.  95,952 rows
// of 64 in bf16 (B4 H12 T1999), one call after another on the same buffers:
// forward 13.2 -> 4.9 us, backward 15.6 -> 5.8 us; 400,000 rows 60.0 -> 16.6 and
// 62.3 -> 23.3.  Both forms give the same bits: sums of eight products per lane
// and a tree over the lanes would take 4.4 and 5.1 us, but its float32 error is
// larger (rms of rstd 3.517e-8 against 3.494e-8) and the flipped 16-bit roundings
// travel through the delta rule's recurrence.
#include <initializer_list>

#include "common.h"
#include "misc_kernels.h"

namespace linatt {

template <typename T>
__global__ __launch_bounds__(256) void l2norm_fwd_kernel(const T* __restrict__ x, T* __restrict__ y,
                                                         float* __restrict__ rstd, int n, int d,
                                                         float eps) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= n) return;
  const T* xr = x + (int64_t)row * d;
  float ss = 0.f;
  for (int e = lane; e < d; e += 64) {
    const float xv = (float)xr[e];
    ss += xv * xv;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  const float r = rsqrtf(ss + eps);
  T* yr = y + (int64_t)row * d;
  for (int e = lane; e < d; e += 64) yr[e] = (T)((float)xr[e] * r);
  if (lane == 0) rstd[row] = r;
}

template <typename T>
__global__ __launch_bounds__(256) void l2norm_bwd_kernel(const T* __restrict__ y,
                                                         const float* __restrict__ rstd,
                                                         const T* __restrict__ dy,
                                                         T* __restrict__ dx, int n, int d) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= n) return;
  const T* yr = y + (int64_t)row * d;
  const T* gr = dy + (int64_t)row * d;
  float dot = 0.f;
  for (int e = lane; e < d; e += 64) dot += (float)yr[e] * (float)gr[e];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) dot += __shfl_xor(dot, off);
  const float r = rstd[row];
  T* xr = dx + (int64_t)row * d;
  for (int e = lane; e < d; e += 64) xr[e] = (T)(r * ((float)gr[e] - (float)yr[e] * dot));
}

// Rows of 64 K elements by groups of eight lanes.  Lane sub of a row's group holds
// elements 64 k + 8 c .. + 7 (k < K) of chunk c = l2_chunk(sub), so that the
// wave-per-row kernels' summation order is kept, bit for bit: the chain over k
// in the lane, xor 32, 16 and 8 of the element index as the three DPP steps
// (lane xor 1, 2 and 7, which l2_chunk maps to chunk xor 4, 2 and 1), xor 4, 2
// and 1 in the lane.  The result does not depend on the pointers' alignment.
constexpr int l2_rows(int K) { return K >= 4 ? 1 : 4 / K; }  // rows in flight: 64 bytes per lane and 16-bit operand
__device__ __forceinline__ int l2_chunk(int sub) {
  const int hi = sub >> 2, lo = sub ^ (7 * hi);
  return 4 * (lo & 1) + 2 * ((lo >> 1) & 1) + hi;
}
__device__ __forceinline__ float l2_sum(float (&p)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) p[j] = group_sum<8>(p[j]);
  return ((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]));
}

// (T)(a r) of a lane's eight elements.  float16 rows of 64 take the product's
// float16 rounding in one step (a mixed-precision fma with +0), as the general
// kernel's loop does for its last odd element; longer rows there go in pairs,
// rounded to float32 first.
template <typename T, int K>
__device__ __forceinline__ v8_t<T> l2_out(const float (&a)[8], float r) {
  v8_t<T> o;
  if constexpr (__is_same(T, _Float16) && K == 1) {
    u32x4 u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned w;
      asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(w) : "v"(a[2 * j]), "v"(r));
      asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(w) : "v"(a[2 * j + 1]), "v"(r));
      u[j] = w;
    }
    o = __builtin_bit_cast(v8_t<T>, u);
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (T)(a[j] * r);
  }
  return o;
}

template <typename T, int K>
__global__ __launch_bounds__(256) void l2norm_fwd_rows_kernel(const T* __restrict__ x, T* __restrict__ y,
                                                              float* __restrict__ rstd, int n, float eps) {
  constexpr int RPB = 32, D = 64 * K, R = l2_rows(K);
  const int sub = threadIdx.x & 7, r0 = blockIdx.x * (R * RPB) + (threadIdx.x >> 3), c8 = 8 * l2_chunk(sub);
  v8_t<T> xv[R][K];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = r0 + i * RPB;
#pragma unroll
    for (int k = 0; k < K; ++k) xv[i][k] = row < n ? ld8<T>(x + (int64_t)row * D + 64 * k + c8) : zero8<T>();
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = r0 + i * RPB;
    float p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = 0.f;
#pragma unroll
      for (int k = 0; k < K; ++k) p[j] = fmaf((float)xv[i][k][j], (float)xv[i][k][j], p[j]);
    }
    const float r = rsqrtf(l2_sum(p) + eps);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      float a[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = (float)xv[i][k][j];
      if (row < n) st8<T>(y + (int64_t)row * D + 64 * k + c8, l2_out<T, K>(a, r));
    }
    if (row < n && sub == 0) rstd[row] = r;
  }
}

template <typename T, int K>
__global__ __launch_bounds__(256) void l2norm_bwd_rows_kernel(const T* __restrict__ y,
                                                              const float* __restrict__ rstd,
                                                              const T* __restrict__ dy,
                                                              T* __restrict__ dx, int n) {
  constexpr int RPB = 32, D = 64 * K, R = l2_rows(K);
  const int sub = threadIdx.x & 7, r0 = blockIdx.x * (R * RPB) + (threadIdx.x >> 3), c8 = 8 * l2_chunk(sub);
  v8_t<T> yv[R][K], gv[R][K];
  float rs[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = r0 + i * RPB;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      yv[i][k] = row < n ? ld8<T>(y + (int64_t)row * D + 64 * k + c8) : zero8<T>();
      gv[i][k] = row < n ? ld8<T>(dy + (int64_t)row * D + 64 * k + c8) : zero8<T>();
    }
    rs[i] = row < n ? rstd[row] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = r0 + i * RPB;
    float p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = 0.f;
#pragma unroll
      for (int k = 0; k < K; ++k) p[j] = fmaf((float)yv[i][k][j], (float)gv[i][k][j], p[j]);
    }
    const float dot = l2_sum(p);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      float a[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = fmaf(-(float)yv[i][k][j], dot, (float)gv[i][k][j]);
      if (row < n) st8<T>(dx + (int64_t)row * D + 64 * k + c8, l2_out<T, K>(a, rs[i]));
    }
  }
}

// 64-element parts per row of the row-group kernels, 0 where they do not apply
inline int l2_parts(int d, std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if ((uintptr_t)p & 15) return 0;
  return d == 64 || d == 128 || d == 256 ? d / 64 : 0;
}
inline int l2_blocks(int n, int K) {
  const int per = 32 * l2_rows(K);
  return (int)(((int64_t)n + per - 1) / per);
}

template <typename T>
hipError_t launch_l2norm_fwd(const void* x, void* y, float* rstd, int n, int d, float eps,
                             hipStream_t s) {
  const int parts = l2_parts(d, {x, y});
  auto go = [&](auto l) {
    constexpr int K = decltype(l)::value;
    l2norm_fwd_rows_kernel<T, K><<<dim3(l2_blocks(n, K)), dim3(256), 0, s>>>((const T*)x, (T*)y, rstd, n, eps);
    return hipGetLastError();
  };
  if (parts == 1) return go(IntC<1>{});
  if (parts == 2) return go(IntC<2>{});
  if (parts == 4) return go(IntC<4>{});
  l2norm_fwd_kernel<T><<<dim3((n + 3) / 4), dim3(256), 0, s>>>((const T*)x, (T*)y, rstd, n, d, eps);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_l2norm_bwd(const void* y, const float* rstd, const void* dy, void* dx, int n,
                             int d, hipStream_t s) {
  const int parts = l2_parts(d, {y, dy, dx});
  auto go = [&](auto l) {
    constexpr int K = decltype(l)::value;
    l2norm_bwd_rows_kernel<T, K><<<dim3(l2_blocks(n, K)), dim3(256), 0, s>>>((const T*)y, rstd, (const T*)dy, (T*)dx,
                                                                             n);
    return hipGetLastError();
  };
  if (parts == 1) return go(IntC<1>{});
  if (parts == 2) return go(IntC<2>{});
  if (parts == 4) return go(IntC<4>{});
  l2norm_bwd_kernel<T><<<dim3((n + 3) / 4), dim3(256), 0, s>>>((const T*)y, rstd, (const T*)dy,
                                                               (T*)dx, n, d);
  return hipGetLastError();
}

#define LINATT_L2_INST(T)                                                                       \
  template hipError_t launch_l2norm_fwd<T>(const void*, void*, float*, int, int, float, hipStream_t); \
  template hipError_t launch_l2norm_bwd<T>(const void*, const float*, const void*, void*, int, int, \
                                           hipStream_t);
LINATT_L2_INST(__bf16)
LINATT_L2_INST(_Float16)
LINATT_L2_INST(float)

}  // namespace linatt
