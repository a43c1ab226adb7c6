// Row L2 normalisation y = x / sqrt(sum x^2 + eps) and its backward
// dx = rstd (dy - y <y, dy>), for the q/k normalisation fla applies inside
// its delta-rule kernels when use_qk_l2norm_in_kernel=True (third-party
// flash-linear-attention==0.5.0, scripts/setup.sh:27 of the reference;
// DeltaNet configs set qk_norm: l2, configs/model/200m/delta_net_200m.yaml:13).
// fp32 arithmetic.
//
// HBM-bound: one read and one write per element forward, two and one
// backward.  Rows of 64, 128 or 256 elements at 16-byte aligned pointers take
// the row-group kernels: d / 8 lanes per row with eight elements each (16-byte
// loads in 16-bit types), kL2Rows rows per lane group whose loads are all
// issued before the first sum, sums by DPP steps inside the group.  Any other
// row length or alignment takes one wave per row with 2-byte (4-byte) accesses:
// at d = 64 that form leaves one element per lane and three quarters of each
// wave's time in the six shuffle steps.  95,952 rows of 64 in bf16 (B4 H12
// T1999): forward 17.9 -> 6.6 us, backward 21.0 -> 7.4 us.
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

constexpr int kL2Rows = 4;

// rows r0, r0 + RPB, .. of the block's kL2Rows * RPB rows; lane sub of the
// row's LPR lanes holds elements 8 sub .. 8 sub + 7
template <typename T, int LPR>
__global__ __launch_bounds__(256) void l2norm_fwd_rows_kernel(const T* __restrict__ x, T* __restrict__ y,
                                                              float* __restrict__ rstd, int n, float eps) {
  constexpr int RPB = 256 / LPR, D = 8 * LPR;
  const int sub = threadIdx.x % LPR, r0 = blockIdx.x * (kL2Rows * RPB) + threadIdx.x / LPR;
  v8_t<T> xv[kL2Rows];
#pragma unroll
  for (int i = 0; i < kL2Rows; ++i) {
    const int row = r0 + i * RPB;
    xv[i] = row < n ? ld8<T>(x + (int64_t)row * D + 8 * sub) : zero8<T>();
  }
#pragma unroll
  for (int i = 0; i < kL2Rows; ++i) {
    const int row = r0 + i * RPB;
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += (float)xv[i][j] * (float)xv[i][j];
    const float r = rsqrtf(group_sum<LPR>(ss) + eps);
    v8_t<T> o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (T)((float)xv[i][j] * r);
    if (row < n) {
      *reinterpret_cast<v8_t<T>*>(y + (int64_t)row * D + 8 * sub) = o;
      if (sub == 0) rstd[row] = r;
    }
  }
}

template <typename T, int LPR>
__global__ __launch_bounds__(256) void l2norm_bwd_rows_kernel(const T* __restrict__ y,
                                                              const float* __restrict__ rstd,
                                                              const T* __restrict__ dy,
                                                              T* __restrict__ dx, int n) {
  constexpr int RPB = 256 / LPR, D = 8 * LPR;
  const int sub = threadIdx.x % LPR, r0 = blockIdx.x * (kL2Rows * RPB) + threadIdx.x / LPR;
  v8_t<T> yv[kL2Rows], gv[kL2Rows];
  float rs[kL2Rows];
#pragma unroll
  for (int i = 0; i < kL2Rows; ++i) {
    const int row = r0 + i * RPB;
    yv[i] = row < n ? ld8<T>(y + (int64_t)row * D + 8 * sub) : zero8<T>();
    gv[i] = row < n ? ld8<T>(dy + (int64_t)row * D + 8 * sub) : zero8<T>();
    rs[i] = row < n ? rstd[row] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < kL2Rows; ++i) {
    const int row = r0 + i * RPB;
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) dot += (float)yv[i][j] * (float)gv[i][j];
    dot = group_sum<LPR>(dot);
    v8_t<T> o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (T)(rs[i] * ((float)gv[i][j] - (float)yv[i][j] * dot));
    if (row < n) *reinterpret_cast<v8_t<T>*>(dx + (int64_t)row * D + 8 * sub) = o;
  }
}

// lanes per row of the row-group kernels, 0 where they do not apply
inline int l2_lanes(int d, std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if ((uintptr_t)p & 15) return 0;
  return d == 64 ? 8 : d == 128 ? 16 : d == 256 ? 32 : 0;
}
inline int l2_blocks(int n, int lpr) {
  const int per = kL2Rows * (256 / lpr);
  return (int)(((int64_t)n + per - 1) / per);
}

template <typename T>
hipError_t launch_l2norm_fwd(const void* x, void* y, float* rstd, int n, int d, float eps,
                             hipStream_t s) {
  const int lpr = l2_lanes(d, {x, y});
  auto go = [&](auto l) {
    constexpr int LPR = decltype(l)::value;
    l2norm_fwd_rows_kernel<T, LPR><<<dim3(l2_blocks(n, LPR)), dim3(256), 0, s>>>((const T*)x, (T*)y, rstd, n, eps);
    return hipGetLastError();
  };
  if (lpr == 8) return go(IntC<8>{});
  if (lpr == 16) return go(IntC<16>{});
  if (lpr == 32) return go(IntC<32>{});
  l2norm_fwd_kernel<T><<<dim3((n + 3) / 4), dim3(256), 0, s>>>((const T*)x, (T*)y, rstd, n, d, eps);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_l2norm_bwd(const void* y, const float* rstd, const void* dy, void* dx, int n,
                             int d, hipStream_t s) {
  const int lpr = l2_lanes(d, {y, dy, dx});
  auto go = [&](auto l) {
    constexpr int LPR = decltype(l)::value;
    l2norm_bwd_rows_kernel<T, LPR><<<dim3(l2_blocks(n, LPR)), dim3(256), 0, s>>>((const T*)y, rstd, (const T*)dy,
                                                                            (T*)dx, n);
    return hipGetLastError();
  };
  if (lpr == 8) return go(IntC<8>{});
  if (lpr == 16) return go(IntC<16>{});
  if (lpr == 32) return go(IntC<32>{});
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
