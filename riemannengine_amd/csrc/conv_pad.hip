// Copies around the tiled kernels for channel counts they do not take: the
// features' rows, the weights and the bias are padded with zeros to
// pad_width, the tiled kernels run on the copies, and the results are cropped.
// The copies are bound by HBM (24 fp32 channels of 200k rows: 45 MB, 12 us).
// Measured on MI355X, 3^3 on 200k rows, against one lane per output and (dW)
// per element of dW: 64->20 bf16 forward 5151 -> 56 us, dX 417 -> 63, dW 60.9
// ms -> 91 us; 24->80 dX 7510 -> 106.
//
// The tiled kernels multiply a missing neighbour's zeros, which a weight (or,
// in dW, a gradient) that is not finite turns into NaN. The copies see every
// such value and set a flag on the device; the finishing kernels then add the
// outputs up again over the pairs that exist, from the unpadded operands.
#include "conv_pad.hpp"

namespace rhip {

namespace {

template <typename T> __device__ __forceinline__ bool finite(T v) {
  const float f = to_f32(v);
  return f - f == 0.f;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void pad_features_kernel(const T *__restrict__ src,
                                                                int64_t n, int c, int cp,
                                                                T *__restrict__ dst, int *zero,
                                                                int *bad) {
  constexpr int VE = 16 / sizeof(T); // elements per thread
  const int64_t t = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (t == 0 && zero)
    *zero = 0;
  const int pieces = cp / VE;
  const int64_t r = t / pieces;
  if (r >= n)
    return;
  const int c0 = static_cast<int>(t - r * pieces) * VE;
  T v[VE];
  bool ok = true;
#pragma unroll
  for (int e = 0; e < VE; ++e) {
    v[e] = c0 + e < c ? src[r * c + c0 + e] : from_f32<T>(0.f);
    ok = ok && finite(v[e]);
  }
  *reinterpret_cast<uint4 *>(dst + r * cp + c0) = *reinterpret_cast<const uint4 *>(v);
  if (bad && !ok)
    *bad = 1;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void pad_weights_kernel(
    const T *__restrict__ w, int K, int cin, int cout, int cp, int np, T *__restrict__ dst,
    const float *__restrict__ bias, float *__restrict__ bias_dst, int *bad) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (bias && t < np)
    bias_dst[t] = t < cout ? bias[t] : 0.f;
  const int64_t row = t / np;
  const int n = static_cast<int>(t - row * np);
  const int64_t k = row / cp;
  const int c = static_cast<int>(row - k * cp);
  if (k >= K)
    return;
  const bool in = c < cin && n < cout;
  const T v = in ? w[(k * cin + c) * cout + n] : from_f32<T>(0.f);
  dst[t] = v;
  if (!finite(v))
    *bad = 1;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void finish_rows_kernel(const T *yp, int np, T *y,
                                                               const PadSum<T> sum,
                                                               const int *__restrict__ bad) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  const int64_t pos = t / sum.ncols;
  const int col = static_cast<int>(t - pos * sum.ncols);
  if (pos >= sum.n_rows)
    return;
  if (*bad == 0) {
    if (yp != y)
      y[t] = yp[pos * np + col];
    return;
  }
  float acc = 0.f;
  for (int k = 0; k < sum.K; ++k) {
    const int32_t id = sum.nbr[k * sum.n_rows + pos];
    if (id < 0)
      continue;
    const T *xr = sum.x + static_cast<int64_t>(id) * sum.C;
    const T *wr = sum.w + static_cast<int64_t>(sum.wperm ? sum.wperm[k] : k) * sum.C * sum.ncols +
                  col * sum.wn;
    for (int c = 0; c < sum.C; ++c)
      acc += to_f32(xr[c]) * to_f32(wr[c * sum.wc]);
  }
  if (sum.bias)
    acc += sum.bias[col];
  y[(sum.order ? sum.order[pos] : pos) * sum.ncols + col] = from_f32<T>(acc);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void finish_weights_kernel(
    const T *__restrict__ dwp, int cp, int np, const T *__restrict__ x, int cin,
    const T *__restrict__ gy, int cout, const int32_t *__restrict__ nbr,
    const int32_t *__restrict__ order, int64_t n_out, int K, T *__restrict__ dw,
    const int *__restrict__ bad) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (t >= static_cast<int64_t>(K) * cin * cout)
    return;
  const int64_t row = t / cout;
  const int co = static_cast<int>(t - row * cout);
  const int64_t k = row / cin;
  const int ci = static_cast<int>(row - k * cin);
  if (*bad == 0) {
    dw[t] = dwp[(k * cp + ci) * np + co];
    return;
  }
  float acc = 0.f;
  for (int64_t p = 0; p < n_out; ++p) {
    const int32_t id = nbr[k * n_out + p];
    if (id >= 0)
      acc += to_f32(x[static_cast<int64_t>(id) * cin + ci]) *
             to_f32(gy[(order ? order[p] : p) * cout + co]);
  }
  dw[t] = from_f32<T>(acc);
}

dim3 blocks_of(int64_t threads) {
  return dim3(static_cast<unsigned>(ceil_div(std::max<int64_t>(threads, 1), kThreads)));
}

} // namespace

template <typename T>
void pad_features(const T *src, int64_t n, int c, int cp, T *dst, int *zero, int *bad,
                  hipStream_t s) {
  hipLaunchKernelGGL((pad_features_kernel<T>), blocks_of(n * cp * static_cast<int64_t>(sizeof(T)) / 16),
                     dim3(kThreads), 0, s, src, n, c, cp, dst, zero, bad);
  RHIP_LAUNCH_CHECK();
}

template <typename T>
void pad_weights(const T *w, int K, int cin, int cout, int cp, int np, T *dst, const float *bias,
                 float *bias_dst, int *bad, hipStream_t s) {
  hipLaunchKernelGGL((pad_weights_kernel<T>), blocks_of(static_cast<int64_t>(K) * cp * np),
                     dim3(kThreads), 0, s, w, K, cin, cout, cp, np, dst, bias, bias_dst, bad);
  RHIP_LAUNCH_CHECK();
}

template <typename T>
void finish_rows(const T *yp, int np, T *y, const PadSum<T> &sum, const int *bad, hipStream_t s) {
  hipLaunchKernelGGL((finish_rows_kernel<T>), blocks_of(sum.n_rows * sum.ncols), dim3(kThreads), 0,
                     s, yp, np, y, sum, bad);
  RHIP_LAUNCH_CHECK();
}

template <typename T>
void finish_weights(const T *dwp, int cp, int np, const T *x, int cin, const T *gy, int cout,
                    const int32_t *nbr, const int32_t *order, int64_t n_out, int K, T *dw,
                    const int *bad, hipStream_t s) {
  hipLaunchKernelGGL((finish_weights_kernel<T>), blocks_of(static_cast<int64_t>(K) * cin * cout),
                     dim3(kThreads), 0, s, dwp, cp, np, x, cin, gy, cout, nbr, order, n_out, K, dw,
                     bad);
  RHIP_LAUNCH_CHECK();
}

#define RHIP_PAD_FOR(T)                                                                          \
  template void pad_features<T>(const T *, int64_t, int, int, T *, int *, int *, hipStream_t);   \
  template void pad_weights<T>(const T *, int, int, int, int, int, T *, const float *, float *,  \
                               int *, hipStream_t);                                              \
  template void finish_rows<T>(const T *, int, T *, const PadSum<T> &, const int *, hipStream_t); \
  template void finish_weights<T>(const T *, int, int, const T *, int, const T *, int,           \
                                  const int32_t *, const int32_t *, int64_t, int, T *,           \
                                  const int *, hipStream_t);
RHIP_PAD_FOR(float)
RHIP_PAD_FOR(__bf16)

} // namespace rhip
