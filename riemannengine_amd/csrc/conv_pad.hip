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
// outputs that are not finite up again over the pairs that exist, from the
// unpadded operands: one lane per output, and in dW, where a sum runs over all
// rows, one wave per 16 x 16 tile on the fp32 matrix cores. With one infinite
// gradient, or all NaN, dW of 64->20 bf16 on 200k rows takes 5.6 ms (one lane
// per element 71, a wave per element 12 and 198).
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
  const int64_t row = sum.order ? sum.order[pos] : pos;
  const T v = yp[row * np + col];
  if (finite(v)) {
    y[row * sum.ncols + col] = v;
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
  y[row * sum.ncols + col] = from_f32<T>(acc);
}

// A wave owns 16 x 16 elements of one offset's dW, a lane four of a column.
template <typename T>
__global__ __launch_bounds__(kThreads) void finish_weights_kernel(
    const T *__restrict__ dwp, int cp, int np, const T *__restrict__ x, int cin,
    const T *__restrict__ gy, int cout, const int32_t *__restrict__ nbr,
    const int32_t *__restrict__ order, int64_t n_out, int K, T *__restrict__ dw,
    const int *__restrict__ bad) {
  const int lane = threadIdx.x & (kWave - 1), i16 = lane & 15, g = lane >> 4;
  const int ct = (cin + 15) / 16, ot = (cout + 15) / 16;
  const int64_t tile = blockIdx.x * static_cast<int64_t>(kWaves) + threadIdx.x / kWave;
  const int64_t k = tile / (ct * ot);
  if (k >= K)
    return; // the whole wave
  const int rem = static_cast<int>(tile - k * (ct * ot));
  const int ci0 = rem / ot * 16, co = rem % ot * 16 + i16;
  const bool col = co < cout;
  T v[4];
  bool ok = true;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int ci = ci0 + 4 * g + e;
    v[e] = col && ci < cin ? dwp[(k * cp + ci) * np + co] : from_f32<T>(0.f);
    ok = ok && finite(v[e]);
  }
  if (*bad != 0 && __any(!ok)) { // uniform
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const bool row = ci0 + i16 < cin;
    for (int64_t p0 = 0; p0 < n_out; p0 += kWave) {
      const int64_t p = p0 + lane;
      const int32_t id = p < n_out ? nbr[k * n_out + p] : -1;
      if (!__any(id >= 0)) // uniform; past here row 0 exists
        continue;
      const int32_t o = id < 0 ? 0 : (order ? order[p] : static_cast<int32_t>(p));
      T a[16], b[16];
      uint32_t has = 0;
#pragma unroll
      for (int s = 0; s < 16; ++s) { // positions 4s + g, at clamped places: all in flight
        const int32_t is = __shfl(id, 4 * s + g), os = __shfl(o, 4 * s + g);
        has |= (is >= 0 ? 1u : 0u) << s;
        a[s] = x[static_cast<int64_t>(max(is, 0)) * cin + min(ci0 + i16, cin - 1)];
        b[s] = gy[static_cast<int64_t>(os) * cout + min(co, cout - 1)];
      }
#pragma unroll
      for (int s = 0; s < 16; ++s) { // zeros on both sides where there is no pair
        const bool pair = (has >> s) & 1u;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(pair && row ? to_f32(a[s]) : 0.f,
                                                   pair && col ? to_f32(b[s]) : 0.f, acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = finite(v[e]) ? v[e] : from_f32<T>(acc[e]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (col && ci0 + 4 * g + e < cin)
      dw[(k * cin + ci0 + 4 * g + e) * cout + co] = v[e];
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
  hipLaunchKernelGGL((finish_weights_kernel<T>),
                     blocks_of(K * ceil_div(cin, 16) * ceil_div(cout, 16) * kWave), dim3(kThreads),
                     0, s, dwp, cp, np, x, cin, gy, cout, nbr, order, n_out, K, dw,
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
