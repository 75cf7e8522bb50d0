// Layers of channel counts the tiled kernels do not take, run on them with
// padded copies of the operands (conv_pad.hip).
#pragma once

#include "conv_device.hpp"

namespace rhip {

// Channels a layer's side is padded to: a width every tiled kernel takes as
// reduction and as columns.
inline int pad_width(int c) {
  for (int w : {32, 64, 128, 192, 256})
    if (c <= w)
      return w;
  return static_cast<int>(ceil_div(c, 64)) * 64;
}

// What the finishing kernels need to add an output up again from the unpadded
// operands: y[p][n] = sum_k sum_c x[nbr[k][p]][c] w[perm(k)][c * wc + n * wn]
// (+ bias[n]), w slices of C * ncols elements.
template <typename T> struct PadSum {
  const T *x, *w;
  int C, ncols;
  int64_t wc, wn;
  const int32_t *wperm;
  const float *bias;
  const int32_t *nbr, *order;
  int64_t n_rows;
  int K;
};

// dst[r][0 .. cp) = src[r][0 .. c), zeros beyond. `zero` (if given) is set to
// 0, `bad` (if given) to 1 where a value is not finite.
template <typename T>
void pad_features(const T *src, int64_t n, int c, int cp, T *dst, int *zero, int *bad,
                  hipStream_t s);

// dst [K][cp][np] from w [K][cin][cout], zeros beyond; bias_dst[0 .. np) from
// bias (either null: none); bad as above.
template <typename T>
void pad_weights(const T *w, int K, int cin, int cout, int cp, int np, T *dst, const float *bias,
                 float *bias_dst, int *bad, hipStream_t s);

// y[r][0 .. ncols) = yp[r][0 .. ncols) of rows of np (yp == y with np ==
// ncols: nothing to move); where *bad, values that are not finite are the sums
// of `sum`.
template <typename T>
void finish_rows(const T *yp, int np, T *y, const PadSum<T> &sum, const int *bad, hipStream_t s);

// dw [K][cin][cout] from dwp [K][cp][np]; where *bad, values that are not
// finite are the sums over the pairs of x[nbr[k][p]][ci] * gy[order[p]][co].
template <typename T>
void finish_weights(const T *dwp, int cp, int np, const T *x, int cin, const T *gy, int cout,
                    const int32_t *nbr, const int32_t *order, int64_t n_out, int K, T *dw,
                    const int *bad, hipStream_t s);

} // namespace rhip
