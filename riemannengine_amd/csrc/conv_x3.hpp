// fp32 forward / input gradient on the bf16 matrix cores (conv_x3.hip).
#pragma once

#include "conv_device.hpp"

namespace rhip {

// Whether the kernel takes a reduction of cred channels to ncols columns over
// K offsets, from n_x to n_rows rows (a forward, else an input gradient).
bool conv_x3_takes(bool forward, int cred, int ncols, int K, int64_t n_x, int64_t n_rows);

// Bytes of the three-part weights for K offsets.
inline size_t conv_x3_weight_bytes(int K, int cred, int ncols) {
  return static_cast<size_t>(K) * cred * ncols * 6;
}

// Splits of the offset axis (1: none) and the floats of their partial sums.
int conv_x3_splits(int64_t n_rows, int cred, int ncols, int K);

// y[order[j]][n] = sum_k x[nbr[k][j]] . w[perm(k)][.][n] (+ bias[n]), the
// weight of channel c and column n at w[k * cred * ncols + c * wc + n * wn].
// wt: conv_x3_weight_bytes; partial: splits * n_rows * ncols floats, or fewer
// for no split.
void conv_x3(const float *x, int64_t n_x, int cred, const float *w, int wc, int wn,
             const int32_t *wperm, int ncols, const float *bias, const int32_t *nbr,
             int64_t n_rows, int K, const int32_t *order, float *y, void *wt, float *partial,
             size_t partial_floats, hipStream_t s);

} // namespace rhip
