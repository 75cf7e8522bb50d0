// Forward / input gradient of maps with few rows (conv_small.hip).
#pragma once

#include "conv_device.hpp"

namespace rhip {

// Whether the small-map kernel runs this pass (forward, else input gradient).
template <typename T>
bool conv_small_takes(bool forward, int64_t n_rows, int64_t n_x, int cred, int ncols, int K);

// y[order[j]][n] = sum_k x[nbr[k][j]] . w[perm(k)][.][n] (+ bias[n]); w slices
// as [cred][ncols] (by_channel, fp32 only) or [ncols][cred].
template <typename T>
void conv_small(const T *x, int64_t n_x, int cred, const T *w, bool by_channel,
                const int32_t *wperm, int ncols, const float *bias, const int32_t *nbr,
                int64_t n_rows, int K, const int32_t *order, T *y, hipStream_t s);

} // namespace rhip
