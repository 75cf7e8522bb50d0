// Thin convolutions (conv_thin.hip): layers with few im2col columns.
#pragma once

#include "conv_device.hpp"

namespace rhip {

// im2col columns (offsets x channels): piece indices stay exact in
// gather_tile's 20-bit reciprocal up to here
constexpr int kThinMaxCols = 1024;

// Whether the thin kernels can run a layer of K offsets over n_x feature
// rows of C reduced channels.
bool conv_thin_takes(int K, int C, int64_t n_x, int elem_bytes);

// y[order[p]][n] = sum_k sum_c x[nbr[k][p]][c] * w[perm(k) * wk + c * wc + n * wn] (+ bias[n])
template <typename T>
void conv_thin(const T *x, int64_t n_x, int C, const T *w, int64_t wk, int64_t wc, int64_t wn,
               const int32_t *wperm, int ncols, const float *bias, const int32_t *nbr,
               int64_t n_rows, int K, const int32_t *order, T *y, hipStream_t s);

// dw[k][c][n] = sum_p x[nbr[k][p]][c] * gy[order[p]][n]; partial holds
// conv_dw_thin_ranges(...) * K * C * cout floats.
int conv_dw_thin_ranges(int K, int C, int cout, int64_t n_rows);
template <typename T>
void conv_dw_thin(const T *x, int64_t n_x, int C, const T *gy, int cout, const int32_t *nbr,
                  int64_t n_rows, int K, const int32_t *order, float *partial, T *dw,
                  hipStream_t s);

} // namespace rhip
