// Thin convolutions: layers whose reduction over offsets and channels is
// short (a network's first layer with its few input channels, 1^D layers
// such as a classifier) and channel counts the tiled kernels of conv.hip do
// not take. Such a layer is one dense product over im2col rows: position p's
// row holds x[nbr[k][p]][c] at r = k * C + c (zeros for a missing
// neighbour), so
//   forward / dX:  Y[p][n]  = sum_r A[p][r] W[r][n]
//   dW:            dW[r][n] = sum_p A[p][r] dY[p][n]
// with A built in LDS, 64 positions at a time, and multiplied on MFMA in the
// features' type with fp32 sums. The zeros of missing neighbours cost MFMA
// work (about 2.5 times the pairs of a surface's 3^3 map), which is small
// against what the walk over the offsets costs in the tiled kernels here.
//
// Weights or gradients that are not finite would turn those zeros into NaN
// (0 * inf): a chunk that holds any is multiplied element by element, over
// the pairs that exist only.
#include <algorithm>
#include <type_traits>

#include "conv_thin.hpp"

namespace rhip {

namespace {

constexpr int kSeg = 64; // positions per LDS tile
constexpr int kRC = 96;  // im2col columns per LDS chunk (a 3^3 layer of 3 channels: 81)
constexpr int kRB = kRC / 16;

template <typename T> constexpr bool kF32 = std::is_same<T, float>::value;

// PB bytes at a buffer offset, as 32-bit words (2 bytes: the low half)
template <int PB> struct PieceOf { using type = uint32_t; };
template <> struct PieceOf<16> { using type = v4u; };
template <int PB>
__device__ __forceinline__ typename PieceOf<PB>::type load_piece(__amdgpu_buffer_rsrc_t r,
                                                                 uint32_t off) {
  if constexpr (PB == 16)
    return __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  else if constexpr (PB == 4)
    return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
  else
    return static_cast<uint32_t>(
        static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0)));
}
template <int PB, typename T>
__device__ __forceinline__ void store_piece(T *p, const typename PieceOf<PB>::type &v) {
  if constexpr (PB == 2)
    *reinterpret_cast<uint16_t *>(p) = static_cast<uint16_t>(v);
  else
    *reinterpret_cast<typename PieceOf<PB>::type *>(p) = v;
}

// whether a 32-bit word of values (one float or two bf16) has one that is
// not finite (all exponent bits set)
template <typename T> __device__ __forceinline__ bool word_bad(uint32_t w) {
  if constexpr (kF32<T>)
    return (w & 0x7f800000u) == 0x7f800000u;
  else
    return (w & 0x7f800000u) == 0x7f800000u || (w & 0x7f80u) == 0x7f80u;
}
template <int PB, typename T>
__device__ __forceinline__ bool piece_bad(const typename PieceOf<PB>::type &v) {
  if constexpr (PB == 16)
    return word_bad<T>(v[0]) || word_bad<T>(v[1]) || word_bad<T>(v[2]) || word_bad<T>(v[3]);
  else
    return word_bad<T>(v);
}

// How a layer's im2col columns split into LDS chunks of at most kRC: up to kc
// whole offsets each, or for C > kRC one offset's channels in `parts` parts
// of cw (a multiple of 32, the last one shorter).
struct Thin {
  int K, C;
  int ppr;       // pieces per feature row
  uint32_t div;  // ceil(2^20 / ppr): piece -> offset
  uint32_t cdiv; // ceil(2^20 / C): column -> offset
  int kc, parts, cw, chunks;
  int64_t blocks; // position tiles
};
struct Chunk {
  int k0, kn, c0, cw; // offsets k0 .. k0 + kn - 1, channels c0 .. c0 + cw - 1
  __device__ int cols() const { return kn * cw; }
};
__device__ __forceinline__ Chunk chunk_of(const Thin &th, int ch) {
  if (th.parts == 1)
    return {ch * th.kc, min(th.kc, th.K - ch * th.kc), 0, th.C};
  const int c0 = (ch % th.parts) * th.cw;
  return {ch / th.parts, 1, c0, min(th.cw, th.C - c0)};
}
// the offset of column r of a chunk
__device__ __forceinline__ int offset_of(const Thin &th, const Chunk &c, int r) {
  return c.k0 + (c.kn == 1 ? 0 : static_cast<int>((static_cast<uint32_t>(r) * th.cdiv) >> 20));
}

// A chunk's im2col columns of positions pos0 .. pos0 + 63 to LDS rows of LDA
// elements. Missing
// neighbours, and with TAIL positions past the end, give zeros without a
// memory access (a row index past the buffer's last). idx(k, position): the
// feature row or -1. Pieces under 16 bytes: lane = position and wave w the
// offsets w, w + 4, ..., so that the table reads are coalesced and an
// offset's row address serves all its pieces; 16-byte pieces go piece-fastest,
// so that a wave reads whole rows. Returns whether a value read was not
// finite (CHECK).
template <typename T, int PB, int LDA, bool CHECK, bool TAIL, typename Idx>
__device__ __forceinline__ bool gather_tile(T *s, __amdgpu_buffer_rsrc_t rx, uint32_t n_x,
                                            int64_t pos0, int64_t n_rows, const Thin &th,
                                            const Chunk &ck, Idx &&idx) {
  constexpr int VE = PB / sizeof(T);
  constexpr int U = 8; // loads in flight per thread
  const uint32_t row_bytes = static_cast<uint32_t>(th.C * sizeof(T));
  const uint32_t c0_bytes = static_cast<uint32_t>(ck.c0 * sizeof(T));
  const int k0 = ck.k0, kn = ck.kn;
  const int tid = threadIdx.x;
  bool bad = false;
  if constexpr (PB < 16) {
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int p = tid & (kSeg - 1);
    const int64_t pos = min(pos0 + p, n_rows - 1);
    const int32_t in = TAIL && pos0 + p >= n_rows ? -1 : 0;
    if (kn < kWaves) { // few offsets: the waves share out their pieces
      const int ppc = ck.cw / VE, items = kn * ppc;
      for (int j0 = wv; j0 < items; j0 += kWaves * U) {
        uint32_t off[U];
        T *dst[U];
#pragma unroll
        for (int u = 0; u < U; ++u) { // past the last piece: the last one again
          const int j = min(j0 + kWaves * u, items - 1);
          const int k = (j >= ppc ? 1 : 0) + (j >= 2 * ppc ? 1 : 0), q = j - k * ppc;
          off[u] = min(static_cast<uint32_t>(idx(k0 + k, pos) | in), n_x) * row_bytes + c0_bytes +
                   static_cast<uint32_t>(q * PB);
          dst[u] = s + p * LDA + k * th.C + q * VE;
        }
        typename PieceOf<PB>::type v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          v[u] = load_piece<PB>(rx, off[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          store_piece<PB>(dst[u], v[u]);
          if constexpr (CHECK)
            bad = bad || piece_bad<PB, T>(v[u]);
        }
      }
      return bad;
    }
    for (int j0 = wv; j0 < kn; j0 += kWaves * U) {
      // past the last offset: the last one again (the same values once more)
      uint32_t off[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        off[u] = min(static_cast<uint32_t>(idx(k0 + min(j0 + kWaves * u, kn - 1), pos) | in),
                     n_x) * row_bytes + c0_bytes;
      T *dst = s + p * LDA;
      for (int q = 0; q < ck.cw / VE; ++q) {
        typename PieceOf<PB>::type v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          v[u] = load_piece<PB>(rx, off[u] + static_cast<uint32_t>(q * PB));
#pragma unroll
        for (int u = 0; u < U; ++u) {
          store_piece<PB>(dst + min(j0 + kWaves * u, kn - 1) * th.C + q * VE, v[u]);
          if constexpr (CHECK)
            bad = bad || piece_bad<PB, T>(v[u]);
        }
      }
    }
  } else {
    const int qn = kn * (ck.cw / VE); // pieces per position
    const int sh = 32 - __builtin_clz(max(qn - 1, 1)); // rounded up to a power of two
    const int count = max((kSeg << sh) / kThreads, 1);
    for (int j0 = 0; j0 < count; j0 += U) {
      uint32_t off[U];
      T *dst[U];
      bool live[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = (j0 + u) * kThreads + tid;
        const int p = min(e >> sh, kSeg - 1), i = min(e & ((1 << sh) - 1), qn - 1);
        live[u] = j0 + u < count && (e >> sh) < kSeg && (e & ((1 << sh) - 1)) < qn;
        const int k = kn == 1 ? 0 : static_cast<int>((static_cast<uint32_t>(i) * th.div) >> 20);
        const int q = i - k * th.ppr;
        const int32_t id = idx(k0 + k, min(pos0 + p, n_rows - 1)) |
                           (live[u] && pos0 + p < n_rows ? 0 : -1);
        off[u] = min(static_cast<uint32_t>(id), n_x) * row_bytes +
                 static_cast<uint32_t>(q * PB) + c0_bytes;
        dst[u] = s + p * LDA + k * th.C + q * VE;
      }
      typename PieceOf<PB>::type v[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        v[u] = load_piece<PB>(rx, off[u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (live[u]) {
          store_piece<PB>(dst[u], v[u]);
          if constexpr (CHECK)
            bad = bad || piece_bad<PB, T>(v[u]);
        }
    }
  }
  return bad;
}

// Y[order[p]][n] = sum_r A[p][r] W[r][n] (+ bias[n]): W[k * C + c][n] at
// w[perm(k) * wk + c * wc + n * wn]. A workgroup owns NT columns and walks
// tiles of 64 positions (wave w: rows 16w .. 16w + 15); chunks of rc columns
// of A and W go through LDS, W only once where one chunk holds it all.
// Bound by the latency of a tile's loads (table, then features). Measured on
// MI355X, kernel alone: a first layer of 194k rows, 3^3, 3->32 bf16, 236 us
// on the one-lane-per-output kernel, 31 here (45 with the offset, table index
// and row address worked out anew for every piece); a 1^3 layer of 96k rows,
// 64->20 fp32, forward and dX 193 us each, 22 here. 1024 workgroups at most,
// so that the staged weights serve three tiles or more on a large map.
template <typename T, int NT, int PB>
__global__ __launch_bounds__(kThreads) void conv_thin_kernel(
    const T *__restrict__ x, int64_t n_x, const Thin th, const T *__restrict__ w, int64_t wk,
    int64_t wc, int64_t wn, const int32_t *__restrict__ wperm, int ncols,
    const float *__restrict__ bias, const int32_t *__restrict__ nbr, int64_t n_rows,
    const int32_t *__restrict__ order, T *__restrict__ y) {
  using M = Mfma<T>;
  using Frag = typename M::Frag;
  constexpr int CH = M::kCh, EPL = CH / 4;
  constexpr int LD = kRC + 16 / sizeof(T);
  constexpr int NB = NT / 16;
  __shared__ __align__(16) T sA[kSeg * LD];
  __shared__ __align__(16) T sB[NT * LD];
  __shared__ int sbad; // 1 + the last chunk staged with a weight that is not finite
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int i16 = lane & 15, g = lane >> 4;
  const int col0 = blockIdx.y * NT;
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(x, n_x * th.C * static_cast<int64_t>(sizeof(T)));
  auto idx = [&](int k, int64_t p) { return nbr[k * n_rows + p]; };
  if (tid == 0)
    sbad = 0;
  // the chunk's weights transposed to [n][r], zeros past its columns (up to a
  // whole MFMA step) and past ncols; the tile's columns past the chunk's zero
  // too. Consecutive threads go along the contiguous axis of w.
  auto stage = [&](const Chunk &ck, int ch) {
    const int cols = ck.cols(), rc = (cols + CH - 1) / CH * CH;
    constexpr int WU = 8;
    const int count = wn == 1 ? rc * NT : NT * kRC; // elements, NT or kRC per row
    for (int e0 = tid; e0 < count; e0 += WU * kThreads) {
      T v[WU];
      int at[WU];
      int k[WU], r[WU], n[WU];
#pragma unroll
      for (int i = 0; i < WU; ++i) {
        const int e = e0 + i * kThreads;
        n[i] = wn == 1 ? e % NT : e / kRC;
        r[i] = wn == 1 ? e / NT : e % kRC;
        const int rr = min(r[i], cols - 1);
        k[i] = offset_of(th, ck, rr);
        at[i] = (ck.c0 + rr - (k[i] - ck.k0) * th.C) * static_cast<int>(wc) +
                min(col0 + n[i], ncols - 1) * static_cast<int>(wn);
      }
      if (wperm) {
#pragma unroll
        for (int i = 0; i < WU; ++i)
          k[i] = wperm[k[i]];
      }
#pragma unroll
      for (int i = 0; i < WU; ++i) // at clamped places, all in flight
        v[i] = w[k[i] * wk + at[i]];
#pragma unroll
      for (int i = 0; i < WU; ++i) {
        const bool in = r[i] < cols && col0 + n[i] < ncols;
        const float f = to_f32(v[i]);
        if (in && !(f - f == 0.f))
          sbad = ch + 1;
        if (r[i] < rc && n[i] < NT)
          sB[n[i] * LD + r[i]] = in ? v[i] : from_f32<T>(0.f);
      }
    }
    for (int p = wv; p < kSeg; p += kWaves)
      if (cols + lane < rc)
        sA[p * LD + cols + lane] = from_f32<T>(0.f);
  };
  for (int64_t t = blockIdx.x; t < th.blocks; t += gridDim.x) {
    const int64_t pos0 = t * kSeg;
    v4f acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      acc[nb] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int ch = 0; ch < th.chunks; ++ch) {
      const Chunk ck = chunk_of(th, ch);
      __syncthreads(); // every wave is done with the previous chunk
      if (th.chunks > 1 || t == blockIdx.x)
        stage(ck, ch);
      // rows past the end repeat the last one; they are not stored
      gather_tile<T, PB, LD, false, false>(sA, rx, static_cast<uint32_t>(n_x), pos0, n_rows, th,
                                           ck, idx);
      __syncthreads();
      if (sbad == ch + 1) { // over the pairs that exist only
        for (int e = 0; e < 4; ++e) {
          const int64_t pos = pos0 + 16 * wv + 4 * g + e;
          for (int r = 0; r < ck.cols() && pos < n_rows; ++r) {
            if (nbr[offset_of(th, ck, r) * n_rows + pos] < 0)
              continue;
            const float a = to_f32(sA[(16 * wv + 4 * g + e) * LD + r]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              acc[nb][e] += a * to_f32(sB[(16 * nb + i16) * LD + r]);
          }
        }
        continue;
      }
#pragma unroll 2
      for (int s = 0; s < ck.cols(); s += CH) {
        const Frag a = *reinterpret_cast<const Frag *>(&sA[(16 * wv + i16) * LD + s + g * EPL]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const Frag b =
              *reinterpret_cast<const Frag *>(&sB[(16 * nb + i16) * LD + s + g * EPL]);
          M::mma(a, b, acc[nb]);
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t pos = pos0 + 16 * wv + 4 * g + e;
      if (pos >= n_rows)
        continue;
      T *dst = y + (order ? order[pos] : pos) * ncols + col0 + i16;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int col = col0 + 16 * nb + i16;
        if (col < ncols)
          dst[16 * nb] = from_f32<T>(acc[nb][e] + (bias ? bias[col] : 0.f));
      }
    }
  }
}

// Partial dW: workgroup (range, chunk, column block) adds A^T dY over the
// 64-position segments range, range + ranges, ... into rows r0 .. r0 + rc of
// its slot partial[range][R][cout]. Wave w owns column block w % NB and
// every (4 / NB)-th 16-row block. The K-major operands of bf16 come from
// row-major LDS tiles through ds_read_b64_tr_b16. Measured on MI355X with the
// reduction, the layers above: 74.5 ms and 32.3 ms on the pair lists with one
// lane per element of dW (each lane a serial walk over its offset's pairs),
// 41 us and 34 us here.
template <typename T, int NT, int PB, int PBY>
__global__ __launch_bounds__(kThreads) void conv_dw_thin_kernel(
    const T *__restrict__ x, int64_t n_x, const Thin th, const T *__restrict__ gy, const Thin ty,
    const int32_t *__restrict__ nbr, int64_t n_rows, const int32_t *__restrict__ order,
    float *__restrict__ partial) {
  constexpr int NB = NT / 16;
  constexpr int WPB = kWaves / NB;           // waves per column block
  constexpr int TPW = (kRB + WPB - 1) / WPB; // row blocks per wave
  // fp32 reads [4s + g][i16]: rows 16 (or 49) banks apart, and 4-byte stores
  // a position per lane want an odd stride
  constexpr int LDA = kF32<T> ? (PB == 16 ? kRC + 16 : kRC + 17) : kRC + 8;
  constexpr int LDY = kF32<T> ? (NT == 16 ? 16 : NT + 16) : NT + 8;
  __shared__ __align__(16) T sA[kSeg * LDA];
  __shared__ __align__(16) T sY[kSeg * LDY];
  __shared__ int64_t sbad; // 1 + the last segment with a gradient that is not finite
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int i16 = lane & 15, g = lane >> 4;
  const int cout = ty.C, n0 = blockIdx.z * NT;
  const Chunk ck = chunk_of(th, blockIdx.y);
  const Chunk cy = {0, 1, n0, min(NT, cout - n0)};
  const int cols = ck.cols(), nrb = (cols + 15) / 16;
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(x, n_x * th.C * static_cast<int64_t>(sizeof(T)));
  const __amdgpu_buffer_rsrc_t ry = buf_rsrc(gy, n_rows * cout * static_cast<int64_t>(sizeof(T)));
  auto idx = [&](int k, int64_t p) { return nbr[k * n_rows + p]; };
  auto row = [&](int, int64_t p) { return order ? order[p] : static_cast<int32_t>(p); };
  const int nb = wv % NB;
  v4f acc[TPW];
#pragma unroll
  for (int j = 0; j < TPW; ++j)
    acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
  if (tid == 0)
    sbad = 0;
  for (int64_t s = blockIdx.x; s < th.blocks; s += gridDim.x) {
    __syncthreads(); // every wave is done with the previous segment
    if (gather_tile<T, PBY, LDY, true, true>(sY, ry, static_cast<uint32_t>(n_rows), s * kSeg,
                                             n_rows, ty, cy, row))
      sbad = s + 1;
    gather_tile<T, PB, LDA, false, true>(sA, rx, static_cast<uint32_t>(n_x), s * kSeg, n_rows, th,
                                         ck, idx);
    __syncthreads();
    if (sbad == s + 1) { // over the pairs that exist only
      for (int j = 0; j < TPW; ++j)
        for (int e = 0; e < 4; ++e) {
          const int r = 16 * (wv / NB + WPB * j) + 4 * g + e;
          for (int p = 0; p < kSeg && r < cols; ++p) {
            const int64_t pos = s * kSeg + p;
            if (pos < n_rows && nbr[offset_of(th, ck, r) * n_rows + pos] >= 0)
              acc[j][e] += to_f32(sA[p * LDA + r]) * to_f32(sY[p * LDY + 16 * nb + i16]);
          }
        }
      continue;
    }
    if constexpr (kF32<T>) {
#pragma unroll 4
      for (int st = 0; st < kSeg / 4; ++st) {
        const float b = sY[(4 * st + g) * LDY + 16 * nb + i16];
#pragma unroll
        for (int j = 0; j < TPW; ++j) {
          const int rb = wv / NB + WPB * j;
          if (rb < nrb)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                sA[(4 * st + g) * LDA + 16 * rb + i16], b, acc[j], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int st = 0; st < kSeg / 32; ++st) {
        const int prow = 32 * st + 8 * g + i16 / 4, pcol = 4 * (i16 % 4);
        const T *py = sY + prow * LDY + 16 * nb + pcol;
        const v4s blo = ds_read_tr16(py), bhi = ds_read_tr16(py + 4 * LDY);
        const v8bf b = __builtin_bit_cast(
            v8bf, __builtin_shufflevector(blo, bhi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int j = 0; j < TPW; ++j) {
          const int rb = wv / NB + WPB * j;
          if (rb < nrb) {
            const T *pa = sA + prow * LDA + 16 * rb + pcol;
            const v4s alo = ds_read_tr16(pa), ahi = ds_read_tr16(pa + 4 * LDA);
            const v8bf a = __builtin_bit_cast(
                v8bf, __builtin_shufflevector(alo, ahi, 0, 1, 2, 3, 4, 5, 6, 7));
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[j], 0, 0, 0);
          }
        }
      }
    }
  }
  float *slot = partial + (static_cast<int64_t>(blockIdx.x) * th.K * th.C + ck.k0 * th.C + ck.c0) *
                              cout;
  const int n = n0 + 16 * nb + i16;
#pragma unroll
  for (int j = 0; j < TPW; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 16 * (wv / NB + WPB * j) + 4 * g + e;
      if (r < cols && n < cout)
        slot[static_cast<int64_t>(r) * cout + n] = acc[j][e];
    }
}

// dw[i] = sum over the slots s of partial[s][i], in a fixed order: a
// workgroup of 16 waves owns 64 elements, wave w sums the slots s = w (mod
// 16) and the 16 sums are added in order.
template <typename T>
__global__ __launch_bounds__(1024) void thin_reduce_kernel(const float *__restrict__ partial,
                                                           int slots, int64_t n,
                                                           T *__restrict__ dw) {
  __shared__ float part[16][kWave];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kWave + lane;
  float sum = 0.f;
  if (i < n) {
#pragma unroll 8
    for (int s = w; s < slots; s += 16)
      sum += partial[s * n + i];
  }
  part[w][lane] = sum;
  __syncthreads();
  if (w != 0 || i >= n)
    return;
  for (int q = 1; q < 16; ++q)
    sum += part[q][lane];
  dw[i] = from_f32<T>(sum);
}

// The largest piece of 16, 4 or 2 bytes that divides a feature row and its
// address.
int piece_bytes(const void *p, int64_t row_bytes) {
  const auto a = reinterpret_cast<uintptr_t>(p) | static_cast<uintptr_t>(row_bytes);
  return a % 16 == 0 ? 16 : (a % 4 == 0 ? 4 : 2);
}

// The chunks of K offsets of C channels, in equal shares.
Thin thin_of(int K, int C, int pieces, int64_t n_rows) {
  auto inv = [](int d) { return static_cast<uint32_t>(((1 << 20) + d - 1) / d); };
  Thin t{K, C, pieces, inv(pieces), inv(C), 1, 1, C, 1, ceil_div(n_rows, kSeg)};
  if (C <= kRC) {
    t.chunks = static_cast<int>(ceil_div(K, kRC / C));
    t.kc = static_cast<int>(ceil_div(K, t.chunks));
    t.chunks = static_cast<int>(ceil_div(K, t.kc));
  } else {
    t.cw = static_cast<int>(ceil_div(ceil_div(C, ceil_div(C, kRC)), 32) * 32);
    t.parts = static_cast<int>(ceil_div(C, t.cw));
    t.chunks = K * t.parts;
  }
  return t;
}

} // namespace

bool conv_thin_takes(int K, int C, int64_t n_x, int elem_bytes) {
  return static_cast<int64_t>(K) * C <= kThinMaxCols && n_x * C * elem_bytes <= kBufMaxBytes;
}

template <typename T>
void conv_thin(const T *x, int64_t n_x, int C, const T *w, int64_t wk, int64_t wc, int64_t wn,
               const int32_t *wperm, int ncols, const float *bias, const int32_t *nbr,
               int64_t n_rows, int K, const int32_t *order, T *y, hipStream_t s) {
  const int pb = piece_bytes(x, static_cast<int64_t>(C) * sizeof(T));
  const Thin th = thin_of(K, C, C * static_cast<int>(sizeof(T)) / pb, n_rows);
  auto go = [&](auto ntc, auto pbc) {
    constexpr int NT = decltype(ntc)::value;
    const dim3 grid(static_cast<unsigned>(std::min<int64_t>(th.blocks, 1024)),
                    static_cast<unsigned>(ceil_div(ncols, NT)));
    hipLaunchKernelGGL((conv_thin_kernel<T, NT, decltype(pbc)::value>), grid, dim3(kThreads), 0,
                       s, x, n_x, th, w, wk, wc, wn, wperm, ncols, bias, nbr, n_rows, order, y);
  };
  using N16 = std::integral_constant<int, 16>;
  using N32 = std::integral_constant<int, 32>;
  using N64 = std::integral_constant<int, 64>;
  auto pick = [&](auto pbc) {
    ncols <= 16 ? go(N16{}, pbc) : (ncols <= 32 ? go(N32{}, pbc) : go(N64{}, pbc));
  };
  if (pb == 16) {
    pick(std::integral_constant<int, 16>{});
  } else if (pb == 4) {
    pick(std::integral_constant<int, 4>{});
  } else {
    if constexpr (!kF32<T>)
      pick(std::integral_constant<int, 2>{});
  }
  RHIP_LAUNCH_CHECK();
}

// Ranges of the thin dW kernel: about 1024 workgroups (four per CU), each
// range at least two segments, at most 512 partial slots.
int conv_dw_thin_ranges(int K, int C, int cout, int64_t n_rows) {
  const int64_t units = thin_of(K, C, 1, 1).chunks * ceil_div(cout, cout <= 32 ? 32 : 64);
  const int64_t segs = ceil_div(std::max<int64_t>(n_rows, 1), kSeg);
  return static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>({512, 1024 / units, ceil_div(segs, 2)})));
}

template <typename T>
void conv_dw_thin(const T *x, int64_t n_x, int C, const T *gy, int cout, const int32_t *nbr,
                  int64_t n_rows, int K, const int32_t *order, float *partial, T *dw,
                  hipStream_t s) {
  const int pb = piece_bytes(x, static_cast<int64_t>(C) * sizeof(T));
  int pby = piece_bytes(gy, static_cast<int64_t>(cout) * sizeof(T));
  if (pby == 4 && !kF32<T>)
    pby = 2;
  const Thin th = thin_of(K, C, C * static_cast<int>(sizeof(T)) / pb, n_rows);
  const Thin ty = thin_of(1, cout, cout * static_cast<int>(sizeof(T)) / pby, n_rows);
  const int ranges = conv_dw_thin_ranges(K, C, cout, n_rows);
  const int64_t n = static_cast<int64_t>(K) * C * cout;
  if (n_rows > 0) {
    auto go = [&](auto ntc, auto pbc, auto pbyc) {
      constexpr int NT = decltype(ntc)::value;
      const dim3 grid(static_cast<unsigned>(ranges), static_cast<unsigned>(th.chunks),
                      static_cast<unsigned>(ceil_div(cout, NT)));
      hipLaunchKernelGGL((conv_dw_thin_kernel<T, NT, decltype(pbc)::value, decltype(pbyc)::value>),
                         grid, dim3(kThreads), 0, s, x, n_x, th, gy, ty, nbr, n_rows, order,
                         partial);
    };
    auto pick_n = [&](auto pbc, auto pbyc) {
      cout <= 16   ? go(std::integral_constant<int, 16>{}, pbc, pbyc)
      : cout <= 32 ? go(std::integral_constant<int, 32>{}, pbc, pbyc)
                   : go(std::integral_constant<int, 64>{}, pbc, pbyc);
    };
    auto pick = [&](auto pbc) {
      using Elem = std::integral_constant<int, sizeof(T)>;
      pby == 16 ? pick_n(pbc, std::integral_constant<int, 16>{}) : pick_n(pbc, Elem{});
    };
    if (pb == 16) {
      pick(std::integral_constant<int, 16>{});
    } else if (pb == 4) {
      pick(std::integral_constant<int, 4>{});
    } else {
      if constexpr (!kF32<T>)
        pick(std::integral_constant<int, 2>{});
    }
    RHIP_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL((thin_reduce_kernel<T>), dim3(static_cast<unsigned>(ceil_div(n, kWave))),
                     dim3(1024), 0, s, partial, n_rows > 0 ? ranges : 0, n, dw);
  RHIP_LAUNCH_CHECK();
}

template void conv_thin<float>(const float *, int64_t, int, const float *, int64_t, int64_t,
                               int64_t, const int32_t *, int, const float *, const int32_t *,
                               int64_t, int, const int32_t *, float *, hipStream_t);
template void conv_thin<__bf16>(const __bf16 *, int64_t, int, const __bf16 *, int64_t, int64_t,
                                int64_t, const int32_t *, int, const float *, const int32_t *,
                                int64_t, int, const int32_t *, __bf16 *, hipStream_t);
template void conv_dw_thin<float>(const float *, int64_t, int, const float *, int, const int32_t *,
                                  int64_t, int, const int32_t *, float *, float *, hipStream_t);
template void conv_dw_thin<__bf16>(const __bf16 *, int64_t, int, const __bf16 *, int,
                                   const int32_t *, int64_t, int, const int32_t *, float *,
                                   __bf16 *, hipStream_t);

} // namespace rhip
