// Output-stationary gather GEMM for maps with few rows. There the other
// kernels are chains of memory round trips: a 64- or 128-row workgroup walks
// its offsets one after another, each stage waiting for its weights, its rows
// and two barriers, on a fraction of the CUs, or splits the offsets over
// workgroups and adds the partial sums in a second launch. Here a workgroup
// owns 16 output rows and its four waves share out the (offset, channel
// chunk) stages of those rows: each wave takes every fourth stage and keeps U
// stages' rows and weights in flight, straight from global memory to MFMA
// operands, with no barrier until the four sums are added in LDS in wave
// order (deterministic, one launch, no partial buffers).
//
// Every workgroup reads the weights of its rows' offsets itself (no copy is
// staged for others), which the L2 serves; that traffic, n_rows / 16 times the
// weights, is what limits the rows (conv_small_takes).
//
// A missing neighbour's row is zeros, which a weight that is not finite turns
// into NaN. A wave whose sums hold a value that is not finite walks its stages
// once more in the same order, each stage's products added only to the rows
// that have the neighbour, and takes those sums from there.
#include <algorithm>
#include <type_traits>

#include "conv_small.hpp"

namespace rhip {

namespace {

constexpr int kRows = 16;

template <typename T, int NT, int U, bool BY_CHANNEL>
__global__ __launch_bounds__(kThreads) void conv_small_kernel(
    const T *__restrict__ x, int64_t n_x, int cred, const T *__restrict__ w,
    const int32_t *__restrict__ wperm, int ncols, const float *__restrict__ bias,
    const int32_t *__restrict__ nbr, int64_t n_rows, int K, const int32_t *__restrict__ order,
    T *__restrict__ y) {
  using M = Mfma<T>;
  using Frag = typename M::Frag;
  constexpr int CH = M::kCh, EPL = CH / 4; // channels per stage, per lane
  constexpr int NB = NT / 16;
  constexpr int LDR = NT + 4;
  static_assert(!BY_CHANNEL || std::is_same<T, float>::value, "one channel per load: fp32");
  __shared__ __align__(16) float sR[kWaves][kRows * LDR];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int i16 = lane & 15, g = lane >> 4;
  const int64_t tile0 = xcd_tile(blockIdx.x) * kRows;
  if (tile0 >= n_rows)
    return; // padding workgroup (uniform)
  const int col0 = blockIdx.y * NT;

  // neighbour indices: lane (i16, g) of slot q holds offset 4q + g of row i16
  // (absent or past the end: -1), and the offsets with any neighbour
  typedef int32_t v8i __attribute__((ext_vector_type(8)));
  v8i v;
  {
    const int64_t pos = tile0 + i16;
    const bool in = pos < n_rows;
    const int64_t pc = in ? pos : n_rows - 1;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int k = 4 * q + g;
      v[q] = nbr[(k < K ? k : K - 1) * n_rows + pc] | ((in && k < K) ? 0 : -1);
    }
  }
  uint32_t m = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const uint64_t bal = __ballot(v[q] >= 0);
#pragma unroll
    for (int gg = 0; gg < 4; ++gg)
      m |= (((bal >> (16 * gg)) & 0xffffull) != 0 ? 1u : 0u) << (4 * q + gg);
  }
  m = __builtin_amdgcn_readfirstlane(m);

  const int nch = cred / CH;
  int cc = 0; // channel chunk of the next stage
  auto advance = [&](int n) {
    cc += n;
    while (cc >= nch && m) {
      cc -= nch;
      m &= m - 1;
    }
  };
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(x, n_x * cred * static_cast<int64_t>(sizeof(T)));
  v4f acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
    acc[nb] = v4f{0.f, 0.f, 0.f, 0.f};
  auto row_of = [&](int k) { // offset k's row for lane row i16
    return __builtin_amdgcn_ds_bpermute(((k & 3) * 16 + i16) * 4, v[k >> 2]);
  };
  auto load_a = [&](int32_t id, int ch) {
    const uint32_t off =
        pick_off(static_cast<uint32_t>(id) * static_cast<uint32_t>(cred * sizeof(T)) +
                     static_cast<uint32_t>((ch * CH + g * EPL) * sizeof(T)),
                 ~(id >> 31));
    return __builtin_bit_cast(Frag, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0));
  };
  auto load_b = [&](int k, int ch, Frag (&b)[NB]) {
    const int64_t kw = wperm ? wperm[k] : k;
    const int c = ch * CH + g * EPL, n = col0 + i16;
    const T *wk = w + kw * cred * ncols + (BY_CHANNEL ? c * ncols + n : n * cred + c);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if constexpr (BY_CHANNEL) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          b[nb][e] = wk[e * ncols + nb * 16];
      } else {
        b[nb] = *reinterpret_cast<const Frag *>(wk + nb * 16 * cred);
      }
    }
  };
  const uint32_t all = m;
  advance(wv);
  while (m) {
    int kj[U], cj[U];
    bool live[U];
#pragma unroll
    for (int u = 0; u < U; ++u) { // past the last stage: the first again, not multiplied
      live[u] = m != 0;
      kj[u] = live[u] ? __builtin_ctz(m) : kj[0];
      cj[u] = live[u] ? cc : cj[0];
      if (live[u])
        advance(kWaves);
    }
    Frag a[U], b[U][NB];
    int32_t id[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      id[u] = row_of(kj[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      a[u] = load_a(id[u], cj[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      load_b(kj[u], cj[u], b[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (live[u]) { // uniform
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          M::mma(a[u], b[u][nb], acc[nb]);
      }
  }
  float check = 0.f; // NaN where a sum is not finite
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      check += 0.f * acc[nb][e];
  if (__any(!(check == 0.f))) { // uniform
    v4f again[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      again[nb] = v4f{0.f, 0.f, 0.f, 0.f};
    m = all;
    cc = 0;
    for (advance(wv); m; advance(kWaves)) {
      const int k = __builtin_ctz(m);
      const Frag a = load_a(row_of(k), cc);
      Frag b[NB];
      load_b(k, cc, b);
      bool has[4]; // rows 4g .. 4g + 3
#pragma unroll
      for (int e = 0; e < 4; ++e)
        has[e] = __builtin_amdgcn_ds_bpermute(((k & 3) * 16 + 4 * g + e) * 4, v[k >> 2]) >= 0;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        v4f t = again[nb];
        M::mma(a, b[nb], t);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          again[nb][e] = has[e] ? t[e] : again[nb][e];
      }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[nb][e] = acc[nb][e] - acc[nb][e] == 0.f ? acc[nb][e] : again[nb][e];
  }
  // D[4g + e][i16] of block nb
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      sR[wv][(4 * g + e) * LDR + nb * 16 + i16] = acc[nb][e];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (kRows * NT + kThreads - 1) / kThreads; ++i) {
    const int e = tid + i * kThreads;
    const int r = e / NT, c = e % NT;
    const int64_t pos = tile0 + r;
    if (r < kRows && pos < n_rows) {
      float sum = sR[0][r * LDR + c];
#pragma unroll
      for (int q = 1; q < kWaves; ++q)
        sum += sR[q][r * LDR + c];
      if (bias)
        sum += bias[col0 + c];
      y[(order ? order[pos] : pos) * ncols + col0 + c] = from_f32<T>(sum);
    }
  }
}

template <typename T> int small_nt(int ncols) {
  return ncols % 64 == 0 ? 64 : (ncols % 32 == 0 ? 32 : 16);
}

} // namespace

template <typename T>
bool conv_small_takes(bool forward, int64_t n_rows, int64_t n_x, int cred, int ncols, int K) {
  if (n_rows < 1 || n_x < 1 || K > 32 || cred % Mfma<T>::kCh != 0 || ncols % 16 != 0 ||
      n_x * cred * static_cast<int64_t>(sizeof(T)) > kBufMaxBytes)
    return false;
  // The weights that all workgroups read together. Measured on MI355X, 3^3
  // forward / input gradient per call with the host's 12 us, the other kernels
  // against this one: fp32 16->32 on 10k rows (36 MB) 20.1 / 18.8 us against
  // 11.6 / 12.2, 32->32 on 10k (72 MB) 20.9 / 21.6 against 13.5 / 15.9, 64->64
  // on 2k (57 MB) 24.8 / 24.8 against 20.1 / 22.1, but on 4.9k (134 MB) 28.0 /
  // 27.9 against 25.7 / 32.0 and 16->32 on 48k (167 MB) 19.4 / 21.4 against
  // 22.6 / 29.8; bf16 32->32 on 10k (36 MB) 18.1 / 15.3 against 14.2 / 11.5, but
  // 64->64 on 4.9k (67 MB) 19.0 / 15.5 against 22.0 / 19.2.
  const bool f32 = std::is_same<T, float>::value;
  const int64_t read = ceil_div(n_rows, kRows) * K * cred * ncols * static_cast<int64_t>(sizeof(T));
  // Of 16 channels that is up to 58k rows, where many short workgroups cost
  // more: fp32 16->16 on 23k rows 20.3 / 20.0 against 13.4 / 13.5, on 37k 13.1
  // against 13.9 (dX), on 48k 16.2 / 14.4 against 17.2 / 16.0, transposed 2^3 on
  // 101k 16.2 / 12 against 14.5 / 15.
  if (n_rows > (f32 && forward && K <= 8 ? 70000 : 40000))
    return false;
  // With a few offsets the other kernels have no chain to shorten, and read
  // the weights a fraction as often. 1^3 in fp32: dX 128->64 on 48k rows (99
  // MB) 13 us against 65, 256->128 on 5k (41 MB) 12 against 19, but 192->192 on
  // 3.1k (29 MB) 16 against 12. The forward, whose weights lie along the lanes
  // and need no transposed copy here, gains longer: 256->128 on 5k 15 against
  // 12, 64->64 on 23k (24 MB) 15 against 13, on 48k (49 MB) 15 against 23. bf16
  // gains nothing there (128->256 on 3.1k 12 against 18).
  if (K < 8)
    return f32 && read <= (forward ? (n_rows <= 10000 ? 45'000'000 : 24'000'000)
                                   : (n_rows <= 4096 ? 33'000'000 : 8'000'000));
  return read <= (f32 ? 100'000'000 : 40'000'000);
}

template <typename T>
void conv_small(const T *x, int64_t n_x, int cred, const T *w, bool by_channel,
                const int32_t *wperm, int ncols, const float *bias, const int32_t *nbr,
                int64_t n_rows, int K, const int32_t *order, T *y, hipStream_t s) {
  const int nt = small_nt<T>(ncols);
  const dim3 grid(static_cast<unsigned>(xcd_grid(ceil_div(n_rows, kRows))),
                  static_cast<unsigned>(ncols / nt));
  auto go = [&](auto ntc, auto uc, auto bc) {
    hipLaunchKernelGGL((conv_small_kernel<T, decltype(ntc)::value, decltype(uc)::value,
                                          decltype(bc)::value>),
                       grid, dim3(kThreads), 0, s, x, n_x, cred, w, wperm, ncols, bias, nbr, n_rows,
                       K, order, y);
  };
  using U4 = std::integral_constant<int, 4>;
  auto pick = [&](auto bc) {
    nt == 64   ? go(std::integral_constant<int, 64>{}, U4{}, bc)
    : nt == 32 ? go(std::integral_constant<int, 32>{}, U4{}, bc)
               : go(std::integral_constant<int, 16>{}, U4{}, bc);
  };
  if constexpr (std::is_same<T, float>::value) {
    if (by_channel) {
      pick(std::true_type{});
      RHIP_LAUNCH_CHECK();
      return;
    }
  }
  pick(std::false_type{});
  RHIP_LAUNCH_CHECK();
}

template bool conv_small_takes<float>(bool, int64_t, int64_t, int, int, int);
template bool conv_small_takes<__bf16>(bool, int64_t, int64_t, int, int, int);
template void conv_small<float>(const float *, int64_t, int, const float *, bool, const int32_t *,
                                int, const float *, const int32_t *, int64_t, int,
                                const int32_t *, float *, hipStream_t);
template void conv_small<__bf16>(const __bf16 *, int64_t, int, const __bf16 *, bool,
                                 const int32_t *, int, const float *, const int32_t *, int64_t,
                                 int, const int32_t *, __bf16 *, hipStream_t);

} // namespace rhip
