// fp32 forward and input gradient on the bf16 matrix cores: the
// output-stationary gather GEMM of conv_os_lds_kernel with each fp32 operand
// as the sum of three bf16 parts.
//
// A float is hi + mid + lo: hi rounds it to bf16 (8 bits), mid rounds the
// rest, lo is what is left. Of the nine products of two such sums the six
// largest are kept (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi); the dropped
// ones are under 2^-25 of the product, below the rounding of one fp32
// multiplication (the method: G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging
// the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019). All sums stay fp32 in the MFMA accumulators. Six
// v_mfma_f32_16x16x32_bf16 take 96 cycles for 32 channels where eight
// v_mfma_f32_16x16x4_f32 take 256. The error against 64-bit sums (2-norm, 3^3,
// normal / ReLU features) is below the fp32 MFMAs': 64->64 9.6e-8 / 7.9e-8
// against 3.8e-7 / 2.7e-7, 256->256 3.7e-7 / 3.0e-7 against 1.1e-6 / 7.5e-7.
//
// Both operands are split after a multiplication by 2^24, and the sums are
// multiplied by 2^-48. The parts of a float are multiples of its last bit, at
// least 2^-149, so scaled they are normal bf16 values, exact down to the
// smallest fp32 (unscaled, the later parts of a value below 2^-110 were bf16
// denormals that hold fewer bits: off by 9e-6 at 2^-118, 4e-2 at 2^-130).
// Where parts cannot represent a value or a scaled sum leaves fp32's range
// (infinities, NaN, operands of 2^103 and sums of 2^80 and more) some part or
// sum is not finite, and so is every output it reaches. A wave that holds such
// an output walks its stages once more on the fp32 matrix cores, each stage's
// products added only to the rows that have the neighbour, and takes from that
// the outputs that are not finite.
#include <algorithm>
#include <type_traits>

#include "conv_x3.hpp"

namespace rhip {

namespace {

constexpr int kMaxK = 128;

constexpr float kScale = 0x1p24f, kUnscale = 0x1p-48f; // operands, sums

struct Parts {
  v8bf hi, mid, lo;
};

// the three bf16 parts of eight floats times kScale
__device__ __forceinline__ Parts split8(const v4f &a, const v4f &b) {
  Parts p;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = (j < 4 ? a[j & 3] : b[j & 3]) * kScale;
    const __bf16 h = static_cast<__bf16>(v);
    const float r = v - static_cast<float>(h);
    const __bf16 m = static_cast<__bf16>(r);
    p.hi[j] = h;
    p.mid[j] = m;
    p.lo[j] = static_cast<__bf16>(r - static_cast<float>(m));
  }
  return p;
}

// Weights times kScale in three parts: wt[k][part][n][c'], the 32 channels of a step in
// the order the gathered rows come in: place 8g + j holds channel 4g + j of
// the step's first 16 for j < 4, else channel 4g + j - 4 of its second 16.
__global__ __launch_bounds__(kThreads) void x3_weights_kernel(const float *__restrict__ w, int wc,
                                                              int wn, int cred, int ncols,
                                                              int64_t total,
                                                              __bf16 *__restrict__ wt) {
  const int64_t i = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  if (i >= total)
    return;
  const int per = cred * ncols;
  const int64_t k = i / per;
  const int rem = static_cast<int>(i - k * per);
  const int n = rem / cred, cp = rem % cred;
  const int g = (cp & 31) >> 3, j = cp & 7;
  const int c = (cp & ~31) + 4 * g + (j < 4 ? j : 12 + j);
  const float v = w[k * per + c * wc + n * wn] * kScale;
  const __bf16 h = static_cast<__bf16>(v);
  const float r = v - static_cast<float>(h);
  const __bf16 m = static_cast<__bf16>(r);
  __bf16 *dst = wt + 3 * k * per + rem;
  dst[0] = h;
  dst[per] = m;
  dst[2 * per] = static_cast<__bf16>(r - static_cast<float>(m));
}

__device__ __forceinline__ bool finite(float v) { return v - v == 0.f; }

// The call's operands as they came (conv_x3).
struct Operands {
  const float *x, *w;
  int wc, wn;
  const int32_t *wperm, *nbr;
  int64_t n_rows;
  int K, cred, ncols;
};

// As conv_os_lds_kernel (indices of a wave's row groups in LDS, offsets
// walked as a bit mask, quad-order gathers, missing neighbours as loads past
// the buffer), RG 16-row groups per wave so that each weight fragment read
// from LDS (three parts, 1.5 times the bytes of fp32) serves RG groups.
// Bound by no single unit: on 410k rows, 64->64, the matrix pipes are busy 0.39
// of the time, the VALU 0.40, LDS 0.15 and 0.21 more in bank conflicts; of 284
// us (with one sum, operands not scaled) a variant without the gathers took
// 218, one without the split into parts 253, one with the hi hi product alone
// 172. Stages of 64 channels at 3 waves
// per SIMD took 293, one row group per wave 309-334, three or four 298.
template <int NT, int RG, int WAVES, int CW, int KQ, bool SPLIT>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(WAVES))) void
conv_x3_kernel(const float *__restrict__ x, int64_t n_x, const __bf16 *__restrict__ wt,
               const Operands ops, const float *__restrict__ bias, const int32_t *__restrict__ nbr,
               int64_t n_rows, int K, const int32_t *__restrict__ order, float *__restrict__ y,
               float *__restrict__ partial) {
  constexpr int CCH = 32; // channels per stage: one MFMA step
  constexpr int NCH = CW / CCH, CSUB = CCH / 16;
  constexpr int LDW = CCH + 8;
  constexpr int ROWS = kWaves * RG * 16;
  constexpr int NB = NT / 16;
  constexpr int PP = NT * (CCH / 8); // 16-byte pieces per staged part
  constexpr int NV = 3 * PP;
  constexpr int NPT = (NV + kThreads - 1) / kThreads;
  constexpr int MW = KQ / 8;
  static_assert(CW % CCH == 0 && CCH % 32 == 0 && KQ % 8 == 0, "whole chunks and steps");
  __shared__ __align__(16) __bf16 sB[3 * NT * LDW];
  __shared__ __align__(16) int32_t sK[kWaves][RG][KQ][kWave];
  __shared__ uint32_t smask[kWaves * RG][MW];

  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i16 = lane & 15;
  const int g = lane >> 4;
  const int ncols = ops.ncols;
  const int64_t tile0 = xcd_tile(blockIdx.x) * ROWS;
  if (tile0 >= n_rows)
    return; // padding workgroup (uniform)
  const int col0 = blockIdx.y * NT;

  uint32_t wmask[MW] = {};
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    const int64_t pos = tile0 + (wv * RG + r) * 16 + i16;
    const bool in = pos < n_rows;
    const int64_t pc = in ? pos : n_rows - 1;
#pragma unroll
    for (int mw = 0; mw < MW; ++mw) {
      int32_t v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int k = 32 * mw + 4 * q + g;
        v[q] = nbr[(k < K ? k : K - 1) * n_rows + pc] | ((in && k < K) ? 0 : -1);
      }
      uint32_t w = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        sK[wv][r][8 * mw + q][lane] = v[q];
        const uint64_t bal = __ballot(v[q] >= 0);
#pragma unroll
        for (int gg = 0; gg < 4; ++gg)
          w |= (((bal >> (16 * gg)) & 0xffffull) != 0 ? 1u : 0u) << (4 * q + gg);
      }
      w = __builtin_amdgcn_readfirstlane(w);
      wmask[mw] |= w;
      if (lane == 0)
        smask[wv * RG + r][mw] = w;
    }
  }
  __syncthreads();
  uint32_t m[MW] = {}; // the workgroup's offsets, walked in ascending order
#pragma unroll
  for (int mw = 0; mw < MW; ++mw) {
#pragma unroll
    for (int i = 0; i < kWaves * RG; ++i)
      m[mw] |= smask[i][mw];
    m[mw] = __builtin_amdgcn_readfirstlane(m[mw]);
  }
  auto lowest = [&]() {
    int k = 0;
#pragma unroll
    for (int mw = MW - 1; mw >= 0; --mw)
      if (m[mw])
        k = 32 * mw + __builtin_ctz(m[mw]);
    return k;
  };

  // the hi hi products, and the five small ones: the first sum then rounds
  // once per 32 channels, and the second's roundings are 2^-8 of that
  v4f acc[RG][NB], low[RG][NB];
#pragma unroll
  for (int r = 0; r < RG; ++r)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      acc[r][nb] = low[r][nb] = v4f{0.f, 0.f, 0.f, 0.f};

  const int rsel = lane >> 2;
  const int tsrc = quad_src(lane);
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(x, n_x * CW * static_cast<int64_t>(sizeof(float)));
  const uint32_t lane_byte = static_cast<uint32_t>((lane & 3) * 16);
  int cc = 0;
  auto advance = [&](int k) {
    if (++cc == NCH) {
      cc = 0;
      m[k >> 5] &= m[k >> 5] - 1;
    }
  };
  int left = 0;
  auto to_first = [&]() { // from all stages to this split's
    if constexpr (SPLIT) {
      left = 0;
#pragma unroll
      for (int mw = 0; mw < MW; ++mw)
        left += __builtin_popcount(m[mw]) * NCH;
      const int s_begin = static_cast<int>(static_cast<int64_t>(left) * blockIdx.z / gridDim.z);
      const int s_end = static_cast<int>(static_cast<int64_t>(left) * (blockIdx.z + 1) / gridDim.z);
      for (int i = 0; i < s_begin; ++i)
        advance(lowest());
      left = s_end - s_begin;
    }
  };
  uint32_t all[MW];
#pragma unroll
  for (int mw = 0; mw < MW; ++mw)
    all[mw] = m[mw];
  to_first();
  auto more = [&]() {
    if constexpr (SPLIT)
      return left > 0;
    uint32_t o = 0;
#pragma unroll
    for (int mw = 0; mw < MW; ++mw)
      o |= m[mw];
    return o != 0;
  };
  while (more()) {
    const int k = lowest(), ch = cc;
    advance(k);
    if constexpr (SPLIT)
      --left;
    uint32_t off[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      const int32_t id = sK[wv][r][k >> 2][(k & 3) * 16 + rsel];
      off[r] = pick_off(static_cast<uint32_t>(id) * static_cast<uint32_t>(CW * sizeof(float)) +
                            static_cast<uint32_t>(ch * CCH * sizeof(float)) + lane_byte,
                        ~(id >> 31));
    }
    const int kw = ops.wperm ? ops.wperm[k] : k;
    const __bf16 *wk = wt + (static_cast<int64_t>(kw) * 3 * ncols + col0) * CW + ch * CCH;
    uint4 wreg[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      const int li = min(static_cast<int>(threadIdx.x) + i * kThreads, NV - 1);
      const int part = li / PP, q = li % PP;
      wreg[i] = *reinterpret_cast<const uint4 *>(
          wk + (part * ncols + q / (CCH / 8)) * CW + (q % (CCH / 8)) * 8);
    }
    v4u a[RG][CSUB];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int sub = 0; sub < CSUB; ++sub)
        a[r][sub] = __builtin_bit_cast(
            v4u, __builtin_amdgcn_raw_buffer_load_b128(
                     rx, off[r] + static_cast<uint32_t>(sub * 64), 0, 0));
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      const int li = threadIdx.x + i * kThreads;
      const int part = li / PP, q = li % PP;
      if (NV % kThreads == 0 || li < NV)
        *reinterpret_cast<uint4 *>(
            &sB[(part * NT + q / (CCH / 8)) * LDW + (q % (CCH / 8)) * 8]) = wreg[i];
    }
    __syncthreads(); // the stage's weights are in LDS
    if ((wmask[k >> 5] >> (k & 31)) & 1u) { // uniform
#pragma unroll
      for (int st = 0; st < CCH / 32; ++st) {
        Parts p[RG];
#pragma unroll
        for (int r = 0; r < RG; ++r)
          p[r] = split8(__builtin_bit_cast(v4f, quad_to_mfma(a[r][2 * st], tsrc)),
                        __builtin_bit_cast(v4f, quad_to_mfma(a[r][2 * st + 1], tsrc)));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const __bf16 *pb = &sB[(nb * 16 + i16) * LDW + st * 32 + g * 8];
          const v8bf bh = *reinterpret_cast<const v8bf *>(pb);
          const v8bf bm = *reinterpret_cast<const v8bf *>(pb + NT * LDW);
          const v8bf bl = *reinterpret_cast<const v8bf *>(pb + 2 * NT * LDW);
          // smallest products first, the row groups' chains alternating
#pragma unroll
          for (int r = 0; r < RG; ++r)
            low[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[r].lo, bh, low[r][nb], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < RG; ++r)
            low[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[r].hi, bl, low[r][nb], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < RG; ++r)
            low[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[r].mid, bm, low[r][nb], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < RG; ++r)
            low[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[r].mid, bh, low[r][nb], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < RG; ++r)
            low[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[r].hi, bm, low[r][nb], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < RG; ++r)
            acc[r][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[r].hi, bh, acc[r][nb], 0, 0, 0);
        }
      }
    }
    __syncthreads(); // every wave is done reading the stage's weights
  }
#pragma unroll
  for (int r = 0; r < RG; ++r)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      acc[r][nb] = (acc[r][nb] + low[r][nb]) * kUnscale;

  float sum = 0.f; // NaN where an output is not finite (0 * v is NaN there)
#pragma unroll
  for (int r = 0; r < RG; ++r)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sum += 0.f * acc[r][nb][e];
  if (__any(!finite(sum))) { // uniform: those outputs from the operands in fp32
    v4f again[RG][NB];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        again[r][nb] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mw = 0; mw < MW; ++mw)
      m[mw] = all[mw];
    cc = 0;
    to_first();
    while (more()) {
      const int k = lowest(), ch = cc;
      advance(k);
      if constexpr (SPLIT)
        --left;
      if (!((wmask[k >> 5] >> (k & 31)) & 1u)) // uniform
        continue;
      const int kw = ops.wperm ? ops.wperm[k] : k;
      v4f b[NB][2]; // channels 16 sub + 4g .. 4g + 3 of the stage, column i16
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            b[nb][sub][e] = ops.w[static_cast<int64_t>(kw) * CW * ncols +
                                  (ch * CCH + 16 * sub + 4 * g + e) * ops.wc +
                                  (col0 + nb * 16 + i16) * ops.wn];
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const int32_t *ids = &sK[wv][r][k >> 2][(k & 3) * 16];
        const int32_t id = ids[i16];
        const uint32_t off = pick_off(
            static_cast<uint32_t>(id) * static_cast<uint32_t>(CW * sizeof(float)) +
                static_cast<uint32_t>(ch * CCH * sizeof(float)) + static_cast<uint32_t>(16 * g),
            ~(id >> 31));
        const int4 has = *reinterpret_cast<const int4 *>(ids + 4 * g); // rows 4g .. 4g + 3
        v4f a[2];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
          a[sub] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                               rx, off + static_cast<uint32_t>(sub * 64), 0, 0));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          v4f t = again[r][nb];
          Mfma<float>::mma(a[0], b[nb][0], t);
          Mfma<float>::mma(a[1], b[nb][1], t);
          again[r][nb] = v4f{has.x >= 0 ? t[0] : again[r][nb][0],
                             has.y >= 0 ? t[1] : again[r][nb][1],
                             has.z >= 0 ? t[2] : again[r][nb][2],
                             has.w >= 0 ? t[3] : again[r][nb][3]};
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[r][nb][e] = finite(acc[r][nb][e]) ? acc[r][nb][e] : again[r][nb][e];
  }

  if constexpr (SPLIT) { // [split][position][column]
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t pos = tile0 + (wv * RG + r) * 16 + 4 * g + e;
        if (pos < n_rows) {
          float *dst = partial + (blockIdx.z * n_rows + pos) * ncols + col0 + i16;
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            dst[nb * 16] = acc[r][nb][e];
        }
      }
    return;
  }
#pragma unroll
  for (int r = 0; r < RG; ++r) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t pos = tile0 + (wv * RG + r) * 16 + 4 * g + e;
      if (pos < n_rows) {
        const int64_t o = order ? order[pos] : pos;
        float *dst = y + o * ncols + col0 + i16;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          float v = acc[r][nb][e];
          if (bias)
            v += bias[col0 + nb * 16 + i16];
          __builtin_nontemporal_store(v, &dst[nb * 16]); // as conv_os_lds_kernel's
        }
      }
    }
  }
}

// The split form's sums in split order, with the bias.
__global__ __launch_bounds__(kThreads) void x3_reduce_kernel(const float *__restrict__ partial,
                                                             int splits, int64_t n_rows, int ncols,
                                                             const float *__restrict__ bias,
                                                             const int32_t *__restrict__ order,
                                                             float *__restrict__ y) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  const int q = ncols / 4;
  const int64_t pos = t / q;
  if (pos >= n_rows)
    return;
  const int c = static_cast<int>(t - pos * q) * 4;
  v4f a = *reinterpret_cast<const v4f *>(partial + pos * ncols + c);
#pragma unroll 4
  for (int z = 1; z < splits; ++z)
    a += *reinterpret_cast<const v4f *>(partial + (z * n_rows + pos) * ncols + c);
  if (bias)
    a += v4f{bias[c], bias[c + 1], bias[c + 2], bias[c + 3]};
  *reinterpret_cast<v4f *>(y + (order ? order[pos] : pos) * ncols + c) = a;
}

int x3_nt(int ncols) { return ncols % 64 == 0 ? 64 : 32; }

// 16-row groups per wave: two share each weight fragment; one where a
// stencil's indices (8 KB of LDS per group and 32 offsets) would leave too
// few workgroups per CU.
constexpr int x3_rg(int K) { return K <= 32 ? 2 : 1; }

template <int NT, int CW, int KQ>
void launch(dim3 grid, bool split, const float *x, int64_t n_x, const __bf16 *wt,
            const Operands &ops, const float *bias, const int32_t *order, float *y, float *partial,
            hipStream_t s) {
  constexpr int RG = x3_rg(4 * KQ), W = RG == 2 ? 4 : 3;
  if (split)
    hipLaunchKernelGGL((conv_x3_kernel<NT, RG, W, CW, KQ, true>), grid, dim3(kThreads), 0, s, x,
                       n_x, wt, ops, bias, ops.nbr, ops.n_rows, ops.K, order, y, partial);
  else
    hipLaunchKernelGGL((conv_x3_kernel<NT, RG, W, CW, KQ, false>), grid, dim3(kThreads), 0, s, x,
                       n_x, wt, ops, bias, ops.nbr, ops.n_rows, ops.K, order, y, nullptr);
}

} // namespace

// Narrow layers stay on the fp32 MFMAs: at 32 reduced channels or 16 to 48
// columns a stage's multiplies are few against its loads and index work, and
// fp32 stages half the bytes. Measured on MI355X, forward, fp32 MFMA against
// this kernel: 64->64 on 410k rows 379 / 291 us, on 48k rows 82 / 68, on 10k
// 43 / 33, on 2k 24 / 25; 96->96 on 101k rows 339 / 260; 128->128 on 10k rows
// 120 / 79; 256->256 on 2k rows 122 / 84; 81 offsets, 64->64, 233k rows 1007 /
// 718; but 32->32 on 200k rows 70 / 67, 64->32 on 200k rows 121 / 125, 64->16
// on 101k rows 46 / 70. (Scaling the operands came after these and costs 1 to
// 3 %: 64->64 on 410k rows 293, 256->256 on 48k 743 -> 758.) The width is a
// template argument, of which each value adds 12 kernels; the five are those
// that networks have most, and other multiples of 32 (160, 224, 320 and on)
// stay on the fp32 MFMAs, where they were not compared.
//
// 32-column tiles split every row's operand again per tile: reductions that
// the fp32 kernel has whole 64-channel stages for take them on maps of up to
// 20,480 rows, where the splits below fill the chip (64->96 on 10k rows 46
// against 45 us on the fp32 MFMAs, 128->96 71 / 89, 256->160 193 / 221; on 29k
// rows 81 / 72, 144 / 140, 499 / 412). 96 and 192 channels it has not.
//
// Maps of up to 8 offsets with about one pair per row of the finer side
// (stride-2 maps, their transposes, 1^D): the staged weights serve few
// products. Measured on stride-2 maps, fp32 MFMA / this kernel: reductions of
// 64 channels never gained (64->64 on 48k rows 14 / 17-24 us, transposed; 64->128
// to 24k rows 27 / 32); the rest gain from about 4e8 pairs x channels x
// columns (192->192 from 15,770 rows 38 / 33, 96->192 from 23k 33 / 28;
// 128->128 from 23k 26.5 / 27), with one neighbour per row also from 40k rows
// only (256->128 to 37k rows 36 / 40, to 48k 43 / 39), or, in the forward, for
// which the fp32 kernel needs a transposed copy, from 20k to 192 columns and
// more (192->192 to 23k 37 / 33, but dX 96->192 21 / 27).
bool conv_x3_takes(bool forward, int cred, int ncols, int K, int64_t n_x, int64_t n_rows) {
  const bool width = cred == 64 || cred == 96 || cred == 128 || cred == 192 ||
                     cred == 256;
  if (!width || ncols < 64 || ncols % 32 != 0 || K > kMaxK || n_x < 1 ||
      n_x * cred * static_cast<int64_t>(sizeof(float)) > kBufMaxBytes)
    return false;
  if (ncols % 64 != 0 && cred % 64 == 0 && cred != 192 && n_rows > 20480)
    return false;
  const int64_t fine = std::max(n_x, n_rows);
  if (K <= 8 && K * std::min(n_x, n_rows) < 4 * fine) // under two pairs a row at best
    return cred > 64 && fine * cred * ncols >= 400'000'000 &&
           (n_rows <= n_x || n_rows >= 40000 || (forward && ncols >= 192 && n_rows >= 20000));
  return true;
}

int conv_x3_splits(int64_t n_rows, int cred, int ncols, int K) {
  if (n_rows <= 0 || ncols % 32 != 0)
    return 1;
  // a 32-column tile is half the work of a 64-column one
  const int64_t blocks = std::max<int64_t>(
      1, ceil_div(n_rows, kWaves * x3_rg(K) * 16) * (ncols / 32) / 2);
  const int64_t stages = static_cast<int64_t>(K) * (cred / 32);
  const int64_t want = (640 + blocks / 2) / blocks; // nearest
  return static_cast<int>(
      std::max<int64_t>(1, std::min<int64_t>({16, want, std::max<int64_t>(1, stages / 8)})));
}

void conv_x3(const float *x, int64_t n_x, int cred, const float *w, int wc, int wn,
             const int32_t *wperm, int ncols, const float *bias, const int32_t *nbr,
             int64_t n_rows, int K, const int32_t *order, float *y, void *wt, float *partial,
             size_t partial_floats, hipStream_t s) {
  if (n_rows == 0)
    return;
  __bf16 *w3 = static_cast<__bf16 *>(wt);
  const int64_t total = static_cast<int64_t>(K) * cred * ncols;
  hipLaunchKernelGGL(x3_weights_kernel, dim3(static_cast<unsigned>(ceil_div(total, kThreads))),
                     dim3(kThreads), 0, s, w, wc, wn, cred, ncols, total, w3);
  RHIP_LAUNCH_CHECK();
  const Operands ops{x, w, wc, wn, wperm, nbr, n_rows, K, cred, ncols};
  int splits = conv_x3_splits(n_rows, cred, ncols, K);
  if (partial == nullptr || partial_floats / (static_cast<size_t>(n_rows) * ncols) <
                                static_cast<size_t>(splits))
    splits = 1;
  const int nt = x3_nt(ncols);
  const dim3 grid(static_cast<unsigned>(xcd_grid(ceil_div(n_rows, kWaves * x3_rg(K) * 16))),
                  static_cast<unsigned>(ncols / nt), static_cast<unsigned>(splits));
  auto go = [&](auto ntc, auto cwc, auto kqc) {
    launch<decltype(ntc)::value, decltype(cwc)::value, decltype(kqc)::value>(
        grid, splits > 1, x, n_x, w3, ops, bias, order, y, partial, s);
  };
  auto pick_k = [&](auto ntc, auto cwc) {
    K <= 32   ? go(ntc, cwc, std::integral_constant<int, 8>{})
    : K <= 96 ? go(ntc, cwc, std::integral_constant<int, 24>{})
              : go(ntc, cwc, std::integral_constant<int, 32>{});
  };
  auto pick_c = [&](auto ntc) {
    switch (cred) {
    case 64: pick_k(ntc, std::integral_constant<int, 64>{}); break;
    case 96: pick_k(ntc, std::integral_constant<int, 96>{}); break;
    case 128: pick_k(ntc, std::integral_constant<int, 128>{}); break;
    case 192: pick_k(ntc, std::integral_constant<int, 192>{}); break;
    default: pick_k(ntc, std::integral_constant<int, 256>{}); break;
    }
  };
  nt == 64 ? pick_c(std::integral_constant<int, 64>{})
           : pick_c(std::integral_constant<int, 32>{});
  RHIP_LAUNCH_CHECK();
  if (splits > 1) {
    hipLaunchKernelGGL(x3_reduce_kernel,
                       dim3(static_cast<unsigned>(ceil_div(n_rows * (ncols / 4), kThreads))),
                       dim3(kThreads), 0, s, partial, splits, n_rows, ncols, bias, order, y);
    RHIP_LAUNCH_CHECK();
  }
}

} // namespace rhip
