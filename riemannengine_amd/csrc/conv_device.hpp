// Device helpers shared by the convolution's translation units: MFMA
// operands, conversions, raw buffer loads and the LDS transpose read.
#pragma once

#include "rhip_internal.hpp"

namespace rhip {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// LDS transpose read: within a 16-lane group, lane i receives the (i % 4)-th
// 16-bit element at the address of lane 4e + i/4 as element e.
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

__device__ __forceinline__ v4s ds_read_tr16(const void *p) {
  // generic LDS pointer -> LDS address space (the low 32 bits are the offset)
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      reinterpret_cast<lds_v4s *>(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p))));
}

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
template <typename T> struct Mfma;

// v_mfma_f32_16x16x4_f32: lane l supplies A[l%16][l/16], B[l/16][l%16];
// D[4*(l/16)+e][l%16] lands in element e. A 16-byte lane load covers four
// consecutive channels, consumed by four MFMAs.
template <> struct Mfma<float> {
  static constexpr int kCh = 16; // channels per wave-wide 16-byte load
  using Frag = v4f;
  __device__ static __forceinline__ Frag load(const float *p) {
    return *reinterpret_cast<const v4f *>(p);
  }
  __device__ static __forceinline__ Frag zero() { return v4f{0.f, 0.f, 0.f, 0.f}; }
  // v where keep, else zeros (bitwise, so the load it masks stays unconditional)
  __device__ static __forceinline__ Frag mask(const Frag &v, bool keep) {
    const uint32_t m = keep ? ~0u : 0u;
    uint4 u = __builtin_bit_cast(uint4, v);
    u.x &= m, u.y &= m, u.z &= m, u.w &= m;
    return __builtin_bit_cast(Frag, u);
  }
  __device__ static __forceinline__ void mma(const Frag &a, const Frag &b, v4f &c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], c, 0, 0, 0);
  }
};

// v_mfma_f32_16x16x32_bf16 (gfx950): lane l supplies eight consecutive
// reduction elements of row l%16 (A) / column l%16 (B), group l/16.
template <> struct Mfma<__bf16> {
  static constexpr int kCh = 32;
  using Frag = v8bf;
  __device__ static __forceinline__ Frag load(const __bf16 *p) {
    return *reinterpret_cast<const v8bf *>(p);
  }
  __device__ static __forceinline__ Frag zero() {
    return __builtin_bit_cast(v8bf, uint4{0u, 0u, 0u, 0u});
  }
  __device__ static __forceinline__ void mma(const Frag &a, const Frag &b, v4f &c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  // v where keep, else zeros (bitwise, so the load it masks stays unconditional)
  __device__ static __forceinline__ Frag mask(const Frag &v, bool keep) {
    const uint32_t m = keep ? ~0u : 0u;
    uint4 u = __builtin_bit_cast(uint4, v);
    u.x &= m, u.y &= m, u.z &= m, u.w &= m;
    return __builtin_bit_cast(Frag, u);
  }
};

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(__bf16 v) { return static_cast<float>(v); }
template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ __bf16 from_f32<__bf16>(float v) {
  return static_cast<__bf16>(v);
}

// Raw buffer loads (stride 0): a load at a byte offset at or past the
// buffer's size returns zero without a memory access, so an absent row needs
// no predicate. Kernels put such offsets at kBufOob, past every buffer they
// make (host code keeps buffers below kBufMaxBytes).
constexpr uint32_t kBufOob = 0x80000000u;
constexpr int64_t kBufMaxBytes = (int64_t(1) << 31) - 256; // offsets stay below kBufOob

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, static_cast<int>(bytes),
                                           0x00020000);
}

// A value the optimiser cannot see through: keeps `load | mask` a bitwise
// OR instead of a select that would become a branch around the load.
__device__ __forceinline__ int32_t opaque(int32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// off where keep is all ones, else kBufOob (keep is 0 or -1)
__device__ __forceinline__ uint32_t pick_off(uint32_t off, int32_t keep) {
  return (off & static_cast<uint32_t>(keep)) | (kBufOob & ~static_cast<uint32_t>(keep));
}

// Gathered rows in quad order. The L1 serves a vector load four lanes at a
// time and looks up one cache line per distinct line among them; in the MFMA
// operand layout (lane (i16, g): row i16, bytes 16g..16g+15 of a 64-byte
// slice) the four lanes of a quad hold four rows, so every lane costs an
// access. Loading lane 4m + c with row m's bytes 16c..16c+15 instead makes
// each quad one 64-byte access (a quarter of the accesses); quad_to_mfma
// then moves lane 4m + c's 16 bytes to lane 16c + m with four ds_bpermute.
__device__ __forceinline__ int quad_src(int lane) { return (4 * (lane & 15) + (lane >> 4)) * 4; }

__device__ __forceinline__ v4u quad_to_mfma(const v4u &v, int src) {
  v4u o;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    o[d] = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int32_t>(v[d])));
  return o;
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

} // namespace rhip
