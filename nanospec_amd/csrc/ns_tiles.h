// Pieces shared by the kernels in which one wave holds 32 tokens x 128 vocab entries of a 256 x 256
// logits tile (thin.hip, emit.hip): lane 32 h + r holds token r's entries 8 k + 4 h .. + 3 of
// chunk k = 0..15, as an accumulator of v_mfma_f32_32x32x16_bf16 leaves them.
#pragma once

#include "ns_gemm.h"
#include "ns_internal.h"

namespace ns {

// LDS image of a wave's 32 rows of 128 entries (teacher, Markov or output rows), written or read
// as whole row pieces and taken chunk by chunk (8 entries).  bf16: 256-byte rows, chunk c at
// c ^ (row & 15), the 8-byte halves of rows 16-31 swapped, so the 32 lanes of a read cover every
// bank once.  fp32: 512-byte rows of 16-byte quads, quad q at q ^ (row & 31).
template <typename TT>
struct Rows;
template <>
struct Rows<uint16_t> {
  static constexpr int kBytes = 32 * 256;
  static constexpr int kLoads = 8;        // 16-byte pieces per lane
  static constexpr int kPer = 8;          // entries per piece
  static __device__ __forceinline__ int row(int i, int lane) { return 4 * i + (lane >> 4); }
  static __device__ __forceinline__ int piece(int lane) { return lane & 15; }
  static __device__ __forceinline__ void put(lds_t* b, int i, int lane, u32x4_t x) {
    const int r = row(i, lane), c = piece(lane);
    if (i >= 4) x = u32x4_t{x[2], x[3], x[0], x[1]};
    *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>(b + r * 256 + ((c ^ (r & 15)) << 4)) = x;
  }
  // byte offset of entries 8 k + 4 h .. + 3 of row r
  static __device__ __forceinline__ int off(int k, int r, int h) {
    return r * 256 + ((k ^ (r & 15)) << 4) + 8 * (h ^ (r >> 4));
  }
  static __device__ __forceinline__ void get(const lds_t* b, int k, int r, int h, float* u) {
    const u32x2_t x = *reinterpret_cast<const __attribute__((address_space(3))) u32x2_t*>(b + off(k, r, h));
    u[0] = bf16_lo(x[0]); u[1] = bf16_hi(x[0]);
    u[2] = bf16_lo(x[1]); u[3] = bf16_hi(x[1]);
  }
  // dl chunk c of row r
  static __device__ __forceinline__ u32x4_t out(const lds_t* b, int r, int c) {
    const u32x4_t x = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(b + r * 256 + ((c ^ (r & 15)) << 4));
    return r >= 16 ? u32x4_t{x[2], x[3], x[0], x[1]} : x;
  }
};
template <>
struct Rows<float> {
  static constexpr int kBytes = 32 * 512;
  static constexpr int kLoads = 16;
  static constexpr int kPer = 4;
  static __device__ __forceinline__ int row(int i, int lane) { return 2 * i + (lane >> 5); }
  static __device__ __forceinline__ int piece(int lane) { return lane & 31; }
  static __device__ __forceinline__ void put(lds_t* b, int i, int lane, u32x4_t x) {
    const int r = row(i, lane), q = piece(lane);
    *reinterpret_cast<__attribute__((address_space(3))) u32x4_t*>(b + r * 512 + ((q ^ r) << 4)) = x;
  }
  static __device__ __forceinline__ int off(int k, int r, int h) { return r * 512 + (((2 * k + h) ^ r) << 4); }
  static __device__ __forceinline__ void get(const lds_t* b, int k, int r, int h, float* u) {
    const u32x4_t x = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t*>(b + off(k, r, h));
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = __uint_as_float(x[e]);
  }
  static __device__ __forceinline__ u32x4_t out(const lds_t* b, int r, int c) {
    const u32x2_t lo = *reinterpret_cast<const __attribute__((address_space(3))) u32x2_t*>(b + off(c, r, 0));
    const u32x2_t hi = *reinterpret_cast<const __attribute__((address_space(3))) u32x2_t*>(b + off(c, r, 1));
    return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
  }
};

// LDS written by some lanes of a wave, read by others of the same wave
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ PairState half_merge(const PairState& s) {
  PairState a, b;
  half_pair(s.mz, a.mz, b.mz);
  half_pair(s.sz, a.sz, b.sz);
  half_pair(s.mu, a.mu, b.mu);
  half_pair(s.su, a.su, b.su);
  half_pair(s.A, a.A, b.A);
  return pair_merge(a, b);
}

__device__ __forceinline__ LseState half_merge(const LseState& s) {
  LseState a, b;
  half_pair(s.m, a.m, b.m);
  half_pair(s.s, a.s, b.s);
  return lse_merge(a, b);
}

// One distribution's online (max, sum-exp) over W values.
template <int W>
__device__ __forceinline__ void lse_update(LseState& st, const float* z) {
  float b = z[0];
#pragma unroll
  for (int i = 1; i < W; ++i) b = fmaxf(b, z[i]);
  const float m = fmaxf(st.m, b);
  const float ml = m * kLog2e;
  float s = st.s * fast_exp2((st.m - m) * kLog2e);
#pragma unroll
  for (int i = 0; i < W; ++i) s += fast_exp2(__builtin_fmaf(z[i], kLog2e, -ml));
  st = {m, s};
}

}  // namespace ns
