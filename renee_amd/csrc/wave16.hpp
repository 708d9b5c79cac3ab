// What the kernels for few rows (small_step.hpp, back_step.hpp) share: 16x16x32 MFMAs on fragments that cross from one layout
// to another through the LDS, and exchanges between lanes eight apart.
#pragma once
#include "pipe_core.hpp"

namespace xfc {

struct Wave16 {
  // The wave's own LDS operations are over; and the workgroup's, with no wait for vector memory.
  static __device__ __forceinline__ void lds_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
  static __device__ __forceinline__ void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
  // Transposing read of a [k][32] image: lane t of each 16 supplies 4 columns of row t / 4 and receives column t of 4 rows.
  static __device__ __forceinline__ half8 read_tr(const half_t* base, int k, int col) {
    const fp16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((XFC_LDS fp16x4_t*)(base + k * 32 + col));
    const fp16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((XFC_LDS fp16x4_t*)(base + (k + 4) * 32 + col));
    half8 f;
#pragma unroll
    for (int e = 0; e < 4; ++e) { f[e] = (half_t)lo[e]; f[4 + e] = (half_t)hi[e]; }
    return f;
  }
  static __device__ __forceinline__ float4v mfma(const half8& a, const half8& b, const float4v& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  // v (16 bytes) of the lane eight away in its row of sixteen; and one of two
  template <class V>
  static __device__ __forceinline__ V across8(const V& v) {
    uint4v q = __builtin_bit_cast(uint4v, v);
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)q[e], 0x128, 0xf, 0xf, true);  // row_ror:8
    return __builtin_bit_cast(V, q);
  }
  template <class V>
  static __device__ __forceinline__ V pick(bool first, const V& x, const V& y) {
    uint4v p = __builtin_bit_cast(uint4v, x);
    const uint4v q = __builtin_bit_cast(uint4v, y);
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = first ? p[e] : q[e];
    return __builtin_bit_cast(V, p);
  }
};

}  // namespace xfc
