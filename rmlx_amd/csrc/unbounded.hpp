// Results of rows with infinities, over again (the GEMVs whose offsets and biases of both signs make a NaN of an infinite activation, (1024 + q) inf -
// 1024 inf, where the sum of the products is an infinity; f32 and bf16 values past the range of f16 are infinities here too).
#pragma once
#include "q4_stream.hpp"

namespace rmlx {
namespace q4 {

// 8 activations as the products take them
__device__ __forceinline__ h8 x_piece(const char* x, int32_t x_dtype, uint32_t k) {
  if (x_dtype == RMLX_DTYPE_F32) {
    h8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (_Float16)reinterpret_cast<const float*>(x)[k + e];
    return v;
  }
  const u4 d = *reinterpret_cast<const u4*>(x + k * 2);
  return __builtin_bit_cast(h8, x_dtype == RMLX_DTYPE_BF16 ? bf16x8_to_f16(d) : d);
}
// (scale * q + bias) * x of a row in f32, over n pieces of 8: those that the list names, or all of them.
template <int BITS>
__device__ __forceinline__ float plain_sum(uint32_t gs_log2, const char* w, const __half* s, const __half* b, const char* x, int32_t x_dtype, const uint16_t* list, uint32_t n) {
  float sum = 0.f;
#pragma unroll 1
  for (uint32_t i = 0; i < n && sum == sum; ++i) {
    const uint32_t k = (list != nullptr ? list[i] : i) * 8;
    const float sc = (float)s[k >> gs_log2], bi = (float)b[k >> gs_log2];
    const h8 v = x_piece(x, x_dtype, k);
    const uint32_t* q = reinterpret_cast<const uint32_t*>(w + k * BITS / 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t v_q = BITS == 4 ? q[0] >> (4 * e) & 15u : q[e >> 2] >> (8 * (e & 3)) & 255u;
      sum = fmaf(fmaf((float)v_q, sc, bi), (float)v[e], sum);
    }
  }
  return sum;
}
// The pieces of a row that hold a value that is not finite, into the wave's list (K / 8 places); their number.
__device__ __forceinline__ uint32_t odd_pieces(const char* x, int32_t x_dtype, uint32_t K, uint32_t lane, uint16_t* list) {
  uint32_t n = 0;
#pragma unroll 1
  for (uint32_t k = 0; k < K; k += 512) {
    bool odd = false;
    if (k + lane * 8 < K) {
      const h8 v = x_piece(x, x_dtype, k + lane * 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) odd = odd || !__builtin_isfinite((float)v[e]);
    }
    const uint64_t mask = __builtin_amdgcn_ballot_w64(odd);
    if (odd) list[n + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0))] = (uint16_t)(k / 8 + lane);
    n += (uint32_t)__builtin_popcountll(mask);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  return n;
}

}  // namespace q4
}  // namespace rmlx
