// Pieces that the MFMA tile GEMMs (qmm_tile.hip, qmm_slice.hip, qmm_twin.hip) share: direct loads into LDS, weight unpacking, tile order.
#pragma once
#include "common.hpp"

namespace rmlx {

struct TileParams {
  const uint32_t* w; const __half* s; const __half* b;
  const uint32_t* w1; const __half* s1; const __half* b1;  // pair: the up matrix
  const __half* x; void* out;
  float* partial;                   // not null: f32 partial sums [splits, M, N]
  uint32_t M, N, K, group_size, tiles_m, tiles_n, splits;
  uint32_t tile_rows;               // rows of a row tile (not of a table's)
  int32_t exact, out_f32, epi_kind, epi_dtype;
  const void* epi;
  // grouped: (expert, first row, rows) per row tile, their number, optional gather of the activation rows, strides per expert
  const uint32_t* tile_tab; const uint32_t* n_tiles; const uint32_t* row_map;
  uint32_t x_rows;
  uint64_t estride_w, estride_s;    // u32 words / halves
};
// The GEMM with waves along k (qmm_slice.hip), for the plans that have four or more (kw)
void launch_qmm_slice(const TileParams& p, uint32_t bits, const TilePlan& plan, dim3 grid, hipStream_t s);
// The GEMM of two workgroups per CU (qmm_twin.hip): tiles of 256 (wn = 8) or 128 columns (wn = 4; not for a pair)
void launch_qmm_twin(const TileParams& p, uint32_t bits, uint32_t wn, dim3 grid, hipStream_t s);

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
struct __attribute__((packed, aligned(2))) u4_any { u4 v; };  // 16 bytes at any even address
struct __attribute__((packed, aligned(2))) u2_any { u2 v; };
struct __attribute__((packed, aligned(2))) h4_any { h4 v; };
struct __attribute__((packed, aligned(4))) f4_any { f4 v; };

__device__ __forceinline__ uint32_t h2bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

constexpr uint32_t kOutside = 0xC0000000u;  // an offset past every buffer (at most 2 GiB): the load returns zero

// 16 (4) bytes per lane from buffer r at byte offset off straight into LDS at lds + 16 (4) * lane
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t off, u4 r) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(off), "s"(r) : "memory", "m0");
}
// the same to base + at and from a uniform byte offset on top
template <uint32_t AT>
__device__ __forceinline__ void dma16_at(uint32_t base, uint32_t off, u4 r, uint32_t more) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(base), "v"(off), "s"(r), "s"(more), "n"(AT)
               : "memory", "scc", "m0");
}
// the same where `cond` (uniform) is not zero; the branch stays inside, so that the loop body remains one block for the scheduler
__device__ __forceinline__ void dma16_if(uint32_t cond, uint32_t lds, uint32_t off, u4 r) {
  asm volatile(
      "s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 .Ldma_skip_%=\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n"
      ".Ldma_skip_%=:" ::"s"(lds), "v"(off), "s"(r), "s"(cond) : "memory", "scc", "m0");
}
template <int N>
__device__ __forceinline__ void wait_dma_and_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
__device__ __forceinline__ u4 rsrc(const void* base, uint64_t bytes) {
  const uint64_t a = (uint64_t)base;
  return (u4){uni((uint32_t)a), uni((uint32_t)(a >> 32)), uni((uint32_t)(bytes > 0x80000000ull ? 0x80000000ull : bytes)), 0x00020000u};
}

// 8 Q4 values of one word -> 8 f16 weights in natural order.  As an e4m3 byte a value below 16 is q / 512 whatever its bits
// (denormal below 8, first exponent from 8 on), so one scaled conversion makes two of them f16, exactly: 13 vector instructions a
// word against 16 with magic-number pairs.
__device__ __forceinline__ h8 weights_q4(uint32_t w, h2 s2, h2 b2) {
  const uint32_t even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
  const uint32_t lo = __builtin_amdgcn_perm(odd, even, 0x05010400u), hi = __builtin_amdgcn_perm(odd, even, 0x07030602u);
  u4 o;
  o.x = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, false) * s2 + b2);
  o.y = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, true) * s2 + b2);
  o.z = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, false) * s2 + b2);
  o.w = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, true) * s2 + b2);
  return __builtin_bit_cast(h8, o);
}
// 8 Q8 values of two words (0x6400 | q is 1024 + q)
__device__ __forceinline__ h8 weights_q8(uint32_t w0, uint32_t w1, h2 s2, h2 b2) {
  const h2 k = {(_Float16)1024.0f, (_Float16)1024.0f};
  u4 o;
  o.x = h2bits((__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u)) - k) * s2 + b2);
  o.y = h2bits((__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u)) - k) * s2 + b2);
  o.z = h2bits((__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u)) - k) * s2 + b2);
  o.w = h2bits((__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u)) - k) * s2 + b2);
  return __builtin_bit_cast(h8, o);
}

// v (the sums of columns c .. c + 3 of a row, `left` of them inside the matrix; o = offset of the first in the output) through the fused
// epilogue: residual add / SwiGLU gate in f32 (quantized.rs:3206-3246).  A lane reads its own outputs' 8 (f32: 16) bytes of the
// operand where it stores the tile; the output may be the operand.  Residual, f16, against f32 sums of the whole output and a second
// kernel: 3001 x 14336 x 4096 406 -> 356 us (without an epilogue 321) and no workspace, 2048 x 4096 x 4096 88 -> 75, 128 x 4096 x 4096
// 15.5 -> 11.8.
__device__ __forceinline__ void tile_epilogue(const TileParams& p, uint64_t o, uint32_t left, f4& v) {
  f4 g = {0.f, 0.f, 0.f, 0.f};
  if (p.epi_dtype == RMLX_DTYPE_F32) {
    const float* q = static_cast<const float*>(p.epi) + o;
    if (left >= 4) g = reinterpret_cast<const f4_any*>(q)->v;
    else
      for (uint32_t e = 0; e < left; ++e) g[e] = q[e];
  } else {
    const _Float16* q = static_cast<const _Float16*>(p.epi) + o;
    if (left >= 4) {
      const h4 w = reinterpret_cast<const h4_any*>(q)->v;
#pragma unroll
      for (int e = 0; e < 4; ++e) g[e] = (float)w[e];
    } else {
      for (uint32_t e = 0; e < left; ++e) g[e] = (float)q[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = p.epi_kind == EPI_RESIDUAL ? v[e] + g[e] : g[e] / (1.0f + __expf(-g[e])) * v[e];
}

// The operand of a k step: weights rounded to f16 (lo unused), or, EXACT, w = scale * q + bias rounded once to f32 and cut into hi + lo
// of 11 bits each, multiplied one after the other (hi towards zero, so that both have one sign; 21 to 22 bits of the weight are kept, of
// weights below 2^-4 the bits down to 2^-24; beyond 131008 the low part overflows).  Costs 16 vector instructions a word and a product per fragment on top:
// 64 rows, 33001 x 2880 47.4 against 35.8 us, 2000 x 20001 x 4096 566 against 341 us; error against 64 bits 2.07e-4 of the result, that of
// rounding it, against 2.75e-4 (E = 16, top-2 experts: 2.2e-4 against 4.4e-4).
struct Weights { h8 hi, lo; };
__device__ __forceinline__ void split_pair(float w0, float w1, h2* hi, h2* lo) {
  const h2 h = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(w0, w1));
  // (-1 from a register that the compiler does not know: w - hi is then one instruction of mixed precision a value, not a conversion, a
  // subtraction and a half)
  float minus;
  asm("s_mov_b32 %0, -1.0" : "=s"(minus));
  *hi = h;
  *lo = (h2){(_Float16)__builtin_fmaf((float)h[0], minus, w0), (_Float16)__builtin_fmaf((float)h[1], minus, w1)};
}
__device__ __forceinline__ Weights split_q4(uint32_t w, float s, float b) {
  const uint32_t even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
  const uint32_t v[2] = {__builtin_amdgcn_perm(odd, even, 0x05010400u), __builtin_amdgcn_perm(odd, even, 0x07030602u)};
  typedef float f2 __attribute__((ext_vector_type(2)));
  Weights o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f2 q = i % 2 == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(v[i / 2], 512.0f, false) : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(v[i / 2], 512.0f, true);
    h2 hi, lo;
    split_pair(__builtin_fmaf(q.x, s, b), __builtin_fmaf(q.y, s, b), &hi, &lo);
    o.hi[2 * i] = hi[0]; o.hi[2 * i + 1] = hi[1]; o.lo[2 * i] = lo[0]; o.lo[2 * i + 1] = lo[1];
  }
  return o;
}
__device__ __forceinline__ Weights split_q8(uint32_t w0, uint32_t w1, float s, float b) {
  Weights o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = i < 2 ? w0 : w1;
    const float q0 = (float)((w >> (i % 2 * 16)) & 0xFFu), q1 = (float)((w >> (i % 2 * 16 + 8)) & 0xFFu);
    h2 hi, lo;
    split_pair(__builtin_fmaf(q0, s, b), __builtin_fmaf(q1, s, b), &hi, &lo);
    o.hi[2 * i] = hi[0]; o.hi[2 * i + 1] = hi[1]; o.lo[2 * i] = lo[0]; o.lo[2 * i + 1] = lo[1];
  }
  return o;
}

struct Tile { uint32_t mt, nt, split, expert, row_lo, rows; bool zeros; };
// Tile of this workgroup; false past the last.
template <uint32_t kBlock>
__device__ __forceinline__ bool tile_of(const TileParams& p, uint32_t tile_rows, Tile* out) {
  // An XCD (workgroup id % 8) takes a run of tiles, in blocks of up to four row tiles by all column tiles; a pair, which is always a grouped launch,
  // row tile by row tile: the activations then stay in the XCD's L2 while the weights, of another expert for nearly every row tile, pass through
  // once (128 experts of 1536 x 4096, 2048 tokens 890 -> 883 us, 512 tokens 474 -> 467; 45 experts of 2048 x 2048, 3503 tokens of 4 picks 513 -> 506).
  const uint32_t tiles_m = p.tile_tab != nullptr ? uni(*p.n_tiles) : p.tiles_m, total = tiles_m * p.tiles_n * p.splits, pid = blockIdx.x;
  if (pid >= total) return false;
  const uint32_t xcd = pid & 7, per = total >> 3, rem = total & 7;
  uint32_t idx = xcd * per + (xcd < rem ? xcd : rem) + (pid >> 3);
  Tile t;
  t.split = idx % p.splits; idx /= p.splits;
  const uint32_t in_block = kBlock * p.tiles_n, first = idx / in_block * kBlock, within = idx % in_block, h = tiles_m - first < kBlock ? tiles_m - first : kBlock;
  t.mt = uni(first + within % h); t.nt = uni(within / h); t.split = uni(t.split);
  t.expert = 0; t.row_lo = t.mt * p.tile_rows; t.zeros = false;
  t.rows = p.M - t.row_lo < p.tile_rows ? p.M - t.row_lo : p.tile_rows;
  if (p.tile_tab != nullptr) {
    t.expert = uni(p.tile_tab[3 * t.mt]); t.row_lo = uni(p.tile_tab[3 * t.mt + 1]);
    const uint32_t n = uni(p.tile_tab[3 * t.mt + 2]);
    t.rows = n & 0x7FFFFFFFu; t.zeros = (n >> 31) != 0;
    if (t.zeros) t.expert = 0;
  }
  t.rows = t.rows < tile_rows ? t.rows : tile_rows;
  *out = t;
  return true;
}

}  // namespace
}  // namespace rmlx
