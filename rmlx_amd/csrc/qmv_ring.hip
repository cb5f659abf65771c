// Streaming GEMV of up to 16 rows per weight row that reads the weights as they lie (4- and 8-bit, group sizes 32 / 64 / 128, any N from a
// tile on, any K of whole groups from 512 to what a workgroup's registers hold of 16 activation rows, 8192 at 4 bits, 4096 at 8 and at group
// size 32): a matrix (DENSE), the rows of the expert that a chunk table names (TABLE), and the
// SwiGLU of its gate and up matrices (PAIR).  The products are exact (integer dot products, scaled in f32).
//
// What bounds it is HBM.  The other multi-row GEMVs load a tile of 16 weight rows as the matrix instruction wants it, 64 bytes of each of
// 16 rows at a time: 4.9 TB/s at best, and 3 to 4 where K is no multiple of 512 (rows then begin in the middle of cache lines).  Here a
// slot of 16 rows is one contiguous piece of the matrix (or H pieces a row), copied to LDS by whole 1 KB wave loads that bypass the
// registers (6.6 TB/s measured for a bare copy of that form), three or four slots ahead; the operands are picked from LDS behind it, whose
// 16-byte chunks are stored xor-ed with a key of the row, since rows a multiple of 128 bytes apart would hit the same banks.
// The activations never pass through LDS: a wave multiplies the same slice of k in every tile, so it keeps its part of the 16 rows in
// registers, in operand order, for as long as its workgroup stays in a chunk (f16, bf16 and f32 are read as they are: no conversion pass).
// One workgroup of eight waves per CU takes an equal share of all weight rows (of all chunks, for a table): no last round that is half
// empty, whatever the number of rows.  A slot costs one barrier; the waves' partial sums of a tile are added through LDS behind the
// products of the next one.
// Routed block, 128 experts, hidden 4096, inner 1536, top 8, 4-bit, group size 64: 12 / 32 / 64 / 128 / 200 tokens 143 / 221 / 247 / 264 / 303 us
// against 165 / 247 / 287 / 348 / 390 on the kernels before (three blocks in turn; floor by its bytes: 193 at 128 tokens); 40 experts, hidden 2944,
// inner 3072, group size 128, 15 / 120 tokens of 4 picks: 93 / 131 against 154 / 252.  8 rows, 33001 x 2880 16.2 us against 20.9; 13 rows, 14336 x 4096,
// 8-bit, four matrices 58.8 against 75.1; 16 rows, 151936 x 4096 66 against 104.  A slot of 16 x 4096 takes 1.25 us with its weights in the caches, 1.35 at the floor of HBM:
// 171 vector instructions per wave and slot, 80 of them unpacking, so both sides are nearly equal.
//
// (the device code below loads with inline assembly where the compiler would wait for the loads of a slot before it lets the next one out;
// the counts behind wait_but are those of the loads that this kernel issues, in order)
#include <cstddef>
#include <type_traits>
#include <utility>

#include "launch.hpp"
#include "q4_stream.hpp"
#include "tile.hpp"
#include "unbounded.hpp"

namespace rmlx {
namespace {

// Beside the arguments that the first loads need (separate ones: those arrive in scalar registers).
struct RingParams {
  void* out;
  uint32_t ld_out, x_rows, spr_inv;   // (2^20 / a row's groups of eight)
  int32_t out_f32;
  const uint32_t* w1; const __half* s1; const __half* b1;
  const uint32_t* row_map; const uint32_t* chunk_tab; const uint32_t* n_chunks;
  uint64_t estride_w, estride_s;
  uint32_t slack;  // weight rows that one more chunk costs a workgroup
  const uint32_t* picks; uint32_t entries, per, per_inv, n_experts;  // GATHER; per_inv: 2^16 / per
};
// rows of one matrix; of the expert that a chunk table names; of its gate and up matrices; of the experts that a list of entries picks
enum { DENSE = 0, TABLE = 1, PAIR = 2, GATHER = 3 };
constexpr uint32_t kMaxEntries = 256, kNoExpert = 0xFFFFFFFEu;
// How the waves share a tile's k: `ks` parts, 2^nt_log2 tiles side by side, the tile of wave i in bits 8 + 3 i
inline uint32_t ring_geometry(uint32_t ks, int32_t x_dtype) {
  uint32_t v = ks | (ks == 1 ? 3u : (ks == 2 ? 2u : (ks <= 4 ? 1u : 0u))) << 4 | (uint32_t)x_dtype << 6;
  for (uint32_t w = 0; w < 8; ++w) v |= (w / ks) << (8 + 3 * w);
  return v;
}

constexpr int kWaves = 8;

template <class F, int... I>
__device__ __forceinline__ void repeat_over(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void repeat(F&& f) { repeat_over(f, std::make_integer_sequence<int, N>{}); }

// 8 nibbles -> f16 0 .. 15 in the order 0, 2, 4, 6, 1, 3, 5, 7 (as an e4m3 byte a value below 16 is q / 512)
__device__ __forceinline__ h8 nibbles(uint32_t w) {
  const uint32_t even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
  u4 o;
  o.x = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(even, 512.0f, false));
  o.y = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(even, 512.0f, true));
  o.z = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(odd, 512.0f, false));
  o.w = h2bits((h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(odd, 512.0f, true));
  return __builtin_bit_cast(h8, o);
}
__device__ __forceinline__ h8 nibble_order(h8 v) {  // the activations in that order
  const u4 d = __builtin_bit_cast(u4, v);
  u4 o;
  o.x = __builtin_amdgcn_perm(d.y, d.x, 0x05040100u);
  o.y = __builtin_amdgcn_perm(d.w, d.z, 0x05040100u);
  o.z = __builtin_amdgcn_perm(d.y, d.x, 0x07060302u);
  o.w = __builtin_amdgcn_perm(d.w, d.z, 0x07060302u);
  return __builtin_bit_cast(h8, o);
}
// 8 bytes -> f16 1024 + q
__device__ __forceinline__ h8 bytes8(uint32_t w0, uint32_t w1) {
  u4 o;
  o.x = __builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u);
  o.y = __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u);
  o.z = __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u);
  o.w = __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u);
  return __builtin_bit_cast(h8, o);
}
// 16 bytes per lane and load straight into LDS, one load behind another from `lds` on (the instruction's offset counts for both addresses, so
// the lanes' are given less 0, 1024, 2048 .. bytes).  One statement: nothing may come between m0 and the loads that use it.
__device__ __forceinline__ void dma_slot(uint32_t lds, const uint32_t (&off)[3], u4 r) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %4, 0 offen nt lds\n\tbuffer_load_dwordx4 %2, %4, 0 offen offset:1024 nt lds\n\t"
               "buffer_load_dwordx4 %3, %4, 0 offen offset:2048 nt lds" ::"s"(lds), "v"(off[0]), "v"(off[1]), "v"(off[2]), "s"(r) : "memory", "m0");
}
__device__ __forceinline__ void dma_slot(uint32_t lds, const uint32_t (&off)[4], u4 r) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %5, 0 offen nt lds\n\tbuffer_load_dwordx4 %2, %5, 0 offen offset:1024 nt lds\n\t"
               "buffer_load_dwordx4 %3, %5, 0 offen offset:2048 nt lds\n\tbuffer_load_dwordx4 %4, %5, 0 offen offset:3072 nt lds"
               ::"s"(lds), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(r) : "memory", "m0");
}
// the buffer from byte `by` on (scalar: the lanes' offsets stay as they are)
__device__ __forceinline__ u4 later(u4 r, uint32_t by) {
  const uint64_t a = ((uint64_t)r.y << 32 | r.x) + by;
  return (u4){uni((uint32_t)a), uni((uint32_t)(a >> 32)), uni(r.z - by), r.w};
}
template <int AT>
__device__ __forceinline__ void load16(u4& d, uint32_t off, u4 r) {
  static_assert(AT >= 0 && AT < 4096, "12 bits of offset");
  asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen offset:%3" : "=v"(d) : "v"(off), "s"(r), "n"(AT) : "memory");
}
__device__ __forceinline__ void hold(u4& d) { asm volatile("" : "+v"(d)::"memory"); }
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ float half_of(uint32_t w, int i) {
  const uint16_t h = (i & 1) ? (uint16_t)(w >> 16) : (uint16_t)(w & 0xFFFFu);
  return (float)__builtin_bit_cast(_Float16, h);
}
// A lane's 8 values of product (u, j) begin at k_lane g + k_of(u, j) of the slice: the four lanes of a row are inside one group.
template <int BITS, int GS>
constexpr uint32_t kLaneK = BITS == 4 ? (GS == 128 ? 32 : (GS == 64 ? 16 : 8)) : (GS == 32 ? 8 : 16);
template <int BITS, int GS>
constexpr uint32_t k_of(int u, int j) {
  if (BITS == 4) return GS == 128 ? u * 128 + j * 8 : (GS == 64 ? u * 128 + (j >> 1) * 64 + (j & 1) * 8 : u * 128 + j * 32);
  return GS == 32 ? u * 64 + j * 32 : u * 64 + j * 8;
}

template <int BITS, int GS, int U, int H>
struct Ring {
  static constexpr int kUnitK = BITS == 4 ? 128 : 64, kProducts = BITS == 4 ? 4 : 2, KU = U * kUnitK;  // KU: k of a wave in a slot
  static constexpr int NG = KU / GS, NB = (NG + 3) / 4, SD = (NG + 1) / 2;  // groups of a wave in a slot, bias products, dwords of scales
  static constexpr uint32_t kWBytes = kWaves * U * 1024, kSBytes = (256 * NG * H + 1023) / 1024 * 1024, kScales = 2 * kSBytes, kSums = kWaves * 1024;
  static constexpr int R = 4 * (kWBytes + kScales) + 2 * kSums <= 160 * 1024 ? 4 : 3;
  static constexpr uint32_t oScales = R * kWBytes, oSums = oScales + R * kScales, kLds = oSums + 2 * kSums;
  static_assert(kLds <= 160 * 1024 && kSBytes <= 4096, "LDS, one load a wave for the scales");
};

// An equal share of all (chunk, weight row) pairs for every workgroup, or, where that is hardly more work for it, of one chunk (a second
// one starts over with empty rings and other activations: about 4 us, in which a CU streams 100 KB).
__device__ __forceinline__ void take_share(uint32_t chunks, uint32_t N, uint32_t slack, uint32_t* pos, uint32_t* end) {
  const uint32_t all = chunks * N, each = all / gridDim.x, more = all - each * gridDim.x, b = blockIdx.x;
  const uint32_t per = chunks == 0 ? 0 : gridDim.x / chunks, part = per == 0 ? 0 : N / per, rest = N - part * per;
  if (per != 0 && part <= each + slack) {
    const uint32_t c = b / per, i = b - c * per;
    *pos = c * N + i * part + (i < rest ? i : rest);
    *end = c < chunks ? *pos + part + (i < rest ? 1 : 0) : *pos;
  } else {
    *pos = b * each + (b < more ? b : more);
    *end = *pos + each + (b < more ? 1 : 0);
  }
  *pos = uni(*pos);
  *end = uni(*end);
}

// The kernel's arguments as they lie in memory.
struct RingArgs {
  const uint32_t* w0; const __half* s0; const __half* b0; const char* x;
  uint32_t N, K, M, geometry, share, over, cpr_inv;
  RingParams p;
};
static_assert(offsetof(RingArgs, geometry) == 44 && offsetof(RingArgs, p) == 64, "the kernel's parameters, one behind another");
// Offsets and biases of both signs make a NaN of an infinite activation, (1024 + q) inf - 1024 inf, where the sum of the products is an
// infinity (f32 and bf16 values past the range of f16 are infinities here too).  A wave that has stored a result that is not finite comes
// here at its end and goes over the results of such rows once more, over the pieces of the row that are not finite (the others do not change
// the sum; over all of it where there are none: then the weights are not finite); what is not finite is stored anew.  The arguments are read again, so that nothing
// is kept for this (as scalar registers they made the others spill), and what it costs the others is a multiply-add for each result:
// gather of 32 x 8 rows 40.6 -> 40.9 us, of 89 x 2 rows over 32 experts of 1664 x 2496 24.3 -> 24.5, 13 rows, 14336 x 4096, 8-bit 59.2 -> 58.9 for four.  A row of 100001 x 4096 with one infinity
// 45 -> 70 us, all 16 rows 142 (3.1 ms with every lane looking through its row for itself).
typedef const __attribute__((address_space(1))) RingArgs* RingArgsPtr;
template <int BITS, int GS, int H, int MODE>
__device__ __forceinline__ void store_unbounded(char* lds, bool spoiled, uint32_t chunks, uint32_t seg_row, uint32_t seg_rows, uint32_t seg_expert) {
  auto args = []() -> RingArgsPtr {                       // (from memory, each time, into vector registers)
    auto a = (RingArgsPtr)(const void*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+v"(a));
    return a;
  };
  const RingArgsPtr a = args();
  const uint32_t N = uni(a->N), K = uni(a->K), geometry = uni(a->geometry), tid = threadIdx.x, wave = uni(tid >> 6), lane = tid & 63;
  const int32_t x_dtype = geometry >> 6 & 3;
  uint16_t* const list = reinterpret_cast<uint16_t*>(lds) + wave * 1024;  // (in the place of the rings, which nobody reads any more)
  // (which results are this lane's: as in the kernel)
  const uint32_t nt_log2 = H == 2 ? 0 : geometry >> 4 & 3, w_log2 = nt_log2 < 2 ? nt_log2 : 2, it = wave * 64 + lane, ot = it >> (8 - w_log2);
  const uint32_t l = it >> (2 - w_log2) & 63, out_m = (l >> 4) * 4 + ((it & ((4 >> w_log2) - 1)) << w_log2), out_c = (ot << 4) + (l & 15);
  uint32_t pos, end, seg = 0;
  if (MODE != DENSE) take_share(MODE == GATHER ? uni(chunks) : uni(*a->p.n_chunks), N, uni(a->p.slack), &pos, &end);
  else {
    const uint32_t share = a->share, over = a->over;
    pos = uni(blockIdx.x * share + (blockIdx.x < over ? blockIdx.x : over));
    end = uni(pos + share + (blockIdx.x < over ? 1 : 0));
  }
#pragma unroll 1
  do {
    const RingArgsPtr a = args();
    const uint32_t chunk = MODE == DENSE ? blockIdx.y : pos / N, r0 = MODE == DENSE ? pos : pos - chunk * N, r1 = end - pos < N - r0 ? r0 + (end - pos) : N;
    pos += r1 - r0;
    uint32_t expert = 0, row0 = chunk * 16, rows = uni(a->M) - row0 < 16u ? uni(a->M) - row0 : 16u;
    if constexpr (MODE == GATHER) {
      expert = __builtin_amdgcn_readlane(seg_expert, seg * 16);
      rows = expert == kNoExpert ? 0u : __builtin_amdgcn_readlane(seg_rows, seg * 16);
    } else if (MODE != DENSE) {
      const uint32_t* const t = a->p.chunk_tab + 3 * chunk;
      expert = uni(t[0]); row0 = uni(t[1]); rows = uni(t[2]);
      if ((rows >> 31) != 0) rows = 0;                    // (zeros)
    }
#pragma unroll 1
    for (uint32_t i = 0; i < rows; ++i) {
      const bool mine = i - out_m < 1u << w_log2 && ot < 1u << nt_log2;
      if (__builtin_amdgcn_ballot_w64(mine && spoiled) == 0) continue;
      const RingArgsPtr a = args();
      uint32_t m = row0 + i, from = m;
      if constexpr (MODE == GATHER) m = from = __builtin_amdgcn_readlane(seg_row, seg * 16 + i);
      else if (MODE != DENSE && a->p.row_map != nullptr) from = uni(a->p.row_map[m]);
      const char* const x = a->x + (uint64_t)from * (K << (x_dtype == RMLX_DTYPE_F32 ? 2 : 1));
      const uint32_t n = q4::odd_pieces(x, x_dtype, K, lane, list);
#pragma unroll 1
      for (uint32_t r = mine ? r0 + out_c : r1; r < r1; r += 16u << nt_log2) {
        auto sum_of = [&](bool up, bool whole) {
          const RingArgsPtr a = args();
          const uint64_t at = (uint64_t)r * (K / GS) + expert * a->p.estride_s;
          const char* const w = reinterpret_cast<const char*>(up ? a->p.w1 : a->w0) + expert * a->p.estride_w * 4 + (uint64_t)r * (K * BITS / 8);
          return q4::plain_sum<BITS>(GS == 32 ? 5 : (GS == 64 ? 6 : 7), w, (up ? a->p.s1 : a->s0) + at, (up ? a->p.b1 : a->b0) + at, x, x_dtype, whole ? nullptr : list, whole ? K / 8 : n);
        };
        float v = sum_of(false, n == 0);
        if constexpr (MODE == PAIR) {
          float u = sum_of(true, n == 0);
          const bool v_ok = __builtin_isfinite(v), u_ok = __builtin_isfinite(u);
          if (v_ok && u_ok) continue;
          if (v_ok) v = sum_of(false, true);
          if (u_ok) u = sum_of(true, true);
          v = q4::silu_f(v) * u;
        } else if (__builtin_isfinite(v)) continue;
        const RingArgsPtr a = args();
        const uint64_t o = (uint64_t)m * a->p.ld_out + r;
        if (MODE != GATHER && a->p.out_f32) static_cast<float*>(a->p.out)[o] = v;
        else static_cast<__half*>(a->p.out)[o] = __float2half(v);
      }
    }
    ++seg;
  } while (MODE != DENSE && pos < end);
}

template <int BITS, int GS, int U, int H, int MODE>
__global__ __launch_bounds__(kWaves * 64, 2) void qmv_ring_kernel(uint64_t w0_, uint64_t s0_, uint64_t b0_, uint64_t x_, uint32_t N,
                                                                  uint32_t K, uint32_t M, uint32_t geometry, uint32_t share, uint32_t over, uint32_t cpr_inv,
                                                                  RingParams p) {
  const uint32_t* const w0 = global_at<uint32_t>(w0_);
  const __half *const s0 = global_at<__half>(s0_), *const b0 = global_at<__half>(b0_);
  const char* const x = global_at<char>(x_);
  const uint32_t spr_inv = p.spr_inv;
  using C = Ring<BITS, GS, U, H>;
  constexpr bool DUAL = MODE == PAIR;
  constexpr int kUnitK = C::kUnitK, kProducts = C::kProducts, KU = C::KU, NG = C::NG, NB = C::NB, SD = C::SD, R = C::R;
  // 4-bit: unpacked to 1024 + q and 64 + q (5 vector instructions a word), the products begin at minus the offsets' share; where there are
  // no registers for that, to q (7 instructions)
  constexpr bool kOffsets = BITS == 4 && GS != 32 && H == 1;
  static_assert(KU % GS == 0, "whole groups");
  __shared__ __align__(1024) char lds[C::kLds];

  const uint32_t tid = threadIdx.x, wave = uni(tid >> 6);
  uint32_t lane = tid & 63;
  const uint32_t KS = geometry & 15, nt_log2 = H == 2 ? 0 : geometry >> 4 & 3, tw = geometry >> (8 + 3 * wave) & 7, kp = wave - tw * KS, NT = 1u << nt_log2;
  const int32_t x_dtype = geometry >> 6 & 3;
  uint32_t pos = 0, end = 0, gather_chunks = 0;
  // GATHER: every workgroup groups the entries by expert itself (a launch of its own for that costs more: 3 us against about 1.5), a stable
  // counting sort over at most 256 of them, all waves alike behind the ranks.  A chunk is 16 rows of one expert's entries one behind another;
  // a workgroup's share lies in at most four of those (at most 256 chunks, an entry has no more than 16 rows, and twice the workgroups are
  // let in): lane 16 s + i keeps row i of the s-th.
  uint32_t seg_row = 0, seg_rows = 0, seg_expert = 0;
  if constexpr (MODE == GATHER) {
    uint32_t* const keys = reinterpret_cast<uint32_t*>(lds);  // in the place of the rings
    uint32_t *const order = keys + kMaxEntries, *const run_chunks = order + kMaxEntries, *const run_rows = run_chunks + kMaxEntries;
    uint32_t* const mine = run_rows + kMaxEntries + wave * 16;
    if (tid < kMaxEntries) {
      const uint32_t e = tid < p.entries ? p.picks[tid] : 0xFFFFFFFFu;
      keys[tid] = tid < p.entries && e >= p.n_experts ? kNoExpert : e;
      run_chunks[tid] = 0;
    }
    q4::lds_barrier();
    if (tid < p.entries) {
      const uint32_t e = keys[tid];
      uint32_t below = 0, before = 0, same = 0;
      for (uint32_t j = 0; j < p.entries; j += 4) {
        const u4 v = *reinterpret_cast<const u4*>(keys + j);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
          below += v[i] < e ? 1u : 0u;
          same += v[i] == e ? 1u : 0u;
          before += v[i] == e && j + i < tid ? 1u : 0u;
        }
      }
      order[below + before] = tid;
      if (before == 0) {
        run_chunks[below] = (same * p.per + 15) / 16;
        run_rows[below] = same * p.per;
      }
    }
    q4::lds_barrier();
    const u4 v = *reinterpret_cast<const u4*>(run_chunks + lane * 4);
    uint32_t inc = v.x + v.y + v.z + v.w;
    const uint32_t own = inc;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = __shfl_up(inc, o, 64);
      if ((int)lane >= o) inc += t;
    }
    gather_chunks = __shfl(inc, 63, 64);
    take_share(uni(gather_chunks), N, p.slack, &pos, &end);
    const uint32_t c0 = pos / N;
    if (lane < 16) mine[lane] = 0;
    uint32_t base = inc - own;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
#pragma unroll
      for (uint32_t sg = 0; sg < 4; ++sg) {
        const uint32_t d = c0 + sg - base, q = lane * 4 + i;
        if (c0 + sg >= base && d < v[i]) {
          mine[4 * sg] = q * p.per + 16 * d;
          mine[4 * sg + 1] = run_rows[q] - 16 * d < 16u ? run_rows[q] - 16 * d : 16u;
          mine[4 * sg + 2] = keys[order[q]];
        }
      }
      base += v[i];
    }
    const u4 m = *reinterpret_cast<const u4*>(mine + (lane >> 4) * 4);
    const uint32_t row = m.x + (lane & 15), q = row * p.per_inv >> 16;
    seg_rows = m.y;
    seg_expert = m.z;
    seg_row = (lane & 15) < m.y ? order[q] * p.per + row - q * p.per : 0;
    wait_lds();
    q4::lds_barrier();                                    // (the rings may be filled)
  } else if (MODE != DENSE) {
    take_share(uni(*p.n_chunks), N, p.slack, &pos, &end);
  } else {
    pos = uni(blockIdx.x * share + (blockIdx.x < over ? blockIdx.x : over));
    end = uni(pos + share + (blockIdx.x < over ? 1 : 0));
  }
  const uint32_t xshift = x_dtype == RMLX_DTYPE_F32 ? 2 : 1;
  const uint32_t lds0 = uni((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  if (pos >= end) return;
  uint32_t seg = 0;
  float spoiled = 0.f;                                    // NaN once the lane has stored a result that is not finite

  do {
    // (what follows from these is worked out where it is used: kept across segments it costs more registers than there are, and the first
    // loads wait for it)
    if (MODE != DENSE) asm volatile("" : "+s"(K), "+v"(lane));
    const uint32_t G = K / GS, row_bytes = K * BITS / 8;
    const uint32_t chunk = MODE == DENSE ? blockIdx.y : pos / N, r0 = MODE == DENSE ? pos : pos - chunk * N, r1 = end - pos < N - r0 ? r0 + (end - pos) : N;
    pos += r1 - r0;
    uint32_t expert = 0, row0 = chunk * 16, rows = M - row0 < 16u ? M - row0 : 16u;
    bool zeros = false;
    if constexpr (MODE == GATHER) {
      expert = __builtin_amdgcn_readlane(seg_expert, seg * 16); rows = __builtin_amdgcn_readlane(seg_rows, seg * 16);
      zeros = expert == kNoExpert;
      if (zeros) expert = 0;
    } else if (MODE != DENSE) {
      expert = uni(p.chunk_tab[3 * chunk]); row0 = uni(p.chunk_tab[3 * chunk + 1]); rows = uni(p.chunk_tab[3 * chunk + 2]);
      zeros = (rows >> 31) != 0;
      rows &= 0x7FFFFFFFu;
      if (zeros) expert = 0;
    }
    auto at = [](const void* q, uint64_t o) { return static_cast<const void*>(static_cast<const char*>(q) + o); };
    const bool mapped = MODE == GATHER || (MODE != DENSE && p.row_map != nullptr);
    auto source_row = [&](uint32_t m) -> uint32_t { return __builtin_amdgcn_ds_bpermute((seg * 16 + m) * 4, seg_row); };  // GATHER
    const uint32_t xrow = K << xshift;
    const void* const x_base = mapped ? static_cast<const void*>(x) : at(x, (uint64_t)row0 * xrow);
    const u4 xr = rsrc(x_base, (uint64_t)(mapped ? p.x_rows : rows) * xrow);
    const uint32_t xm = lane & 15;                        // of the lane's row, and its place in a product
    uint32_t x_row = xm;
    if constexpr (MODE == GATHER) x_row = source_row(xm);
    else if (mapped && xm < rows) x_row = p.row_map[row0 + xm];
    const uint32_t x_lane = xm < rows ? x_row * xrow + ((lane >> 4) * kLaneK<BITS, GS> << xshift) : kOutside;

    // ---- activations: this wave's part of every slot, in operand order (k past the row, rows past the chunk: zeros from the range check) ----
    u4 xv[H][U][kProducts];
    auto groups_of = [&](int h) -> uint32_t { const uint32_t k0 = (h * KS + kp) * KU; return k0 < K ? (K - k0) / GS : 0; };
    auto request_x = [&]() {
      repeat<H>([&](auto h) {
        const uint32_t groups = groups_of(h), base = groups != 0 ? x_lane + (h * KS + kp) * KU * 2 : kOutside;  // (never a sum with x_lane: it wraps)
        if (groups >= (uint32_t)NG || groups == 0) {
          repeat<U>([&](auto u) {
            repeat<kProducts>([&](auto j) { load16<k_of<BITS, GS>(decltype(u)::value, decltype(j)::value) * 2>(xv[h][u][j], base, xr); });
          });
        } else {
          repeat<U>([&](auto u) {
            repeat<kProducts>([&](auto j) {
              constexpr uint32_t gi = (decltype(u)::value * kUnitK + decltype(j)::value * 32) / GS;
              load16<k_of<BITS, GS>(decltype(u)::value, decltype(j)::value) * 2>(xv[h][u][j], gi < groups ? base : kOutside, xr);
            });
          });
        }
      });
    };
    auto load_x_f32 = [&]() {
      const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>((uint64_t)uni(xr.y) << 32 | uni(xr.x)), 0, (int)uni(xr.z), 0x00020000);
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < kProducts; ++j) {
            const uint32_t k = (h * KS + kp) * KU + k_of<BITS, GS>(u, j);
            const uint32_t off = (uint32_t)((u * kUnitK + j * 32) / GS) < groups_of(h) ? x_lane + k * 4 : kOutside;
            const u4 lo = __builtin_amdgcn_raw_buffer_load_b128(xb, off, 0, 0), hi = __builtin_amdgcn_raw_buffer_load_b128(xb, off + 16, 0, 0);
            const f4 l = __builtin_bit_cast(f4, lo), g = __builtin_bit_cast(f4, hi);
            h8 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) { o[e] = (_Float16)l[e]; o[4 + e] = (_Float16)g[e]; }
            xv[h][u][j] = __builtin_bit_cast(u4, o);
          }
    };
    auto hold_x = [&]() {  // (behind the wait: nothing reads the registers before)
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < kProducts; ++j) hold(xv[h][u][j]);
    };
    if (x_dtype == RMLX_DTYPE_F32) load_x_f32();
    else request_x();

    // ---- loads of a slot: one part (of H) of the k of 16 NT rows of one matrix, shared by the waves ------------------------------------------
    // LDS holds the slot's 16-byte chunks row by row, xor-ed with a key of the row so that operand reads spread over the banks.
    const uint32_t cpr = H == 1 ? row_bytes / 16 : KS * U * 4;  // chunks of a row in a slot
    const uint32_t kshift = cpr % 16 == 0 ? 0 : (cpr % 8 == 0 ? 1 : 2), kmask = cpr % 16 == 0 ? 15 : (cpr % 8 == 0 ? 7 : (cpr % 4 == 0 ? 3 : 0));
    const uint64_t ew = (uint64_t)expert * p.estride_w * 4 + (uint64_t)r0 * row_bytes, es = (uint64_t)expert * p.estride_s * 2;
    const uint64_t wbytes = (uint64_t)(r1 - r0) * row_bytes;
    const u4 wr0 = rsrc(at(w0, ew), wbytes), wr1 = DUAL ? rsrc(at(p.w1, ew), wbytes) : wr0;
    // (waves 0 to 3 load the scales, 4 to 7 the biases: the rows' groups as they lie, 1 KB each)
    const u4 sr0 = rsrc(at(wave < 4 ? s0 : b0, es), (uint64_t)N * G * 2), sr1 = DUAL ? rsrc(at(wave < 4 ? p.s1 : p.b1, es), (uint64_t)N * G * 2) : sr0;
    const uint32_t tiles = (r1 - r0 + (16u << nt_log2) - 1) >> (4 + nt_log2), slots = tiles * H * (DUAL ? 2 : 1);
    uint32_t w_from[U];                                   // where a lane's bytes of a load come from: chunk 64 (wave U + u) + lane of the slot
    {
      const uint32_t i0 = wave * (U * 64) + lane, dr = 64 * cpr_inv >> 20, dc = 64 - dr * cpr;
      uint32_t r = i0 * cpr_inv >> 20, c = i0 - r * cpr;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        w_from[u] = r < 16u << nt_log2 ? r * row_bytes + ((c ^ (r >> kshift & kmask)) * 16) - u * 1024 : kOutside;  // (the load adds it)
        r += dr;
        c += dc;
        if (c >= cpr) { c -= cpr; ++r; }
      }
    }
    const uint32_t s_rows = (16u << nt_log2) * G * 2, s_last = N * G * 2 - ((s_rows + 15) & ~15u);  // bytes of a tile's groups; the last place to load them from
    // (their chunks are xor-ed with a key of the matrix row where rows lie a multiple of 64 bytes apart; tiles begin 16 rows apart, except
    // the one that is loaded from the last place)
    const uint32_t spr = G / 8, sshift = spr % 16 == 0 ? 0 : (spr % 8 == 0 ? 1 : 2), smask = G % 32 != 0 ? 0 : (spr % 16 == 0 ? 15 : (spr % 8 == 0 ? 7 : 3));
    auto skey = [&](uint32_t r) -> uint32_t { return r >> sshift & smask; };
    uint32_t s_from = (wave & 3) * 1024 + lane * 16, s_from_last = s_from;
    if (smask != 0) {
      const uint32_t i = (wave & 3) * 64 + lane, r = i * spr_inv >> 20, c = i - r * spr;
      s_from = (r * spr + (c ^ skey(r0 + r))) * 16;
      s_from_last = (r * spr + (c ^ skey(N - (16u << nt_log2) + r))) * 16;
    }
    auto scales_at = [&](uint32_t tile) -> uint32_t { return (r0 + (tile << (4 + nt_log2))) * G * 2; };
    const bool has_s = (wave & 3) * 1024 < C::kSBytes;
    uint32_t iq = 0, iplace = 0, splace = 0;              // the next slot to go out, its places in the rings
    auto issue = [&](bool first) {                        // (first: its tile's scales go out with it)
      if (iq >= slots) return;                            // (an empty load costs 16 cycles of the address unit all the same)
      const uint32_t tm = iq / H, t = DUAL ? tm >> 1 : tm;
      const bool up = DUAL && (tm & 1) != 0;
      const u4 wr = later(up ? wr1 : wr0, (t << (4 + nt_log2)) * row_bytes + (H == 1 ? 0 : iq % H * cpr * 16));
      if (first && has_s) {
        const uint32_t sa = scales_at(t);
        dma16(lds0 + C::oScales + splace * C::kScales + (wave < 4 ? 0 : C::kSBytes) + (wave & 3) * 1024, sa < s_last ? s_from : s_from_last,
              later(up ? sr1 : sr0, sa < s_last ? sa : s_last));
      }
      if (first) splace = splace == R - 1 ? 0 : splace + 1;
      dma_slot(lds0 + iplace * C::kWBytes + wave * U * 1024, w_from, wr);
      iplace = iplace == R - 1 ? 0 : iplace + 1;
      ++iq;
    };
    repeat<R>([&](auto i) { issue(H == 1 || decltype(i)::value % H == 0); });

    asm volatile("" : "+v"(lane));
    const uint32_t n = lane & 15, g = lane >> 4, row = (tw < NT ? tw * 16 : 0) + n;
    h8 xa[H][U][kProducts];
    float xs[H][NB];                                      // sums per (row, group): of group g NB + j of the lane's row
    f4 base[kOffsets ? NG : 1];                           // minus the offsets' share of a group's products, in accumulator layout
    q4::Q4Consts qc{0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    asm volatile("" : "+s"(qc.m0), "+s"(qc.m1), "+v"(qc.k0), "+v"(qc.k1));
    auto prepare_x = [&]() {
      h8 ones = {(_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1, (_Float16)1};
      const u4 offs = {0xE400E400u, 0xD400D400u, 0xE400E400u, 0xD400D400u};
      if (x_dtype == RMLX_DTYPE_BF16) {
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < kProducts; ++j) xv[h][u][j] = q4::bf16x8_to_f16(xv[h][u][j]);
      }
      const f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < H; ++h) {
#pragma unroll
        for (int j = 0; j < NB; ++j) xs[h][j] = 0.f;
        f4 sum = zero;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < kProducts; ++j) {
            const h8 v = __builtin_bit_cast(h8, xv[h][u][j]);
            const int k = u * kUnitK + j * 32, gi = k / GS;
            const bool first = k % GS == 0, last = (k + 32) % GS == 0;
            xa[h][u][j] = BITS != 4 ? v : (kOffsets ? __builtin_bit_cast(h8, q4::permute_x8(xv[h][u][j])) : nibble_order(v));
            sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, v, first ? zero : sum, 0, 0, 0);
            if constexpr (kOffsets) base[gi] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[h][u][j], __builtin_bit_cast(h8, offs), first ? zero : base[gi], 0, 0, 0);
            if (last) {
#pragma unroll
              for (int b = 0; b < NB; ++b) xs[h][b] = gi % NB == b && g == (uint32_t)(gi / NB) ? sum[0] : xs[h][b];
            }
          }
      }
    };

    // ---- operands of a slot ----------------------------------------------------------------------------------------------------
    // byte of the wave's part of the row -> place in the slot
    auto place = [&](uint32_t byte) -> uint32_t { return row * (cpr * 16) + (((kp * (U * 4) + (byte >> 4)) ^ (row >> kshift & kmask)) << 4) + (byte & 15); };
    constexpr int kParts = (BITS == 4 && GS == 128) || (BITS == 8 && GS != 32) ? 1 : ((BITS == 4 ? GS == 64 : GS == 32) ? 2 : 4);  // reads of a load's chunks
    constexpr bool kWide = NG % 8 == 0 || NG == 4;         // (a part's groups are whole 8 or 16 bytes of a row)
    uint32_t w_at[U][kParts], s_at[H][kWide ? SD / 4 + 1 : SD], b_at[H][NB];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < kParts; ++q) w_at[u][q] = place(u * 64 + q * (64 / kParts) + g * (16 / kParts));
    const bool even = G % 2 == 0 && NG % 2 == 0;          // (a row's groups then begin at whole dwords)
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const uint32_t g0 = (h * KS + kp) * NG;
      auto group_at = [&](uint32_t i) -> uint32_t {       // place of group i of the lane's row
        return smask == 0 ? (row * G + i) * 2 : ((row * spr + ((i >> 3) ^ skey(r0 + row))) * 8 + (i & 7)) * 2;
      };
      if constexpr (kWide) {
#pragma unroll
        for (int i = 0; i < (NG + 7) / 8; ++i) s_at[h][i] = group_at(g0 + 8 * i);
      } else {
#pragma unroll
        for (int i = 0; i < SD; ++i) s_at[h][i] = group_at(g0 + 2 * i);
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {                      // (past the row: its last group; the activations' sum is 0)
        const uint32_t i = g0 + g * NB + j;
        b_at[h][j] = C::kSBytes + group_at(i < G ? i : G - 1);
      }
    }
    uint32_t rq = 0, rplace = 0, qplace = 0;              // the next slot to be read, its places in the rings
    struct Operands { uint32_t w[U][4], s[SD]; float b[NB]; };
    auto read = [&](Operands& o, auto hc) {
      constexpr int h = decltype(hc)::value;
      const char* wt = lds + rplace * C::kWBytes;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (kParts == 1) {
          const u4 v = *reinterpret_cast<const u4*>(wt + w_at[u][0]);
          o.w[u][0] = v.x; o.w[u][1] = v.y; o.w[u][2] = v.z; o.w[u][3] = v.w;
        } else if constexpr (kParts == 2) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const u2 v = *reinterpret_cast<const u2*>(wt + w_at[u][q]);
            o.w[u][2 * q] = v.x; o.w[u][2 * q + 1] = v.y;
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) o.w[u][q] = *reinterpret_cast<const uint32_t*>(wt + w_at[u][q]);
        }
      }
      const uint32_t sa = scales_at(DUAL ? rq / H >> 1 : rq / H), early = sa < s_last ? 0 : sa - s_last;
      const char* st = lds + C::oScales + qplace * C::kScales + early;
      if (kWide && smask != 0) {
        if constexpr (NG == 4) {
          const u2 v = *reinterpret_cast<const u2*>(st + s_at[h][0]);
          o.s[0] = v.x; o.s[1] = v.y;
        } else {
#pragma unroll
          for (int i = 0; i < SD / 4; ++i) {
            const u4 v = *reinterpret_cast<const u4*>(st + s_at[h][i]);
            o.s[4 * i] = v.x; o.s[4 * i + 1] = v.y; o.s[4 * i + 2] = v.z; o.s[4 * i + 3] = v.w;
          }
        }
      } else if (even) {
#pragma unroll
        for (int i = 0; i < SD; ++i) o.s[i] = *reinterpret_cast<const uint32_t*>(st + (kWide ? s_at[h][0] + i * 4 : s_at[h][kWide ? 0 : i]));
      } else {                                            // (rows of any even length, never keyed)
        const uint32_t a = (uint32_t)(st - lds) + s_at[h][0], sh = (a & 2) * 8;
        uint32_t d[SD + 1];
#pragma unroll
        for (int i = 0; i <= SD; ++i) d[i] = *reinterpret_cast<const uint32_t*>(lds + (a & ~3u) + i * 4);
#pragma unroll
        for (int i = 0; i < SD; ++i) o.s[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], sh);
      }
      const uint32_t valid = groups_of(h);
      if (valid < (uint32_t)NG) {  // (the groups behind the row are those of another one)
#pragma unroll
        for (int i = 0; i < SD; ++i) o.s[i] &= (uint32_t)(2 * i) < valid ? ((uint32_t)(2 * i + 1) < valid ? 0xFFFFFFFFu : 0xFFFFu) : 0u;
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        o.b[j] = half_of(*reinterpret_cast<const uint16_t*>(st + b_at[h][j]), 0);
        if constexpr (BITS == 8)  // the operands are 1024 + q
          o.b[j] = fmaf(half_of(*reinterpret_cast<const uint16_t*>(st + b_at[h][j] - C::kSBytes), 0), -1024.0f, o.b[j]);
      }
      rplace = rplace == R - 1 ? 0 : rplace + 1;
      if (h == H - 1) qplace = qplace == R - 1 ? 0 : qplace + 1;
      ++rq;
    };
    f4 acc;
    // Group by group; a group's sums are scaled behind the products of the next one, whose latency that covers.
    auto multiply = [&](const Operands& o, auto hc) {
      constexpr int h = decltype(hc)::value, kOf = GS / 32;  // kOf: products of a group
      const f4 zero = {0.f, 0.f, 0.f, 0.f};
      if (h == 0) acc = zero;
      f4 dot[2];
#pragma unroll
      for (int gi = 0; gi <= NG; ++gi) {
        if (gi < NG) {
#pragma unroll
          for (int q = 0; q < kOf; ++q) {
            const int u = (gi * kOf + q) / kProducts, j = (gi * kOf + q) % kProducts;
            h8 wv;
            if constexpr (kOffsets) wv = __builtin_bit_cast(h8, q4::unpack_q4_word(o.w[u][j], qc));
            else if constexpr (BITS == 4) wv = nibbles(o.w[u][j]);
            else wv = bytes8(o.w[u][(2 * j) & 3], o.w[u][(2 * j + 1) & 3]);
            dot[gi & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[h][u][j], wv, q == 0 ? (kOffsets ? base[kOffsets ? gi : 0] : zero) : dot[gi & 1], 0, 0, 0);
          }
        }
        if (gi > 0) {
          const float sc = half_of(o.s[(gi - 1) >> 1], gi - 1);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[i] = fmaf(sc, dot[(gi - 1) & 1][i], acc[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[h][j], o.b[j], acc, 0, 0, 0);
    };

    // ---- the waves' sums of a tile, added in wave order; lane (n, g): rows 4 g + 0 .. 3, column n --------------------------------------
    // Each of the NT tiles has 8 / NT places (waves without a part put zeros into those that no part has).  A thread takes one, two or
    // four rows of a lane (one, two, more tiles side by side); it reads them before the products of the next tile and stores behind.
    const bool idle = tw >= NT;
    const uint32_t put = C::oSums + ((idle ? (nt_log2 == 0 ? wave : (wave & 1) * 4 + 3) : (tw << (3 - nt_log2)) + kp) * 64 + lane) * 16;
    const uint32_t w_log2 = nt_log2 < 2 ? nt_log2 : 2, it = wave * 64 + lane;
    const uint32_t l = it >> (2 - w_log2) & 63, part = it & ((4 >> w_log2) - 1), ot = it >> (8 - w_log2);  // (ot >= NT: nothing to do)
    const uint32_t get = C::oSums + (((ot << (3 - nt_log2)) * 64 + l) << 4) + (part << w_log2) * 4;
    const uint32_t out_m = (l >> 4) * 4 + (part << w_log2), out_c = (ot << 4) + (l & 15);
    const uint32_t out_rows = ot < NT && out_m < rows ? rows - out_m : 0;
    const uint64_t out_at = (uint64_t)(row0 + out_m) * p.ld_out + r0 + out_c;
    f4 gate;
    float term[8];
    uint32_t term_row[4];                                 // GATHER: the rows of x and of the result
    auto sums_read = [&](uint32_t tm) {
      if constexpr (MODE == GATHER) {
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e)
          if (e < 1u << w_log2) term_row[e] = source_row(out_m + e);
      }
      const char* q = lds + get + (tm & 1) * C::kSums;
      if (nt_log2 == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) term[i] = *reinterpret_cast<const float*>(q + i * 1024);
      } else if (nt_log2 == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const u2 v = *reinterpret_cast<const u2*>(q + i * 1024);
          term[2 * i] = __uint_as_float(v.x); term[2 * i + 1] = __uint_as_float(v.y);
        }
      } else {
        const f4 v0 = *reinterpret_cast<const f4*>(q), v1 = nt_log2 == 2 ? *reinterpret_cast<const f4*>(q + 1024) : (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) { term[e] = v0[e]; term[4 + e] = v1[e]; }
      }
    };
    auto sums_store = [&](uint32_t tm) {
      f4 v = {0.f, 0.f, 0.f, 0.f};
      if (nt_log2 == 0) v[0] = ((term[0] + term[1]) + (term[2] + term[3])) + ((term[4] + term[5]) + (term[6] + term[7]));
      else if (nt_log2 == 1) {
        v[0] = (term[0] + term[2]) + (term[4] + term[6]);
        v[1] = (term[1] + term[3]) + (term[5] + term[7]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = term[e] + term[4 + e];
      }
      const int w = 1 << w_log2;
      if (DUAL) {
        if ((tm & 1) == 0) { gate = v; return; }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < w) v[e] = q4::silu_f(gate[e]) * v[e];
      }
      const uint32_t c = (DUAL ? tm >> 1 : tm) << (4 + nt_log2);
      if (out_rows == 0 || c + out_c >= r1 - r0) return;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < w) spoiled = fmaf(v[e], 0.f, spoiled);
      if constexpr (MODE == GATHER) {
        __half* q = static_cast<__half*>(p.out) + r0 + out_c + c;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (e < w && (uint32_t)e < out_rows) q[(uint64_t)term_row[e] * p.ld_out] = __float2half(zeros ? 0.f : v[e]);
      } else if (p.out_f32) {
        float* q = static_cast<float*>(p.out) + out_at + c;
#pragma unroll
        for (int e = 0; e < 4; ++e, q += p.ld_out)
          if (e < w && (uint32_t)e < out_rows) *q = zeros ? 0.f : v[e];
      } else {
        __half* q = static_cast<__half*>(p.out) + out_at + c;
#pragma unroll
        for (int e = 0; e < 4; ++e, q += p.ld_out)
          if (e < w && (uint32_t)e < out_rows) *q = __float2half(zeros ? 0.f : v[e]);
      }
    };

    // `count` slots may still be on their way, `left` of them at most exist (those of a slot: U loads, and one of its tile's scales with its
    // first; near the end the scales' loads are not counted, so one or two more loads are waited for)
    auto wait_but = [&](auto firsts, auto count, uint32_t left) {
      constexpr int all = decltype(count)::value * U;
      if (left >= (uint32_t)decltype(count)::value) {
        if (has_s) wait_loads<all + decltype(firsts)::value>();
        else wait_loads<all>();
      } else if (decltype(count)::value > 1 && left != 0) wait_loads<U>();
      else wait_loads<0>();
    };
    using std::integral_constant;
    wait_but(integral_constant<int, (R + H - 1) / H>{}, integral_constant<int, R>{}, slots);
    hold_x();
    prepare_x();
    // Slot s is multiplied from registers while slot s + 1 is read from LDS; the barrier behind it says that everybody has read slot
    // s + 1, whose place the loads of slot s + 1 + R then take, and that slot s + 2 has arrived.
    Operands o[2];
    wait_but(integral_constant<int, H == 1 ? R - 2 : (R - 2 + 1) / 2>{}, integral_constant<int, R - 2>{}, slots > 2 ? slots - 2 : 0);
    q4::lds_barrier();
    read(o[0], integral_constant<int, 0>{});
    q4::lds_barrier();
    issue(H == 1 || R % H == 0);
    for (uint32_t s2 = 0; s2 < slots; s2 += 2) {
      repeat<2>([&](auto sc) {
        constexpr int s = decltype(sc)::value, h = H == 1 ? 0 : s;
        if (s2 + s >= slots) return;
        const uint32_t tm = (s2 + s) / H;
        if (s2 + s + 1 < slots) read(o[(s + 1) & 1], integral_constant<int, H == 1 ? 0 : (s + 1) & 1>{});
        if (h == 0 && tm > 0 && ot < NT) sums_read(tm - 1);  // (uniform: whole waves)
        multiply(o[s], integral_constant<int, h>{});
        if (h == H - 1) *reinterpret_cast<f4*>(lds + put + (tm & 1) * C::kSums) = idle ? (f4){0.f, 0.f, 0.f, 0.f} : acc;
        if (h == 0 && tm > 0 && ot < NT) sums_store(tm - 1);
        // slots s + 3 .. s + R may still be on their way
        wait_but(integral_constant<int, H == 1 ? R - 2 : (R % 2 == 0 ? (R - 2) / 2 : (R - 3) / 2 + ((s + 3) % 2 == 0 ? 1 : 0))>{}, integral_constant<int, R - 2>{},
                 slots > s2 + s + 3 ? slots - (s2 + s + 3) : 0);
        q4::lds_barrier();
        issue(H == 1 || (s + 1 + R) % H == 0);
      });
    }
    if (ot < NT) {
      sums_read(slots / H - 1);
      sums_store(slots / H - 1);
    }
    wait_loads<0>();
    if (MODE != DENSE) q4::lds_barrier();  // (the rings are free again)
    ++seg;
  } while (MODE != DENSE && pos < end);
  if (__builtin_amdgcn_ballot_w64(spoiled != spoiled) != 0)
    store_unbounded<BITS, GS, H, MODE>(lds, spoiled != spoiled, gather_chunks, seg_row, seg_rows, seg_expert);
}

struct RingLaunch { const QmvArgs* a; uint32_t geometry, share, over, wgs, chunks, cpr_inv; RingParams p; };
template <int BITS, int GS, int U, int H, int MODE>
void launch_ring(const RingLaunch& l, hipStream_t s) {
  Launch<qmv_ring_kernel<BITS, GS, U, H, MODE>>::go(dim3(l.wgs, l.chunks), dim3(kWaves * 64), 0, s, address(l.a->w0), address(l.a->s0),
                                                    address(l.a->b0), address(l.a->x), l.a->N, l.a->K, l.a->M, l.geometry, l.share, l.over, l.cpr_inv, l.p);
}
template <int BITS, int GS, int U, int H>
void launch_mode(const RingLaunch& l, hipStream_t s) {
  if constexpr (BITS == 4)
    if (l.p.picks != nullptr) { launch_ring<BITS, GS, U, H, GATHER>(l, s); return; }
  if (l.a->dual) launch_ring<BITS, GS, U, H, PAIR>(l, s);
  else if (l.a->chunk_tab != nullptr) launch_ring<BITS, GS, U, H, TABLE>(l, s);
  else launch_ring<BITS, GS, U, H, DENSE>(l, s);
}
// How a row is split over the waves: `h` slots of `ks` parts of `u` loads (128 values at 4 bits, 64 at 8), the split with the fewest empty
// loads and idle waves; rows in two slots only where one does not hold them (twice the barriers and the registers of the activations; at
// 4 bits and group size 32 there are not enough of those, and three loads are no whole groups of 128 8-bit values).
struct RingPlan { uint32_t ks, u, h; };
bool ring_plan(uint32_t K, uint32_t gs, uint32_t bits, RingPlan* out) {
  const uint32_t per = bits == 4 ? 128 : 64, units = (K + per - 1) / per;
  double best = 0;
  for (uint32_t h = 1; h <= 2; ++h)
    for (uint32_t u : {4u, 3u}) {
      const uint32_t ks = (units + u * h - 1) / (u * h);
      if (ks > 8 || units < u * h || (h == 2 && (u != 4 || best > 0 || (bits == 4 && gs == 32))) || (u == 3 && bits == 8 && gs == 128)) continue;
      const double e = (double)units / (ks * u * h) * (ks * (8 / ks)) / 8;  // loads that are not empty, waves that have any
      if (e > best + 1e-6) { best = e; *out = RingPlan{ks, u, h}; }
    }
  return best > 0;
}
template <int BITS, int GS>
void launch_slice(const RingLaunch& l, const RingPlan& plan, hipStream_t s) {
  if constexpr (BITS == 8 || GS != 32)
    if (plan.h == 2) { launch_mode<BITS, GS, 4, 2>(l, s); return; }
  if constexpr (BITS == 4 || GS != 128)
    if (plan.u == 3) { launch_mode<BITS, GS, 3, 1>(l, s); return; }
  launch_mode<BITS, GS, 4, 1>(l, s);
}

}  // namespace

bool qmv_ring_supported(uint32_t N, uint32_t K, uint32_t group_size, uint32_t bits) {
  if ((bits != 4 && bits != 8) || (group_size != 32 && group_size != 64 && group_size != 128) || N == 0 || K < 512 || K % group_size != 0) return false;
  RingPlan plan;
  if (!ring_plan(K, group_size, bits, &plan)) return false;
  // (a tile's groups are loaded in whole 16-byte pieces from inside the matrix)
  return N >= 16u * (8 / plan.ks) && (uint64_t)N * K * bits / 8 <= 0x80000000ull && (uint64_t)N * (K / group_size) * 2 < 0x7FFF0000ull;
}

// What the launches have in common: the split of a row and the constants of the kernel's divisions
static void ring_split(const QmvArgs& a, uint32_t bits, uint32_t gs, int32_t x_dtype, RingPlan* plan, RingLaunch* l) {
  RingParams& p = l->p;
  l->a = &a;
  l->wgs = ctx().num_cus;
  p.out = a.out; p.row_map = a.row_map; p.chunk_tab = a.chunk_tab; p.n_chunks = a.n_chunks_dev;
  p.w1 = a.w1; p.s1 = a.s1; p.b1 = a.b1;
  p.estride_w = a.expert_stride_w; p.estride_s = a.expert_stride_s;
  p.ld_out = a.ld_out; p.out_f32 = a.out_f32;
  ring_plan(a.K, gs, bits, plan);
  l->geometry = ring_geometry(plan->ks, x_dtype);
  const uint32_t cpr = plan->h == 1 ? a.K * bits / 128 : plan->ks * plan->u * 4;
  p.slack = 102400 / (a.K * bits / 8);
  l->cpr_inv = ((1u << 20) + cpr - 1) / cpr;
  if (a.K / gs >= 8) p.spr_inv = ((1u << 20) + a.K / gs / 8 - 1) / (a.K / gs / 8);
}
static int32_t launch_format(const RingLaunch& l, const RingPlan& plan, uint32_t bits, uint32_t gs, hipStream_t s) {
  if (bits == 4) {
    if (gs == 32) launch_slice<4, 32>(l, plan, s);
    else if (gs == 64) launch_slice<4, 64>(l, plan, s);
    else launch_slice<4, 128>(l, plan, s);
  } else {
    if (gs == 32) launch_slice<8, 32>(l, plan, s);
    else if (gs == 64) launch_slice<8, 64>(l, plan, s);
    else launch_slice<8, 128>(l, plan, s);
  }
  RMLX_HIP_CHECK(take_launch_error());
  return RMLX_OK;
}

// Workgroups over the rows of a matrix: one per CU, or a few less where a workgroup's share is within 3 KB of a power of two and its 128th part
// more, or less, from 512 KB on: walked side by side, such shares keep to a part of the memory channels (8 rows, 8-bit, us, by what the share
// is beyond the power, KB: 512 KB, K = 2048, 0 / 2 / 4 / 6 / 8 25.9 / 28.3 / 35.3 / 26.8 / 26.7; 1 MB, K = 4096, 0 / 4 / 6 / 8 / 10 / 12 / 16 45.8 / 48.0 /
// 51.7 / 58.6 / 52.0 / 48.2 / 47.5, -8 52.0; 2 MB, 8 / 16 / 24 89.4 / 102.6 / 90.1; 256 KB, 1 / 2 / 3 16.8 / 17.9 / 17.3).  33001 x 4096, 2 / 16 rows 33.3 /
// 34.5 us on all CUs, 25.9 / 27.3 on two less.
static uint32_t ring_workgroups(uint64_t bytes) {
  const uint32_t cus = ctx().num_cus;
  for (uint32_t w = cus; w + 8 > cus && w > 0; --w) {
    const uint64_t share = bytes / w;
    uint64_t p = 512 << 10;
    while (p + p / 2 < share) p *= 2;
    const int64_t past = (int64_t)(share > p ? share - p : p - share) - (int64_t)(p / 128);
    if (past < -3072 || past > 3072) return w;
  }
  return cus;
}

int32_t launch_qmv_ring(const QmvArgs& a, uint32_t bits, int32_t x_dtype, uint32_t x_rows, hipStream_t s) {
  const uint32_t gs = a.group_size == 0 ? 64 : a.group_size, size = x_dtype == RMLX_DTYPE_F32 ? 4 : 2;
  if (!qmv_ring_supported(a.N, a.K, gs, bits) || (a.dual != 0 && a.chunk_tab == nullptr) || (a.row_map != nullptr && (uint64_t)x_rows * a.K * size > 0x80000000ull))
    return fail(RMLX_INVALID_SHAPE, "streaming qmv: unsupported shape N=%u K=%u bits=%u group_size=%u, %u rows", a.N, a.K, bits, gs, x_rows);
  RingLaunch l{};
  RingPlan plan;
  ring_split(a, bits, gs, x_dtype, &plan, &l);
  l.p.x_rows = x_rows;
  if (a.chunk_tab != nullptr) {
    if (a.max_chunks == 0) return RMLX_OK;
    if ((uint64_t)a.max_chunks * a.N > 0xFFFFFFFFull) return fail(RMLX_INVALID_SHAPE, "streaming qmv: too many row chunks (%u)", a.max_chunks);
    l.chunks = 1;
  } else {
    if (a.M == 0) return RMLX_OK;
    l.chunks = (a.M + 15) / 16;
    l.wgs = ring_workgroups((uint64_t)a.N * a.K * bits / 8);
    l.share = a.N / l.wgs;
    l.over = a.N - l.share * l.wgs;
  }
  return launch_format(l, plan, bits, gs, s);
}

bool qmv_ring_gather_supported(uint32_t N, uint32_t K, uint32_t group_size, uint32_t entries, uint32_t per, uint32_t n_experts, int32_t x_dtype) {
  const uint64_t rows = (uint64_t)entries * per;
  // (a workgroup's share lies in at most four chunks: there are at most twice as many of these as workgroups)
  const uint64_t chunks = rows / 16 + (entries < n_experts ? entries : n_experts + 1);
  return per >= 1 && per <= 16 && entries <= kMaxEntries && n_experts < kNoExpert && qmv_ring_supported(N, K, group_size, 4) &&
         chunks <= 2 * (uint64_t)ctx().num_cus && chunks * N <= 0xFFFFFFFFull && rows * K * (x_dtype == RMLX_DTYPE_F32 ? 4 : 2) <= 0x80000000ull;
}

int32_t launch_qmv_ring_gather(const QmvArgs& a, const uint32_t* picks, uint32_t entries, uint32_t per, uint32_t n_experts, int32_t x_dtype, hipStream_t s) {
  const uint32_t gs = a.group_size;
  if (!qmv_ring_gather_supported(a.N, a.K, gs, entries, per, n_experts, x_dtype))
    return fail(RMLX_INVALID_SHAPE, "streaming qmv: unsupported gather N=%u K=%u group_size=%u, %u x %u rows", a.N, a.K, gs, entries, per);
  RingLaunch l{};
  RingPlan plan;
  ring_split(a, 4, gs, x_dtype, &plan, &l);
  l.chunks = 1;
  l.p.x_rows = entries * per;
  l.p.picks = picks; l.p.entries = entries; l.p.per = per; l.p.per_inv = (65536 + per - 1) / per; l.p.n_experts = n_experts;
  return launch_format(l, plan, 4, gs, s);
}

}  // namespace rmlx
