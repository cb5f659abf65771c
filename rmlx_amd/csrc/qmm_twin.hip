// GEMM of two workgroups per CU: four waves and 80 KB of LDS each, so that one multiplies while the other starts up or stores.  Dense launches
// and routed experts where its price is below the other tiles' (qmm_tile.hip: twin_limit; api.cpp: tile_expert_rows).
//
// A tile is 32 MI activation rows by 128 NI weight rows; every wave owns 32 NI weight rows over all activation rows and all k, so a weight is
// unpacked once per tile, into the operand registers, and at NI = 2 an activation read from LDS feeds two products (half the reads of the
// eight-wave tiles of qmm_tile.hip; of a pair: one of the gate, one of the up matrix, so silu(gate) * up needs no exchange between waves).
// Stages of 64 k by direct loads into LDS: activations in two places (a stage's place is free once its last operands are in registers, a
// quarter before its products end: there stands the loop's one barrier, and the loads of the stage after next go out), weights in three
// (they come from HBM once where every expert has one row tile: with two places their latency showed), 8-bit in two.  The instructions of a k step are pinned
// in chunks of an activation fragment: its NI products, its next read, its share of the unpacking and, behind the barrier, one load.
// Rows past the tile are loaded as zeros (products with zeros cost less power than with repeats; no traffic), k past the row as well.
//
// What bounds it: power and vector issue, as qmm_tile.hip (128 experts of 128 rows: matrix unit 0.65 of the cycles busy in gate / up, 0.51 in down, five vector
// instructions a product, at 1.45 to 1.6 GHz), but not the ends of a tile: those take 7 to 9 us of every tile of a lone workgroup per CU (2560 rows, 16384 x 1536:
// eight-wave tiles 145 us, here 119; 1551 rows, 11328 x 4544 185 / 155).  With a workgroup of eight waves that splits k in two instead (same LDS reads): 130 us, its sums meet
// in LDS behind the loop.  Routed block, 2048 tokens, top-8 of 128 experts of 1536 x 4096: 872 -> 777 us, in turn on one card
// (the card's power moves both by 5 % from one to another).
// NI = 1 (up to seven fragments) fills the chip with half the columns: 300 rows, 16384 x 4096 58.7 (256 columns) / 56.5 (128 columns, three stages) / 49.2.
#include <type_traits>

#include "tile.hpp"

namespace rmlx {
namespace {

constexpr uint32_t kStageK = 64, kWaves = 4;
template <int BITS> constexpr uint32_t kWSlots = BITS == 4 ? 3 : 2;
// LDS of a tile of 32 mi rows by 128 NI columns: two stages of activations, three (8-bit: two) of packed weights, two units of scales and biases
template <int BITS, int NI>
constexpr uint32_t twin_lds(int mi) {
  const uint32_t cols = 128 * NI, loop = 2 * mi * 32 * kStageK * 2 + kWSlots<BITS> * cols * kStageK * BITS / 8 + 2 * cols * 32;
  const uint32_t out = mi * 32 * cols * 2;
  return loop > out ? loop : out;
}

template <int BITS, int NI, int MI, bool DUAL>
__device__ __forceinline__ void twin_body(const TileParams p, const Tile t_, char* const lds) {
  static_assert(!DUAL || NI == 2, "a wave of a pair multiplies gate and up rows");
  constexpr uint32_t BM = 32 * MI, BN = 128 * NI, BNO = DUAL ? BN / 2 : BN, KB = kStageK, kWaveCols = 32 * NI;
  constexpr uint32_t kRound = kWaves * 1024, kUnitBytes = BN * 32;
  constexpr uint32_t kARow = KB * 2, kWRow = KB * BITS / 8, kABytes = BM * kARow, kWBytes = BN * kWRow, oW = 2 * kABytes, oS = oW + kWSlots<BITS> * kWBytes, kNS = kWSlots<BITS>;
  constexpr int NA = kABytes / kRound, NW = kWBytes / kRound, CW = kWRow / 16;
  const uint32_t tid = threadIdx.x, lane = tid & 63, r = lane & 31, hh = lane >> 5, wave = uni(tid >> 6);
  const uint32_t lds0 = uni((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  const uint32_t K = p.K, G = K / p.group_size, row_bytes = K * BITS / 8;
  const uint32_t rows = t_.rows, row_lo = t_.row_lo, n0 = t_.nt * BNO, cols = p.N - n0 < BNO ? p.N - n0 : BNO;
  const uint32_t stages = (K + KB - 1) / KB, s0 = uni(stages * t_.split / p.splits), s1 = uni(stages * (t_.split + 1) / p.splits);

  // ---- where a wave's loads come from -----------------------------------------------------------------------------------
  // Chunks of a row lie xor-ed with its number, on the address that a lane loads from, so that operand reads spread over the banks.
  auto at = [](const void* q, uint64_t o) { return static_cast<const void*>(static_cast<const char*>(q) + o); };
  const bool mapped = p.row_map != nullptr;  // (of a grouped launch: rows from anywhere in x, which is at most 2 GiB then)
  const u4 xr = mapped ? rsrc(p.x, (uint64_t)p.x_rows * K * 2) : rsrc(at(p.x, (uint64_t)row_lo * K * 2), (uint64_t)rows * K * 2);
  const uint32_t a_row = wave * 8 + lane / 8, ca16 = ((lane % 8) ^ ((a_row >> 1) & 7)) * 16;  // (a load of a wave: 8 rows)
  uint32_t aoff[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) {
    uint32_t m = q * 32 + a_row;
    const bool in = m < rows;
    if (mapped) m = p.row_map[row_lo + (in ? m : 0)];
    aoff[q] = in ? m * K * 2 + ca16 : kOutside;
  }
  // weights: LDS row li = column li of the tile; of a pair: column 32 (li / 64) + li % 32 of the gate (li & 32 = 0) or up matrix
  auto w_key = [](uint32_t li) -> uint32_t { return CW == 4 ? (li >> 2) & 3 : (li >> 3) & 1; };
  auto col_of = [&](uint32_t li) -> uint32_t { const uint32_t c = DUAL ? (li >> 6) * 32 + (li & 31) : li; return c < cols ? c : cols - 1; };
  const uint64_t wbase = (uint64_t)t_.expert * p.estride_w * 4 + (uint64_t)n0 * row_bytes;
  constexpr uint32_t kWPiece = 64 / CW;
  const uint32_t w_li = wave * kWPiece + lane / CW, cw16 = ((lane % CW) ^ w_key(w_li)) * 16;
  u4 wr[NW];
  uint32_t woff[NW];
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    wr[q] = rsrc(at(DUAL && ((q * kWaves + wave) * kWPiece & 32) != 0 ? p.w1 : p.w, wbase), (uint64_t)cols * row_bytes);
    woff[q] = col_of(q * kWaves * kWPiece + w_li) * row_bytes + cw16;
  }
  // scales and biases: 16 bytes (eight groups) a row, a unit's scales before its biases.  A unit that would run past the row starts earlier;
  // where a row has fewer groups, the last rows' loads start earlier.
  const uint64_t sbase = (uint64_t)t_.expert * p.estride_s * 2;
  auto sb_row = [&](uint32_t c) -> uint32_t {
    const uint32_t o = (n0 + c) * G * 2, last = p.N * G * 2 - 16;
    return o < last || G >= 8 ? o : last;
  };
  const bool s_up = DUAL && (wave & 2) != 0;
  const u4 sr = rsrc(at(NI == 1 && wave >= 2 ? p.b : (s_up ? p.s1 : p.s), sbase), (uint64_t)p.N * G * 2);
  const u4 br = rsrc(at(s_up ? p.b1 : p.b, sbase), (uint64_t)p.N * G * 2);
  const uint32_t s_c = (wave & (DUAL || NI == 1 ? 1 : 3)) * 64 + lane, soff = sb_row(s_c < cols ? s_c : cols - 1);
  const uint32_t gshift = p.group_size == 32 ? 5 : (p.group_size == 64 ? 6 : 7), ushift = gshift - 3;  // stage -> unit
  auto unit_start = [&](uint32_t unit) { return G < 8 ? 0u : (unit * 8 < G - 8 ? unit * 8 : G - 8); };
  auto dma_sb = [&](uint32_t cond, uint32_t u) {
    const uint32_t to = lds0 + oS + (u & 1) * kUnitBytes + wave * 1024, from = soff + unit_start(u) * 2;
    dma16_if(uni(cond), to, from, sr);
    if constexpr (NI == 2) dma16_if(uni(cond), to + BN * 16, from, br);
  };

  // what goes out next: activations ta bytes and weights tw bytes into their rows.  Past the end of the row, or of this split, a lane's
  // offset goes out of range for good
  const uint32_t base = lds0 + wave * 1024, a_end = s1 * kARow < K * 2 ? s1 * kARow : K * 2, w_end = s1 * kWRow < row_bytes ? s1 * kWRow : row_bytes;
  uint32_t ta = s0 * kARow, tw = s0 * kWRow, w_slot = 0;
  auto dma_a = [&](auto slotc, auto qc) {
    constexpr int q = decltype(qc)::value;
    if constexpr (q < NA) dma16_at<decltype(slotc)::value * kABytes + q * kRound>(base, aoff[q], xr, ta);
  };
  auto dma_w = [&](auto qc) {
    constexpr int q = decltype(qc)::value;
    dma16_at<oW + q * kRound>(base + w_slot, woff[q], wr[q], tw);
  };
  auto clip = [&] {
    if (ta + kARow > a_end || tw + kWRow > w_end) {
#pragma unroll
      for (int q = 0; q < NA; ++q) aoff[q] = ta + ca16 < a_end ? aoff[q] : kOutside;
#pragma unroll
      for (int q = 0; q < NW; ++q) woff[q] = tw + cw16 < w_end ? woff[q] : kOutside;
    }
  };
  auto a_next = [&] { ta += kARow; };
  auto w_next = [&] { tw += kWRow; w_slot = w_slot == (kNS - 1) * kWBytes ? 0 : w_slot + kWBytes; };
  auto each = [&](auto n, auto f) {
    auto go = [&](auto self, auto q) {
      if constexpr (decltype(q)::value < decltype(n)::value) {
        f(q);
        self(self, std::integral_constant<int, decltype(q)::value + 1>{});
      }
    };
    go(go, std::integral_constant<int, 0>{});
  };

  // ---- operands: lane (r, hh) of k step j multiplies k = 32 hh + 8 j .. + 7 of the stage ------------------------------------------
  constexpr int WW = BITS;  // words of a lane, stage and weight row
  uint32_t a_rd[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) a_rd[j] = r * kARow + (((hh * 4 + j) ^ ((r >> 1) & 7)) * 16);
  uint32_t w_rd[WW / 4];
#pragma unroll
  for (int v = 0; v < WW / 4; ++v) w_rd[v] = oW + (wave * kWaveCols + r) * kWRow + ((hh * (WW / 4) + v) ^ w_key(r)) * 16;
  uint32_t sb_rd[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) {
    const uint32_t c = DUAL ? wave * 32 + r : wave * kWaveCols + ni * 32 + r, cc = c < cols ? c : cols - 1;
    sb_rd[ni] = oS + ((DUAL ? ni * 128 : 0) + c) * 16 + ((n0 + cc) * G * 2 - sb_row(cc));
  }
  const uint32_t own_group = p.group_size == 32 ? hh * 2 : 0;  // (the lane's half of a stage is a group of its own)
  // bytes of the group's place in its row (of the last group, past the end), and what a unit that starts earlier adds
  const uint32_t gb_last = (G - 1) * 2, unit_last = (G - 1) / 8 * 16, early = unit_last - unit_start((G - 1) / 8) * 2;
  uint32_t t_read = s0;
  uint32_t wq[NI][WW], sraw[NI], braw[NI];
  uint32_t r_slot = 0;
  auto load_w = [&] {
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int v = 0; v < WW / 4; ++v) {
        const u4 q = *reinterpret_cast<const u4*>(lds + r_slot + w_rd[v] + ni * 32 * kWRow);
        wq[ni][4 * v] = q.x; wq[ni][4 * v + 1] = q.y; wq[ni][4 * v + 2] = q.z; wq[ni][4 * v + 3] = q.w;
      }
    r_slot = r_slot == (kNS - 1) * kWBytes ? 0 : r_slot + kWBytes;
    const uint32_t gb = ((t_read * KB) >> gshift) * 2, x = gb < gb_last ? gb : gb_last, so = (x & 15) + (x / 16 & 1) * kUnitBytes + (x >= unit_last ? early : 0);
    const uint32_t own = x < gb_last ? own_group : 0;
    ++t_read;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      sraw[ni] = *reinterpret_cast<const uint16_t*>(lds + sb_rd[ni] + own + so);
      braw[ni] = *reinterpret_cast<const uint16_t*>(lds + sb_rd[ni] + own + so + BN * 16);
    }
  };
  h2 s2[NI], b2[NI];
  auto pick_sb = [&] {
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const _Float16 sv = __builtin_bit_cast(_Float16, (uint16_t)sraw[ni]), bv = __builtin_bit_cast(_Float16, (uint16_t)braw[ni]);
      s2[ni] = (h2){sv, sv};
      b2[ni] = (h2){bv, bv};
    }
  };
  // pair c of the 8 weights of k step j (two vector instructions and the share of the word's four or five)
  uint32_t even[NI], odd[NI], bytes[NI];
  auto unpack = [&](h8& o, int ni, int j, int c) {
    h2 q;
    if constexpr (BITS == 4) {
      if (c == 0) { even[ni] = wq[ni][j % WW] & 0x0F0F0F0Fu; odd[ni] = (wq[ni][j % WW] >> 4) & 0x0F0F0F0Fu; }
      if (c % 2 == 0) bytes[ni] = __builtin_amdgcn_perm(odd[ni], even[ni], c == 0 ? 0x05010400u : 0x07030602u);
      q = c % 2 == 0 ? (h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(bytes[ni], 512.0f, false) : (h2)__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(bytes[ni], 512.0f, true);
    } else {
      const h2 k = {(_Float16)1024.0f, (_Float16)1024.0f};
      q = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, wq[ni][(2 * j + c / 2) % WW], c % 2 == 0 ? 0x04010400u : 0x04030402u)) - k;
    }
    const h2 v = q * s2[ni] + b2[ni];
    o[2 * c] = v[0]; o[2 * c + 1] = v[1];
  };
  auto read_a = [&](uint32_t slot, int i, int j) -> h8 { return *reinterpret_cast<const h8*>(lds + slot * kABytes + a_rd[j] + i * 32 * kARow); };

  f16v acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][ni][e] = 0.f;

  // ---- k loop: behind the barrier in stage t, activations of stage t + 2 and weights of stage t + kNS go out -------------------
  const uint32_t umask = (1u << ushift) - 1;
  {
    clip();
    dma_sb(1, s0 >> ushift);
#pragma unroll
    for (uint32_t i = 1; i < kNS; ++i) dma_sb(((s0 + i) & umask) == 0, (s0 + i) >> ushift);
    using std::integral_constant;
    auto weights = [&] { each(integral_constant<int, NW>{}, dma_w); w_next(); };
    weights();
    each(integral_constant<int, NA>{}, [&](auto q) { dma_a(integral_constant<int, 0>{}, q); });
    a_next();
    clip();
    weights();
    each(integral_constant<int, NA>{}, [&](auto q) { dma_a(integral_constant<int, 1>{}, q); });
    a_next();
    clip();
    if constexpr (kNS > 2) {
      weights();
      clip();
    }
  }
  wait_dma_and_barrier<NA + NW * (kNS - 1)>();
  h8 a[MI];
  h8 wf[NI];
  load_w();
#pragma unroll
  for (int i = 0; i < MI; ++i) a[i] = read_a(0, i, 0);
  pick_sb();
#pragma unroll
  for (int c = 0; c < 4 * NI; ++c) unpack(wf[c / 4], c / 4, 0, c % 4);
  uint32_t t = s0;
  auto step = [&](auto ic) -> bool {
    constexpr int I = decltype(ic)::value;
    auto kstep = [&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (j == 3) {
        wait_dma_and_barrier<NW * (kNS - 2)>();  // stage t has been read by all, stage t + 1 has arrived
        load_w();
        dma_sb(((t + kNS) & umask) == 0, (t + kNS) >> ushift);
      }
      h8 wx[NI];
      constexpr int kFirst = j < 3 ? 0 : (MI > 3 ? 2 : MI - 1);
      auto chunk = [&](auto self, auto ic2) {
        constexpr int i = decltype(ic2)::value;
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) acc[i][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[ni], a[i], acc[i][ni], 0, 0, 0);
        a[i] = j < 3 ? read_a(I, i, j + 1) : read_a(I ^ 1, i, 0);
        if constexpr (j == 3) {
          if constexpr (i == kFirst) pick_sb();
          dma_a(ic, ic2);
          if constexpr (i == MI - 1) {
            each(std::integral_constant<int, NW>{}, dma_w);
            a_next();
            w_next();
          }
        }
#pragma unroll
        for (int c = 0; c < 4 * NI; ++c)
          if (kFirst + c * (MI - kFirst) / (4 * NI) == i) unpack(wx[c / 4], c / 4, (j + 1) & 3, c % 4);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i + 1 < MI) self(self, std::integral_constant<int, i + 1>{});
      };
      chunk(chunk, std::integral_constant<int, 0>{});
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) {
        wf[ni] = wx[ni];
        if constexpr (j == 3) asm volatile("" : "+v"(wf[ni]));  // (unpacked here, between the products, not behind the loop's branches)
      }
    };
    kstep(std::integral_constant<int, 0>{});
    kstep(std::integral_constant<int, 1>{});
    kstep(std::integral_constant<int, 2>{});
    kstep(std::integral_constant<int, 3>{});
    clip();
    return ++t < s1;
  };
  while (step(std::integral_constant<int, 0>{}) && step(std::integral_constant<int, 1>{})) {
  }
  wait_dma_and_barrier<0>();

  if (t_.zeros) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][ni][e] = 0.f;
  }

  // ---- store: fragment (i, ni) of a lane holds activation row 32 i + r, weight rows 8 eg + 4 hh + 0 .. 3 of the wave's 32
  constexpr uint32_t U = BNO / 8, kKey = U < 32 ? U - 1 : 31;
  // (no plan splits K; without the choice of partial sums here the f32 store is laid out otherwise and down projections are slower, 15 experts of 1024 x 512,
  // group size 32, 343 rows each 56.6 / 62.4 us, 128 of 4096 x 1536, 128 rows 770 / 778)
  const bool f32 = !DUAL && (p.partial != nullptr || p.out_f32);
  float* const o32 = p.partial != nullptr ? p.partial + (uint64_t)t_.split * p.M * p.N : static_cast<float*>(p.out);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const uint32_t m = i * 32 + r;
    auto put = [&](f4 v, uint32_t c) {  // columns c .. c + 3 of row m
      if (f32) {
        if (m >= rows) return;
        float* q = o32 + (uint64_t)(row_lo + m) * p.N + n0 + c;
        if (c + 4 <= cols) reinterpret_cast<f4_any*>(q)->v = v;
        else
          for (uint32_t e = 0; e < 4; ++e)
            if (c + e < cols) q[e] = v[e];
      } else {
        if (!DUAL && p.epi_kind != EPI_NONE && m < rows && c < cols) tile_epilogue(p, (uint64_t)(row_lo + m) * p.N + n0 + c, cols - c, v);
        const h2 lo = {(_Float16)v[0], (_Float16)v[1]}, hi = {(_Float16)v[2], (_Float16)v[3]};
        *reinterpret_cast<u2*>(lds + (m * U + ((c >> 3) ^ (m & kKey))) * 16 + (c & 4) * 2) = (u2){h2bits(lo), h2bits(hi)};
      }
    };
#pragma unroll
    for (int eg = 0; eg < 4; ++eg) {
      auto sum = [&](int ni) { return (f4){acc[i][ni][eg * 4], acc[i][ni][eg * 4 + 1], acc[i][ni][eg * 4 + 2], acc[i][ni][eg * 4 + 3]}; };
      if constexpr (DUAL) {
        const f4 g = sum(0);
        f4 v = sum(1);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= g[e] / (1.0f + __expf(-g[e]));
        put(v, wave * 32 + 8 * eg + 4 * hh);
        __builtin_amdgcn_sched_barrier(0);
      } else {
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) put(sum(ni), wave * kWaveCols + ni * 32 + 8 * eg + 4 * hh);
      }
    }
  }
  if (f32) return;
  __syncthreads();
  for (uint32_t g = tid; g < BM * U; g += kWaves * 64) {
    const uint32_t m = g / U, u = g % U, c = u * 8;
    if (m >= rows || c >= cols) continue;
    const u4 v = *reinterpret_cast<const u4*>(lds + (m * U + (u ^ (m & kKey))) * 16);
    __half* q = static_cast<__half*>(p.out) + (uint64_t)(row_lo + m) * p.N + n0 + c;
    if (c + 8 <= cols) {
      reinterpret_cast<u4_any*>(q)->v = v;
    } else {
      const h8 hv = __builtin_bit_cast(h8, v);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (c + e < cols) reinterpret_cast<_Float16*>(q)[e] = hv[e];
    }
  }
}

template <int BITS, int NI, int MIMAX, bool DUAL>
__global__ __launch_bounds__(256, 2) __attribute__((aligned(16384))) void qmm_twin_kernel(TileParams p) {
  __shared__ __align__(1024) char lds[twin_lds<BITS, NI>(MIMAX)];
  static_assert(sizeof(lds) <= 80 * 1024, "two workgroups per CU");
  Tile t;
  if (!tile_of<DUAL ? 1 : 4>(p, MIMAX * 32, &t)) return;
  const uint32_t frags = (t.rows + 31) / 32;
  auto go = [&](auto self, auto mi) {
    constexpr int MI = decltype(mi)::value;
    if (MI == MIMAX || frags <= MI) twin_body<BITS, NI, MI, DUAL>(p, t, lds);
    else if constexpr (MI < MIMAX) self(self, std::integral_constant<int, MI + 1>{});
  };
  go(go, std::integral_constant<int, 1>{});
}
}  // namespace
void launch_qmm_twin(const TileParams& p, uint32_t bits, uint32_t wn, dim3 grid, hipStream_t s) {
  auto go = [&](auto b) {
    constexpr int B = decltype(b)::value;
    if (p.w1 != nullptr) hipLaunchKernelGGL((qmm_twin_kernel<B, 2, B == 4 ? 5 : 4, true>), grid, dim3(256), 0, s, p);
    else if (wn == 8) hipLaunchKernelGGL((qmm_twin_kernel<B, 2, B == 4 ? 5 : 4, false>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((qmm_twin_kernel<B, 1, 7, false>), grid, dim3(256), 0, s, p);
  };
  if (bits == 4) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 8>{});
}
}  // namespace rmlx
