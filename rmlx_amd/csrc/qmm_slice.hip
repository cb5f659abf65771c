// GEMM of small tiles whose waves share a tile's k: 32 or 64 activation rows x 64 WN weight rows on eight waves, KG = 8 / WN of
// them along k (four waves for 8-bit experts).  A stage holds 16 KS KG k of both operands in LDS; wave (wn, kg) multiplies its 64
// weight rows with all activation rows over 16 KS k of it, and the KG partial sums meet in LDS at the end.
//
// Against the tiles of qmm_tile.hip, where every wave runs all k over 32 weight rows: two waves per SIMD at a few workgroups per
// chip, a weight fragment pair per activation read (half the LDS reads), a barrier per 128 or 256 k instead of 64.  Loads travel
// straight into LDS; ring places are compile-time constants (the loop is unrolled over the ring) and offsets along k sit in scalar
// registers, because at this size a wave's own instruction chain is the limit: 45 scalar instructions a stage instead of 25 cost 10 %.
// What bounds it: with loads, barriers and operand reads all taken out, the unpacking and the products of a 64 x 128 x 4096 tile
// still take 10 us, of 15.5 us in the whole kernel; products and unpacking overlap (measured: 6 vector instructions in the shadow of
// every product cost nothing), the LDS reads between two barriers do not.  Reading operands one stage ahead into a second register
// set (25.2 against 23.1 us at 512 x 4096 x 4096), a barrier inside the stage, sixteen waves (25.1) and scales turned by group in
// LDS (24.3) were no faster; rings of less than two stages of distance are (latency of about 1 us per stage).
// Measured, 4096 x 4096, 4-bit, weights from HBM, tiles of qmm_tile.hip / these: 32 rows 18.8 / 11.2 us, 64 rows 20.7 / 11.2, 256
// rows 21.1 / 14.8; 512 rows 26.9 / 23.1; 13 rows, 14336 x 4096, 8-bit 26.0 / 17.1; 128 rows, 12288 x 4096 25.6 / 21.6, 8-bit
// 29.2 / 27.9.  On 530 shapes of 9 to 1200 rows the best of both is 7 to 18 % ahead of those tiles alone (against the older GEMMs: see the
// dispatch; 32 rows, 4096 x 4096 stay on the register-weights GEMM at 9.1).
#include <type_traits>

#include "tile.hpp"

namespace rmlx {
namespace {

// LDS: S stages of activations (64 KG bytes a row) and packed weights (4 KG BITS bytes a row), a ring of scales and biases (units of
// eight groups)
constexpr int slice_units(int kb, int S) { const int n = ((S - 1) * kb + 255) / 256 + 1; return n <= 2 ? 2 : (n <= 4 ? 4 : 8); }
constexpr uint32_t slice_lds(int bits, int mi, int wn, int kg, int ks, int S) {
  const int kb = 16 * ks * kg;
  return S * (mi * 32 * kb * 2 + wn * 64 * kb * bits / 8) + slice_units(kb, S) * wn * 2048;
}
constexpr uint32_t slice_lds_all(int bits, int mi, int wn, int kg, int ks, int S) {
  const uint32_t loop = slice_lds(bits, mi, wn, kg, ks, S), sums = wn * kg * 8192 + mi * 32 * wn * 64 * 2;
  return loop > sums ? loop : sums;
}

template <int BITS, int MI, int WN, int KG, int KS, int S, bool DUAL, bool EXACT>
__device__ __forceinline__ void slice_body(const TileParams p, const Tile t_, char* const lds) {
  constexpr int kWaves = WN * KG, BM = 32 * MI, BN = 64 * WN, BNO = DUAL ? BN / 2 : BN, KB = 16 * KS * KG;
  constexpr uint32_t kRound = kWaves * 1024, kUnitBytes = WN * 2048;
  constexpr uint32_t kARow = KB * 2, kWRow = KB * BITS / 8, kABytes = BM * kARow, kWBytes = BN * kWRow, kStage = kABytes + kWBytes;
  constexpr int CA = kARow / 16, CW = kWRow / 16;              // 16-byte chunks of a stage row
  constexpr int NA = kABytes / kRound, NW = kWBytes / kRound, NL = NA + NW, kUnits = slice_units(KB, S);
  static_assert(NA * kRound == kABytes && NW * kRound == kWBytes && kWaves >= 4, "whole rounds of the waves");
  constexpr uint32_t oS = S * kStage;
  const uint32_t tid = threadIdx.x, lane = tid & 63, r = lane & 31, hh = lane >> 5, wave = uni(tid >> 6), wn = wave % WN, kg = wave / WN;
  const uint32_t lds0 = uni((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  const uint32_t K = p.K, G = K / p.group_size, row_bytes = K * BITS / 8;
  const uint32_t rows = t_.rows, row_lo = t_.row_lo, n0 = t_.nt * BNO, cols = p.N - n0 < BNO ? p.N - n0 : BNO;
  const uint32_t stages = (K + KB - 1) / KB, s0 = uni(stages * t_.split / p.splits), s1 = uni(stages * (t_.split + 1) / p.splits);

  // ---- where a wave's loads come from -----------------------------------------------------------------------------------
  // Chunks of a row lie xor-ed with its number, so that operand reads spread over the banks; the xor is made on the address that a
  // lane loads from.  Rows past the tile's last repeat it; k past the row is loaded as zeros.
  auto at = [](const void* q, uint64_t o) { return static_cast<const void*>(static_cast<const char*>(q) + o); };
  const bool mapped = p.row_map != nullptr;  // (of a grouped launch: rows from anywhere in x, which is at most 2 GiB then)
  const u4 xr = mapped ? rsrc(p.x, (uint64_t)p.x_rows * K * 2) : rsrc(at(p.x, (uint64_t)row_lo * K * 2), (uint64_t)rows * K * 2);
  constexpr uint32_t kAPiece = 64 / CA, kWPiece = 64 / CW;    // rows of a 1 KB load
  static_assert(kWaves * kAPiece % 16 == 0 && kWaves * kWPiece % 16 == 0, "one xor for all loads of a lane");
  const uint32_t a_row = wave * kAPiece + lane / CA, ca16 = ((lane % CA) ^ (a_row & 15)) * 16;
  uint32_t aoff[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) {
    uint32_t m = q * kWaves * kAPiece + a_row;
    m = m < rows ? m : rows - 1;
    if (mapped) m = p.row_map[row_lo + m];
    aoff[q] = m * K * 2 + ca16;
  }
  // LDS row li of the weights: column wn 64 + ni 32 + r of the tile; of a pair: column wn 32 + r of the gate (ni = 0) or up matrix
  auto w_key = [](uint32_t li) -> uint32_t { return CW == 4 ? (li >> 2) & 3 : (CW == 8 ? (li >> 1) & 7 : li & 15); };
  auto col_of = [&](uint32_t li) -> uint32_t { const uint32_t c = DUAL ? (li >> 6) * 32 + (li & 31) : li; return c < cols ? c : cols - 1; };
  const uint64_t wbase = (uint64_t)t_.expert * p.estride_w * 4 + (uint64_t)n0 * row_bytes;
  const uint32_t w_li = wave * kWPiece + lane / CW, cw16 = ((lane % CW) ^ w_key(w_li)) * 16;
  u4 wr[NW];
  uint32_t woff[NW];
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    wr[q] = rsrc(at(DUAL && ((q * kWaves + wave) * kWPiece & 32) != 0 ? p.w1 : p.w, wbase), (uint64_t)cols * row_bytes);
    woff[q] = col_of(q * kWaves * kWPiece + w_li) * row_bytes + cw16;
  }
  // scales and biases: 16 bytes (eight groups) a row; waves 0 and 1 load the scales of half of the rows each, 2 and 3 the biases.  A
  // unit that would run past the row starts earlier; where a row has fewer groups, the last rows' loads start earlier.
  constexpr uint32_t kHalf = BN / 2;
  const uint64_t sbase = (uint64_t)t_.expert * p.estride_s * 2;
  auto sb_row = [&](uint32_t c) -> uint32_t {
    const uint32_t o = (n0 + c) * G * 2, last = p.N * G * 2 - 16;
    return o < last || G >= 8 ? o : last;
  };
  const bool s_up = DUAL && (wave & 1) != 0;
  const u4 sr = rsrc(at(wave & 2 ? (s_up ? p.b1 : p.b) : (s_up ? p.s1 : p.s), sbase), (uint64_t)p.N * G * 2);
  const uint32_t s_c = (DUAL ? 0 : (wave & 1) * kHalf) + lane % kHalf, soff = sb_row(s_c < cols ? s_c : cols - 1);
  const uint32_t gshift = p.group_size == 32 ? 5 : (p.group_size == 64 ? 6 : 7);
  const uint32_t ushift = gshift + 3 - (KB == 256 ? 8 : 7);      // stage -> unit
  auto unit_start = [&](uint32_t unit) { return G < 8 ? 0u : (unit * 8 < G - 8 ? unit * 8 : G - 8); };
  auto dma_sb = [&](uint32_t u) {
    if (kHalf == 64 || lane < kHalf) dma16(lds0 + oS + u % kUnits * kUnitBytes + wave * kHalf * 16, soff + unit_start(u) * 2, sr);
  };
  // the next stage to go out: byte offset of its activations in a row (of its last stage, past the end) and bytes left from there
  const uint32_t ta_last = (s1 - 1) * kARow;
  uint32_t ta = s0 * kARow;
  int32_t left = (int32_t)(K * 2 - ta);
  const int32_t ca = ca16, cw = cw16 * (16 / BITS);
  const uint32_t base = lds0 + wave * 1024;
  auto dma_stage = [&](auto slotc) {
    constexpr uint32_t kSlot = decltype(slotc)::value * kStage;
    const uint32_t tw = ta * BITS / 16;
    const bool a_ok = ca < left, w_ok = cw < left;
    dma16_at<kSlot>(base, a_ok ? aoff[0] : kOutside, xr, ta);
    if constexpr (NA > 1) dma16_at<kSlot + kRound>(base, a_ok ? aoff[1] : kOutside, xr, ta);
    if constexpr (NA > 2) dma16_at<kSlot + 2 * kRound>(base, a_ok ? aoff[2] : kOutside, xr, ta);
    if constexpr (NA > 3) dma16_at<kSlot + 3 * kRound>(base, a_ok ? aoff[3] : kOutside, xr, ta);
    dma16_at<kSlot + kABytes>(base, w_ok ? woff[0] : kOutside, wr[0], tw);
    if constexpr (NW > 1) dma16_at<kSlot + kABytes + kRound>(base, w_ok ? woff[1] : kOutside, wr[1], tw);
    if constexpr (NW > 2) dma16_at<kSlot + kABytes + 2 * kRound>(base, w_ok ? woff[2] : kOutside, wr[2], tw);
    if constexpr (NW > 3) dma16_at<kSlot + kABytes + 3 * kRound>(base, w_ok ? woff[3] : kOutside, wr[3], tw);
    static_assert(NA <= 4 && NW <= 4, "loads of a stage");
    left = ta < ta_last ? left - (int32_t)kARow : 0;
    ta = ta < ta_last ? ta + kARow : ta_last;
  };

  // ---- operands: lane (r, hh) of k step j multiplies k = 16 KS kg + 8 KS hh + 8 j .. + 7 of the stage ---------------------------
  struct Ops { h8 a[MI][KS]; uint32_t w[2][KS * BITS / 4]; uint32_t s[2], b[2]; };
  uint32_t a_rd[KS], sb_rd[2];
#pragma unroll
  for (int j = 0; j < KS; ++j) a_rd[j] = r * kARow + (((kg * 2 * KS + hh * KS + j) ^ (r & 15)) * 16);
  constexpr int kWLane = KS * BITS, NWP = (kWLane + 15) / 16;  // a lane's bytes, and the reads they take
  uint32_t w_rd[NWP];
#pragma unroll
  for (int v = 0; v < NWP; ++v) {
    const uint32_t at = (kg * 2 + hh) * kWLane + v * 16;
    w_rd[v] = kABytes + (wn * 64 + r) * kWRow + ((at / 16) ^ w_key(r)) * 16 + at % 16;
  }
  const uint32_t own_group = KS == 4 && p.group_size == 32 ? hh * 2 : 0;  // (of 64 k of a wave: the lane's half is a group of its own)
#pragma unroll
  for (int ni = 0; ni < 2; ++ni) {
    const uint32_t c = col_of(wn * 64 + ni * 32 + r);
    const uint32_t piece = DUAL ? ni : (wn * 64 + ni * 32) / kHalf, pos = DUAL ? wn * 32 + r : (wn * 64 + ni * 32) % kHalf + r;
    sb_rd[ni] = oS + piece * kHalf * 16 + pos * 16 + ((n0 + c) * G * 2 - sb_row(c));
  }
  // bytes of the group's place in its row (of the last group, past the end), and what a unit that starts earlier adds
  const uint32_t gb_step = (KB >> gshift) * 2, gb_last = (G - 1) * 2, unit_last = (G - 1) / 8 * 16, early = unit_last - unit_start((G - 1) / 8) * 2;
  uint32_t gb = ((s0 * KB + kg * KS * 16) >> gshift) * 2;
  auto fetch = [&](Ops& o, uint32_t slot) {
    const char* st = lds + slot * kStage;
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      if constexpr (kWLane == 8) {
        const u2 v = *reinterpret_cast<const u2*>(st + w_rd[0] + ni * 32 * kWRow);
        o.w[ni][0] = v.x; o.w[ni][1] = v.y;
      } else {
#pragma unroll
        for (int q = 0; q < NWP; ++q) {
          const u4 v = *reinterpret_cast<const u4*>(st + w_rd[q] + ni * 32 * kWRow);
          o.w[ni][4 * q] = v.x; o.w[ni][4 * q + 1] = v.y; o.w[ni][4 * q + 2] = v.z; o.w[ni][4 * q + 3] = v.w;
        }
      }
    }
    const uint32_t x = gb < gb_last ? gb : gb_last, so = (x & 15) + x / 16 % kUnits * kUnitBytes + (x >= unit_last ? early : 0);
    const uint32_t own = KS == 4 && x < gb_last ? own_group : 0;
    gb += gb_step;
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      o.s[ni] = *reinterpret_cast<const uint16_t*>(lds + sb_rd[ni] + own + so);
      o.b[ni] = *reinterpret_cast<const uint16_t*>(lds + sb_rd[ni] + own + so + kHalf * 32);
    }
#pragma unroll
    for (int j = 0; j < KS; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i) o.a[i][j] = *reinterpret_cast<const h8*>(st + a_rd[j] + i * 32 * kARow);
  };
  f16v acc[MI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][ni][e] = 0.f;
  auto compute = [&](const Ops& o) {
#pragma unroll
    for (int j = 0; j < KS; ++j)
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        const _Float16 sv = __builtin_bit_cast(_Float16, (uint16_t)o.s[ni]), bv = __builtin_bit_cast(_Float16, (uint16_t)o.b[ni]);
        const h2 s2 = {sv, sv}, b2 = {bv, bv};
        Weights w;
        if constexpr (EXACT && BITS == 4) w = split_q4(o.w[ni][j], (float)sv, (float)bv);
        else if constexpr (EXACT) w = split_q8(o.w[ni][2 * j], o.w[ni][2 * j + 1], (float)sv, (float)bv);
        else if constexpr (BITS == 4) w.hi = weights_q4(o.w[ni][j], s2, b2);
        else w.hi = weights_q8(o.w[ni][2 * j], o.w[ni][2 * j + 1], s2, b2);
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[i][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w.hi, o.a[i][j], acc[i][ni], 0, 0, 0);
        if constexpr (EXACT)
#pragma unroll
          for (int i = 0; i < MI; ++i) acc[i][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w.lo, o.a[i][j], acc[i][ni], 0, 0, 0);
      }
  };

  // ---- k loop: stage t + S - 1 goes out, into the place that stage t - 1 has left, while stage t is multiplied ---------------
  const uint32_t umask = (1u << ushift) - 1;
  auto sb_from = [&](uint32_t t) { return wave < 4 ? ((t + umask) >> ushift) : 0x7FFFFFFFu >> ushift; };  // first unit that begins at or after stage t
  {
    if (wave < 4) {
      if ((s0 & umask) != 0) dma_sb(s0 >> ushift);
      for (uint32_t u = (s0 + umask) >> ushift; (u << ushift) < s0 + S - 1; ++u) dma_sb(u);
    }
    auto first = [&](auto self, auto i) {
      constexpr int I = decltype(i)::value;
      if constexpr (I < S - 1) { dma_stage(i); self(self, std::integral_constant<int, I + 1>{}); }
    };
    first(first, std::integral_constant<int, 0>{});
  }
  uint32_t unit = sb_from(s0 + S - 1), unit_at = unit << ushift;  // the next unit of scales to go out, with this stage
  uint32_t t = s0;
  auto step = [&](auto ic) -> bool {
    constexpr int I = decltype(ic)::value;
    wait_dma_and_barrier<(S - 2) * NL>();
    if (t + (S - 1) == unit_at) {
      dma_sb(unit);
      ++unit;
      unit_at += umask + 1;
    }
    Ops o;
    fetch(o, I);
    dma_stage(std::integral_constant<int, (I + S - 1) % S>{});
    compute(o);
    return ++t < s1;
  };
  auto round = [&](auto self, auto ic) -> bool {
    constexpr int I = decltype(ic)::value;
    if constexpr (I == S) return true;
    else return step(ic) && self(self, std::integral_constant<int, I + 1>{});
  };
  while (round(round, std::integral_constant<int, 0>{})) {
  }
  wait_dma_and_barrier<0>();

  // ---- the KG sums of a value, added in order: fragment row by fragment row through LDS ------------------------------------
  // lane (r, hh) of fragment (i, ni): activation row 32 i + r, weight rows 8 eg + 4 hh + 0 .. 3 of the 32
  constexpr uint32_t U = BNO / 8, kKey = U < 32 ? U - 1 : 31;  // 16-byte units of an output row, xor-ed with the row
  f4* const sums = reinterpret_cast<f4*>(lds);
  char* const outs = lds + kWaves * 8192;
  const bool f32 = !DUAL && (p.partial != nullptr || p.out_f32);
  float* const o32 = p.partial != nullptr ? p.partial + (uint64_t)t_.split * p.M * p.N : static_cast<float*>(p.out);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    if (i > 0) __syncthreads();
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int eg = 0; eg < 4; ++eg)
        sums[((wave * 2 + ni) * 4 + eg) * 64 + lane] = (f4){acc[i][ni][eg * 4], acc[i][ni][eg * 4 + 1], acc[i][ni][eg * 4 + 2], acc[i][ni][eg * 4 + 3]};
    __syncthreads();
    auto total = [&](uint32_t ni, uint32_t eg) {
      f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int z = 0; z < KG; ++z) v += sums[(((z * WN + wn) * 2 + ni) * 4 + eg) * 64 + lane];
      return v;
    };
    const uint32_t m = i * 32 + r;
    auto put = [&](f4 v, uint32_t c) {  // columns c .. c + 3 of row m
      if (t_.zeros) v = (f4){0.f, 0.f, 0.f, 0.f};
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
        *reinterpret_cast<u2*>(outs + (m * U + ((c >> 3) ^ (m & kKey))) * 16 + (c & 4) * 2) = (u2){h2bits(lo), h2bits(hi)};
      }
    };
    if constexpr (DUAL) {
#pragma unroll
      for (int q = 0; q < (KG < 4 ? 4 / KG : 1); ++q) {
        const uint32_t eg = q * KG + kg;
        if (eg >= 4) break;
        const f4 g = total(0, eg);
        f4 v = total(1, eg);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= g[e] / (1.0f + __expf(-g[e]));
        put(v, wn * 32 + 8 * eg + 4 * hh);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8 / KG; ++q) {
        const uint32_t u = q * KG + kg;
        put(total(u / 4, u % 4), wn * 64 + u / 4 * 32 + 8 * (u % 4) + 4 * hh);
      }
    }
  }
  if (f32) return;
  __syncthreads();
  for (uint32_t g = tid; g < BM * U; g += kWaves * 64) {
    const uint32_t m = g / U, u = g % U, c = u * 8;
    if (m >= rows || c >= cols) continue;
    const u4 v = *reinterpret_cast<const u4*>(outs + (m * U + (u ^ (m & kKey))) * 16);
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

template <int BITS, int MIMAX, int WN, int KG, int KS, int S, int WPE, bool DUAL, bool EXACT>
__global__ __launch_bounds__(WN * KG * 64, WPE) void qmm_slice_kernel(TileParams p) {
  __shared__ __align__(1024) char lds[slice_lds_all(BITS, MIMAX, WN, KG, KS, S)];
  Tile t;
  if (!tile_of<DUAL ? 1 : 4>(p, MIMAX * 32, &t)) return;
  if (MIMAX == 2 && t.rows > 32) slice_body<BITS, MIMAX, WN, KG, KS, S, DUAL, EXACT>(p, t, lds);
  else slice_body<BITS, 1, WN, KG, KS, S, DUAL, EXACT>(p, t, lds);
}

template <int BITS, int MI, int WN, int KG, int KS, int S, bool DUAL>
void launch_one(const TileParams& p, dim3 grid, hipStream_t s) {
  // (two workgroups per CU where their LDS allows it)
  constexpr int kWpe = slice_lds_all(BITS, MI, WN, KG, KS, S) <= 80 * 1024 ? WN * KG / 2 : WN * KG / 4;
  if (p.exact) hipLaunchKernelGGL((qmm_slice_kernel<BITS, MI, WN, KG, KS, S, kWpe, DUAL, true>), grid, dim3(WN * KG * 64), 0, s, p);
  else hipLaunchKernelGGL((qmm_slice_kernel<BITS, MI, WN, KG, KS, S, kWpe, DUAL, false>), grid, dim3(WN * KG * 64), 0, s, p);
}

template <int BITS>
void launch_plan(const TileParams& p, const TilePlan& plan, dim3 grid, hipStream_t s) {
  constexpr bool q4 = BITS == 4;
  if (plan.wn == 2 && plan.mi == 1) launch_one<BITS, 1, 1, 8, 2, q4 ? 3 : 4, false>(p, grid, s);
  else if (plan.wn == 2) launch_one<BITS, 2, 1, 8, 2, 3, false>(p, grid, s);
  else if (plan.mi == 1) launch_one<BITS, 1, 2, 4, 4, q4 ? 4 : 3, false>(p, grid, s);
  else launch_one<BITS, 2, 2, 4, q4 ? 4 : 2, q4 ? 3 : 4, false>(p, grid, s);
}

}  // namespace

void launch_qmm_slice(const TileParams& p, uint32_t bits, const TilePlan& plan, dim3 grid, hipStream_t s) {
  if (bits == 4) launch_plan<4>(p, plan, grid, s);
  else launch_plan<8>(p, plan, grid, s);
}

int32_t launch_qmm_slice_grouped(const GroupedQmmArgs& a, uint32_t x_rows, hipStream_t s) {
  if (!qmm_tile_supported(a.N, a.K, a.group_size, a.bits) || (a.row_map != nullptr && !qmm_tile_maps_rows(x_rows, a.K)))
    return fail(RMLX_INVALID_SHAPE, "grouped qmm: unsupported shape N=%u K=%u bits=%u group_size=%u, %u rows", a.N, a.K, a.bits, a.group_size, x_rows);
  if (a.max_tiles == 0) return RMLX_OK;
  TileParams p{};
  p.w = a.w; p.s = a.s; p.b = a.b; p.w1 = a.w1; p.s1 = a.s1; p.b1 = a.b1;
  p.x = a.x; p.out = a.out; p.N = a.N; p.K = a.K; p.group_size = a.group_size;
  p.out_f32 = a.out_f32; p.exact = a.exact;
  p.tile_tab = a.tile_tab; p.n_tiles = a.n_tiles_dev; p.row_map = a.row_map; p.x_rows = x_rows;
  p.estride_w = a.expert_stride_w; p.estride_s = a.expert_stride_s;
  p.splits = 1;
  const uint32_t cols = a.w1 != nullptr ? 32 : 64;
  p.tiles_n = (a.N + cols - 1) / cols;
  const uint64_t wgs = (uint64_t)a.max_tiles * p.tiles_n;
  if (wgs > 0x7FFFFFFFull) return fail(RMLX_INVALID_SHAPE, "grouped qmm: grid too large");
  const dim3 grid((unsigned)wgs);
  if (a.bits == 4) {
    if (a.w1 != nullptr) launch_one<4, 1, 1, 8, 2, 3, true>(p, grid, s);
    else launch_one<4, 1, 1, 8, 2, 3, false>(p, grid, s);
  } else {
    if (a.w1 != nullptr) launch_one<8, 1, 1, 4, 2, 4, true>(p, grid, s);
    else launch_one<8, 1, 1, 4, 2, 4, false>(p, grid, s);
  }
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

}  // namespace rmlx
