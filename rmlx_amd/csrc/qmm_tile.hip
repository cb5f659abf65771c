// GEMM of large tiles: every 4- / 8-bit matrix the type admits at group size 32 / 64 / 128, any number of rows on either side, any K
// of whole groups; f16 activations, f32 accumulation on 32x32x16 MFMAs.
//
// A tile is 32 MI activation rows x 32 WN weight rows; wave w owns weight rows 32 w .. 32 w + 31 over all activation rows, so that a
// weight is unpacked once per tile, into the operand registers.  Everything else is arranged so that the vector ALU and the
// registers carry nothing but that unpacking:
//   - activations, packed weights, scales and biases all travel by direct loads into LDS (16 bytes per lane, 1 KB per wave), two
//     steps of 64 k ahead; LDS slots are xor-ed by row, and the xor is made on the address that a lane loads from;
//   - weights come 64 bytes of a row at a time (4-bit: two steps' worth), scales and biases eight groups at a time (dword loads
//     per 128 k cost 5 %: their 64 lanes touch 64 cache lines each);
//   - rows past the tile repeat its last row, k past the row is loaded as zeros by the range check: no other handling of ragged
//     sizes in the loop; the store goes through LDS in whole rows;
//   - the last row tile of a launch, and every tile of a grouped one, runs the loop built for the fragments it has (1 .. MI).
// K may be split over two groups of waves in the workgroup (KW = 2, one round of small tiles: 512 x 4096 x 4096 26.5 us against 29.5
// us with two workgroups and a second kernel) and over workgroups.
//
// What bounds it: power.  At 8192^3 with random data the chip runs at 1.5 GHz instead of 2.4 (a zero-filled launch is 1.5 x as
// fast in the same number of cycles; at 3001 x 14336 x 4096 1.6 GHz, with the matrix unit busy for 70 % of those cycles), so time follows the energy of a step, not its cycles: 64 unpacking instructions per wave
// and step cost 15 % and the operand reads 10 % of the launch.  That is why the large tile gives each wave all 256 rows of a few
// weight rows (2 x 4 waves of 128 x 64, half the LDS reads but every weight unpacked twice: 1143 against 1217 TFLOP/s).
// 8192^3: 903 us (1217 TFLOP/s; the library's f16 product of normal values 1515 with its second operand laid out as the weights are here, 1304 with it
// row-major, 1805 on zeros); 4096^3 122 us against 158 us on the 128 x 128 K-split tiles;
// 3001 x 14336 x 4096 bf16 416 -> 332 us.  Small tiles are bound by the unpacking of a lone wave per SIMD (7.6 cycles per dependent
// vector instruction: 0.33 of the 0.39 us of a 64-row step); most sizes that would use them are on qmm_slice.hip.
#include <cmath>
#include <type_traits>

#include "tile.hpp"

namespace rmlx {
namespace {

// (deeper rings measured no faster at any tile size: the distance of two steps covers the latency)
constexpr int kStages = 3;

// LDS of a tile: S activation stages of 64 k, a ring of packed weights (4-bit: (S + 1) / 2 rounds of 128 k, 8-bit: S steps of
// 64 k; 64 bytes a row either way) and a ring of scales and biases (eight groups = 16 bytes a row each)
template <int BITS, int WN>
constexpr uint32_t tile_lds(int mi, int S) {
  const int BN = WN * 32, R = (S + 1) / 2, pieces = (mi * 4 + WN - 1) / WN * WN;  // (of 1 KB: whole rounds of the waves)
  return S * pieces * 1024 + (BITS == 4 ? R : S) * BN * 64 + (R > 2 ? 3 : 2) * BN * 32;
}
template <int BITS, int WN, int MIMAX, int KW>
constexpr uint32_t kernel_lds() {
  uint32_t most = MIMAX * 32 * WN * 32 * 2;  // the f16 tile on its way out
  for (int mi = 1; mi <= MIMAX; ++mi) {
    const uint32_t v = KW * tile_lds<BITS, WN>(mi, kStages);
    most = v > most ? v : most;
  }
  return most;
}

template <int BITS, int WN, int MI, int KW, bool DUAL, bool EXACT>
__device__ __forceinline__ void tile_body(const TileParams p, const Tile t_, char* lds) {
  constexpr int BM = MI * 32, BN = WN * 32, BNO = DUAL ? BN / 2 : BN, S = kStages, R = (S + 1) / 2;
  constexpr int kThreads = WN * KW * 64, kPieces = (BM / 8 + WN - 1) / WN * WN;
  constexpr uint32_t kABytes = kPieces * 1024, kWBytes = BN * 64, kWSlots = BITS == 4 ? R : S, kSbBytes = BN * 32, kSbSlots = R > 2 ? 3 : 2;
  constexpr int NA = kPieces / WN, NWI = BN / 16 / WN;  // loads per wave of a stage and of a weight slot (of scales: one)
  constexpr int WV = BITS == 4 ? 1 : 2;                                   // 16-byte pieces of a lane's weights per step
  static_assert(S * kABytes + kWSlots * kWBytes + kSbSlots * kSbBytes == tile_lds<BITS, WN>(MI, S), "LDS");
  constexpr uint32_t oW = S * kABytes, oS = oW + kWSlots * kWBytes;
  const uint32_t tid = threadIdx.x, lane = tid & 63, kg = KW > 1 ? uni((tid >> 6) / WN) : 0, wv = uni(tid >> 6) - kg * WN, r = lane & 31, hh = lane >> 5;
  char* const lds_all = lds;
  lds += kg * tile_lds<BITS, WN>(MI, S);  // every k range of the workgroup has rings of its own
  const uint32_t lds0 = uni((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  const uint32_t K = p.K, G = K / p.group_size, row_bytes = K * BITS / 8;
  const uint32_t rows = t_.rows, row_lo = t_.row_lo, n0 = t_.nt * BNO, cols = p.N - n0 < BNO ? p.N - n0 : BNO;
  // rounds of 128 k: of this split, then of this wave group (n_rounds each: the last group's may run past the split's end)
  const uint32_t rounds = (K + 127) / 128, s0 = uni(rounds * t_.split / p.splits), s1 = uni(rounds * (t_.split + 1) / p.splits);
  const uint32_t n_rounds = (s1 - s0 + KW - 1) / KW, r0 = s0 + kg * n_rounds, r1 = r0 + n_rounds < s1 ? r0 + n_rounds : s1;
  const uint32_t kend2 = (r1 * 128 < K ? r1 * 128 : K) * 2;

  // ---- where a wave's loads come from ---------------------------------------------------------------------------
  const uint64_t wbase = (uint64_t)t_.expert * p.estride_w * 4 + (uint64_t)n0 * row_bytes;
  const uint64_t sbase = (uint64_t)t_.expert * p.estride_s * 2;  // (of the whole matrix)
  auto at = [](const void* q, uint64_t o) { return static_cast<const void*>(static_cast<const char*>(q) + o); };
  // activations: a piece = 8 rows of 128 bytes; the 16-byte chunk is xor-ed with the row so that the operand reads spread over
  // the banks.  Rows past the tile's last repeat it.
  const uint32_t ca = (lane & 7) ^ ((((wv & 1) * 8 + (lane >> 3)) >> 1) & 7);
  const bool mapped = p.row_map != nullptr;  // (of a grouped launch: rows from anywhere in x, which is at most 2 GiB then)
  const u4 xr = mapped ? rsrc(p.x, (uint64_t)p.x_rows * K * 2) : rsrc(at(p.x, (uint64_t)row_lo * K * 2), (uint64_t)rows * K * 2);
  uint32_t aoff[NA];
#pragma unroll
  for (int q = 0; q < NA; ++q) {
    uint32_t m = (q * WN + wv) * 8 + (lane >> 3);
    m = m < rows ? m : rows - 1;
    if (mapped) m = p.row_map[row_lo + m];
    aoff[q] = m * K * 2;
  }
  // weights: a piece = 16 rows of 64 bytes.  A pair's tile holds BN / 2 gate rows, then the same rows of the up matrix.
  auto tile_row = [&](uint32_t li) { const uint32_t c = DUAL ? li % BNO : li; return c < cols ? c : cols - 1; };
  const uint32_t cw = (lane & 3) ^ ((lane >> 4) & 3);
  u4 wr[NWI];
  uint32_t woff[NWI];
#pragma unroll
  for (int q = 0; q < NWI; ++q) {
    const uint32_t li0 = (q * WN + wv) * 16;
    wr[q] = rsrc(at(DUAL && li0 >= BNO ? p.w1 : p.w, wbase), (uint64_t)cols * row_bytes);
    woff[q] = tile_row(li0 + (lane >> 2)) * row_bytes;
  }
  // scales and biases: a piece = 16 bytes (eight groups) of 64 rows, all scales before all biases.  A unit of eight groups that
  // would run past the row starts earlier.
  const uint32_t s_li0 = wv % (BN / 64) * 64;
  const bool s_up = DUAL && s_li0 >= BNO;
  const u4 sr = rsrc(at(wv >= BN / 64 ? (s_up ? p.b1 : p.b) : (s_up ? p.s1 : p.s), sbase), (uint64_t)p.N * G * 2);
  // (fewer than eight groups in a row: a load runs into the next rows, and the last rows' starts earlier)
  auto sb_row = [&](uint32_t li) {
    const uint32_t o = (n0 + tile_row(li)) * G * 2, last = p.N * G * 2 - 16;
    return o < last || G >= 8 ? o : last;
  };
  const uint32_t soff = sb_row(s_li0 + lane);
  const uint32_t gshift = p.group_size == 32 ? 5 : (p.group_size == 64 ? 6 : 7), ushift = gshift - 4;  // k -> group, round -> unit
  auto unit_start = [&](uint32_t unit) { return G < 8 ? 0u : (unit * 8 < G - 8 ? unit * 8 : G - 8); };
  auto dma_a = [&](uint32_t t, uint32_t stage, int q) {
    const uint32_t kb = t * 128 + ca * 16;
    const bool ok = kb < kend2;  // (k past the row, or past this split's last round: zeros)
    dma16(lds0 + stage + (q * WN + wv) * 1024, ok ? aoff[q] + kb : kOutside, xr);
  };
  auto dma_w = [&](uint32_t unit, uint32_t slot, int q) {
    uint32_t kb = unit * 64 + cw * 16;
    kb = kb < row_bytes - 16 ? kb : row_bytes - 16;
    dma16(lds0 + oW + slot * kWBytes + (q * WN + wv) * 1024, woff[q] + kb, wr[q]);
  };
  auto dma_s = [&](uint32_t cond, uint32_t unit) {
    dma16_if(uni(cond), lds0 + oS + unit % kSbSlots * kSbBytes + wv * 1024, soff + unit_start(unit) * 2, sr);
  };
  // Loads go out in groups: group t = step t's activations and, 8-bit, weights; an even one also the weights of round t / 2
  // (4-bit) and, where a unit begins with it, its scales.  part k of 3.
  auto dma_group = [&](auto roundc, uint32_t t, uint32_t stage, uint32_t wslot, int part) {
    constexpr bool kRound = decltype(roundc)::value;
    constexpr int kW = (BITS == 8 || kRound) ? NWI : 0;
#pragma unroll
    for (int q = 0; q < NA + kW; ++q) {
      if (part >= 0 && q % 3 != part) continue;
      if (q < NA) dma_a(t, stage, q);
      else dma_w(BITS == 8 ? t : t / 2, wslot, q - NA);
    }
    if (kRound && (part < 0 || part == 2)) dma_s(t == 2 * r0 || ((t / 2) & ((1u << ushift) - 1)) == 0, (t / 2) >> ushift);
  };

  // ---- operands: lane (r, hh) of k step k multiplies k = 32 hh + 8 k .. + 7 of the 64 ----------------------------------
  uint32_t a_rd[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) a_rd[k] = r * 128 + (((4 * hh + k) ^ ((r >> 1) & 7)) * 16);
  auto read_a = [&](uint32_t stage, int i, int k) -> h8 { return *reinterpret_cast<const h8*>(lds + stage + a_rd[k] + i * 4096); };
  const uint32_t w_rd = oW + (wv * 32 + r) * 64, w_key = (r >> 2) & 3;
  u4 wq[WV];
  auto load_wq = [&](uint32_t slot, int par) {
#pragma unroll
    for (int v = 0; v < WV; ++v) {
      const uint32_t c = BITS == 4 ? 2 * par + hh : 2 * hh + v;
      wq[v] = *reinterpret_cast<const u4*>(lds + slot * kWBytes + w_rd + ((c ^ w_key) * 16));
    }
  };
  uint32_t sraw, braw;
  const uint32_t sb_rd = oS + (wv * 32 + r) * 16 + ((n0 + tile_row(wv * 32 + r)) * G * 2 - sb_row(wv * 32 + r));
  auto load_sb = [&](uint32_t t) {  // group of step t (group size 32: of the lane's half of it)
    const uint32_t unit = t * 64 >> (gshift + 3);
    uint32_t g = (t * 64 + (gshift == 5 ? hh * 32 : 0)) >> gshift;
    g = (g < G ? g : G - 1) - unit_start(unit);  // (0 .. 7)
    const char* q = lds + (unit % kSbSlots) * kSbBytes + sb_rd + g * 2;
    sraw = *reinterpret_cast<const uint16_t*>(q);
    braw = *reinterpret_cast<const uint16_t*>(q + BN * 16);
  };
  h2 s2, b2;
  auto pick_sb = [&]() {
    s2 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(sraw, sraw, 0x01000100u));
    b2 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(braw, braw, 0x01000100u));
  };
  auto word = [](const u4& v, int c) -> uint32_t { return c == 0 ? v.x : (c == 1 ? v.y : (c == 2 ? v.z : v.w)); };
  auto operand = [&](int k) -> Weights {
    Weights w;
    if constexpr (EXACT && BITS == 4) w = split_q4(word(wq[0], k), (float)s2[0], (float)b2[0]);
    else if constexpr (EXACT) w = split_q8(word(wq[(k >> 1) % WV], 2 * (k & 1)), word(wq[(k >> 1) % WV], 2 * (k & 1) + 1), (float)s2[0], (float)b2[0]);
    else if constexpr (BITS == 4) w.hi = weights_q4(word(wq[0], k), s2, b2);
    else w.hi = weights_q8(word(wq[(k >> 1) % WV], 2 * (k & 1)), word(wq[(k >> 1) % WV], 2 * (k & 1) + 1), s2, b2);
    return w;
  };

  f16v acc[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;

  // ---- k loop ------------------------------------------------------------------------------------------------------
  constexpr bool kAhead = MI <= 4;
  constexpr int kStep = NA + (BITS == 8 ? NWI : 0), kRound = BITS == 4 ? NWI : 0;  // (scales not counted: a wait then covers one load more than it has to)
  const uint32_t t0 = 2 * r0;
  uint32_t slot8 = 0, slot_r = 0;  // ring positions: step (activation stage, 8-bit weights), round (4-bit weights)
#pragma unroll
  for (int t = 0; t < (kAhead ? S : S - 1); ++t) {
    if (t % 2 == 0) dma_group(std::true_type{}, t0 + t, t * kABytes, BITS == 8 ? t : t / 2, -1);
    else dma_group(std::false_type{}, t0 + t, t * kABytes, t, -1);
  }
  if constexpr (kAhead) {
    // Few fragments: a group of matrix instructions is shorter than an LDS read.  All operands of a step are read during the step
    // before, each into the registers that its predecessor has just left; group t + S goes out during step t into step t's slots.
    wait_dma_and_barrier<(S - 2) * kStep + (R - 1) * kRound>();  // groups 0 and 1 have arrived
    h8 bf[4][MI];
    Weights wf;
    load_sb(t0);
    load_wq(0, 0);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < MI; ++i) bf[k][i] = read_a(0, i, k);
    pick_sb();
    wf = operand(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // stage 0 has been read
    auto step = [&](auto parc, uint32_t t, uint32_t round) {
      constexpr int par = decltype(parc)::value;
      const uint32_t slot_nxt = slot8 == S - 1 ? 0u : slot8 + 1, round_nxt = slot_r == R - 1 ? 0u : slot_r + 1;
      const uint32_t nxt = slot_nxt * kABytes;
      u4 wq_now[WV];
#pragma unroll
      for (int v = 0; v < WV; ++v) wq_now[v] = wq[v];
      load_wq(BITS == 4 ? (par ? round_nxt : slot_r) : slot_nxt, par ^ 1);
      load_sb(t + 1);
      u4 wq_nxt[WV];
#pragma unroll
      for (int v = 0; v < WV; ++v) { wq_nxt[v] = wq[v]; wq[v] = wq_now[v]; }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf.hi, bf[k][i], acc[i], 0, 0, 0);
          if constexpr (!EXACT) bf[k][i] = read_a(nxt, i, k);
        }
        if constexpr (EXACT)
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf.lo, bf[k][i], acc[i], 0, 0, 0);
            bf[k][i] = read_a(nxt, i, k);
          }
        if (k < 3) {
          wf = operand(k + 1);
          dma_group(std::integral_constant<bool, par == 1>{}, t + S, slot8 * kABytes, BITS == 8 ? slot8 : slot_r, k);
        } else {
#pragma unroll
          for (int v = 0; v < WV; ++v) wq[v] = wq_nxt[v];
          pick_sb();
          wf = operand(0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      wait_dma_and_barrier<(S - 2) * kStep + (par == 0 ? R - 2 : R - 1) * kRound>();  // group t + 2 has arrived
      slot8 = slot_nxt;
      if constexpr (par == 1) slot_r = round_nxt;
    };
    for (uint32_t round = r0; round < r0 + n_rounds; ++round) {
      step(std::integral_constant<int, 0>{}, 2 * round, round);
      step(std::integral_constant<int, 1>{}, 2 * round + 1, round);
    }
  } else {
    // Group t + S - 1 goes out during step t, between its matrix instructions, into the slots that step t - 1 has left.
    wait_dma_and_barrier<(S - 2) * kStep + (R - 2) * kRound>();
    h8 bf[MI];
    Weights wf;
    load_sb(t0);
    load_wq(0, 0);
#pragma unroll
    for (int i = 0; i < MI; ++i) bf[i] = read_a(0, i, 0);
    pick_sb();
    wf = operand(0);

    uint32_t stage = 0;
    auto step = [&](auto parc, uint32_t t, uint32_t round) {
      constexpr int par = decltype(parc)::value;
      const uint32_t slot_nxt = slot8 == S - 1 ? 0u : slot8 + 1, round_nxt = slot_r == R - 1 ? 0u : slot_r + 1;
      const uint32_t slot_prv = slot8 == 0 ? S - 1 : slot8 - 1, round_prv = slot_r == 0 ? R - 1 : slot_r - 1;
      const uint32_t nxt = slot_nxt * kABytes;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        h8 bn[MI];
        Weights wn;
        if (k < 3) {
#pragma unroll
          for (int i = 0; i < MI; ++i) bn[i] = read_a(stage, i, k + 1);
          wn = operand(k + 1);
          dma_group(std::integral_constant<bool, par == 0>{}, t + S - 1, slot_prv * kABytes, BITS == 8 ? slot_prv : round_prv, k);
        } else {
          // everything of step t + 1 has arrived; the S - 2 groups after it may still be on their way
          wait_dma_and_barrier<(S - 2) * kStep + (par == 0 ? R - 1 : R - 2) * kRound>();
          load_sb(t + 1);
          load_wq(BITS == 4 ? (par ? round_nxt : slot_r) : slot_nxt, par ^ 1);
#pragma unroll
          for (int i = 0; i < MI; ++i) bn[i] = read_a(nxt, i, 0);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf.hi, bf[i], acc[i], 0, 0, 0);
        if constexpr (EXACT)
#pragma unroll
          for (int i = 0; i < MI; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf.lo, bf[i], acc[i], 0, 0, 0);
        if (k == 3) {
          pick_sb();
          wn = operand(0);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) bf[i] = bn[i];
        wf = wn;
        __builtin_amdgcn_sched_barrier(0);
      }
      stage = nxt;
      slot8 = slot_nxt;
      if constexpr (par == 1) slot_r = round_nxt;
    };
    for (uint32_t round = r0; round < r0 + n_rounds; ++round) {
      step(std::integral_constant<int, 0>{}, 2 * round, round);
      step(std::integral_constant<int, 1>{}, 2 * round + 1, round);
    }
  }
  wait_dma_and_barrier<0>();
  lds = lds_all;
  if constexpr (KW > 1) {  // the sums of the k ranges meet in LDS, added in range order
    static_assert(KW == 2, "k ranges");
    f4* g = reinterpret_cast<f4*>(lds) + wv * MI * 256 + lane;
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int eg = 0; eg < 4; ++eg) g[(i * 4 + eg) * 64] = (f4){acc[i][eg * 4], acc[i][eg * 4 + 1], acc[i][eg * 4 + 2], acc[i][eg * 4 + 3]};
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int eg = 0; eg < 4; ++eg) {
          const f4 v = g[(i * 4 + eg) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][eg * 4 + e] += v[e];
        }
    }
    __syncthreads();
  }

  // ---- store: fragment i of a lane holds activation row 32 i + r, weight rows 32 wv + 8 eg + 4 hh + 0 .. 3 of the tile -----
  if (!DUAL && (p.partial != nullptr || p.out_f32)) {
    if (kg != 0) return;
    float* o = p.partial != nullptr ? p.partial + (uint64_t)t_.split * p.M * p.N : static_cast<float*>(p.out);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const uint32_t m = i * 32 + r;
      if (m >= rows) continue;
      float* const om = o + (uint64_t)(row_lo + m) * p.N + n0;
#pragma unroll
      for (int eg = 0; eg < 4; ++eg) {
        const uint32_t c = wv * 32 + 8 * eg + 4 * hh;
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = t_.zeros ? 0.f : acc[i][eg * 4 + e];
        if (c + 4 <= cols) reinterpret_cast<f4_any*>(om + c)->v = v;
        else
          for (uint32_t e = 0; e < 4; ++e)
            if (c + e < cols) om[c + e] = v[e];
      }
    }
    return;
  }
  if constexpr (DUAL) {  // the gate waves hand their sums to the waves with the same columns of the up matrix
    f4* g = reinterpret_cast<f4*>(lds) + (wv % (WN / 2)) * MI * 256 + lane;
    if (wv < WN / 2) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int eg = 0; eg < 4; ++eg) g[(i * 4 + eg) * 64] = (f4){acc[i][eg * 4], acc[i][eg * 4 + 1], acc[i][eg * 4 + 2], acc[i][eg * 4 + 3]};
    }
    __syncthreads();
    if (wv >= WN / 2) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int eg = 0; eg < 4; ++eg) {
          const f4 v = g[(i * 4 + eg) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][eg * 4 + e] *= v[e] / (1.0f + __expf(-v[e]));
        }
    }
    __syncthreads();
  }
  constexpr uint32_t U = BNO / 8, kKey = U < 32 ? U - 1 : 31;  // 16-byte units of an output row of the tile, xor-ed with the row
  if (kg == 0 && (!DUAL || wv >= WN / 2)) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const uint32_t m = i * 32 + r;
#pragma unroll
      for (int eg = 0; eg < 4; ++eg) {
        const uint32_t c = (DUAL ? wv - WN / 2 : wv) * 32 + 8 * eg + 4 * hh;
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = t_.zeros ? 0.f : acc[i][eg * 4 + e];
        if (!DUAL && p.epi_kind != EPI_NONE && m < rows && c < cols) tile_epilogue(p, (uint64_t)(row_lo + m) * p.N + n0 + c, cols - c, v);
        const h2 lo = {(_Float16)v[0], (_Float16)v[1]}, hi = {(_Float16)v[2], (_Float16)v[3]};
        *reinterpret_cast<u2*>(lds + (m * U + ((c >> 3) ^ (m & kKey))) * 16 + hh * 8) = (u2){h2bits(lo), h2bits(hi)};
      }
    }
  }
  __syncthreads();
  for (uint32_t g = tid; g < BM * U; g += kThreads) {
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

// Starts on a 16 KB line: the same instructions at another place ran up to 3 % slower (64 KB of instruction cache for two CUs; 1433 rows,
// 9792 x 960, 8 bits: 41.7 us unaligned, 41.4 / 40.9 / 40.7 on lines of 1 / 4 / 16 KB, 40.4 at the best place seen).
template <int BITS, int WN, int MIMAX, int KW, bool DUAL, bool EXACT>
__global__ __launch_bounds__(WN * KW * 64, 2) __attribute__((aligned(16384))) void qmm_tile_kernel(TileParams p) {
  __shared__ __align__(1024) char lds[kernel_lds<BITS, WN, MIMAX, KW>()];
  Tile t;
  if (!tile_of<DUAL ? 1 : 4>(p, MIMAX * 32, &t)) return;
  const uint32_t frags = (t.rows + 31) / 32;
  auto go = [&](auto mi) {
    constexpr int MI = decltype(mi)::value;
    if constexpr (MI <= MIMAX) tile_body<BITS, WN, MI, KW, DUAL, EXACT>(p, t, lds);
  };
  using std::integral_constant;
  switch (frags) {
    case 1: go(integral_constant<int, 1>{}); break;
    case 2: go(integral_constant<int, 2>{}); break;
    case 3: go(integral_constant<int, 3>{}); break;
    case 4: go(integral_constant<int, 4>{}); break;
    case 5: go(integral_constant<int, 5>{}); break;
    case 6: go(integral_constant<int, 6>{}); break;
    case 7: go(integral_constant<int, 7>{}); break;
    default: go(integral_constant<int, 8>{}); break;
  }
}

// out[i] = epilogue(sum of the partial sums, in split order); four outputs per thread
__global__ __launch_bounds__(256) void tile_splits_sum_kernel(TileParams p) {
  const uint64_t i = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4, total = (uint64_t)p.M * p.N;
  if (i >= total) return;
  const uint32_t n = total - i < 4 ? (uint32_t)(total - i) : 4;
  f4 v = {0.f, 0.f, 0.f, 0.f};
  for (uint32_t z = 0; z < p.splits; ++z) {
    const float* q = p.partial + z * total + i;
    if (n == 4) v += reinterpret_cast<const f4_any*>(q)->v;
    else
      for (uint32_t e = 0; e < n; ++e) v[e] += q[e];
  }
  if (p.epi_kind != EPI_NONE) tile_epilogue(p, i, n, v);
  _Float16* out = static_cast<_Float16*>(p.out) + i;
  const h2 o[2] = {{(_Float16)v[0], (_Float16)v[1]}, {(_Float16)v[2], (_Float16)v[3]}};
  if (n == 4) {
    reinterpret_cast<u2_any*>(out)->v = (u2){h2bits(o[0]), h2bits(o[1])};
  } else {
    for (uint32_t e = 0; e < n; ++e) out[e] = o[e / 2][e % 2];
  }
}

template <int BITS, bool EXACT>
void launch_tile_as(const TileParams& p, const TilePlan& plan, dim3 grid, hipStream_t s) {
  if (p.w1 != nullptr) {
    if (plan.mi == 8) hipLaunchKernelGGL((qmm_tile_kernel<BITS, 8, 8, 1, true, EXACT>), grid, dim3(512), 0, s, p);
    else if (plan.mi == 4) hipLaunchKernelGGL((qmm_tile_kernel<BITS, 4, 4, 1, true, EXACT>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((qmm_tile_kernel<BITS, 4, 2, 1, true, EXACT>), grid, dim3(256), 0, s, p);
  }
  else if (plan.wn == 8 && plan.mi == 8) hipLaunchKernelGGL((qmm_tile_kernel<BITS, 8, 8, 1, false, EXACT>), grid, dim3(512), 0, s, p);
  else if (plan.wn == 8) hipLaunchKernelGGL((qmm_tile_kernel<BITS, 8, 4, 1, false, EXACT>), grid, dim3(512), 0, s, p);
  else if (plan.mi == 4 && plan.kw == 1) hipLaunchKernelGGL((qmm_tile_kernel<BITS, 4, 4, 1, false, EXACT>), grid, dim3(256), 0, s, p);
  else if (plan.mi == 4) hipLaunchKernelGGL((qmm_tile_kernel<BITS, 4, 4, 2, false, EXACT>), grid, dim3(512), 0, s, p);
  else if (plan.kw == 1) hipLaunchKernelGGL((qmm_tile_kernel<BITS, 4, 2, 1, false, EXACT>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((qmm_tile_kernel<BITS, 4, 2, 2, false, EXACT>), grid, dim3(512), 0, s, p);
}

template <int BITS>
void launch_tile(const TileParams& p, const TilePlan& plan, dim3 grid, hipStream_t s) {
  if (p.exact) launch_tile_as<BITS, true>(p, plan, grid, s);
  else launch_tile_as<BITS, false>(p, plan, grid, s);
}

}  // namespace

bool qmm_tile_supported(uint32_t N, uint32_t K, uint32_t group_size, uint32_t bits) {
  return (bits == 4 || bits == 8) && (group_size == 32 || group_size == 64 || group_size == 128) && N > 0 && K > 0 && K % group_size == 0 &&
         (uint64_t)N * (K / group_size) >= 8 && (uint64_t)N * (K / group_size) <= (1u << 29) && K <= (1u << 20);
}

// The plan with the shortest estimated launch.  A workgroup's time is its number of 64-k steps times the length of a step, which
// grows with the 32-row fragments of the tile and with the workgroups that share a CU (`step` holds (constant, per fragment) for
// 1, 2, .. of them); fragments cost half as much on an idle chip as on a full one, where the clock falls.  A launch adds its start
// and end, a K split the kernel that adds up the partial sums.  Fitted to about 15000 timed launches (780 shapes, every plan and
// split): 6 % mean error, and the picks are 1.3 % slower on average than the fastest plan; the rows of two workgroups per CU to 200 shapes of 17 rows and more.
// (kw >= 4: waves along k, steps of `k` values; mi_most: two workgroups per CU, qmm_twin.hip, tiles of mi to mi_most fragments)
struct Cost { uint32_t wn, mi, kw; int per_cu; double start, step[3][2], sum, sum_per_mi; uint32_t k, mi_most; };
static const Cost kCosts[2][12] = {
    {{8, 8, 1, 1, 8.19, {{0.503, 0.118}}, 7.46, 1.10},
     {8, 4, 1, 1, 3.71, {{0.428, 0.110}}, 4.90, 1.74},
     {4, 4, 1, 2, 4.64, {{0.270, 0.073}, {0.531, 0.083}}, 3.39, 1.59},
     {4, 2, 1, 3, 3.50, {{0.300, 0.057}, {0.490, 0.053}, {0.707, 0.074}}, 3.49, 1.88},
     {4, 4, 2, 1, 5.09, {{0.356, 0.159}}, 3.52, 2.07},
     {4, 2, 2, 1, 3.90, {{0.398, 0.146}}, 3.46, 2.43},
     {2, 1, 8, 2, 4.14, {{0.256, 0.271}, {1.023, 0.000}}, 3.00, 0.10, 256},
     {2, 2, 8, 1, 5.20, {{0.089, 0.370}}, 2.80, 0.00, 256},
     {4, 1, 4, 1, 4.56, {{0.201, 0.751}}, 3.20, 1.04, 256},
     {4, 2, 4, 1, 5.46, {{0.296, 0.467}}, 2.87, 1.33, 256},
     {8, 3, 1, 2, 5.86, {{0.365, 0.171}, {0.572, 0.278}}, 0, 0, 0, 5},
     {4, 3, 1, 2, 4.85, {{0.269, 0.098}, {0.358, 0.153}}, 0, 0, 0, 7}},
    {{8, 8, 1, 1, 7.26, {{0.608, 0.104}}, 8.71, 1.34},
     {8, 4, 1, 1, 3.33, {{0.516, 0.102}}, 5.39, 1.89},
     {4, 4, 1, 2, 4.87, {{0.352, 0.047}, {0.628, 0.091}}, 3.44, 1.65},
     {4, 2, 1, 3, 3.36, {{0.349, 0.055}, {0.702, 0.000}, {1.128, 0.000}}, 3.53, 2.00},
     {4, 4, 2, 1, 4.87, {{0.517, 0.141}}, 3.57, 2.17},
     {4, 2, 2, 1, 3.44, {{0.519, 0.139}}, 4.01, 2.62},
     {2, 1, 8, 1, 4.61, {{0.000, 0.671}}, 2.59, 0.00, 256},
     {2, 2, 8, 1, 5.17, {{0.061, 0.452}}, 2.30, 0.00, 256},
     {4, 1, 4, 1, 4.56, {{0.032, 1.080}}, 3.39, 0.00, 256},
     {4, 2, 4, 1, 5.28, {{0.156, 0.302}}, 3.22, 0.64, 128},
     {8, 3, 1, 2, 3.81, {{0.571, 0.154}, {0.722, 0.256}}, 0, 0, 0, 4},
     {4, 3, 1, 2, 3.84, {{0.330, 0.105}, {0.395, 0.173}}, 0, 0, 0, 7}}};
// A launch of `tiles` workgroups, `steps` steps of 64 k each, `frags` fragments high on average
static double rounds_us(const Cost& c, double tiles, double frags, double steps) {
  const double cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
  const double load = tiles / cus, full = std::floor(load / c.per_cu), rest = load - full * c.per_cu;
  double t = steps * full * (c.step[c.per_cu - 1][0] + c.step[c.per_cu - 1][1] * frags);
  if (rest > 1e-9) {
    const double* s = c.step[(int)std::ceil(rest - 1e-9) - 1];
    t += steps * (s[0] + s[1] * frags * (full > 0 || load >= 1 ? 1.0 : 0.5 + 0.5 * load));
  }
  return t;
}

// What the estimate of two workgroups per CU, in `wn` * 32 columns, may be of the best other plan's for them to be ahead: the table's errors differ from
// tile to tile (it has the 256 x 256 tile too long against the others and the tiles of 128 rows by 256 columns too short, over short rows above all).  Of 615
// shapes of 65 to 4096 rows timed in both forms these lines take 205, 12 % faster on average, four of them 2 to 5 % slower (the best choice: 311, 10 %).
static double twin_limit(const TilePlan& other, uint32_t wn, uint32_t M, uint32_t K) {
  const bool is_short = K <= 640;
  if (other.kw > 1 || other.splits > 1) return 0.95;
  if (other.wn == 8 && other.mi == 8) return wn == 8 ? (is_short ? 1.03 : 0.98) : (M <= 320 ? 0.8 : 0.87);
  if (other.wn == 8) return wn == 8 ? (is_short ? 1.13 : 1.03) : (is_short ? 1.07 : 1.01);
  return wn == 8 ? (is_short ? 1.02 : 0.98) : 0.95;
}
enum { PLAN_ROUNDED = 0, PLAN_EXACT = 1, PLAN_TWIN = 2 };  // any kernel, those with exact weights, two workgroups per CU only
static TilePlan estimate_plan(uint32_t M, uint32_t N, uint32_t K, uint32_t bits, int kind, double* us) {
  const bool exact = kind == PLAN_EXACT;
  constexpr double kExactStep = 1.5;  // two products: 8 to 64 rows 1.35 to 1.45 x, 300 to 2000 rows 1.55 to 1.65
  const double cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
  const uint32_t rounds = (K + 127) / 128;
  TilePlan best{4, 2, 1, 1};
  double best_us = 1e30;
  auto price = [&](const Cost& c, uint32_t mi) {
    const uint64_t tm = (M + mi * 32 - 1) / (mi * 32), tiles = tm * ((N + c.wn * 32 - 1) / (c.wn * 32));
    const double frags = (double)((M + 31) / 32) / (double)tm;
    for (uint32_t splits : {1u, 2u, 3u, 4u, 6u, 8u}) {
      const uint32_t stages = c.k != 0 ? (K + c.k - 1) / c.k : 0;
      if (splits > 1 && (c.mi_most != 0 || rounds < 2 * splits * c.kw || (double)(tiles * splits) > 1.6 * c.per_cu * cus || (uint64_t)splits * M * N > (1u << 27))) break;
      const double steps = c.k != 0 ? (stages + splits - 1) / splits : 2.0 * ((((rounds + splits - 1) / splits) + c.kw - 1) / c.kw);
      double t = rounds_us(c, (double)(tiles * splits), frags, steps);
      t = c.start + (exact ? kExactStep : 1.0) * t;
      if (splits > 1) t += c.sum + c.sum_per_mi * splits * ((double)M * N / (1 << 20));
      if (t < best_us) { best_us = t; best = TilePlan{c.wn, mi, c.kw, splits, c.mi_most != 0}; }
    }
  };
  for (const Cost& c : kCosts[bits == 8])
    if (kind != PLAN_TWIN && c.mi_most == 0 && !(c.k != 0 && c.mi == 2 && M <= 32)) price(c, c.mi);
  *us = best_us;  // (the dispatch's lines were drawn for these: a shorter estimate must not send a call to a kernel that is longer still)
  if (exact) return best;
  // Two workgroups per CU (rounded weights only), without a K split (timed 4 to 15 % slower than the plans of the other kernels: 2398 rows, 896 x 10432 76
  // against 68 us).  Up to 64 rows only over rows of up to 1024 values (8 rows, 117760 x 640, 8-bit 24.6 / 21.7; but 9 rows, 22016 x 14336 41 / 57, 21 rows, 62144 x
  // 11328 108 / 153), in 256 columns.
  const TilePlan other = best;
  const double other_us = best_us;
  best_us = 1e30;
  for (const Cost& c : kCosts[bits == 8])
    for (uint32_t mi = c.mi; mi <= c.mi_most; ++mi)
      if (M > 64 || c.wn == 8 || kind == PLAN_TWIN) price(c, mi);
  if (kind == PLAN_TWIN) return best;
  if (M <= 64) return K <= 1024 && best_us < 1.05 * other_us ? best : other;
  if (M <= 96 && K > 2048) return other;  // (72 rows, 117312 x 3200, group size 32 91 / 102)
  return best_us < twin_limit(other, best.wn, M, K) * other_us ? best : other;
}

// (about 1 us of arithmetic, asked for twice per call by launches that take 5: the last plans of a thread are kept)
TilePlan qmm_tile_plan(uint32_t M, uint32_t N, uint32_t K, uint32_t bits, bool exact, double* us) {
  struct Kept { uint32_t M, N, K, bits; TilePlan plan; double us; };
  thread_local Kept kept[64] = {};
  const uint32_t kind = bits + (exact ? 1 : 0);
  Kept& e = kept[(M * 31 + N * 7 + K + kind) & 63];
  if (e.M != M || e.N != N || e.K != K || e.bits != kind) {
    e.plan = estimate_plan(M, N, K, bits, exact ? PLAN_EXACT : PLAN_ROUNDED, &e.us);
    e.M = M; e.N = N; e.K = K; e.bits = kind;
  }
  if (us != nullptr) *us = e.us;
  return e.plan;
}

TilePlan qmm_twin_plan(uint32_t M, uint32_t N, uint32_t K, uint32_t bits) {
  double us;
  return estimate_plan(M, N, K, bits, PLAN_TWIN, &us);
}

double qmm_tile_grouped_us(uint32_t bits, bool twin, uint32_t tile_rows, double row_tiles, double frags, uint32_t N, uint32_t K) {
  const uint32_t wn = twin || tile_rows == 256 ? 8 : 4, mi = twin ? 3 : tile_rows / 32;
  for (const Cost& c : kCosts[bits == 8])
    if (c.wn == wn && c.mi == mi && c.kw == 1 && (c.mi_most != 0) == twin)
      return c.start + rounds_us(c, row_tiles * ((N + wn * 32 - 1) / (wn * 32)), frags, 2.0 * ((K + 127) / 128));
  return 1e30;
}

size_t qmm_tile_workspace_bytes(const TilePlan& plan, uint32_t M, uint32_t N) {
  return plan.splits > 1 ? (size_t)plan.splits * M * N * sizeof(float) : 0;
}

int32_t launch_qmm_tile(const QmmArgs& a, const TilePlan& plan, hipStream_t s) {
  if (!qmm_tile_supported(a.N, a.K, a.group_size, a.bits) || a.x_dtype != RMLX_DTYPE_F16)
    return fail(RMLX_INVALID_SHAPE, "qmm: unsupported shape N=%u K=%u bits=%u group_size=%u", a.N, a.K, a.bits, a.group_size);
  if (a.M == 0) return RMLX_OK;
  TileParams p{};
  p.w = a.w; p.s = a.s; p.b = a.b;
  p.x = static_cast<const __half*>(a.x);
  p.out = a.out; p.M = a.M; p.N = a.N; p.K = a.K; p.group_size = a.group_size;
  // Row tiles of equal height, to a fragment of 32 rows: worth it only where the highest gets lower (1050 rows, 21673 x 4224, 8-bit 221 -> 204 us, 316 rows,
  // 26560 x 2432 59 -> 51).  Heights that differ by one where it does not cost up to 6 % (926 rows, 2496 x 5120, 8-bit 41.0 / 42.9 with tiles of three and
  // four fragments, 320 rows, 5568 x 12032 70 / 73).
  const uint32_t frags = (a.M + 31) / 32;
  p.tiles_m = (frags + plan.mi - 1) / plan.mi;
  p.tile_rows = (frags + p.tiles_m - 1) / p.tiles_m * 32;
  p.tiles_m = (a.M + p.tile_rows - 1) / p.tile_rows;
  p.tiles_n = (a.N + plan.wn * 32 - 1) / (plan.wn * 32);
  p.splits = plan.splits;
  p.partial = plan.splits > 1 ? static_cast<float*>(a.workspace) : nullptr;
  p.epi_kind = a.epi_kind; p.epi = a.epi; p.epi_dtype = a.epi_dtype; p.exact = a.exact;
  const uint64_t wgs = (uint64_t)p.tiles_m * p.tiles_n * p.splits;
  if (wgs > 0x7FFFFFFFull) return fail(RMLX_INVALID_SHAPE, "qmm: grid too large");
  if (plan.twin) launch_qmm_twin(p, a.bits, plan.wn, dim3((unsigned)wgs), s);
  else if (plan.kw >= 4) launch_qmm_slice(p, a.bits, plan, dim3((unsigned)wgs), s);
  else if (a.bits == 4) launch_tile<4>(p, plan, dim3((unsigned)wgs), s);
  else launch_tile<8>(p, plan, dim3((unsigned)wgs), s);
  RMLX_HIP_CHECK(hipGetLastError());
  if (p.partial != nullptr) {
    const uint64_t quads = ((uint64_t)p.M * p.N + 3) / 4;
    hipLaunchKernelGGL(tile_splits_sum_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, p);
    RMLX_HIP_CHECK(hipGetLastError());
  }
  return RMLX_OK;
}

int32_t launch_qmm_tile_grouped(const GroupedQmmArgs& a, uint32_t x_rows, hipStream_t s) {
  if (!qmm_tile_supported(a.N, a.K, a.group_size, a.bits) || (a.row_map != nullptr && !qmm_tile_maps_rows(x_rows, a.K)))
    return fail(RMLX_INVALID_SHAPE, "grouped qmm: unsupported shape N=%u K=%u bits=%u group_size=%u, %u rows", a.N, a.K, a.bits, a.group_size, x_rows);
  if (a.twin && (a.exact || a.tile_rows > (a.bits == 4 ? 160u : 128u)))
    return fail(RMLX_RUNTIME_ERROR, "grouped qmm: two workgroups per CU take rounded weights and row tiles of up to 160 rows (8-bit: 128), got %u", a.tile_rows);
  if (a.max_tiles == 0) return RMLX_OK;
  if (a.tile_rows == 32) return launch_qmm_slice_grouped(a, x_rows, s);
  TileParams p{};
  p.w = a.w; p.s = a.s; p.b = a.b; p.w1 = a.w1; p.s1 = a.s1; p.b1 = a.b1;
  p.x = a.x; p.out = a.out; p.N = a.N; p.K = a.K; p.group_size = a.group_size;
  p.out_f32 = a.out_f32; p.exact = a.exact;
  p.tile_tab = a.tile_tab; p.n_tiles = a.n_tiles_dev; p.row_map = a.row_map; p.x_rows = x_rows;
  p.estride_w = a.expert_stride_w; p.estride_s = a.expert_stride_s;
  p.splits = 1;
  const TilePlan plan{a.tile_rows == 256 || a.twin ? 8u : 4u, a.tile_rows / 32, 1, 1, a.twin != 0};
  const uint32_t cols = plan.wn * 32 / (a.w1 != nullptr ? 2 : 1);
  p.tiles_n = (a.N + cols - 1) / cols;
  const uint64_t wgs = (uint64_t)a.max_tiles * p.tiles_n;
  if (wgs > 0x7FFFFFFFull) return fail(RMLX_INVALID_SHAPE, "grouped qmm: grid too large");
  if (plan.twin) launch_qmm_twin(p, a.bits, plan.wn, dim3((unsigned)wgs), s);
  else if (a.bits == 4) launch_tile<4>(p, plan, dim3((unsigned)wgs), s);
  else launch_tile<8>(p, plan, dim3((unsigned)wgs), s);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

bool qmm_tile_maps_rows(uint32_t x_rows, uint32_t K) { return (uint64_t)x_rows * K * 2 <= 0x80000000ull; }

}  // namespace rmlx
