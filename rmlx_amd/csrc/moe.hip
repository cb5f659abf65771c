// MoE routing and data-movement kernels for gfx950.
//
//   topk_route_kernel   -- moe_topk_route_f32 (crates/rmlx-core/src/ops/topk_route.rs:212-359)
//   moe_sort_kernel     -- histogram + exclusive scan (moe_prefix_scan_u32, topk_route.rs:373-388)
//                          + the stable token->expert grouping the reference builds on the host
//                          (crates/rmlx-nn/src/moe.rs:1439-1447), done on the device
//   index_gather / scatter_weighted_add / silu_gate / combine
//                       -- crates/rmlx-core/src/ops/moe_kernels.rs:46-223, ops/silu.rs:142-166
#include "common.hpp"
#include "route.hpp"

namespace rmlx {
namespace {

constexpr int kMaxExperts = kMaxSortedExperts;  // LDS histogram capacity of the sort kernel

// ---- routing: one wave per token (route.hpp) --------------------------------------------------
// (`lds_idx`: optional copy of the picks in workgroup memory, for a sort fused behind the routing)
__device__ __forceinline__ void route_token(const float* __restrict__ logits, const float* __restrict__ bias,
                                            uint32_t E, uint32_t K, int renorm, uint32_t* __restrict__ out_idx,
                                            float* __restrict__ out_w, uint32_t row, uint32_t lane,
                                            uint32_t* lds_idx) {
  uint32_t my_idx;
  float my_w;
  route::token_picks(logits, bias, E, K, renorm, row, lane, my_idx, my_w);
  if (lane < K) {
    out_idx[(size_t)row * K + lane] = my_idx;
    out_w[(size_t)row * K + lane] = my_w;
    if (lds_idx != nullptr) lds_idx[row * K + lane] = my_idx;
  }
}

__global__ __launch_bounds__(64) void topk_route_kernel(const float* __restrict__ logits,
                                                        const float* __restrict__ bias, uint32_t E,
                                                        uint32_t K, int renorm, uint32_t* __restrict__ out_idx,
                                                        float* __restrict__ out_w) {
  route_token(logits, bias, E, K, renorm, out_idx, out_w, blockIdx.x, threadIdx.x, nullptr);
}

// ---- histogram + scan + stable counting sort -----------------------------------------------
// Deterministic by construction.  A workgroup places `portion` assignments; each of its 16 waves owns a run of them and a column of counters
// (one per expert) in LDS: it counts its run, thread e turns the counts of expert e into its offset plus an exclusive prefix over what lies
// before the wave, and the wave walks its run once more, in order and with nobody else's cursors to wait for: position = the wave's cursor of
// the expert + rank among the 64 lanes (by ballots over the bits of the id), so ids of one expert keep their original order
// (numpy.argsort(kind="stable")).  Bound by the chain of one wave's iterations and its scattered stores, so from 2048 assignments on there are
// several workgroups (at most 32, see sort_portion): each counts everybody's assignments itself, before and behind its portion, which costs less than
// meeting in a second launch.  The first one writes the tables.  16384 assignments over 128 experts 24 to 37 us in one workgroup, 11 to 13 now.
// A workgroup alone (SHARED: false) has no counts of others to clear and read (a routed block of 96 assignments 27.9 us with them, 27.6 without).
__device__ __forceinline__ uint32_t block_exclusive_scan_1024(uint32_t v, uint32_t* wave_tot, uint32_t* total) {
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o, 64);
    if ((int)lane >= o) inc += t;
  }
  __syncthreads();  // wave_tot may still be read by a previous scan
  if (lane == 63) wave_tot[wave] = inc;
  __syncthreads();
  uint32_t base = 0, all = 0;
  for (uint32_t w = 0; w < 16; ++w) {
    const uint32_t t = wave_tot[w];
    if (w < wave) base += t;
    all += t;
  }
  *total = all;
  return base + inc - v;
}

template <bool SHARED>
__global__ __launch_bounds__(1024) void moe_sort_kernel(const uint32_t* __restrict__ idx, uint32_t n_assign,
                                                        uint32_t E, uint32_t top_k, uint32_t* __restrict__ sorted,
                                                        uint32_t* __restrict__ sorted_tok,
                                                        uint32_t* __restrict__ inv, uint32_t* __restrict__ counts,
                                                        uint32_t* __restrict__ offsets,
                                                        uint32_t* __restrict__ chunk_tab,
                                                        uint32_t* __restrict__ n_chunks, uint32_t chunk_rows,
                                                        uint32_t* __restrict__ split_tab, uint32_t* __restrict__ split_n,
                                                        uint32_t split_cap, uint32_t portion) {
  __shared__ uint32_t wave_tot[16];
  __shared__ uint32_t cur[16][kMaxExperts];  // per wave and expert: count of the wave's run, then its running cursor
  __shared__ uint32_t others[SHARED ? 2 * kMaxExperts : 1];  // assignments before and behind this workgroup's
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t first = SHARED ? blockIdx.x * portion : 0, last = first + portion < n_assign ? first + portion : n_assign;
  const uint32_t run = portion / 16, begin = first + wave * run < last ? first + wave * run : last, end = begin + run < last ? begin + run : last;
#pragma unroll
  for (int w = 0; w < 16; ++w) cur[w][tid] = 0;  // kMaxExperts == blockDim.x
  if constexpr (SHARED) others[tid] = others[kMaxExperts + tid] = 0;
  __syncthreads();
  if constexpr (SHARED) {
    auto count = [&](uint32_t from, uint32_t to, uint32_t* into) {
#pragma unroll 8
      for (uint32_t i = from + tid; i < to; i += 1024) {
        const uint32_t e = idx[i];
        if (e < E) atomicAdd(&into[e], 1u);
      }
    };
    count(0, first, others);
    count(last, n_assign, others + kMaxExperts);
  }
#pragma unroll 4
  for (uint32_t i = begin + lane; i < end; i += 64) {
    const uint32_t e = idx[i];
    if (e < E) atomicAdd(&cur[wave][e], 1u);
  }
  __syncthreads();
  // thread e owns expert e: offsets, counts, its chunks of at most chunk_rows rows
  uint32_t earlier = 0, my_cnt = 0;
  if constexpr (SHARED) {
    earlier = others[tid];
    my_cnt = earlier + others[kMaxExperts + tid];
  }
#pragma unroll
  for (int w = 0; w < 16; ++w) my_cnt += cur[w][tid];
  uint32_t total_rows, total_chunks;
  const uint32_t my_off = block_exclusive_scan_1024(my_cnt, wave_tot, &total_rows);
  const uint32_t my_chunks = (my_cnt + chunk_rows - 1) / chunk_rows;
  const uint32_t my_chunk0 = block_exclusive_scan_1024(my_chunks, wave_tot, &total_chunks);
  uint32_t before = my_off + earlier;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    const uint32_t c = cur[w][tid];
    cur[w][tid] = before;
    before += c;
  }
  const bool writes = !SHARED || blockIdx.x == 0;
  if (writes && tid < E) {
    if (offsets != nullptr) offsets[tid] = my_off;
    if (counts != nullptr) counts[tid] = my_cnt;
    if (chunk_tab != nullptr) {
      // (row tiles of 64 rows and more: an expert's rows in equal shares of whole 32-row fragments)
      const uint32_t per = chunk_rows < 64 || my_chunks < 2 ? chunk_rows : ((my_cnt + 31) / 32 + my_chunks - 1) / my_chunks * 32;
      for (uint32_t c = 0; c < my_chunks; ++c) {
        const uint32_t left = my_cnt > per * c ? my_cnt - per * c : 0;
        chunk_tab[3 * (my_chunk0 + c) + 0] = tid;
        chunk_tab[3 * (my_chunk0 + c) + 1] = my_off + per * c;
        chunk_tab[3 * (my_chunk0 + c) + 2] = left < per ? left : per;
      }
    }
  }
  if (writes && tid == 0) {
    if (offsets != nullptr) offsets[E] = total_rows;
    if (n_chunks != nullptr) *n_chunks = total_chunks;
  }
  // A second pair of tables that splits the experts by their row count: up to 8 rows -> one chunk in the first table
  // (split_cap entries), more -> chunks of at most 16 rows in the second (behind the first); split_n = the two lengths.
  if (writes && split_tab != nullptr) {
    uint32_t n_small, n_big;
    const uint32_t small = my_cnt >= 1 && my_cnt <= 8 ? 1u : 0u, big = my_cnt > 8 ? (my_cnt + 15) / 16 : 0u;
    const uint32_t small0 = block_exclusive_scan_1024(small, wave_tot, &n_small);
    const uint32_t big0 = block_exclusive_scan_1024(big, wave_tot, &n_big);
    if (small) {
      split_tab[3 * small0 + 0] = tid;
      split_tab[3 * small0 + 1] = my_off;
      split_tab[3 * small0 + 2] = my_cnt;
    }
    uint32_t* bt = split_tab + 3 * (size_t)split_cap;
    for (uint32_t c = 0; c < big; ++c) {
      bt[3 * (big0 + c) + 0] = tid;
      bt[3 * (big0 + c) + 1] = my_off + 16 * c;
      bt[3 * (big0 + c) + 2] = my_cnt - 16 * c < 16 ? my_cnt - 16 * c : 16;
    }
    if (tid == 0) { split_n[0] = n_small; split_n[1] = n_big; }
  }
  if (sorted == nullptr && sorted_tok == nullptr) return;
  __syncthreads();

  const int e_bits = 32 - __builtin_clz(E | 1u);  // bits that tell valid expert ids apart
  const uint64_t lanes_below = (1ull << lane) - 1ull;
  uint32_t e_next = begin + lane < end ? idx[begin + lane] : 0xFFFFFFFFu;
  for (uint32_t base = begin; base < end; base += 64) {
    const uint32_t e = e_next, i = base + lane;
    e_next = i + 64 < end ? idx[i + 64] : 0xFFFFFFFFu;  // in flight during this turn
    const bool valid = e < E;
    // rank among the wave's 64 assignments, and how many of them share the expert: the lanes holding the same
    // expert are the intersection, over the bits of the id, of the lanes that agree with this one on that bit
    uint64_t peers = __ballot(valid);
    for (int bit = 0; bit < e_bits; ++bit) {
      const uint64_t set = __ballot((e >> bit) & 1u);
      peers &= ((e >> bit) & 1u) ? set : ~set;
    }
    const uint32_t rank = (uint32_t)__popcll(peers & lanes_below), same_total = (uint32_t)__popcll(peers);
    if (valid) {
      const uint32_t pos = cur[wave][e] + rank;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // every lane has read before the last of its peers moves the cursor
      if (rank + 1 == same_total) cur[wave][e] = pos + 1;
      if (sorted != nullptr) sorted[pos] = i;
      if (sorted_tok != nullptr) sorted_tok[pos] = i / top_k;
      if (inv != nullptr) inv[i] = pos;
    } else if (inv != nullptr && i < end) {
      inv[i] = 0xFFFFFFFFu;  // an expert id outside [0, E): the combine step skips the assignment
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// At most 64 assignments (decode-sized batches): one wave, no barriers.  Lane i owns assignment i; ranks,
// offsets and chunk positions are counted with readlane loops over the other lanes.  Same outputs as above.
__device__ __forceinline__ void sort_small(uint32_t lane, uint32_t n, uint32_t e, uint32_t E, uint32_t top_k,
                                           uint32_t* __restrict__ sorted, uint32_t* __restrict__ sorted_tok,
                                           uint32_t* __restrict__ inv, uint32_t* __restrict__ counts,
                                           uint32_t* __restrict__ offsets, uint32_t* __restrict__ chunk_tab,
                                           uint32_t* __restrict__ n_chunks) {
  const bool valid = e < E;  // (lanes past the n assignments hold an invalid expert)
  uint32_t rank = 0, same = 0, less = 0, n_valid = 0;
  for (int j = 0; j < (int)n; ++j) {
    const uint32_t ej = (uint32_t)__builtin_amdgcn_readlane((int)e, j);
    if (ej >= E) continue;  // uniform
    ++n_valid;
    same += ej == e ? 1u : 0u;
    rank += (ej == e && j < (int)lane) ? 1u : 0u;
    less += ej < e ? 1u : 0u;
  }
  const uint32_t pos = less + rank;
  if (valid && sorted != nullptr) {
    sorted[pos] = lane;
    if (sorted_tok != nullptr) sorted_tok[pos] = lane / top_k;
    if (inv != nullptr) inv[lane] = pos;
  }
  if (!valid && lane < n && inv != nullptr) inv[lane] = 0xFFFFFFFFu;  // skipped by the combine step
  // the first assignment of every expert writes the expert's chunks; chunks of lower experts come first
  const bool leader = valid && rank == 0;
  const uint32_t my_chunks = leader ? (same + 7) / 8 : 0u;
  uint32_t chunks_before = 0, total_chunks = 0;
  for (int j = 0; j < (int)n; ++j) {
    const uint32_t cj = (uint32_t)__builtin_amdgcn_readlane((int)my_chunks, j);
    if (cj == 0) continue;  // uniform
    const uint32_t ej = (uint32_t)__builtin_amdgcn_readlane((int)e, j);
    total_chunks += cj;
    chunks_before += ej < e ? cj : 0u;
  }
  if (leader && chunk_tab != nullptr) {
    for (uint32_t c = 0; c < my_chunks; ++c) {
      chunk_tab[3 * (chunks_before + c) + 0] = e;
      chunk_tab[3 * (chunks_before + c) + 1] = less + 8 * c;
      chunk_tab[3 * (chunks_before + c) + 2] = same - 8 * c < 8u ? same - 8 * c : 8u;
    }
  }
  if (lane == 0 && n_chunks != nullptr) *n_chunks = total_chunks;
  if (counts != nullptr || offsets != nullptr) {
    for (uint32_t ee = lane; ee < E; ee += 64) {
      uint32_t c = 0, o = 0;
      for (int j = 0; j < 64; ++j) {
        const uint32_t ej = (uint32_t)__builtin_amdgcn_readlane((int)e, j);
        c += ej == ee ? 1u : 0u;
        o += ej < ee ? 1u : 0u;
      }
      if (counts != nullptr) counts[ee] = c;
      if (offsets != nullptr) offsets[ee] = o;
    }
    if (lane == 0 && offsets != nullptr) offsets[E] = n_valid;
  }
}

__global__ __launch_bounds__(64) void moe_sort_small_kernel(const uint32_t* __restrict__ idx, uint32_t n_assign,
                                                            uint32_t E, uint32_t top_k, uint32_t* __restrict__ sorted,
                                                            uint32_t* __restrict__ sorted_tok,
                                                            uint32_t* __restrict__ inv, uint32_t* __restrict__ counts,
                                                            uint32_t* __restrict__ offsets,
                                                            uint32_t* __restrict__ chunk_tab,
                                                            uint32_t* __restrict__ n_chunks) {
  const uint32_t lane = threadIdx.x;
  sort_small(lane, n_assign, lane < n_assign ? idx[lane] : 0xFFFFFFFFu, E, top_k, sorted, sorted_tok, inv, counts, offsets,
             chunk_tab, n_chunks);
}

// Routing and grouping of a decode-sized batch in one launch: at most 8 tokens and 64 assignments.  Wave t
// routes token t and leaves its picks in workgroup memory; after the barrier wave 0 sorts them.
__global__ __launch_bounds__(512) void route_sort_small_kernel(const float* __restrict__ logits,
                                                               const float* __restrict__ bias, uint32_t T, uint32_t E,
                                                               uint32_t K, int renorm, uint32_t* __restrict__ out_idx,
                                                               float* __restrict__ out_w, uint32_t* __restrict__ sorted,
                                                               uint32_t* __restrict__ sorted_tok,
                                                               uint32_t* __restrict__ inv,
                                                               uint32_t* __restrict__ chunk_tab,
                                                               uint32_t* __restrict__ n_chunks) {
  __shared__ uint32_t picks[64];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave < T) route_token(logits, bias, E, K, renorm, out_idx, out_w, wave, lane, picks);
  __syncthreads();
  if (wave == 0)
    sort_small(lane, T * K, lane < T * K ? picks[lane] : 0xFFFFFFFFu, E, K, sorted, sorted_tok, inv, nullptr, nullptr,
               chunk_tab, n_chunks);
}

__global__ void index_gather_kernel(const __half* __restrict__ src, uint32_t d, const uint32_t* __restrict__ idx,
                                    uint32_t src_rows, __half* __restrict__ dst) {
  const uint32_t i = blockIdx.x;
  const uint32_t r = idx[i];
  for (uint32_t c = threadIdx.x; c < d; c += blockDim.x)
    dst[(size_t)i * d + c] = r < src_rows ? src[(size_t)r * d + c] : __float2half(0.f);
}

// One workgroup per destination row: assignments are visited in ascending order, so the f32
// sum of a row is reproducible.
__global__ void scatter_weighted_add_kernel(const __half* __restrict__ src, uint32_t n, uint32_t d,
                                            const uint32_t* __restrict__ tok, const float* __restrict__ w,
                                            __half* __restrict__ dst) {
  const uint32_t t = blockIdx.x;
  for (uint32_t c = threadIdx.x; c < d; c += blockDim.x) {
    float acc = __half2float(dst[(size_t)t * d + c]);
    for (uint32_t i = 0; i < n; ++i)
      if (tok[i] == t) acc += w[i] * __half2float(src[(size_t)i * d + c]);
    dst[(size_t)t * d + c] = __float2half(acc);
  }
}

__global__ void silu_gate_kernel(const __half* __restrict__ g, const __half* __restrict__ u,
                                 __half* __restrict__ out, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    const float x = __half2float(g[i]);
    out[i] = __float2half(x / (1.0f + __expf(-x)) * __half2float(u[i]));
  }
}

// out[r, c] = silu(g[r*ld + c]) * u[r*ld + c]: gate and up halves of one [rows, ld] matrix
__global__ void silu_gate_strided_kernel(const __half* __restrict__ g, const __half* __restrict__ u, uint32_t ld,
                                         __half* __restrict__ out, uint32_t rows, uint32_t cols) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x, n = (size_t)rows * cols;
  for (; i < n; i += stride) {
    const size_t r = i / cols, c = i % cols;
    const float x = __half2float(g[r * ld + c]);
    out[i] = __float2half(x / (1.0f + __expf(-x)) * __half2float(u[r * ld + c]));
  }
}

// assignments in their own order: token of assignment a is a / top_k, its position is a
__global__ void identity_positions_kernel(uint32_t* __restrict__ tok, uint32_t* __restrict__ inv, uint32_t n, uint32_t top_k) {
  const uint32_t a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a < n) {
    tok[a] = a / top_k;
    inv[a] = a;
  }
}

// out[t,:] = sum_k w[t*K+k] * y[inv[t*K+k],:], k ascending, f32.  grid = (T, column blocks of 1024):
// every thread owns four columns, loads its rows of all top_k experts first and sums in order.  Bound by the rows of y, which are read once (2048
// tokens of 8 experts, D = 4096: 285 MB in 46 us, 6.2 TB/s; 55 us with loads that stay in the caches).
// Assignments whose position is not below n_rows (the grouping kernels mark an expert id outside
// [0, E) that way) contribute nothing.
typedef float f4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ y,
                                                          const uint32_t* __restrict__ inv,
                                                          const float* __restrict__ weights, uint32_t top_k,
                                                          uint32_t D, uint32_t n_rows, __half* __restrict__ out) {
  const uint32_t t = blockIdx.x;
  const uint32_t c = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c >= D) return;
  float w[8];
  float4 v[8];
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    w[k] = 0.f;
    v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (k < top_k) {
      const uint32_t pos = inv[(size_t)t * top_k + k];
      if (pos < n_rows) {
        w[k] = weights[(size_t)t * top_k + k];
        const f4 r = __builtin_nontemporal_load(reinterpret_cast<const f4*>(y + (size_t)pos * D + c));  // (read once)
        v[k] = make_float4(r[0], r[1], r[2], r[3]);
      }
    }
  }
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    if (k < top_k) { acc.x += w[k] * v[k].x; acc.y += w[k] * v[k].y; acc.z += w[k] * v[k].z; acc.w += w[k] * v[k].w; }
  }
  const __half2 lo = __floats2half2_rn(acc.x, acc.y), hi = __floats2half2_rn(acc.z, acc.w);
  uint2 o;
  o.x = *reinterpret_cast<const uint32_t*>(&lo);
  o.y = *reinterpret_cast<const uint32_t*>(&hi);
  *reinterpret_cast<uint2*>(out + (size_t)t * D + c) = o;
}

// The same sum over f16 rows in assignment order (no grouping: row t*K+k is pick k of token t): out[t,:] = sum_k
// w[t*K+k] * y[t*K+k,:], k ascending, f32; an assignment whose expert id lies outside [0, E) contributes nothing.
__global__ __launch_bounds__(256) void moe_combine_rows_f16_kernel(const __half* __restrict__ y,
                                                                   const uint32_t* __restrict__ idx,
                                                                   const float* __restrict__ weights, uint32_t top_k,
                                                                   uint32_t D, uint32_t E, __half* __restrict__ out) {
  const uint32_t t = blockIdx.x;
  const uint32_t c = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c >= D) return;
  float w[8];
  uint2 v[8];
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    w[k] = 0.f;
    v[k] = make_uint2(0u, 0u);
    if (k < top_k) {
      const size_t a = (size_t)t * top_k + k;
      if (idx[a] < E) {
        w[k] = weights[a];
        v[k] = *reinterpret_cast<const uint2*>(y + a * D + c);
      }
    }
  }
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    if (k < top_k) {
      const float2 lo = __half22float2(*reinterpret_cast<const __half2*>(&v[k].x)), hi = __half22float2(*reinterpret_cast<const __half2*>(&v[k].y));
      acc.x += w[k] * lo.x; acc.y += w[k] * lo.y; acc.z += w[k] * hi.x; acc.w += w[k] * hi.y;
    }
  }
  const __half2 lo = __floats2half2_rn(acc.x, acc.y), hi = __floats2half2_rn(acc.z, acc.w);
  uint2 o;
  o.x = *reinterpret_cast<const uint32_t*>(&lo);
  o.y = *reinterpret_cast<const uint32_t*>(&hi);
  *reinterpret_cast<uint2*>(out + (size_t)t * D + c) = o;
}

}  // namespace

int32_t launch_topk_route(const float* logits, const float* bias, uint32_t T, uint32_t E, uint32_t K,
                          int renorm, uint32_t* idx, float* w, uint32_t* counts, uint32_t* offsets,
                          hipStream_t s) {
  if (T > 0) {
    hipLaunchKernelGGL(topk_route_kernel, dim3(T), dim3(64), 0, s, logits, bias, E, K, renorm, idx, w);
    RMLX_HIP_CHECK(hipGetLastError());
  }
  if ((counts != nullptr || offsets != nullptr) && T * K <= 64 && E <= (uint32_t)kMaxExperts) {
    hipLaunchKernelGGL(moe_sort_small_kernel, dim3(1), dim3(64), 0, s, idx, T * K, E, K, (uint32_t*)nullptr,
                       (uint32_t*)nullptr, (uint32_t*)nullptr, counts, offsets, (uint32_t*)nullptr,
                       (uint32_t*)nullptr);
    RMLX_HIP_CHECK(hipGetLastError());
  } else if (counts != nullptr || offsets != nullptr) {
    hipLaunchKernelGGL(moe_sort_kernel<false>, dim3(1), dim3(1024), 0, s, idx, T * K, E, K, (uint32_t*)nullptr,
                       (uint32_t*)nullptr, (uint32_t*)nullptr, counts, offsets, (uint32_t*)nullptr,
                       (uint32_t*)nullptr, 8u, (uint32_t*)nullptr, (uint32_t*)nullptr, 0u, (T * K + 1023) / 1024 * 1024);
    RMLX_HIP_CHECK(hipGetLastError());
  }
  return RMLX_OK;
}

bool route_sort_fusable(uint32_t T, uint32_t E, uint32_t K) {
  return T >= 1 && T <= 8 && T * K <= 64 && E <= 256 && K >= 1 && K <= 8;
}

int32_t launch_route_sort_small(const float* logits, const float* bias, uint32_t T, uint32_t E, uint32_t K,
                                int renorm, uint32_t* idx, float* w, uint32_t* sorted, uint32_t* sorted_tok,
                                uint32_t* inv, uint32_t* chunk_tab, uint32_t* n_chunks, hipStream_t s) {
  if (!route_sort_fusable(T, E, K)) return fail(RMLX_RUNTIME_ERROR, "route_sort_small: T=%u E=%u K=%u not supported", T, E, K);
  hipLaunchKernelGGL(route_sort_small_kernel, dim3(1), dim3(64 * T), 0, s, logits, bias, T, E, K, renorm, idx, w, sorted,
                     sorted_tok, inv, chunk_tab, n_chunks);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

// Assignments per workgroup of the sort: one workgroup for every 1024 assignments, at most 32, their equal shares rounded up to whole 1024s (a
// wave's run is whole 64s).  So a number a little past a step leaves the last ones little or nothing: 2049 are 2048 and 1, 32769 are 16 portions
// of 2048 and one of 1.
static uint32_t sort_portion(uint32_t n_assign) {
  const uint32_t wgs = n_assign / 1024 < 1 ? 1 : (n_assign / 1024 > 32 ? 32 : n_assign / 1024), each = (n_assign + wgs - 1) / wgs;
  return (each + 1023) / 1024 * 1024;
}

int32_t launch_moe_sort(const uint32_t* idx, uint32_t n_assign, uint32_t E, uint32_t top_k, uint32_t* sorted,
                        uint32_t* sorted_tok, uint32_t* inv, uint32_t* counts, uint32_t* offsets,
                        uint32_t* chunk_tab, uint32_t* n_chunks, uint32_t chunk_rows, hipStream_t s, uint32_t* split_tab,
                        uint32_t* split_n, uint32_t split_cap) {
  if (E > (uint32_t)kMaxExperts)
    return fail(RMLX_INVALID_SHAPE, "moe_sort: n_experts (%u) exceeds maximum %d", E, kMaxExperts);
  if (chunk_rows == 0) return fail(RMLX_RUNTIME_ERROR, "moe_sort: chunk_rows must be non-zero");
  if (n_assign <= 64 && chunk_rows == 8 && split_tab == nullptr)  // the one-wave kernel writes chunks of 8 rows
    hipLaunchKernelGGL(moe_sort_small_kernel, dim3(1), dim3(64), 0, s, idx, n_assign, E, top_k ? top_k : 1u, sorted,
                       sorted_tok, inv, counts, offsets, chunk_tab, n_chunks);
  else {
    const uint32_t portion = sort_portion(n_assign), wgs = n_assign == 0 ? 1 : (n_assign + portion - 1) / portion;
    hipLaunchKernelGGL(wgs > 1 ? moe_sort_kernel<true> : moe_sort_kernel<false>, dim3(wgs), dim3(1024), 0, s, idx, n_assign, E, top_k ? top_k : 1u,
                       sorted, sorted_tok, inv, counts, offsets, chunk_tab, n_chunks, chunk_rows, split_tab, split_n, split_cap, portion);
  }
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

int32_t launch_index_gather(const __half* src, uint32_t d, const uint32_t* idx, uint32_t n, uint32_t src_rows,
                            __half* dst, hipStream_t s) {
  if (n == 0 || d == 0) return RMLX_OK;
  hipLaunchKernelGGL(index_gather_kernel, dim3(n), dim3(256), 0, s, src, d, idx, src_rows, dst);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

int32_t launch_scatter_weighted_add(const __half* src, uint32_t n, uint32_t d, const uint32_t* tok,
                                    const float* w, __half* dst, uint32_t dst_rows, hipStream_t s) {
  if (n == 0 || d == 0 || dst_rows == 0) return RMLX_OK;
  hipLaunchKernelGGL(scatter_weighted_add_kernel, dim3(dst_rows), dim3(256), 0, s, src, n, d, tok, w, dst);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

int32_t launch_silu_gate(const __half* g, const __half* u, __half* out, size_t n, hipStream_t s) {
  if (n == 0) return RMLX_OK;
  size_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(silu_gate_kernel, dim3((unsigned)blocks), dim3(256), 0, s, g, u, out, n);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

int32_t launch_silu_gate_strided(const __half* g, const __half* u, uint32_t ld, __half* out, uint32_t rows,
                                 uint32_t cols, hipStream_t s) {
  const size_t n = (size_t)rows * cols;
  if (n == 0) return RMLX_OK;
  size_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(silu_gate_strided_kernel, dim3((unsigned)blocks), dim3(256), 0, s, g, u, ld, out, rows, cols);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

int32_t launch_identity_positions(uint32_t* tok, uint32_t* inv, uint32_t n, uint32_t top_k, hipStream_t s) {
  if (n == 0) return RMLX_OK;
  hipLaunchKernelGGL(identity_positions_kernel, dim3((n + 255) / 256), dim3(256), 0, s, tok, inv, n, top_k);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

int32_t launch_moe_combine(const float* y, const uint32_t* inv, const float* weights, uint32_t T, uint32_t top_k,
                           uint32_t D, __half* out, hipStream_t s) {
  if (T == 0) return RMLX_OK;
  if (top_k > 8 || D % 4 != 0) return fail(RMLX_INVALID_SHAPE, "moe_combine: top_k <= 8 and D %% 4 == 0 required (top_k=%u D=%u)", top_k, D);
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T, (D + 1023) / 1024), dim3(256), 0, s, y, inv, weights, top_k, D, T * top_k, out);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

int32_t launch_moe_combine_rows_f16(const __half* y, const uint32_t* idx, const float* weights, uint32_t T, uint32_t top_k,
                                    uint32_t D, uint32_t E, __half* out, hipStream_t s) {
  if (T == 0) return RMLX_OK;
  if (top_k > 8 || D % 4 != 0) return fail(RMLX_INVALID_SHAPE, "moe_combine: top_k <= 8 and D %% 4 == 0 required (top_k=%u D=%u)", top_k, D);
  hipLaunchKernelGGL(moe_combine_rows_f16_kernel, dim3(T, (D + 1023) / 1024), dim3(256), 0, s, y, idx, weights, top_k, D, E, out);
  RMLX_HIP_CHECK(hipGetLastError());
  return RMLX_OK;
}

}  // namespace rmlx
