// Grouped quantized matmul over expert segments (the gather-qmm of the MoE block), for gfx950.
//
// out[p, n] = sum_k act[row(p), k] * W_e[n, k]  for every sorted position p in expert e's
// segment, where W_e is affine int4 g64 (w = s*q + b, bf16 s/b per 64 along k) or bf16.
// Epilogues: fused SwiGLU over the gate|up row halves (-> bf16 h), plain bf16, or float32.
//
// Reference: mx.gather_qmm(x, packed, scale, bias, rhs_indices=exp, transpose=True,
// group_size=64, bits=4) at src/quanta/qwen35/moe.py:117-123 and the sorted variant
// src/quanta/dsv4/moe.py:114-124; SwiGLU src/quanta/qwen35/moe.py:59-63 (gate = first I rows,
// up = last I rows); bf16 sibling mx.gather_mm src/quanta/qwen35/moe.py:66-82; the shared
// expert's dense bf16 matmuls src/quanta/qwen35/moe.py:145-151; router logits
// src/quanta/qwen35/moe.py:47.
//
// Two regimes, activations as the MFMAs' A operand (token rows) and weights as the B operand (weight
// rows as columns):
//  * small-M ("decode"): 16x16x32 MFMAs, 16-token m-tiles; each wavefront streams one 16-row weight tile (two
//    for SwiGLU) straight from HBM into registers with one contiguous 1 KiB dwordx4 load per
//    superblock, and never materialises a dequantised weight. For int4 it multiplies the raw
//    codes (as bf16 128+q, exact) on v_mfma_f32_16x16x32_bf16 and applies the per-group affine
//    map on the 16x16 result:
//      sum_k x_k (s q_k + b) = s * sum_k x_k (128+q_k) + (b - 128 s) * sum_k x_k,
//    with sum_k x_k from one extra MFMA against a ones fragment. Optional split-K across the
//    workgroup's wavefronts, reduced through LDS.
//  * large-M ("prefill"): prefill.hip.
#include <type_traits>

#include "qmoe_internal.h"
#include "route_common.h"
#include "small_body.h"
#include "../../include/quanta_moe.h"

namespace qmoe {

// (SlotRoute, resolve_mtile, act_row, store_out and small_body live in small_body.h)

template <int FMT, int EPI, int W, int CPW, int JPW, int MT>
__global__ void __launch_bounds__(W > 4 ? 64 * W : 256)
__attribute__((amdgpu_waves_per_eu(SmallCfg<FMT, EPI, W, CPW, JPW>::WPE)))
qmm_small_kernel(QmmArgs a, int n_jobs) {
  __shared__ f32x4_t red[SmallCfg<FMT, EPI, W, CPW, JPW, MT>::RED];
  small_body<FMT, EPI, W, CPW, JPW, MT>(a, n_jobs, blockIdx.x, blockIdx.y, red);
}

// The routed gate_up of a slot-major batch with its routing (grid.y = N*k slots).
template <int W, int JPW, int VPL, int DEEP>
__global__ void __launch_bounds__(W > 4 ? 64 * W : 256)
__attribute__((amdgpu_waves_per_eu(SmallCfg<FMT_INT4, EPI_SWIGLU, W, 1, JPW>::WPE)))
qmm_route_gate_up_kernel(QmmArgs a, int n_jobs, SlotRoute route) {
  __shared__ f32x4_t red[SmallCfg<FMT_INT4, EPI_SWIGLU, W, 1, JPW, 1>::RED];
  __shared__ u32x4 xlds[DEEP > 0 ? (W > 4 ? W : 4) * DEEP * 16 : 1];
  __shared__ int route_e;
  small_body<FMT_INT4, EPI_SWIGLU, W, 1, JPW, 1, false, VPL, DEEP>(a, n_jobs, blockIdx.x, blockIdx.y,
                                                                    red, &route, xlds, &route_e);
}

// The same with the shared expert's int8 down projection (a2: W2 * CPW2 chunks, W2 wavefronts
// per job each summing CPW2 of them, one m-tile per wavefront) in the launch, on a flat grid of
// 4-wavefront workgroups: the routed gate_up's job blocks x slots first, then the shared down's
// job blocks x m-tiles.
template <int W, int JPW, int VPL, int DEEP, int W2, int CPW2 = 1>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(SmallCfg<FMT_INT4, EPI_SWIGLU, W, 1, JPW>::WPE)))
qmm_route_gate_up_shdown_kernel(QmmArgs a, int n_jobs, SlotRoute route, int gx1, int64_t n1,
                                QmmArgs a2, int n_jobs2, int gx2) {
  static_assert(W <= 4 && W2 <= 4, "one 4-wavefront workgroup shape for both products");
  constexpr int R1 = SmallCfg<FMT_INT4, EPI_SWIGLU, W, 1, JPW, 1>::RED;
  constexpr int R2 = SmallCfg<FMT_INT8, EPI_BF16, W2, CPW2, 1, 1>::RED;
  __shared__ f32x4_t red[R1 > R2 ? R1 : R2];
  __shared__ u32x4 xlds[DEEP > 0 ? 4 * DEEP * 16 : 1];
  __shared__ int route_e;
  const int64_t b = blockIdx.x;
  if (b < n1) {
    small_body<FMT_INT4, EPI_SWIGLU, W, 1, JPW, 1, false, VPL, DEEP>(
        a, n_jobs, static_cast<int>(b % gx1), static_cast<int>(b / gx1), red, &route, xlds, &route_e);
  } else {
    const int64_t b2 = b - n1;
    small_body<FMT_INT8, EPI_BF16, W2, CPW2, 1, 1>(a2, n_jobs2, static_cast<int>(b2 % gx2),
                                                   static_cast<int>(b2 / gx2), red);
  }
}

// The routing tail (RouteTail). Counts go on tagged workspace words, (kRouteTailTag << 20) |
// count: an atomic add, and a word found without the tag (a fresh workspace) is replaced by a
// tagged count of 1 (compare-and-swap), or counted on once another workgroup has tagged it; the
// add that landed on the untagged word is discarded with it. Returns the count after this one.
__device__ __forceinline__ int tail_count(unsigned long long* w) {
  constexpr unsigned long long kMask = (1ull << 20) - 1;
  const unsigned long long old = __hip_atomic_fetch_add(w, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((old >> 20) == kRouteTailTag) return static_cast<int>((old & kMask) + 1);
  unsigned long long cur = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  unsigned long long want;
  do {
    want = ((cur >> 20) == kRouteTailTag) ? cur + 1 : ((kRouteTailTag << 20) | 1ull);
  } while (!__hip_atomic_compare_exchange_strong(w, &cur, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT));
  return static_cast<int>(want & kMask);
}

// This workgroup's stores are complete (s_waitcnt 0, then the barrier); thread 0 counts it on
// *w and the workgroup learns the count.
__device__ __forceinline__ int tail_arrive(unsigned long long* w) {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  __shared__ int s_cnt;
  if (threadIdx.x == 0) s_cnt = tail_count(w);
  __syncthreads();
  return s_cnt;
}

// Bounded wait of the workgroup until *w holds a tagged count of at least `target`; a wait that
// runs out adds to *timeouts and returns (the kernel always ends).
__device__ __forceinline__ void tail_wait(const unsigned long long* w, int target, uint32_t* timeouts) {
  if (threadIdx.x == 0) {
    uint32_t n = 0;
    for (;;) {
      const unsigned long long v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((v >> 20) == kRouteTailTag && static_cast<int>(v & ((1ull << 20) - 1)) >= target) break;
      __builtin_amdgcn_s_sleep(2);
      if (++n >= kWaitLimit) {
        __hip_atomic_fetch_add(timeouts, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
  }
  __syncthreads();
}

// Ranker r of R: tokens r, r + R, ... one wavefront each, with coherent loads of the logits; the
// top-k launch's outputs (idx coherently, read by the last ranker), and the ids into `ids` (LDS)
// when one workgroup ranks every token.
template <int VPL>
__device__ __forceinline__ void route_tail_rank(const RouteTail& T, int r, int R, int32_t* ids) {
  const int lane = threadIdx.x & 63;
  const int nw = blockDim.x >> 6;
  const int k = T.P.k;
  for (int t = r + R * (threadIdx.x >> 6); t < T.N; t += R * nw) {
    const float* row = T.logits + static_cast<int64_t>(t) * T.ld;
    // (the shared gate's logit is loaded before the ranking, so its latency overlaps it)
    const float sgl = (T.P.has_sg && lane == 0) ? logit_ld<true>(row + T.P.E) : 0.f;
    int id;
    float wsel;
    topk_token<VPL, false, true>(row, T.P, lane, id, wsel);
    if (lane < k) {
      __hip_atomic_store(T.idx + t * k + lane, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      T.w[t * k + lane] = wsel;
      if (ids) ids[t * k + lane] = id;
    }
    if (T.P.has_sg && lane == 0) T.sg[t] = 1.0f / (1.0f + expf(-sgl));
  }
}

// Exclusive scan of one value per thread across the workgroup (1 to 16 wavefronts); tmp holds
// 33 ints and is free again on return.
__device__ __forceinline__ int tail_scan(int v, int* tmp, int& total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off);
    if (lane >= off) incl += o;
  }
  if (lane == 63) tmp[wid] = incl;
  __syncthreads();
  if (wid == 0) {
    const int s = lane < nw ? tmp[lane] : 0;
    int si = s;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      const int o = __shfl_up(si, off);
      if (lane >= off) si += o;
    }
    if (lane < nw) tmp[16 + lane] = si - s;
    if (lane == nw - 1) tmp[32] = si;
  }
  __syncthreads();
  const int r = tmp[16 + wid] + incl - v;
  total = tmp[32];
  __syncthreads();
  return r;
}

// The stable permute of the N * k slots by expert (N <= 64), the permute launch's outputs for
// 16-row m-tiles: counts, offsets and the m-tile prefix (E + 1 entries each with the totals),
// the tile descriptors {expert, first sorted position, rows, 0} with -1 sentinels up to
// max_tiles, and sorted / inv. A slot's stable rank within its expert is the number of earlier
// tokens that chose the expert (top-k experts of a token are distinct): the popcount of the
// expert's 64-bit token mask below the token. Thread i owns experts [i * ve, i * ve + ve).
__device__ __forceinline__ void route_tail_permute(const RouteTail& T, const int32_t* ids,
                                                   unsigned long long* mask, int* hist, int* offs,
                                                   int* tmp) {
  const int E = T.P.E, k = T.P.k, mc = T.N * k, tid = threadIdx.x, nthr = blockDim.x;
  for (int e = tid; e < E; e += nthr) {
    hist[e] = 0;
    mask[e] = 0ull;
  }
  __syncthreads();
  for (int m = tid; m < mc; m += nthr) {
    const int e = ids[m];
    atomicAdd(&hist[e], 1);
    atomicOr(&mask[e], 1ull << (m / k));
  }
  __syncthreads();
  const int ve = (E + nthr - 1) / nthr;   // at most 2 (E <= 512 and 256 threads or more)
  int c[2], rows = 0, tiles = 0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int e = tid * ve + j;
    c[j] = (j < ve && e < E) ? hist[e] : 0;
    rows += c[j];
    tiles += (c[j] + kSmallMTile - 1) / kSmallMTile;
  }
  int rows_total, tiles_total;
  int ex = tail_scan(rows, tmp, rows_total);
  int tex = tail_scan(tiles, tmp, tiles_total);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int e = tid * ve + j;
    if (j >= ve || e >= E) break;
    T.counts[e] = c[j];
    T.offsets[e] = ex;
    T.tile_off[e] = tex;
    offs[e] = ex;
    const int nt = (c[j] + kSmallMTile - 1) / kSmallMTile;
    for (int i = 0; i < nt; ++i)
      reinterpret_cast<int4*>(T.tile_map)[tex + i] =
          make_int4(e, ex + i * kSmallMTile, min(kSmallMTile, c[j] - i * kSmallMTile), 0);
    ex += c[j];
    tex += nt;
  }
  if (tid == 0) {
    T.offsets[E] = rows_total;
    T.tile_off[E] = tiles_total;
  }
  for (int t = tiles_total + tid; t < T.max_tiles; t += nthr)
    reinterpret_cast<int4*>(T.tile_map)[t] = make_int4(-1, 0, 0, 0);
  __syncthreads();
  for (int m = tid; m < mc; m += nthr) {
    const int e = ids[m], t = m / k;
    const int pos = offs[e] + __popcll(mask[e] & ((1ull << t) - 1ull));
    T.sorted[pos] = m;
    T.inv[m] = pos;
  }
}

// The rankers' part of the tail; the last ranker to finish then sorts the slots by expert and
// resets the counters.
__device__ __forceinline__ void route_tail_run(const RouteTail& T, int r, int R) {
  // dynamic LDS: token masks [E] (8 bytes each), histogram [E], offsets [E], scan scratch [34],
  // slot ids [N * k]
  extern __shared__ unsigned long long tail_lds[];
  unsigned long long* mask = tail_lds;
  int* hist = reinterpret_cast<int*>(mask + T.P.E);
  int* offs = hist + T.P.E;
  int* tmp = offs + T.P.E;
  int32_t* ids = tmp + 34;
  int32_t* own = (R == 1) ? ids : nullptr;
  switch (T.vpl) {
    case 1: route_tail_rank<1>(T, r, R, own); break;
    case 2: route_tail_rank<2>(T, r, R, own); break;
    case 4: route_tail_rank<4>(T, r, R, own); break;
    default: route_tail_rank<8>(T, r, R, own); break;
  }
  if (R > 1) {
    if (tail_arrive(T.ctr + 1) != R) return;
    // the last ranker: every slot's expert, from the rankers' coherent stores
    for (int m = threadIdx.x; m < T.N * T.P.k; m += blockDim.x)
      ids[m] = static_cast<int32_t>(__hip_atomic_load(T.idx + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }
  __syncthreads();
  route_tail_permute(T, ids, mask, hist, offs, tmp);
  if (threadIdx.x == 0) {
    __hip_atomic_store(T.ctr, kRouteTailTag << 20, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(T.ctr + 1, kRouteTailTag << 20, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Two dense products over the same activation rows in one launch (the router logits, tiled
// bf16, and the shared expert's gate_up, tiled bf16 or int8 as FMT2): job blocks [0, gx1) run
// the first, the rest the second. Both use the same K, so the same chunking W, and each keeps the
// arithmetic of its own launch.
// NORM: both products RMSNorm their activation rows on the fly (QmmArgs::norm_w), and the first
// product's job 0 writes the normalised rows (norm_out).
// TAIL: the routing tail (RouteTail) after the router workgroups' products.
template <int EPI1, int EPI2, int W, int MT, bool NORM = false, int FMT2 = FMT_BF16, bool TAIL = false>
__global__ void __launch_bounds__(W > 4 ? 64 * W : 256)
qmm_small_pair_kernel(QmmArgs a1, int n_jobs1, int gx1, QmmArgs a2, int n_jobs2, RouteTail T) {
  constexpr int R1 = SmallCfg<FMT_BF16, EPI1, W, 1, 1, MT>::RED;
  constexpr int R2 = SmallCfg<FMT2, EPI2, W, 1, 1, MT>::RED;
  constexpr int RR = R1 > R2 ? R1 : R2;
  // (NORM: behind the chunk sums, the norm's chunk sums [WAVES][MT][16] floats)
  constexpr int WAVES = W > 4 ? W : 4;
  __shared__ f32x4_t red[RR + (NORM ? (WAVES * MT * 16 + 3) / 4 : 0)];
  // the decode dataflow kernel's counters (kSyncStride words apart), cleared for the launch that
  // follows this one
  if (a1.zero_words && blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = threadIdx.x; i < a1.n_zero; i += blockDim.x) a1.zero_words[i * kSyncStride] = 0u;
  if (static_cast<int>(blockIdx.x) < gx1) {
    // (TAIL: the logits go out with coherent stores, read by the last router workgroup)
    small_body<FMT_BF16, EPI1, W, 1, 1, MT, NORM, 0, 0, TAIL ? kCohOut : 0>(a1, n_jobs1, blockIdx.x,
                                                                          blockIdx.y, red);
    if constexpr (TAIL) {
      // the last R router workgroups to finish rank the tokens, the first of them once all
      // router workgroups have stored their logits
      const int arrival = tail_arrive(T.ctr);
      if (arrival > T.total - T.rankers) {
        if (T.rankers > 1) tail_wait(T.ctr, T.total, T.timeouts);
        route_tail_run(T, T.total - arrival, T.rankers);
      }
    }
  } else {
    small_body<FMT2, EPI2, W, 1, 1, MT, NORM>(a2, n_jobs2, blockIdx.x - gx1, blockIdx.y, red);
  }
}

// The routed gate_up (int4 SwiGLU over the permuted m-tiles, small-regime shape W/CPW/JPW) and
// the shared expert's down projection (int8 codes, K = its intermediate size, one dense segment
// of N rows; W2 * CPW2 chunks, W2 wavefronts per job each summing CPW2 of them, MT2 m-tiles per
// wavefront) in one launch of 4-wavefront workgroups on a flat grid: the gate_up's job blocks x
// m-tiles first, the shared down's after them. Each keeps the arithmetic of its own launch, so
// the outputs are those of the two launches bit for bit.
template <int W, int CPW, int JPW, int W2, int MT2, int CPW2 = 1>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(SmallCfg<FMT_INT4, EPI_SWIGLU, W, CPW, JPW>::WPE)))
qmm_gate_up_shdown_kernel(QmmArgs a1, int n_jobs1, int gx1, int64_t n1, QmmArgs a2, int n_jobs2,
                          int gx2) {
  constexpr int R1 = SmallCfg<FMT_INT4, EPI_SWIGLU, W, CPW, JPW, 1>::RED;
  constexpr int R2 = SmallCfg<FMT_INT8, EPI_BF16, W2, CPW2, 1, MT2>::RED;
  __shared__ f32x4_t red[R1 > R2 ? R1 : R2];
  const int64_t b = blockIdx.x;
  if (b < n1) {
    small_body<FMT_INT4, EPI_SWIGLU, W, CPW, JPW, 1>(a1, n_jobs1, static_cast<int>(b % gx1),
                                                     static_cast<int>(b / gx1), red);
  } else {
    const int64_t b2 = b - n1;
    small_body<FMT_INT8, EPI_BF16, W2, CPW2, 1, MT2>(a2, n_jobs2, static_cast<int>(b2 % gx2),
                                                     static_cast<int>(b2 / gx2), red);
  }
}

// ---------------------------------------------------------------- fp16 activation copy
// One wavefront per row, the row held in registers (RPL 16-byte pieces per lane): absmax by a
// wavefront reduction, then act16 = fp16(act * 2^(14 - e)) with 2^(e-1) <= absmax < 2^e, so every
// value sits below 2^14 and all bf16 values within 2^28 of the row maximum convert exactly.
// row_sinv = 2^(e - 14) undoes it on the product (a power of two: exact). The maximum is exact in
// any order, so the result does not depend on the launch shape.
// With a HotRows filter only the hot experts' sorted rows are read and written (a cold row may still be
// being written by the other chain): three dependent loads per row.
__device__ __forceinline__ bool act16_skip(int64_t row, const HotRows& hot) {
  return hot.sorted && hot.counts[hot.idx[hot.sorted[row]]] <= hot.split;
}
template <int RPL>
__global__ void __launch_bounds__(256) act_to_f16_kernel(const uint16_t* __restrict__ act, int K,
                                                         int64_t rows,
                                                         uint16_t* __restrict__ act16,
                                                         float* __restrict__ row_sinv, HotRows hot) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows || act16_skip(row, hot)) return;   // whole wavefront
  const u32x4* src = reinterpret_cast<const u32x4*>(act + row * K);
  const int n8 = K / 8;
  u32x4 v[RPL];
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int c = lane + 64 * i;
    v[i] = (c < n8) ? src[c] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      m = fmaxf(m, fabsf(bf16lo_to_f32(v[i][j])));
      m = fmaxf(m, fabsf(bf16hi_to_f32(v[i][j])));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  int ex = 0;
  if (m > 0.f && m <= 3.4e38f) frexpf(m, &ex);   // m = f * 2^ex, f in [0.5, 1)
  const int sh = (m > 0.f && m <= 3.4e38f) ? 14 - ex : 0;
  if (lane == 0) row_sinv[row] = ldexpf(1.0f, -sh);
  u32x4* dst = reinterpret_cast<u32x4*>(act16 + row * K);
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int c = lane + 64 * i;
    if (c < n8) {
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f16x2_t h = {static_cast<_Float16>(ldexpf(bf16lo_to_f32(v[i][j]), sh)),
                           static_cast<_Float16>(ldexpf(bf16hi_to_f32(v[i][j]), sh))};
        o[j] = __builtin_bit_cast(uint32_t, h);
      }
      dst[c] = o;
    }
  }
}

// Rows longer than 8192: one workgroup per row, the row read twice (absmax, then convert).
__global__ void __launch_bounds__(256) act_to_f16_wide_kernel(const uint16_t* __restrict__ act, int K,
                                                         uint16_t* __restrict__ act16,
                                                         float* __restrict__ row_sinv, HotRows hot) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  if (act16_skip(row, hot)) return;   // whole workgroup
  const u32x4* src = reinterpret_cast<const u32x4*>(act + row * K);
  const int n8 = K / 8;
  float m = 0.f;
  for (int i = threadIdx.x; i < n8; i += 256) {
    const u32x4 v = src[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      m = fmaxf(m, fabsf(bf16lo_to_f32(v[j])));
      m = fmaxf(m, fabsf(bf16hi_to_f32(v[j])));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  int ex = 0;
  if (m > 0.f && m <= 3.4e38f) frexpf(m, &ex);   // m = f * 2^ex, f in [0.5, 1)
  const int sh = (m > 0.f && m <= 3.4e38f) ? 14 - ex : 0;
  if (threadIdx.x == 0) row_sinv[row] = ldexpf(1.0f, -sh);
  u32x4* dst = reinterpret_cast<u32x4*>(act16 + row * K);
  for (int i = threadIdx.x; i < n8; i += 256) {
    const u32x4 v = src[i];
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f16x2_t h = {static_cast<_Float16>(ldexpf(bf16lo_to_f32(v[j]), sh)),
                         static_cast<_Float16>(ldexpf(bf16hi_to_f32(v[j]), sh))};
      o[j] = __builtin_bit_cast(uint32_t, h);
    }
    dst[i] = o;
  }
}

int launch_act_to_f16(const uint16_t* act, int64_t rows, int K, uint16_t* act16, float* row_sinv,
                      hipStream_t stream, const HotRows& hot) {
  if (rows <= 0) return 0;
  if (K % 8) return fail("act_to_f16: K % 8 == 0 required");
  if (K > 8 * 64 * 16) {
    if (rows > 0x7fffffff) return fail("act_to_f16: too many rows");
    act_to_f16_wide_kernel<<<static_cast<unsigned>(rows), 256, 0, stream>>>(act, K, act16, row_sinv, hot);
    return check_launch("act_to_f16");
  }
  if (rows > (int64_t(1) << 32)) return fail("act_to_f16: too many rows");
  const int rpl = (K / 8 + 63) / 64;   // 16-byte pieces per lane
#define QMOE_A16(R) act_to_f16_kernel<R><<<grid, 256, 0, stream>>>(act, K, rows, act16, row_sinv, hot)
  const unsigned grid = static_cast<unsigned>((rows + 3) / 4);
  if (rpl <= 2) QMOE_A16(2);
  else if (rpl <= 4) QMOE_A16(4);
  else if (rpl <= 8) QMOE_A16(8);
  else if (rpl <= 14) QMOE_A16(14);
  else QMOE_A16(16);
#undef QMOE_A16
  return check_launch("act_to_f16");
}


// ============================================================================ launcher
// Small-kernel launch shape. The chunk count CH depends on K only (the summation order); the
// launch picks how many 16-row tiles a wavefront streams (JPW) and how many wavefronts share a
// job's chunks (W = CH or CH / 2, so CPW = 1 or 2): the most work per wavefront that still
// leaves kSmallMinWaves wavefronts, else the most wavefronts.
constexpr int64_t kSmallMinWaves = 5120;
// Fewest m-tiles for which dense bf16 products run two m-tiles per wavefront.
constexpr int64_t kSmallMt2MinTiles = 4;
template <int FMT, int EPI, int W, int CPW, int JPW>
static void launch_small_k(const QmmArgs& a, int64_t mtiles, hipStream_t stream) {
  constexpr int WAVES = W > 4 ? W : 4;
  const int n_jobs = ((EPI == EPI_SWIGLU) ? a.n_rows / 32 : a.n_rows / 16) / JPW;
  const int jobs_per_wg = WAVES / W;
  // dense products over kSmallMt2MinTiles or more m-tiles: two per wavefront (weights read, and
  // int8 weights dequantized, once per 32 rows; below that, halving the grid leaves CUs idle)
  if constexpr (fmt_dense(FMT)) {
    if (mtiles >= kSmallMt2MinTiles && !a.offsets && !a.tile_map) {
      dim3 grid((n_jobs + jobs_per_wg - 1) / jobs_per_wg, static_cast<unsigned>((mtiles + 1) / 2));
      qmm_small_kernel<FMT, EPI, W, CPW, JPW, 2><<<grid, 64 * WAVES, 0, stream>>>(a, n_jobs);
      return;
    }
  }
  dim3 grid((n_jobs + jobs_per_wg - 1) / jobs_per_wg, static_cast<unsigned>(mtiles));
  qmm_small_kernel<FMT, EPI, W, CPW, JPW, 1><<<grid, 64 * WAVES, 0, stream>>>(a, n_jobs);
}

struct SmallShape {
  int jpw, w, cpw;
};

// (SwiGLU wavefronts hold two tiles per job: JPW 4 would exceed the register budget)
// (int6 wavefronts hold at most two tiles: four spill at the three-wavefront register budget)
static SmallShape pick_small_shape(int fmt, int epi, int ch, int64_t mtiles, int jobs) {
  if (!fmt_quant(fmt)) return SmallShape{1, ch, 1};
  const int jmax = (fmt == FMT_INT6) ? ((epi == EPI_SWIGLU) ? 1 : 2) : ((epi == EPI_SWIGLU) ? 2 : 4);
  SmallShape best{1, ch, 1};
  int64_t best_waves = mtiles * jobs * ch, best_work = 1;
  bool best_ok = best_waves >= kSmallMinWaves;
  for (int jpw = 1; jpw <= jmax; jpw *= 2) {
    if (jobs % jpw) continue;
    for (int cpw = 1; cpw <= 2 && cpw <= ch; cpw *= 2) {
      const int w = ch / cpw;
      const int64_t waves = mtiles * (jobs / jpw) * w;
      const int64_t work = static_cast<int64_t>(jpw) * cpw;
      const bool ok = waves >= kSmallMinWaves;
      const bool better = ok ? (!best_ok || work > best_work || (work == best_work && jpw > best.jpw))
                             : (!best_ok && waves > best_waves);
      if (better) {
        best = SmallShape{jpw, w, cpw};
        best_waves = waves;
        best_work = work;
        best_ok = ok;
      }
    }
  }
  return best;
}

template <int FMT, int EPI, int W, int CPW>
static void launch_small_j(const QmmArgs& a, int jpw, int64_t mtiles, hipStream_t stream) {
  if constexpr (FMT == FMT_INT6) {
    if (EPI != EPI_SWIGLU && jpw == 2)
      launch_small_k<FMT, EPI, W, CPW, (EPI == EPI_SWIGLU) ? 1 : 2>(a, mtiles, stream);
    else
      launch_small_k<FMT, EPI, W, CPW, 1>(a, mtiles, stream);
  } else if constexpr (FMT == FMT_INT4 || FMT == FMT_INT3) {
    if (EPI != EPI_SWIGLU && jpw == 4)
      launch_small_k<FMT, EPI, W, CPW, (EPI == EPI_SWIGLU) ? 2 : 4>(a, mtiles, stream);
    else if (jpw == 2)
      launch_small_k<FMT, EPI, W, CPW, 2>(a, mtiles, stream);
    else
      launch_small_k<FMT, EPI, W, CPW, 1>(a, mtiles, stream);
  } else {
    launch_small_k<FMT, EPI, W, 1, 1>(a, mtiles, stream);
  }
}

template <int FMT, int EPI>
static void launch_small(const QmmArgs& a, const SmallShape& sh, int64_t mtiles,
                         hipStream_t stream) {
  if constexpr (fmt_quant(FMT)) {
    if (sh.cpw == 2) {
      if (sh.w == 2) launch_small_j<FMT, EPI, 2, 2>(a, sh.jpw, mtiles, stream);
      else launch_small_j<FMT, EPI, 1, 2>(a, sh.jpw, mtiles, stream);
    } else {
      if (sh.w == 4) launch_small_j<FMT, EPI, 4, 1>(a, sh.jpw, mtiles, stream);
      else if (sh.w == 2) launch_small_j<FMT, EPI, 2, 1>(a, sh.jpw, mtiles, stream);
      else launch_small_j<FMT, EPI, 1, 1>(a, sh.jpw, mtiles, stream);
    }
  } else {
    switch (sh.w) {
      case 16: launch_small_j<FMT, EPI, 16, 1>(a, sh.jpw, mtiles, stream); break;
      case 8: launch_small_j<FMT, EPI, 8, 1>(a, sh.jpw, mtiles, stream); break;
      case 4: launch_small_j<FMT, EPI, 4, 1>(a, sh.jpw, mtiles, stream); break;
      case 2: launch_small_j<FMT, EPI, 2, 1>(a, sh.jpw, mtiles, stream); break;
      default: launch_small_j<FMT, EPI, 1, 1>(a, sh.jpw, mtiles, stream); break;
    }
  }
}

// Slot-major routed gate_up with its routing (qmm_route_gate_up_kernel): int4 weights, SwiGLU,
// the decode kernel's chunking (W = CH wavefronts per job, one chunk each, one tile pair each).
template <int W, int VPL>
static void launch_route_k(const QmmArgs& a, int64_t mc, const SlotRoute& R, hipStream_t stream,
                           const QmmArgs* sdn = nullptr, int w2 = 0) {
  constexpr int WAVES = W > 4 ? W : 4;
  const int n_jobs = a.n_rows / 32;
  const int jobs_per_wg = WAVES / W;
  if (sdn) {   // (the caller checked w2 and the m-tile count)
    const int gx1 = (n_jobs + jobs_per_wg - 1) / jobs_per_wg;
    const int64_t n1 = static_cast<int64_t>(gx1) * mc;
    // (eight chunks: four wavefronts of two per job)
    const int wv2 = (w2 == 8) ? 4 : w2;
    const int n_jobs2 = sdn->n_rows / 16, gx2 = (n_jobs2 + 4 / wv2 - 1) / (4 / wv2);
    const int64_t n2 = static_cast<int64_t>(gx2) * ((sdn->dense_rows + kSmallMTile - 1) / kSmallMTile);
    const dim3 g(static_cast<unsigned>(n1 + n2));
#define QMOE_RSD(D, W2_, CPW2_)                                                                  \
  qmm_route_gate_up_shdown_kernel<W, 1, VPL, D, W2_, CPW2_><<<g, 256, 0, stream>>>(a, n_jobs, R, gx1, n1, \
                                                                                 *sdn, n_jobs2, gx2)
    // (one chunk per job, W = 1, means fewer than 8 superblocks: never the deep form)
    if constexpr (W > 1) {
      if (a.K / 128 == 8 * W) {
        if (w2 == 8) QMOE_RSD(8, 4, 2); else if (w2 == 4) QMOE_RSD(8, 4, 1); else QMOE_RSD(8, 2, 1);
        return;
      }
    }
    if (w2 == 8) QMOE_RSD(0, 4, 2); else if (w2 == 4) QMOE_RSD(0, 4, 1); else QMOE_RSD(0, 2, 1);
#undef QMOE_RSD
    return;
  }
  dim3 grid((n_jobs + jobs_per_wg - 1) / jobs_per_wg, static_cast<unsigned>(mc));
  // every weight load of a wavefront's chunk in flight at once when the chunk is 8 superblocks
  if constexpr (W > 1) {
    if (a.K / 128 == 8 * W) {
      qmm_route_gate_up_kernel<W, 1, VPL, 8><<<grid, 64 * WAVES, 0, stream>>>(a, n_jobs, R);
      return;
    }
  }
  qmm_route_gate_up_kernel<W, 1, VPL, 0><<<grid, 64 * WAVES, 0, stream>>>(a, n_jobs, R);
}
template <int W>
static void launch_route_w(const QmmArgs& a, int64_t mc, const SlotRoute& R, int vpl, hipStream_t stream,
                           const QmmArgs* sdn, int w2) {
  switch (vpl) {
    case 1: launch_route_k<W, 1>(a, mc, R, stream, sdn, w2); break;
    case 2: launch_route_k<W, 2>(a, mc, R, stream, sdn, w2); break;
    case 4: launch_route_k<W, 4>(a, mc, R, stream, sdn, w2); break;
    default: launch_route_k<W, 8>(a, mc, R, stream, sdn, w2); break;
  }
}

bool route_gate_up_fits(int E, int k) { return E <= 512 && k <= 64; }

int64_t route_gate_up_workgroups(int K, int n_rows, int64_t mc) {
  const int nsb = K / 128;
  const int W = (nsb >= 32) ? 4 : (nsb >= 8) ? 2 : 1;   // launch_route_gate_up's chunking
  const int jobs_per_wg = 4 / W, n_jobs = n_rows / 32;
  return static_cast<int64_t>((n_jobs + jobs_per_wg - 1) / jobs_per_wg) * mc;
}

int launch_route_gate_up(const QmmArgs& a, int N, const float* logits, int ld, const float* bias,
                         int E, int k, int scoring, int n_group, int topk_group, int norm_topk,
                         float scale, int has_sg, int32_t* idx, float* w, float* sg,
                         int32_t* tile_map, int64_t max_tiles, int32_t* sorted, int32_t* inv,
                         hipStream_t stream, const QmmArgs* sdn) {
  const int64_t mc = static_cast<int64_t>(N) * k;
  if (!route_gate_up_fits(E, k) || a.K % 128 || a.n_rows % 32 || mc <= 0 || mc > 65535 ||
      max_tiles < mc || max_tiles > (int64_t(1) << 30) || a.slot_of || a.offsets)
    return fail("qmm(route): outside the slot-major routed gate_up");
  SlotRoute R{logits, ld, topk_params(bias, E, k, scoring, n_group, topk_group, norm_topk, scale, has_sg),
              idx, w, sg, reinterpret_cast<int4*>(tile_map), static_cast<int>(max_tiles), sorted, inv,
              static_cast<int>(mc), 1};
  const int nsb = a.K / 128;
  const int ch = (nsb >= 32) ? 4 : (nsb >= 8) ? 2 : 1;   // the int4 chunk rule of launch_qmm
  const int vpl = topk_vpl(E);
  int w2 = 0;
  if (sdn) {
    if (sdn->K % 64 || sdn->n_rows % 16 || !sdn->sb || sdn->offsets || sdn->tile_map ||
        sdn->dense_rows <= 0)
      return fail("qmm(route): the shared down is one dense int8 segment");
    w2 = bf16_chunks(sdn->K);
    // one m-tile per wavefront below kSmallMt2MinTiles m-tiles, as its own launch would run it
    if ((w2 != 2 && w2 != 4 && w2 != 8) ||
        (sdn->dense_rows + kSmallMTile - 1) / kSmallMTile >= kSmallMt2MinTiles)
      return 1;   // no compiled combination: the caller launches the shared down apart
  }
  if (ch == 4) launch_route_w<4>(a, mc, R, vpl, stream, sdn, w2);
  else if (ch == 2) launch_route_w<2>(a, mc, R, vpl, stream, sdn, w2);
  else launch_route_w<1>(a, mc, R, vpl, stream, sdn, w2);
  return check_launch("qmm(route)");
}

// SPLIT: the second product's gate and up tiles as jobs of their own with the bf16 epilogue, the
// [gate | up] rows for a consumer that forms the gated activation (the decode dataflow launch's
// H unit): twice the workgroups, each with one tile's dequant, for the launches whose time this
// product sets.
template <int W, int FMT2, bool TAIL = false, bool SPLIT = false>
static void launch_pair_w(const QmmArgs& a1, const QmmArgs& a2, int64_t mtiles, hipStream_t stream,
                          RouteTail T = RouteTail{}) {
  constexpr int WAVES = W > 4 ? W : 4;
  constexpr int JPWG = WAVES / W;
  constexpr int EPI2 = SPLIT ? EPI_BF16 : EPI_SWIGLU;
  // fp32 epilogue jobs; SwiGLU jobs (a gate and an up tile) or, split, single tiles
  const int n1 = a1.n_rows / 16, n2 = a2.n_rows / (SPLIT ? 16 : 32);
  const int gx1 = (n1 + JPWG - 1) / JPWG, gx2 = (n2 + JPWG - 1) / JPWG;
  const bool mt2 = mtiles >= kSmallMt2MinTiles;   // two m-tiles per wavefront, as in launch_small_k
  const dim3 g(gx1 + gx2, static_cast<unsigned>(mt2 ? (mtiles + 1) / 2 : mtiles));
  size_t lds = 0;
  if (TAIL) {
    T.total = gx1 * static_cast<int>(g.y);
    lds = route_tail_lds_bytes(T.P.E, T.N, T.P.k);
    // rankers: one token per workgroup (its first wavefront), up to kRouteTailMaxRankers and
    // the router workgroups; c2 at 32 tokens: 294.1 us per layer against 299.5 with one token
    // per wavefront of two rankers (16 wavefronts ranking on one compute unit take about four
    // times as long as one)
    T.rankers = std::min(std::min(T.N, kRouteTailMaxRankers), T.total);
  }
  // (NORM: the norm weights in the same dynamic LDS, used before the tail's)
  if (a1.norm_w) lds = std::max(lds, static_cast<size_t>(a1.K) * 2);
#define QMOE_PAIR(MT, NORM) \
  qmm_small_pair_kernel<EPI_F32, EPI2, W, MT, NORM, FMT2, TAIL><<<g, 64 * WAVES, lds, stream>>>(a1, n1, gx1, a2, n2, T)
  if (a1.norm_w) {
    if (mt2) QMOE_PAIR(2, true); else QMOE_PAIR(1, true);
  } else {
    if (mt2) QMOE_PAIR(2, false); else QMOE_PAIR(1, false);
  }
#undef QMOE_PAIR
}

template <int FMT2, bool SPLIT>
static void launch_pair_f(const QmmArgs& a1, const QmmArgs& a2, int64_t mtiles, hipStream_t stream) {
  switch (bf16_chunks(a1.K)) {
    case 16: launch_pair_w<16, FMT2, false, SPLIT>(a1, a2, mtiles, stream); break;
    case 8: launch_pair_w<8, FMT2, false, SPLIT>(a1, a2, mtiles, stream); break;
    case 4: launch_pair_w<4, FMT2, false, SPLIT>(a1, a2, mtiles, stream); break;
    case 2: launch_pair_w<2, FMT2, false, SPLIT>(a1, a2, mtiles, stream); break;
    default: launch_pair_w<1, FMT2, false, SPLIT>(a1, a2, mtiles, stream); break;
  }
}

bool pair_norm_fusable(int K, int64_t rows) {
  const int W = bf16_chunks(K);
  const int64_t mtiles = (rows + kSmallMTile - 1) / kSmallMTile;
  const bool mt2 = mtiles >= kSmallMt2MinTiles;
  const int nks = K / 32, steps = (nks + W - 1) / W;
  if (K % 32 || W < 4) return false;
  // one load batch per chunk: the norm's sums overlap the first weight loads (c2, 32 tokens:
  // 16.2 us against the plain launch's 11.0); longer chunks only for one or two tokens, where
  // the separate norm launch costs a kernel boundary more than the fused pass does
  return steps <= (mt2 ? 4 : 8) || (rows <= 2 && steps <= 16);
}

int launch_qmm_pair_route(const QmmArgs& a1, const QmmArgs& a2, hipStream_t stream, int fmt2,
                          const RouteTail& tail) {
  if (a1.offsets || a2.offsets || a1.dense_rows != a2.dense_rows || a1.K != a2.K || a1.K % 32 ||
      a1.n_rows % 16 || a2.n_rows % 32 || a1.dense_rows <= 0)
    return fail("qmm pair: two dense products over the same rows and K required");
  if (fmt2 != FMT_BF16 && fmt2 != FMT_INT8) return fail("qmm pair: the second product is bf16 or int8");
  if (fmt2 == FMT_INT8 && (a1.K % 64 || !a2.sb)) return fail("qmm pair: int8 weights need K % 64 == 0 and sb");
  if ((a1.norm_w != nullptr) != (a2.norm_w != nullptr) || a2.norm_out)
    return fail("qmm pair: the fused norm applies to both products; the first writes the rows");
  if (a1.norm_w && !pair_norm_fusable(a1.K, a1.dense_rows))
    return fail("qmm pair: the fused norm needs one job per workgroup and one load batch per chunk");
  const int mc = tail.N * tail.P.k;
  if (tail.N != a1.dense_rows || tail.N > kRouteTailMaxTokens || tail.P.E <= 0 ||
      tail.P.E > kRouteTailMaxExperts || tail.P.k <= 0 || tail.P.k > 64 || tail.P.k > tail.P.E ||
      !tail.ctr || !tail.timeouts || tail.logits != a1.out ||
      tail.ld != a1.ld_out || !tail.counts || !tail.tile_map || tail.words != (tail.N + 31) / 32 ||
      tail.vpl != topk_vpl(tail.P.E) ||
      tail.max_tiles < mtile_upper_bound(mc, tail.P.E, kSmallMTile))
    return fail("qmm pair (routing tail): bad routing arguments");
  const int64_t mtiles = (a1.dense_rows + kSmallMTile - 1) / kSmallMTile;
#define QMOE_PAIR_T(W)                                                                     \
  if (fmt2 == FMT_INT8) launch_pair_w<W, FMT_INT8, true>(a1, a2, mtiles, stream, tail);     \
  else launch_pair_w<W, FMT_BF16, true>(a1, a2, mtiles, stream, tail);
  switch (bf16_chunks(a1.K)) {
    case 16: QMOE_PAIR_T(16) break;
    case 8: QMOE_PAIR_T(8) break;
    case 4: QMOE_PAIR_T(4) break;
    case 2: QMOE_PAIR_T(2) break;
    default: QMOE_PAIR_T(1) break;
  }
#undef QMOE_PAIR_T
  return check_launch("qmm pair (routing tail)");
}

__device__ uint32_t g_route_timeouts;

uint32_t* route_tail_timeouts_ptr() {
  uint32_t* p = nullptr;
  return hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(g_route_timeouts)) == hipSuccess ? p : nullptr;
}

uint32_t route_tail_timeouts() {
  uint32_t v = 0;
  if (hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_route_timeouts), sizeof(v), 0, hipMemcpyDeviceToHost) != hipSuccess)
    return 0xFFFFFFFFu;
  return v;
}

int launch_qmm_pair_bf16(const QmmArgs& a1, const QmmArgs& a2, hipStream_t stream, int fmt2, bool split) {
  if (a1.offsets || a2.offsets || a1.dense_rows != a2.dense_rows || a1.K != a2.K || a1.K % 32 ||
      a1.n_rows % 16 || a2.n_rows % 32 || a1.dense_rows <= 0)
    return fail("qmm pair: two dense products over the same rows and K required");
  if (fmt2 != FMT_BF16 && fmt2 != FMT_INT8) return fail("qmm pair: the second product is bf16 or int8");
  if (fmt2 == FMT_INT8 && (a1.K % 64 || !a2.sb)) return fail("qmm pair: int8 weights need K % 64 == 0 and sb");
  if ((a1.norm_w != nullptr) != (a2.norm_w != nullptr) || a2.norm_out)
    return fail("qmm pair: the fused norm applies to both products; the first writes the rows");
  if (a1.norm_w && !pair_norm_fusable(a1.K, a1.dense_rows))
    return fail("qmm pair: the fused norm needs one job per workgroup and one load batch per chunk");
  const int64_t mtiles = (a1.dense_rows + kSmallMTile - 1) / kSmallMTile;
  if (mtiles > 65535) return fail("qmm pair: too many m-tiles for one launch");
  if (split && a2.ld_out < a2.n_rows) return fail("qmm pair: split gate_up rows hold both halves");
  if (fmt2 == FMT_INT8) {
    if (split) launch_pair_f<FMT_INT8, true>(a1, a2, mtiles, stream);
    else launch_pair_f<FMT_INT8, false>(a1, a2, mtiles, stream);
  } else {
    if (split) launch_pair_f<FMT_BF16, true>(a1, a2, mtiles, stream);
    else launch_pair_f<FMT_BF16, false>(a1, a2, mtiles, stream);
  }
  return check_launch("qmm pair");
}

template <int W, int CPW, int JPW, int W2, int MT2, int CPW2 = 1>
static int launch_gsd(const QmmArgs& a1, int64_t mtiles1, const QmmArgs& a2, int64_t mtiles2,
                      hipStream_t stream) {
  static_assert(W <= 4 && W2 <= 4, "one 4-wavefront workgroup shape for both products");
  const int n_jobs1 = a1.n_rows / 32 / JPW, gx1 = (n_jobs1 + 4 / W - 1) / (4 / W);
  const int n_jobs2 = a2.n_rows / 16, gx2 = (n_jobs2 + 4 / W2 - 1) / (4 / W2);
  const int64_t n1 = static_cast<int64_t>(gx1) * mtiles1;
  const int64_t n2 = static_cast<int64_t>(gx2) * ((MT2 == 2) ? (mtiles2 + 1) / 2 : mtiles2);
  if (n1 + n2 > 0x7fffffff) return fail("qmm(gate_up + shared down): grid too large");
  qmm_gate_up_shdown_kernel<W, CPW, JPW, W2, MT2, CPW2>
      <<<dim3(static_cast<unsigned>(n1 + n2)), 256, 0, stream>>>(a1, n_jobs1, gx1, n1, a2, n_jobs2, gx2);
  return check_launch("qmm(gate_up + shared down)");
}

int launch_gate_up_shared_down(const QmmArgs& a1, int64_t mtiles1, const QmmArgs& a2,
                               hipStream_t stream) {
  if (a1.K % 128 || a1.n_rows % 32 || !a1.tile_map || mtiles1 <= 0 || mtiles1 > 65535 ||
      a2.K % 64 || a2.n_rows % 16 || !a2.sb || a2.offsets || a2.tile_map || a2.dense_rows <= 0)
    return fail("qmm(gate_up + shared down): routed int4 gate_up and a dense int8 product required");
  const int nsb = a1.K / 128;
  const int ch = (nsb >= 32) ? 4 : (nsb >= 8) ? 2 : 1;   // launch_qmm's int4 chunk rule
  const SmallShape sh = pick_small_shape(FMT_INT4, EPI_SWIGLU, ch, mtiles1, a1.n_rows / 32);
  const int w2 = bf16_chunks(a2.K);
  const int64_t mtiles2 = (a2.dense_rows + kSmallMTile - 1) / kSmallMTile;
  const bool mt2 = mtiles2 >= kSmallMt2MinTiles;   // as launch_small_k for dense products
#define QMOE_GSD(W, CPW, JPW, W2)                                                    \
  if (sh.w == W && sh.cpw == CPW && sh.jpw == JPW && w2 == W2)                        \
    return mt2 ? launch_gsd<W, CPW, JPW, W2, 2>(a1, mtiles1, a2, mtiles2, stream)     \
               : launch_gsd<W, CPW, JPW, W2, 1>(a1, mtiles1, a2, mtiles2, stream);
  // c2-like shapes (H 4096, shared intermediate 1024). With two m-tiles per wavefront the
  // shared down does not fit beside this gate_up shape's registers (c2 N=64 461 vs 445 us), so
  // it runs one m-tile per wavefront there (the same sums: m-tiles are independent)
  if (sh.w == 2 && sh.cpw == 2 && sh.jpw == 2 && w2 == 4)
    return launch_gsd<2, 2, 2, 4, 1>(a1, mtiles1, a2, mtiles2, stream);
  QMOE_GSD(4, 1, 2, 4)
  QMOE_GSD(4, 1, 1, 4)
  QMOE_GSD(2, 1, 1, 2)   // c1-like shapes (H 2048, shared intermediate 512)
  QMOE_GSD(2, 1, 2, 2)
#undef QMOE_GSD
  // c3-like shapes (H 7168, shared intermediate 2048: eight chunks, four wavefronts of two, one
  // m-tile per wavefront)
  if (w2 == 8) {
    if (sh.w == 2 && sh.cpw == 2 && sh.jpw == 2) return launch_gsd<2, 2, 2, 4, 1, 2>(a1, mtiles1, a2, mtiles2, stream);
    if (sh.w == 4 && sh.cpw == 1 && sh.jpw == 2) return launch_gsd<4, 1, 2, 4, 1, 2>(a1, mtiles1, a2, mtiles2, stream);
    if (sh.w == 4 && sh.cpw == 1 && sh.jpw == 1) return launch_gsd<4, 1, 1, 4, 1, 2>(a1, mtiles1, a2, mtiles2, stream);
  }
  return 1;   // no compiled combination: the caller launches the two products apart
}

int launch_qmm(const QmmArgs& a, int fmt, int epi, int regime, int64_t mtile_bound,
               hipStream_t stream) {
  if (a.K <= 0 || a.n_rows <= 0) return fail("qmm: empty problem");
  if (mtile_bound <= 0) return 0;
  if (regime == kRegimeDense) return launch_dense(a, fmt, epi, stream);
  if (mtile_bound > 65535) return fail("qmm: too many m-tiles for one launch");
  if (a.expert_map && !fmt_quant(fmt))
    return fail("qmm: an expert map needs int3/int4/int6 weights");
  const bool two_acts = (regime == QMOE_REGIME_SMALL) ? a.act_hi != nullptr : a.act16_hi != nullptr;
  if (two_acts) {
    if (!fmt_quant(fmt) || epi == EPI_SWIGLU || a.slot_of)
      return fail("qmm: a second activation needs quantized weights, a non-SwiGLU epilogue and "
                  "rows by sorted position");
    if (a.split_tile <= 0 || a.split_tile % 4 || a.split_tile >= a.n_rows / 16)
      return fail("qmm: split_tile must be a positive multiple of 4 inside the weight tiles");
    if (regime != QMOE_REGIME_SMALL &&
        (!fmt_quant(fmt) || !a.row_sinv_hi || a.split_tile % 16))
      return fail("qmm(large): a second activation needs int3/int4/int6 weights, its row scales "
                  "and split_tile % 16 == 0");
  }
  if (regime == QMOE_REGIME_SMALL) {
    if (fmt_quant(fmt) && a.K % 128) return fail("qmm: int3/int4/int6 need K % 128 == 0");
    if (fmt == FMT_BF16 && a.K % 32) return fail("qmm: bf16 needs K % 32 == 0");
    if (fmt == FMT_INT8 && (a.K % 64 || !a.sb)) return fail("qmm: int8 needs K % 64 == 0 and sb");
    if (a.n_rows % (epi == EPI_SWIGLU ? 32 : 16)) return fail("qmm: weight rows not a tile multiple");
    // The chunk count depends on the shape only (never on the token count), so a row's
    // summation order, and therefore its result, is the same at every batch size (batch
    // invariance). int3/int4/int6 chunks hold >= 4 superblocks (int3, whose superblocks are
    // 3/4 the bytes of int4's: >= 16 at K = 4096, where two chunks measured faster than four);
    // bf16 (router, shared expert) chunks ~8 32-deep steps, one wavefront each, which spreads
    // the few dense row tiles over enough wavefronts.
    int ch;
    if (fmt_quant(fmt)) {
      const int nsb = a.K / 128;
      ch = (nsb >= (fmt == FMT_INT3 ? 64 : 32)) ? 4 : (nsb >= 8) ? 2 : 1;
    } else {
      ch = bf16_chunks(a.K);
    }
    const int jobs = (epi == EPI_SWIGLU) ? a.n_rows / 32 : a.n_rows / 16;
    const SmallShape sh = pick_small_shape(fmt, epi, ch, mtile_bound, jobs);
#define QMOE_SMALL(F, P) launch_small<F, P>(a, sh, mtile_bound, stream)
    if (fmt == FMT_INT4) {
      if (epi == EPI_SWIGLU) QMOE_SMALL(FMT_INT4, EPI_SWIGLU);
      else if (epi == EPI_BF16) QMOE_SMALL(FMT_INT4, EPI_BF16);
      else QMOE_SMALL(FMT_INT4, EPI_F32);
    } else if (fmt == FMT_INT6) {
      if (epi == EPI_SWIGLU) QMOE_SMALL(FMT_INT6, EPI_SWIGLU);
      else if (epi == EPI_BF16) QMOE_SMALL(FMT_INT6, EPI_BF16);
      else QMOE_SMALL(FMT_INT6, EPI_F32);
    } else if (fmt == FMT_INT3) {
      if (epi == EPI_SWIGLU) QMOE_SMALL(FMT_INT3, EPI_SWIGLU);
      else if (epi == EPI_BF16) QMOE_SMALL(FMT_INT3, EPI_BF16);
      else QMOE_SMALL(FMT_INT3, EPI_F32);
    } else if (fmt == FMT_INT8) {
      if (epi == EPI_SWIGLU) QMOE_SMALL(FMT_INT8, EPI_SWIGLU);
      else if (epi == EPI_BF16) QMOE_SMALL(FMT_INT8, EPI_BF16);
      else QMOE_SMALL(FMT_INT8, EPI_F32);
    } else {
      if (epi == EPI_SWIGLU) QMOE_SMALL(FMT_BF16, EPI_SWIGLU);
      else if (epi == EPI_BF16) QMOE_SMALL(FMT_BF16, EPI_BF16);
      else QMOE_SMALL(FMT_BF16, EPI_F32);
    }
#undef QMOE_SMALL
  } else {
    if (fmt == FMT_INT8)
      return fail("qmm(large): int8 weights run in the small regime only (expand them to bf16 "
                  "for the large kernels)");
    if (a.K % 128) return fail("qmm(large): K % 128 == 0 required");
    if (a.dense_mtile && (a.offsets || a.tile_map || a.dense_mtile % 16 || a.dense_mtile < 16 ||
                          a.dense_mtile > kLargeMTile || fmt != FMT_BF16))
      return fail("qmm(large): dense_mtile is a multiple of 16 up to 128, for one dense bf16 segment");
    if (a.n_rows % 256) return fail("qmm(large): weight rows % 256 == 0 required");
    const bool qf = fmt_quant(fmt);
    if (qf && (!a.act16 || !a.row_sinv))
      return fail("qmm(large): int3/int4/int6 weights need the fp16 activation copy");
    if (qf && !a.row_exp)
      return fail("qmm(large): int3/int4/int6 weights need their row exponents (qmoe_row_exponents)");
    const int rc = launch_large(a, fmt, epi, mtile_bound, stream);
    if (rc) return rc;
  }
  return check_launch("qmm");
}

}  // namespace qmoe
