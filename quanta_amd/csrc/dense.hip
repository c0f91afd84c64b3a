// Dense products of batches above the decode sizes: the shared expert's gate_up and down projections over
// more than 256 tokens (tiled bf16 or int8 weights). The router's logits have a kernel of their own
// (prefill.hip): their sums must not depend on how K is cut.
//
// Reference: the shared expert's matmuls src/quanta/qwen35/moe.py:145-151.
//
// Each wavefront holds a 64-token x 64-weight-row tile (SwiGLU: 32 gate + 32 up rows; 4 x 4 16x16
// blocks) and reads its fragments straight from L2 in 64-deep stages, two in registers. KS of the
// workgroup's 8 wavefronts cut K between them (at least four stages each where K has them), their
// partial sums meeting in LDS, added in wavefront order; the other 8 / KS take neighbouring weight
// rows. What bounds these products is latency: they are too small to fill the chip with the large
// kernel's 128 x 256 tiles, whose workgroups each walk all of K behind a barrier per 128 (c1 at 391
// tokens: 14 to 32 workgroups), while the decode kernel's 32 x 16 tiles read four times the bytes
// from L2. Int8 weights are dequantized in registers, without a pass that expands them.
#include "qmoe_internal.h"
#include "small_body.h"
#include "../../include/quanta_moe.h"

namespace qmoe {

constexpr int kDmWaves = 8;
constexpr int kDmTile = 64;
constexpr size_t kDmLdsBytes = static_cast<size_t>(kDmWaves) * 16 * 64 * 16;   // 128 KiB

template <int FMT>
struct DmStage {
  u32x4 x[2][4];            // activation fragments [32-deep step][m-block]
  DenseFrag<FMT> w[2][4];   // weight fragments [step][tile]
};

template <int FMT, int EPI, int KS>
__global__ void __launch_bounds__(64 * kDmWaves) __attribute__((amdgpu_waves_per_eu(2)))
qmm_dense_kernel(QmmArgs a, int n_tok, int n_rb, int n_wg) {
  extern __shared__ f32x4_t dm_part[];   // [wave][m-block * 4 + tile][lane]
  constexpr int NR = kDmWaves / KS;      // row blocks per workgroup
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // workgroup i runs on XCD i % 8: each XCD takes a run of tiles, token blocks fastest, or weight
  // rows fastest when the activations are the larger operand, so that its L2 reads its share of the
  // larger operand once
  const int per = (n_wg + 7) / 8;
  const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per || id >= n_wg) return;
  const int n_rw = (n_rb + NR - 1) / NR;
  const bool by_tok = kDmTile * n_tok > a.n_rows;
  const int tb = by_tok ? id / n_rw : id % n_tok;
  const int rw = (by_tok ? id % n_rw : id / n_tok) * NR + wave / KS;
  const bool rb_ok = rw < n_rb;   // (past the end: the last block, not stored)
  const int rb = min(rw, n_rb - 1);
  const int kpart = wave % KS;
  const int mrow = lane & 15, lg = lane >> 4;
  const int rows = static_cast<int>(a.dense_rows);
  // 32-bit byte offsets from wave-uniform bases (launch_dense bounds the activations to 4 GiB)
  const char* xb = reinterpret_cast<const char*>(a.act);
  uint32_t xo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = kDmTile * tb + 16 * i + mrow;   // (past the end: row 0, never stored)
    xo[i] = static_cast<uint32_t>(t < rows ? t : 0) * (2u * a.K) + 16u * lg;
  }
  const char* wb[4];
  const char* wsb[4];
  constexpr int FB = (FMT == FMT_INT8) ? 8 : 16;   // bytes of a lane's fragment
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int tile = (EPI == EPI_SWIGLU) ? (t < 2 ? 2 * rb + t : a.n_rows / 32 + 2 * rb + t - 2) : 4 * rb + t;
    wb[t] = static_cast<const char*>(a.codes) + static_cast<int64_t>(tile) * (a.K / 32) * 64 * FB;
    wsb[t] = reinterpret_cast<const char*>(a.sb) + static_cast<int64_t>(tile) * (a.K / 64) * 64;
  }
  const uint32_t wo = static_cast<uint32_t>(lane) * FB, so = 4u * mrow;
  const int ns = a.K / 64;
  const int s0 = kpart * ns / KS, s1 = (kpart + 1) * ns / KS;
  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto load = [&](DmStage<FMT>& g, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) g.x[h][i] = *reinterpret_cast<const u32x4*>(xb + (128 * s + 64 * h) + xo[i]);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const char* p = wb[t] + static_cast<int64_t>(s) * 2 * 64 * FB;
      if constexpr (FMT == FMT_INT8) {
        const uint32_t sb = *reinterpret_cast<const uint32_t*>(wsb[t] + static_cast<int64_t>(s) * 64 + so);
        g.w[0][t] = DenseFrag<FMT>{*reinterpret_cast<const u32x2*>(p + wo), sb};
        g.w[1][t] = DenseFrag<FMT>{*reinterpret_cast<const u32x2*>(p + 64 * FB + wo), sb};
      } else {
        g.w[0][t] = DenseFrag<FMT>{*reinterpret_cast<const u32x4*>(p + wo)};
        g.w[1][t] = DenseFrag<FMT>{*reinterpret_cast<const u32x4*>(p + 64 * FB + wo)};
      }
    }
  };
  auto compute = [&](const DmStage<FMT>& g) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16x8_t B = as_bf16x8(dense_bf16<FMT>(g.w[h][t]));
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i][t] = mfma16(as_bf16x8(g.x[h][i]), B, acc[i][t]);
        // (int8: one fragment's dequant at a time; hoisted together they spill)
        if (FMT == FMT_INT8) __builtin_amdgcn_sched_barrier(0);
      }
  };
  if (s0 < s1) {
    DmStage<FMT> st[2];
    load(st[0], s0);
    int s = s0;
    for (; s + 2 < s1; s += 2) {
      load(st[1], s + 1);
      __builtin_amdgcn_sched_barrier(0);
      compute(st[0]);
      load(st[0], s + 2);
      __builtin_amdgcn_sched_barrier(0);
      compute(st[1]);
    }
    if (s + 1 < s1) {
      load(st[1], s + 1);
      __builtin_amdgcn_sched_barrier(0);
      compute(st[0]);
      compute(st[1]);
    } else {
      compute(st[0]);
    }
  }
  // the tile's outputs: m-block mb, columns of the tile pair (t, t + 2)
  auto store = [&](int mb, int t, const f32x4_t& v0, const f32x4_t& v1) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = kDmTile * tb + 16 * mb + 4 * lg + j;
      if (row >= rows) continue;
      if (EPI == EPI_SWIGLU) {
        store_out<EPI>(a, row, 32 * rb + 16 * t + mrow, v0[j], v1[j]);
      } else {
        store_out<EPI>(a, row, 64 * rb + 16 * t + mrow, v0[j], 0.f);
        store_out<EPI>(a, row, 64 * rb + 16 * t + 32 + mrow, v1[j], 0.f);
      }
    }
  };
  if constexpr (KS == 1) {
    if (rb_ok) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) store(i, t, acc[i][t], acc[i][t + 2]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) dm_part[(wave * 16 + 4 * i + t) * 64 + lane] = acc[i][t];
    __syncthreads();
    // the row block's KS wavefronts share its 4 x 2 tile pairs (SwiGLU: a gate tile and its up tile)
    const int w0 = wave - kpart;
    if (rb_ok) {
#pragma unroll
      for (int u = 0; u < 8 / KS; ++u) {
        const int mb = (kpart * (8 / KS) + u) >> 1, t = (kpart * (8 / KS) + u) & 1;
        f32x4_t v[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          v[q] = dm_part[(w0 * 16 + 4 * mb + t + 2 * q) * 64 + lane];
#pragma unroll
          for (int w = 1; w < KS; ++w) {
            const f32x4_t o = dm_part[((w0 + w) * 16 + 4 * mb + t + 2 * q) * 64 + lane];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[q][j] += o[j];
          }
        }
        store(mb, t, v[0], v[1]);
      }
    }
  }
}

template <int FMT, int EPI, int KS>
static int launch_dense_k(const QmmArgs& a, hipStream_t stream) {
  const size_t lds = KS > 1 ? kDmLdsBytes : 0;
  const hipError_t err =
      hipFuncSetAttribute(reinterpret_cast<const void*>(qmm_dense_kernel<FMT, EPI, KS>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
  if (err != hipSuccess) return fail(std::string("qmm(dense): LDS attribute: ") + hipGetErrorString(err));
  const int64_t n_tok = (a.dense_rows + kDmTile - 1) / kDmTile, n_rb = a.n_rows / kDmTile;
  constexpr int NR = kDmWaves / KS;
  const int64_t n_wg = n_tok * ((n_rb + NR - 1) / NR);
  if (n_wg > (int64_t(1) << 30)) return fail("qmm(dense): product too large for one launch");
  qmm_dense_kernel<FMT, EPI, KS><<<dim3(static_cast<unsigned>((n_wg + 7) / 8 * 8)), 64 * kDmWaves, lds, stream>>>(
      a, static_cast<int>(n_tok), static_cast<int>(n_rb), static_cast<int>(n_wg));
  return 0;
}
template <int FMT, int EPI>
static int launch_dense_e(const QmmArgs& a, hipStream_t stream) {
  // at least four 64-deep stages per wavefront
  if (a.K >= 2048) return launch_dense_k<FMT, EPI, 8>(a, stream);
  if (a.K >= 1024) return launch_dense_k<FMT, EPI, 4>(a, stream);
  if (a.K >= 512) return launch_dense_k<FMT, EPI, 2>(a, stream);
  return launch_dense_k<FMT, EPI, 1>(a, stream);
}

int launch_dense(const QmmArgs& a, int fmt, int epi, hipStream_t stream) {
  if (!fmt_dense(fmt) || epi == EPI_F32 || a.offsets || a.tile_map || a.dense_rows <= 0 || a.act_stride || a.norm_w)
    return fail("qmm(dense): one dense bf16 or int8 segment, bf16 out");
  if (a.K % 64 || a.n_rows % kDmTile || (fmt == FMT_INT8 && !a.sb))
    return fail("qmm(dense): K % 64 == 0 and weight rows % 64 == 0 required (int8: scale/bias)");
  if (a.dense_rows * a.K > kDenseMaxActs) return fail("qmm(dense): activations beyond 4 GiB");
#define QMOE_DENSE(F) \
  (epi == EPI_SWIGLU ? launch_dense_e<F, EPI_SWIGLU>(a, stream) : launch_dense_e<F, EPI_BF16>(a, stream))
  const int rc = (fmt == FMT_INT8) ? QMOE_DENSE(FMT_INT8) : QMOE_DENSE(FMT_BF16);
#undef QMOE_DENSE
  return rc ? rc : check_launch("qmm(dense)");
}

}  // namespace qmoe
