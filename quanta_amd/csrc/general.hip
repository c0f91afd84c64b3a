// The block for inputs outside the fast path's formats: float32 activations, float32 scale/bias
// triplets, group sizes 32/64/128 at any hidden size, code widths 2-8, dense float32 or bf16
// expert stacks. It follows the reference's dtype flow exactly:
//   logits = f32(x) @ f32(gate)^T                                  (src/quanta/qwen35/moe.py:47)
//   gu = qmm(x_T, experts_gate_up) in T, the experts' dtype: the scale/bias dtype of a packed
//        triplet ("the qmm output follows the baked scale dtype", :98-104) or the dtype of a
//        dense stack (x cast to it, :77)
//   h = silu(g) * u in T; d = qmm(h, experts_down) in T               (:59-63, :121-123)
//   routed = sum_s f32(d) * w                                          (:191)
//   shared = f32(down(silu(xd Wg^T) * (xd Wu^T))) * sigmoid(f32(x) . f32(g)), xd = x cast to the
//            shared weights' dtype                                     (:145-151)
//   y = cast_x(routed + shared)                                        (:201-202)
// as the reference's own float32 parity gates run it (parity/qwen35_forward_test.py:213-271:
// hidden 32, group size 32, float32 throughout). Four launches (six with a shared expert, seven with a gated
// one, whose logit is a product of its own): router, top-k,
// gate_up with its gated activation, down with the combine; one wavefront per output (fixed-order
// wavefront sums, fp32 accumulation), the affine weight s*q + b evaluated in fp32 per element from
// the LSB-first packed code stream. These shapes are small (the parity configs); the fast path
// serves the bf16 g64 production formats.
#include <math.h>

#include "qmoe_internal.h"
#include "route_common.h"
#include "../../include/quanta_moe.h"

namespace qmoe {

__device__ __forceinline__ float gen_ld(const void* p, int64_t i, int dt) {
  return dt == QMOE_DT_F32 ? static_cast<const float*>(p)[i]
                           : bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
}
__device__ __forceinline__ float gen_round(float v, int dt) {
  return dt == QMOE_DT_F32 ? v : bf16_to_f32(f32_to_bf16(v));
}
__device__ __forceinline__ void gen_st(void* p, int64_t i, float v, int dt) {
  if (dt == QMOE_DT_F32) static_cast<float*>(p)[i] = v;
  else static_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
}

// Weights of the products: a dense [rows][K] stack (BITS 0; `dense_dt`) or affine codes with a scale
// and a bias per group of 2^gshift along K.
struct GenW {
  const uint32_t* packed;
  const void* scale;
  const void* bias;
  const void* dense;
  int sb_dt, dense_dt, gshift, K;
};

// Every product is one wavefront per output (or per few outputs over the same activations). At these sizes
// the launch is a chain of dependent loads, so where K is a multiple of 8 (PIECES; packed K always is) lane l
// takes the 8-element pieces l, l + 64, ... of K: a row of 512 is one round of loads, where element-strided
// lanes took eight. Other K, dense only, keep the strided lanes: there a piece is eight scattered loads (100 x 60,
// 200 bf16 tokens: 53 us per call, 108 in pieces).
//
// A piece is loaded as 16-byte words at its elements' alignment, since the caller's tensors may start anywhere:
// global loads take any address (2048 x 1024 float32, 64 tokens, tensors 4 bytes off: 852 us, 4478 element by
// element).
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));

// Elements 8c .. 8c + 7 of the row at element offset `base`, rounded to `round` when that differs from
// their dtype (the reference's cast to the weights' dtype).
__device__ __forceinline__ void gen_x8(const void* act, int64_t base, int c, int dt, int round, float (&x)[8]) {
  if (dt == QMOE_DT_F32) {
    const f32x4_u* p = reinterpret_cast<const f32x4_u*>(static_cast<const float*>(act) + base + 8 * c);
    const f32x4_u lo = p[0], hi = p[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[j] = lo[j];
      x[4 + j] = hi[j];
    }
  } else {
    const u32x4_u v = *reinterpret_cast<const u32x4_u*>(static_cast<const uint16_t*>(act) + base + 8 * c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[2 * j] = bf16lo_to_f32(v[j]);
      x[2 * j + 1] = bf16hi_to_f32(v[j]);
    }
  }
  if (round != dt) {
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = gen_round(x[j], round);
  }
}

// acc + x . W[row][8c .. 8c + 7], the affine weight fma(s, q, b) formed in fp32 per element. Eight
// codes of any width start on a byte and span at most two words.
template <int BITS>
__device__ __forceinline__ float gen_dot8(const GenW& w, int64_t row, int c, const float (&x)[8], float acc) {
  if constexpr (BITS > 0) {
    const uint32_t* p = w.packed + row * (static_cast<int64_t>(w.K) * BITS / 32);
    const int bit = 8 * BITS * c, sh = bit & 31;
    uint64_t v = p[bit >> 5];
    if (sh + 8 * BITS > 32) v |= static_cast<uint64_t>(p[(bit >> 5) + 1]) << 32;
    v >>= sh;
    const int64_t g = row * (w.K >> w.gshift) + ((8 * c) >> w.gshift);
    const float s = gen_ld(w.scale, g, w.sb_dt), b = gen_ld(w.bias, g, w.sb_dt);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t q = static_cast<uint32_t>(v >> (j * BITS)) & ((1u << BITS) - 1u);
      acc = fmaf(x[j], fmaf(s, static_cast<float>(q), b), acc);
    }
  } else {
    float y[8];
    gen_x8(w.dense, row * w.K, c, w.dense_dt, w.dense_dt, y);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc = fmaf(x[j], y[j], acc);
  }
  return acc;
}

// This lane's part of x . W_i[rows[i]] (i < M): x the row at element offset `base`, rounded to `round`.
template <int BITS, bool PIECES, int M>
__device__ __forceinline__ void gen_dots(const void* act, int64_t base, int dt, int round, const GenW* const (&w)[M],
                                         const int64_t (&rows)[M], int lane, float (&acc)[M]) {
  static_assert(PIECES || BITS == 0, "packed rows are whole pieces");
  const int K = w[0]->K;
  if constexpr (PIECES) {
    for (int c = lane; 8 * c < K; c += 64) {
      float x[8];
      gen_x8(act, base, c, dt, round, x);
#pragma unroll
      for (int i = 0; i < M; ++i) acc[i] = gen_dot8<BITS>(*w[i], rows[i], c, x, acc[i]);
    }
  } else {
    for (int k = lane; k < K; k += 64) {
      float x = gen_ld(act, base + k, dt);
      if (round != dt) x = gen_round(x, round);
#pragma unroll
      for (int i = 0; i < M; ++i) acc[i] = fmaf(x, gen_ld(w[i]->dense, rows[i] * K + k, w[i]->dense_dt), acc[i]);
    }
  }
}

template <int M>
__device__ __forceinline__ void gen_wave_sum(float (&v)[M]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < M; ++i) v[i] += __shfl_xor(v[i], off);
}

// out[r][col0 + o] = a(r) . W[o], a = the activation row r (the router's and the shared expert's
// down products).
struct GenMv {
  const void* act;
  int act_dt, act_round;     // QMOE_DT_*; act_round: the dtype the activation is cast to first
  int64_t rows;
  int n_out;
  GenW w;
  void* out;
  int out_dt;
  int64_t ld_out;
  int col0;
};

template <bool PIECES>
__global__ void __launch_bounds__(256) gen_matvec_kernel(GenMv a) {
  const int lane = threadIdx.x & 63;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (gid >= a.rows * a.n_out) return;   // whole wavefronts exit together; no barriers below
  const int64_t r = gid / a.n_out;
  const int o = static_cast<int>(gid - r * a.n_out);
  float acc[1] = {0.f};
  gen_dots<0, PIECES, 1>(a.act, r * a.w.K, a.act_dt, a.act_round, {&a.w}, {o}, lane, acc);
  gen_wave_sum(acc);
  if (lane == 0) gen_st(a.out, r * a.ld_out + a.col0 + o, acc[0], a.out_dt);
}

// h[r][i] = glu(g, u) in dtype dt: g and u the products of activation row r / row_div with weight
// rows e(r) n2 + i and that + up (or row i of w_up), each rounded to dt as the reference's
// materialised gate_up is.
struct GenGu {
  const void* act;
  int act_dt, act_round;
  const int32_t* row_expert;  // [rows] expert of each output row (nullable: expert 0)
  int row_div;
  int64_t rows;
  int n, n2, up;
  GenW w, w_up;
  void* h;
  int dt, glu;
  float alpha, limit;
};

template <int BITS, bool PIECES>
__global__ void __launch_bounds__(256) gen_gate_up_kernel(GenGu a) {
  const int lane = threadIdx.x & 63;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (gid >= a.rows * a.n) return;
  const int64_t r = gid / a.n;
  const int i = static_cast<int>(gid - r * a.n);
  const int e = a.row_expert ? a.row_expert[r] : 0;   // (-1: no expert, zeros)
  const int64_t row = static_cast<int64_t>(e) * a.n2 + i;
  const int64_t base = r / a.row_div * a.w.K;
  float v[2] = {0.f, 0.f};
  if (e >= 0)
    gen_dots<BITS, PIECES, 2>(a.act, base, a.act_dt, a.act_round, {&a.w, &a.w_up}, {row, row + a.up}, lane, v);
  gen_wave_sum(v);
  if (lane == 0)
    gen_st(a.h, r * a.n + i, glu_f(gen_round(v[0], a.dt), gen_round(v[1], a.dt), a.glu, a.alpha, a.limit), a.dt);
}

// y[t][j] = cast_x(sum_s f32(d_s) * w[t][s] + f32(sh[t][j]) * sg[t]), d_s = h[t*k+s] . W_e[j] rounded
// to dtype dt (the reference's materialised down output), slots in order.
struct GenDn {
  const void* h;
  int dt;
  const int32_t* idx;
  const float* wt;
  int64_t N;
  int k, H;
  GenW w;
  const void* sh;
  int sh_dt;
  const float* sg;
  void* y;
  int y_dt;
};

template <int BITS, bool PIECES>
__global__ void __launch_bounds__(256) gen_down_combine_kernel(GenDn a) {
  const int lane = threadIdx.x & 63;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (gid >= a.N * a.H) return;
  const int64_t t = gid / a.H;
  const int j = static_cast<int>(gid - t * a.H);
  float out = 0.f;
  constexpr int SB = 4;   // slots whose loads and sums run together
  for (int s0 = 0; s0 < a.k; s0 += SB) {
    float v[SB];
#pragma unroll
    for (int i = 0; i < SB; ++i) {
      float d[1] = {0.f};
      if (s0 + i < a.k) {
        const int64_t m = t * a.k + s0 + i;
        const int e = a.idx[m];
        if (e >= 0)
          gen_dots<BITS, PIECES, 1>(a.h, m * a.w.K, a.dt, a.dt, {&a.w}, {static_cast<int64_t>(e) * a.H + j}, lane, d);
      }
      v[i] = d[0];
    }
    gen_wave_sum(v);
#pragma unroll
    for (int i = 0; i < SB; ++i)
      if (s0 + i < a.k) out += gen_round(v[i], a.dt) * a.wt[t * a.k + s0 + i];
  }
  if (lane == 0) {
    if (a.sh) out += gen_ld(a.sh, gid, a.sh_dt) * (a.sg ? a.sg[t] : 1.0f);
    gen_st(a.y, gid, out, a.y_dt);
  }
}

static int gen_grid(int64_t waves, unsigned* grid) {
  if ((waves + 3) / 4 > 0x7fffffff) return fail("general: product too large");
  *grid = static_cast<unsigned>((waves + 3) / 4);
  return 0;
}

static int gen_matvec(const GenMv& a, hipStream_t stream) {
  unsigned grid;
  if (int rc = gen_grid(a.rows * a.n_out, &grid)) return rc;
  if (!grid) return 0;
  if (a.w.K % 8 == 0) gen_matvec_kernel<true><<<grid, 256, 0, stream>>>(a);
  else gen_matvec_kernel<false><<<grid, 256, 0, stream>>>(a);
  return check_launch("general matvec");
}

// launch KERNEL<bits, pieces> for a code width (0: dense)
#define QMOE_GEN(KERNEL, bits, grid, stream, a)                                                               \
  do {                                                                                                        \
    switch (bits) {                                                                                           \
      case 0:                                                                                                 \
        if (a.w.K % 8 == 0) KERNEL<0, true><<<grid, 256, 0, stream>>>(a);                                     \
        else KERNEL<0, false><<<grid, 256, 0, stream>>>(a);                                                   \
        break;                                                                                                \
      case 2: KERNEL<2, true><<<grid, 256, 0, stream>>>(a); break;                                            \
      case 3: KERNEL<3, true><<<grid, 256, 0, stream>>>(a); break;                                            \
      case 4: KERNEL<4, true><<<grid, 256, 0, stream>>>(a); break;                                            \
      case 5: KERNEL<5, true><<<grid, 256, 0, stream>>>(a); break;                                            \
      case 6: KERNEL<6, true><<<grid, 256, 0, stream>>>(a); break;                                            \
      case 8: KERNEL<8, true><<<grid, 256, 0, stream>>>(a); break;                                            \
      default: return fail("general: bits must be 2, 3, 4, 5, 6 or 8");                                       \
    }                                                                                                         \
  } while (0)

static int gen_gate_up(const GenGu& a, int bits, hipStream_t stream) {
  unsigned grid;
  if (int rc = gen_grid(a.rows * a.n, &grid)) return rc;
  if (!grid) return 0;
  QMOE_GEN(gen_gate_up_kernel, bits, grid, stream, a);
  return check_launch("general gate_up");
}

static int gen_down_combine(const GenDn& a, int bits, hipStream_t stream) {
  unsigned grid;
  if (int rc = gen_grid(a.N * a.H, &grid)) return rc;
  QMOE_GEN(gen_down_combine_kernel, bits, grid, stream, a);
  return check_launch("general down + combine");
}

// The run-every-expert form (the reference's sparse=False oracle, moe.py:127-142): every token
// runs every expert e (idx_all[t][e] = e) and the combine weights are the routing weights
// scattered onto the chosen experts, zero elsewhere.
__global__ void __launch_bounds__(256) gen_scatter_kernel(const int32_t* idx, const float* w, int N,
                                                          int k, int E, int32_t* idx_all,
                                                          float* w_all) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= N) return;
  for (int e = 0; e < E; ++e) {
    idx_all[static_cast<int64_t>(t) * E + e] = e;
    w_all[static_cast<int64_t>(t) * E + e] = 0.f;
  }
  for (int s = 0; s < k; ++s) {
    const int e = idx[static_cast<int64_t>(t) * k + s];
    if (e >= 0 && e < E) w_all[static_cast<int64_t>(t) * E + e] = w[static_cast<int64_t>(t) * k + s];
  }
}

struct GenLayout {
  size_t logits, idx, w, sg, idx_all, w_all, h, sh, so, total;
};
static int dt_bytes(int dt) { return dt == QMOE_DT_F32 ? 4 : 2; }
// The routed experts' compute dtype: a dense stack's own dtype (x is cast to it, moe.py:77); for
// packed codes the promotion of x's and the scales' dtypes (mx.gather_qmm's result type).
static int routed_dtype(const qmoe_general_config_t& c) {
  if (!c.experts_packed) return c.expert_dtype;
  return (c.x_dtype == QMOE_DT_F32 || c.expert_dtype == QMOE_DT_F32) ? QMOE_DT_F32 : QMOE_DT_BF16;
}
// Slots per token of the routed stage: top_k, or every expert for the run-every-expert form.
static int routed_slots(const qmoe_general_config_t& c) { return c.dense_all ? c.n_experts : c.top_k; }
static GenLayout gen_layout(const qmoe_general_config_t& c, int64_t N) {
  GenLayout L{};
  size_t o = 0;
  auto take = [&](size_t b) {
    const size_t at = o;
    o = align256(o + b);
    return at;
  };
  const int64_t mc = N * routed_slots(c);
  const int te = dt_bytes(routed_dtype(c)), ts = dt_bytes(c.shared_dtype);
  L.logits = take(static_cast<size_t>(N) * (c.n_experts + 1) * 4);
  L.idx = take(static_cast<size_t>(N) * c.top_k * 4);
  L.w = take(static_cast<size_t>(N) * c.top_k * 4);
  L.sg = take(static_cast<size_t>(N) * 4);
  L.idx_all = take(c.dense_all ? static_cast<size_t>(mc) * 4 : 0);
  L.w_all = take(c.dense_all ? static_cast<size_t>(mc) * 4 : 0);
  L.h = take(static_cast<size_t>(mc) * c.inter * te);
  L.sh = take(static_cast<size_t>(N) * c.shared_inter * ts);
  L.so = take(static_cast<size_t>(N) * c.hidden * ts);
  L.total = o;
  return L;
}

int validate_routing(int N, int H, int E, int k, int scoring, int n_group, int topk_group);

static bool dt_ok(int dt) { return dt == QMOE_DT_BF16 || dt == QMOE_DT_F32; }

static int gen_validate(const qmoe_general_config_t& c) {
  int rc = validate_routing(1, c.hidden, c.n_experts, c.top_k, c.scoring, c.n_group, c.topk_group);
  if (rc) return rc;
  if (c.top_k > 64) return fail("general: top_k <= 64 required");
  if (!dt_ok(c.x_dtype) || !dt_ok(c.gate_dtype) || !dt_ok(c.expert_dtype) || !dt_ok(c.shared_dtype) ||
      !dt_ok(c.shared_gate_dtype))
    return fail("general: dtypes must be QMOE_DT_BF16 or QMOE_DT_F32");
  if (c.inter <= 0 || c.shared_inter < 0) return fail("general: inter > 0, shared_inter >= 0 required");
  if (c.norm_topk < QMOE_NORM_NONE || c.norm_topk > QMOE_NORM_MULTI) return fail("general: bad norm_topk");
  if (c.act < QMOE_ACT_SILU || c.act > QMOE_ACT_SWIGLU_OAI) return fail("general: unknown act");
  if (c.act != QMOE_ACT_SILU && !(c.act_limit > 0.f)) return fail("general: act_limit must be > 0");
  if (c.experts_packed) {
    if (c.bits < 2 || c.bits > 8 || c.bits == 7) return fail("general: bits must be 2, 3, 4, 5, 6 or 8");
    if (c.group_size != 32 && c.group_size != 64 && c.group_size != 128)
      return fail("general: group_size must be 32, 64 or 128");
    if (c.hidden % c.group_size || c.inter % c.group_size)
      return fail("general: hidden and inter must be multiples of group_size");
    if ((static_cast<int64_t>(c.hidden) * c.bits) % 32 || (static_cast<int64_t>(c.inter) * c.bits) % 32)
      return fail("general: packed rows must fill whole 32-bit words");
  } else if (c.experts_packed != 0) {
    return fail("general: experts_packed must be 0 or 1");
  }
  if (c.dense_all != 0 && c.dense_all != 1) return fail("general: dense_all must be 0 or 1");
  if (c.shared_gated != 0 && c.shared_gated != 1) return fail("general: shared_gated must be 0 or 1");
  return 0;
}

}  // namespace qmoe

using namespace qmoe;

extern "C" size_t qmoe_forward_general_workspace(const qmoe_general_config_t* cfg, int64_t N) {
  if (!cfg || N <= 0) return 0;
  return gen_layout(*cfg, N).total;
}

extern "C" int qmoe_forward_general(const qmoe_general_config_t* cfg, const qmoe_general_weights_t* wts,
                                    const void* x, int64_t N, void* y, void* ws, size_t ws_bytes,
                                    void* stream_) {
  if (!cfg || !wts || !x || !y || !ws) return fail("qmoe_forward_general: null pointer");
  const qmoe_general_config_t& c = *cfg;
  int rc = gen_validate(c);
  if (rc) return rc;
  if (N <= 0 || N > 65535) return fail("qmoe_forward_general: 0 < N <= 65535 tokens per call");
  const GenLayout L = gen_layout(c, N);
  if (ws_bytes < L.total) return fail("qmoe_forward_general: workspace too small");
  if (!wts->gate || !wts->gu || !wts->dn) return fail("qmoe_forward_general: missing weights");
  if (c.experts_packed && (!wts->gu_scale || !wts->gu_bias || !wts->dn_scale || !wts->dn_bias))
    return fail("qmoe_forward_general: packed experts need scale and bias");
  const bool shared = c.shared_inter > 0;
  if (shared && (!wts->sh_gate || !wts->sh_up || !wts->sh_down))
    return fail("qmoe_forward_general: missing shared expert");
  if (shared && c.shared_gated && !wts->sh_expert_gate)
    return fail("qmoe_forward_general: a gated shared expert needs sh_expert_gate");
  hipStream_t st = static_cast<hipStream_t>(stream_);
  char* base = static_cast<char*>(ws);
  float* logits = reinterpret_cast<float*>(base + L.logits);
  int32_t* idx = reinterpret_cast<int32_t*>(base + L.idx);
  float* wv = reinterpret_cast<float*>(base + L.w);
  float* sg = reinterpret_cast<float*>(base + L.sg);
  const int n = static_cast<int>(N), H = c.hidden, E = c.n_experts, I = c.inter, Is = c.shared_inter;
  if (c.dense_all && c.experts_packed)
    return fail("qmoe_forward_general: the run-every-expert form takes dense stacks only");
  const int has_sg = (shared && c.shared_gated) ? 1 : 0;
  const int ld = E + 1;

  // router logits in f32 (column E: the shared expert's gate logit)
  auto dense_w = [](const void* p, int dt, int K) {
    GenW w{};
    w.dense = p; w.dense_dt = dt; w.K = K;
    return w;
  };
  GenMv r{};
  r.act = x; r.act_dt = c.x_dtype; r.act_round = c.x_dtype;
  r.rows = N; r.n_out = E; r.w = dense_w(wts->gate, c.gate_dtype, H);
  r.out = logits; r.out_dt = QMOE_DT_F32; r.ld_out = ld;
  if ((rc = gen_matvec(r, st))) return rc;
  if (has_sg) {
    GenMv g = r;
    g.n_out = 1; g.w = dense_w(wts->sh_expert_gate, c.shared_gate_dtype, H); g.col0 = E;
    if ((rc = gen_matvec(g, st))) return rc;
  }
  rc = launch_topk(logits, ld, wts->router_bias, n, E, c.top_k, c.scoring, c.n_group, c.topk_group,
                   c.norm_topk, c.routed_scale, has_sg, idx, wv, sg, st);
  if (rc) return rc;

  // routed experts in their dtype T
  const int T = routed_dtype(c);
  const int ks = routed_slots(c);
  const int64_t mc = N * ks;
  const int32_t* ridx = idx;
  const float* rw = wv;
  if (c.dense_all) {
    int32_t* ia = reinterpret_cast<int32_t*>(base + L.idx_all);
    float* wa = reinterpret_cast<float*>(base + L.w_all);
    gen_scatter_kernel<<<dim3((n + 255) / 256), 256, 0, st>>>(idx, wv, n, c.top_k, E, ia, wa);
    if ((rc = check_launch("general scatter"))) return rc;
    ridx = ia;
    rw = wa;
  }
  void* h = base + L.h;
  const int bits = c.experts_packed ? c.bits : 0;
  auto expert_w = [&](const void* p, const void* scale, const void* bias, int K) {
    GenW w = dense_w(bits ? nullptr : p, c.expert_dtype, K);
    if (bits) {
      w.packed = static_cast<const uint32_t*>(p); w.scale = scale; w.bias = bias; w.sb_dt = c.expert_dtype;
      w.gshift = (c.group_size == 32) ? 5 : (c.group_size == 64) ? 6 : 7;
    }
    return w;
  };
  GenGu e{};
  e.act = x; e.act_dt = c.x_dtype; e.act_round = T; e.row_expert = ridx; e.row_div = ks; e.rows = mc;
  e.n = I; e.n2 = 2 * I; e.up = I;
  e.w = e.w_up = expert_w(wts->gu, wts->gu_scale, wts->gu_bias, H);
  e.h = h; e.dt = T; e.glu = c.act; e.alpha = c.act_alpha; e.limit = c.act_limit;
  if ((rc = gen_gate_up(e, bits, st))) return rc;

  // shared expert in its weights' dtype S
  void* so = nullptr;
  if (shared) {
    const int S = c.shared_dtype;
    void* sh = base + L.sh;
    so = base + L.so;
    GenGu s{};
    s.act = x; s.act_dt = c.x_dtype; s.act_round = S; s.row_div = 1; s.rows = N; s.n = s.n2 = Is;
    s.w = dense_w(wts->sh_gate, S, H);
    s.w_up = dense_w(wts->sh_up, S, H);
    s.h = sh; s.dt = S; s.glu = c.act; s.alpha = c.act_alpha; s.limit = c.act_limit;
    if ((rc = gen_gate_up(s, 0, st))) return rc;
    GenMv sd{};
    sd.act = sh; sd.act_dt = S; sd.act_round = S; sd.rows = N; sd.n_out = H;
    sd.w = dense_w(wts->sh_down, S, Is);
    sd.out = so; sd.out_dt = S; sd.ld_out = H;
    if ((rc = gen_matvec(sd, st))) return rc;
  }
  // routed down, weighted combine, gated shared expert and the cast to x's dtype
  GenDn dn{};
  dn.h = h; dn.dt = T; dn.idx = ridx; dn.wt = rw; dn.N = N; dn.k = ks; dn.H = H;
  dn.w = expert_w(wts->dn, wts->dn_scale, wts->dn_bias, I);
  dn.sh = so; dn.sh_dt = c.shared_dtype; dn.sg = has_sg ? sg : nullptr;
  dn.y = y; dn.y_dt = c.x_dtype;
  return gen_down_combine(dn, bits, st);
}
