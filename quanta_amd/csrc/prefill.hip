// Large-M ("prefill") products over 128-position m-tiles, for gfx950: the routed experts' gate_up and down
// above the decode sizes, router logits there, and large dense bf16 products (router, shared expert).
//
// Reference: mx.gather_qmm over sorted rows src/quanta/dsv4/moe.py:114-124 and
// src/quanta/qwen35/moe.py:117-123; SwiGLU src/quanta/qwen35/moe.py:59-63; bf16 experts
// (mx.gather_mm) src/quanta/qwen35/moe.py:66-82; shared expert src/quanta/qwen35/moe.py:145-151.
//
// Quantized weights (prefill_kernel) are dequantised to fp16 in registers from an LDS copy of their tiled
// layout and multiplied on v_mfma_f32_32x32x16_f16 against an exactly scaled fp16 copy of the
// activations; bf16 weights (qmm_large_kernel) run v_mfma_f32_16x16x32_bf16.
#include <type_traits>

#include "qmoe_internal.h"
#include "small_body.h"
#include "../../include/quanta_moe.h"

namespace qmoe {

constexpr int kPfThreads = 512;                    // 8 wavefronts, two per SIMD
constexpr int kPfABytes = 128 * 128 * 2;           // one superblock of 128 rows of activations: 32 KiB

// LDS byte offset of a pointer into the kernel's dynamic LDS (the low 32 bits of its generic
// address), made wave-uniform for M0
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p)));
}
// Global -> LDS copy: each lane's 16 bytes at src land at lds_off + 16 * lane.
// M0 is saved and restored around the copy.
__device__ __forceinline__ void dma16(const void* src, uint32_t lds_off) {
  uint32_t saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(saved) : "v"(src), "s"(lds_off) : "memory");
}
// The same copy, and one of 4 bytes per lane, from a wave-uniform base address (a scalar register pair) plus a
// 32-bit per-lane offset: the base costs no vector registers.
__device__ __forceinline__ void dma16s(const void* sbase, uint32_t voff, uint32_t lds_off) {
  uint32_t saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(saved) : "v"(voff), "s"(sbase), "s"(lds_off) : "memory");
}
__device__ __forceinline__ void dma4s(const void* sbase, uint32_t voff, uint32_t lds_off) {
  uint32_t saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
               "global_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(saved) : "v"(voff), "s"(sbase), "s"(lds_off) : "memory");
}
// Wait until at most N of this wavefront's vector-memory operations are outstanding (they complete in
// issue order).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

// Workgroup barrier for the load rings: this wavefront's LDS reads drained (lgkmcnt 0), then
// s_barrier. Unlike __syncthreads() it carries no release fence, whose vmcnt(0) would also wait
// for the loads still in flight for later superblocks; the data each barrier publishes has been
// waited for explicitly (wait_vmcnt) by the wavefront that loaded it.
__device__ __forceinline__ void lg_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A lane's row data for the prologue, loaded and waited for in one asm block before any DMA is issued:
// two weight-row exponent bytes and the row scale of its activation row. The compiler then sees
// ready values and never guards their later uses with a vmcnt wait, which it cannot tell from the
// DMA prefetch's own (those waits would drain the prefetch every superblock).
struct RowLoads {
  int ex[2];
  float rs;
};
__device__ __forceinline__ RowLoads load_rows_now(const int8_t* e0, const int8_t* e1, const float* rs) {
  int v0, v1;
  float f;
  asm volatile("global_load_sbyte %0, %3, off\n\tglobal_load_sbyte %1, %4, off\n\t"
               "global_load_dword %2, %5, off\n\ts_waitcnt vmcnt(0)"
               : "=&v"(v0), "=&v"(v1), "=&v"(f)
               : "v"(e0), "v"(e1), "v"(rs)
               : "memory");
  return RowLoads{{v0, v1}, f};
}

// int4 -> fp16 dequant of the prefill kernels, one packed register (two weights) per VALU FMA.
// A code nibble masked in place is an fp16 subnormal: at bits 0-3 of a half it reads q * 2^-24,
// at bits 4-7 q * 2^-20, so fma(code, s * 2^(e+24) or s * 2^(e+20), b * 2^e) yields
// fp16(2^e (s q + b)) with a single rounding (the product is exact inside the FMA). e = row_exp
// - kDeqShift: row_exp puts the row's largest magnitude in [2^13, 2^14), which bounds
// s * 2^row_exp below 2^15 / 15 (15 s = (15 s + b) - b), so the larger scale factor, s *
// 2^(row_exp + 4), stays below 2^15.1 < 65504; the weights themselves lie below 2^-6 and keep
// fp16's full precision down to 2^-8 of the row maximum, below that an absolute 2^-20 of it
// (fp16 subnormals; the MFMAs take them exactly). Pairs 2 and 3 share one 8-bit shift.
constexpr int kDeqShift = 20;
struct DeqSb {
  f16x2_t s_lo, s_hi, b;   // scale for nibbles at bits 0-3 / 4-7 of each half, bias
};
// A weight row's (scale, bias) pair of one scale group as fp16 (s * 2^(e+24), b * 2^e) in one register.
__device__ __forceinline__ uint32_t deq_conv(uint32_t sbw, int e) {
  const f32x2_t v = {ldexpf(bf16lo_to_f32(sbw), e + 24), ldexpf(bf16hi_to_f32(sbw), e)};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}
__device__ __forceinline__ DeqSb deq_sb(uint32_t w) {
  const f16x2_t v = __builtin_bit_cast(f16x2_t, w);
  const f16x2_t lo = {v.x, v.x};
  return DeqSb{lo, lo * f16x2_t{static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)}, f16x2_t{v.y, v.y}};
}
// nibble pair j (0..3) of code word w: weights k = j and j+4 of the word's two 16-bit halves
__device__ __forceinline__ uint32_t deq_pair(uint32_t w, int j, const DeqSb& d) {
  const uint32_t src = (j >= 2) ? (w >> 8) : w;
  const f16x2_t q = __builtin_bit_cast(f16x2_t, src & ((j & 1) ? 0x00F000F0u : 0x000F000Fu));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, (j & 1) ? d.s_hi : d.s_lo, d.b));
}

// int6 pair j (0..3) of step half h: the nibble pair of word w as deq_pair takes it (even j at
// bits 0-3 of each half, odd j in place at bits 4-7, pairs 2 and 3 sharing one 8-bit shift), its
// two high bits from the group's high-bit word hw (bits 2j + 8h and 16 + 2j + 8h, as
// unpack_q128_6) moved just above the nibble: each half holds the 6-bit code q as the fp16
// subnormal q * 2^-24 (even j) or 16 q * 2^-24 (odd j, scaled by s_hi). row_exp bounds
// s * 2^row_exp below 2^15 / 63, so both scale factors stay below 2^19 / 63.
__device__ __forceinline__ uint32_t deq_pair6(uint32_t w, uint32_t hw, int h, int j, const DeqSb& d) {
  const uint32_t src = (j >= 2) ? (w >> 8) : w;
  const bool odd = (j & 1) != 0;
  const int hs = 2 * j + 8 * h - (odd ? 8 : 4);   // right shift of the high bits (left if < 0)
  const uint32_t hb = (hs >= 0) ? (hw >> hs) : (hw << -hs);
  const uint32_t v = (src & (odd ? 0x00F000F0u : 0x000F000Fu)) | (hb & (odd ? 0x03000300u : 0x00300030u));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, v),
                                                                odd ? d.s_hi : d.s_lo, d.b));
}

// int3 pair q (0..15) of the lane's three code words, as unpack_q128_3: the 3-bit codes at bits
// 0-2 of each half, the fp16 subnormal q * 2^-24. (int3 dequantizes with a shift one larger than
// kDeqShift: row_exp bounds s * 2^row_exp below 2^15 / 7, so s * 2^(e+24) stays below 2^18 / 7.)
__device__ __forceinline__ uint32_t deq_pair3(uint32_t w0, uint32_t w1, uint32_t w2, int q,
                                             const DeqSb& d) {
  const uint32_t w = (q < 5) ? w0 : (q < 10) ? w1 : w2;
  const uint32_t v = (q < 15) ? (w >> (3 * (q % 5))) & 0x00070007u
                              : ((w0 >> 15) & 0x00010001u) | ((w1 >> 14) & 0x00020002u) |
                                    ((w2 >> 13) & 0x00040004u);
  return __builtin_bit_cast(uint32_t,
                            __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, v), d.s_lo, d.b));
}

// ============================================================================ quantized weights
// Workgroup tile: 128 sorted positions x 256 NB weight rows (SwiGLU: half gate, half up rows), one
// 128-deep k superblock per iteration. 8 wavefronts side by side along the weight rows: wavefront w
// owns all 128 positions (4 m-blocks of 32) and NB n-blocks of 32 weight rows (two 16-row tiles;
// SwiGLU: NB = 2 a gate and an up block, NB = 1 a gate and an up tile), 64 NB accumulators per
// lane. Every weight is dequantized once per workgroup.
//
// What bounds it is instruction issue beside the MFMAs, and on partly filled tiles the weights' own
// work (copy, scale conversion, dequant of 256 NB rows x K), which a tile pays whatever its fill.
// The 32x32x16 MFMAs halve the instructions of the 16x16x32 form, and with two lane groups instead of
// four over the rows each lane converts one (scale, bias) pair per n-block and swaps: per superblock and
// wavefront 64 MFMAs and 32 conversion operations where 128 and 64 were. The first MFMA of a
// superblock waits for 16 instead of 32 weights per lane.
// Measured against the 16x16x32 form with its loads in one burst and two slots (128 experts of R rows,
// c2's int4 gate_up, us): R = 128 303 -> 286, 96 217 -> 199, 64 176 -> 154, 40 153 -> 145, 32 135 -> 126,
// 17 129 -> 118 (the 4.7 MB of each expert at 5.1 TB/s); 32-row blocks cost R = 72 192 -> 198 and 104
// 244 -> 254. int6 (NB = 1) R = 20 199 -> 180, 128 430 -> 401. Without loads and dequant it runs at 1.25
// PFLOP/s, what a large library product reaches on this card.
//
// All streaming loads go global -> LDS directly (global_load_lds_dwordx4 / _dword, inline assembly), into
// a ring of slots of one superblock each, three wherever they fit in LDS (PfCfg::slots: tiles of any size for
// int3 and int4 with NB = 1, up to 96 rows for int6 and for int3 with NB = 2, up to 64 for int4 with NB = 2), else
// two: loads one or two superblocks ahead, issued between the MFMAs. At the end of superblock p every
// wavefront waits for its own loads of p+1, and one barrier publishes slot p+1 and retires slot p. A
// slot holds
//  * A, 8 KiB per m-block: wavefront w loads rows 16w .. 16w+15, a 64-byte piece q (16-byte chunks 4q .. 4q+3
//    of a row's 128 values) per instruction and row, so a row's four lanes read one line; lane l
//    fetches chunk (l % 4) ^ ((l / 16) % 4) of its row, which spreads a fragment read's rows (64
//    bytes apart) over all banks;
//  * weights, per wavefront: its tiles' code blocks (verbatim copies of the tiled layout), their
//    scale/bias, and int6's high-bit planes.
//
// k order: step n = 4 s1 + c (s1: the superblock's scale group; c = 0..3) multiplies, in lane half hh,
// the eight codes of word (2 s1 + c % 2) of the tiled layout's lane group 2 hh + c / 2, i.e. chunk
// 8 s1 + 4 hh + c of the row. Both NB follow it, superblocks in order with one fp32 accumulator per
// output, so they give identical results.
template <int FMT, int NB>
struct PfCfg {
  static constexpr int NT = 2 * NB;                                                  // 16-row tiles per wavefront
  static constexpr int SBB = (FMT == FMT_INT6) ? 1536 : (FMT == FMT_INT3) ? 768 : 1024;   // tile superblock
  static constexpr int CB = (FMT == FMT_INT3) ? 768 : 1024;                          // its codes (int6: nibbles)
  static constexpr int HB = (FMT == FMT_INT6) ? 512 : 0;                             // int6 high-bit plane
  static constexpr int BWAVE = NT * (CB + 128 + HB);
  static constexpr int LOADS = (FMT == FMT_INT3 ? 3 * NT : NT) + NB + (FMT == FMT_INT6 ? NB : 0);   // per wavefront
  // slots of a tile of MB m-blocks: three where they fit in LDS (loads two superblocks ahead), else two
  static constexpr int slot(int mb) { return 8192 * mb + 8 * BWAVE; }
  static constexpr int slots(int mb) { return 3 * slot(mb) <= 160 * 1024 - 512 ? 3 : 2; }
  static constexpr int ring(int mb) { return slots(mb) * slot(mb); }
  static constexpr int max2(int x, int y) { return x > y ? x : y; }
  static constexpr int ROWTAB = max2(max2(ring(1), ring(2)), max2(ring(3), ring(4)));   // 128 row scales
  static constexpr int LDS = ROWTAB + 512;
};

template <int FMT, int EPI, int NB>
__global__ void __launch_bounds__(kPfThreads, 1) prefill_kernel(QmmArgs a) {
  using C = PfCfg<FMT, NB>;
  constexpr int DS = (FMT == FMT_INT3) ? kDeqShift + 1 : kDeqShift;   // row_exp - e
  extern __shared__ u32x4 lds[];
  char* lds_c = reinterpret_cast<char*>(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  // wave index as a scalar: per-wave decisions are uniform (scalar) branches
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int e, m0, m_cnt;
  // XCD-aware tile order. Workgroups are dispatched round-robin over the 8 XCDs, so linear id i runs
  // on XCD i % 8 as that XCD's (i / 8)-th workgroup. Each XCD takes groups of G m-tiles x all nbk
  // weight-row blocks (G * nbk <= 32, one workgroup per CU of the XCD): the blocks of an m-tile share
  // its activation slices through the XCD's L2, and the G m-tiles share the weight slices.
  const int nbk = a.n_rows / (256 * NB);
  const int G = (nbk >= 32) ? 1 : 32 / nbk;
  const int wi = blockIdx.x, xcd = wi & 7, kx = wi >> 3;
  const int gk = kx / (G * nbk), rk = kx - gk * (G * nbk);
  const int mt = (gk * 8 + xcd) * G + rk / nbk;
  const int cb = rk % nbk;
  if (mt >= a.mtiles || !resolve_mtile(a, mt, kLargeMTile, e, m0, m_cnt)) return;
  // (one stack of a projection whose experts have different widths: the others' m-tiles exit)
  if (a.expert_map) {
    e = a.expert_map[e];
    if (e < 0) return;
  }
  const int64_t ebase = static_cast<int64_t>(e) * (a.n_rows / 16);
  const int nsb = a.K / 128;
  const int mb_act = __builtin_amdgcn_readfirstlane((m_cnt + 31) >> 5);   // 1..4
  // (AWQ: the weight blocks from split_tile on read the second activation copy)
  const bool hi = a.act16_hi && 16 * NB * cb >= a.split_tile;
  const uint16_t* act16 = hi ? a.act16_hi : a.act16;
  const float* row_sinv = hi ? a.row_sinv_hi : a.row_sinv;

  // activation source: this wavefront's 16 rows, four lanes each. Rows past the tile and rows whose
  // activation row is invalid read activation row 0 (the former are never stored, the latter are
  // written as zeros by the epilogue). A wavefront whose rows all lie past the tile loads none.
  const bool a_on = 16 * wave < m_cnt;
  const int arow_r = 16 * wave + (lane >> 2);
  const int64_t arow = (arow_r < m_cnt) ? act_row(a, m0 + arow_r) : -1;
  const char* arow_ptr = reinterpret_cast<const char*>(act16 + (arow >= 0 ? arow : 0) * static_cast<int64_t>(a.K)) +
                         16 * ((lane & 3) ^ ((lane >> 4) & 3));
  const uint32_t lds_base = lds_offset(lds);

  // this wavefront's weight tiles; tile bases are wave-uniform (scalar registers)
  const int r32 = lane & 31, hh = lane >> 5, r16 = lane & 15, half = r32 >> 4;
  auto tile_of = [&](int t) {
    if (EPI == EPI_SWIGLU) {
      if (NB == 2) return (t < 2) ? 16 * cb + 2 * wave + t : a.n_rows / 32 + 16 * cb + 2 * wave + (t - 2);
      return (t == 0) ? 8 * cb + wave : a.n_rows / 32 + 8 * cb + wave;
    }
    return (16 * cb + 2 * wave) * NB + t;
  };
  const char* wtile[C::NT];
  const char* wsb[C::NT];
#pragma unroll
  for (int t = 0; t < C::NT; ++t) {
    const int64_t tb = (ebase + tile_of(t)) * nsb;
    wtile[t] = static_cast<const char*>(a.codes) + tb * C::SBB;
    wsb[t] = reinterpret_cast<const char*>(a.sb) + tb * 128;
  }
  // the lane's weight rows' exponents (one per n-block) and the activation row's scale in one round
  // trip; wavefront w publishes the scales of its rows for the epilogue (-1: no data), before the
  // first barrier
  float* row_tab = reinterpret_cast<float*>(lds_c + C::ROWTAB);
  int rex[NB];   // the dequant exponent e of the lane's weight row (deq_sb)
  {
    const int8_t* e0 = a.row_exp + (ebase + tile_of(0) + half * (tile_of(1) - tile_of(0))) * 16 + r16;
    const int8_t* e1 = (NB == 2) ? a.row_exp + (ebase + tile_of(C::NT - 2) + half) * 16 + r16 : e0;
    const RowLoads rl = load_rows_now(e0, e1, row_sinv + (arow >= 0 ? arow : 0));
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) rex[nb] = rl.ex[nb] - DS;
    if (a_on && (lane & 3) == 0) row_tab[arow_r] = (arow >= 0) ? rl.rs : -1.0f;
  }
  // scale/bias and high-bit copies: lanes 0-31 take an n-block's first tile, lanes 32-63 its second
  const int64_t t_step = static_cast<int64_t>(tile_of(1) - tile_of(0)) * nsb;
  const uint32_t sb_voff = static_cast<uint32_t>(hh * t_step * 128 + 4 * r32);
  const uint32_t hb_voff = static_cast<uint32_t>(hh * t_step * C::SBB + 16 * r32);

  // load u of superblock p into the slot at byte `slot`: the weights' C::LOADS, then A's 4 (when a_on)
  auto issue = [&](int p, int slot, int u, auto mbc) __attribute__((always_inline)) {
    constexpr int AB = 8192 * decltype(mbc)::value;
    constexpr int NC = (FMT == FMT_INT3) ? 3 * C::NT : C::NT;
    const uint32_t dst = lds_base + slot + AB + wave * C::BWAVE;
    if (u < NC) {
      if (FMT == FMT_INT3)   // 768 B per tile: three dword copies
        dma4s(wtile[u / 3] + static_cast<int64_t>(p) * C::SBB + 256 * (u % 3), 4 * lane,
              dst + u / 3 * C::CB + 256 * (u % 3));
      else
        dma16s(wtile[u] + static_cast<int64_t>(p) * C::SBB, 16 * lane, dst + u * C::CB);
    } else if (u < NC + NB) {
      const int nb = u - NC;
      dma4s(wsb[2 * nb] + static_cast<int64_t>(p) * 128, sb_voff, dst + C::NT * C::CB + 256 * nb);
    } else if (u < C::LOADS) {
      const int nb = u - NC - NB;
      dma16s(wtile[2 * nb] + static_cast<int64_t>(p) * C::SBB + 1024, hb_voff, dst + C::NT * (C::CB + 128) + 1024 * nb);
    } else if (a_on) {
      const int q = u - C::LOADS;
      dma16(arow_ptr + 256 * p + 64 * q, lds_base + slot + (4 * wave + q) * 1024);
    }
  };

  f32x16_t acc[4][NB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[i][nb][j] = 0.f;

  // LDS offsets of the lane's fragments in a slot: its row's chunk c of m-block 0, its weight row
  int la[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) la[c] = half * 4096 + hh * 1024 + r16 * 64 + 16 * (c ^ ((r16 >> 2) & 3));
  const int lg0 = 2 * hh * 16 + r16;   // the row's first source lane in a tile (the second: + 16)

  // One superblock: eight 16-deep steps of MB groups; group i issues the NB MFMAs of m-block i, the LDS
  // read of the A fragment PD groups ahead, its share of the next step's 4 NB dequant units (n-block
  // u / 4, pair u % 4) and (LD) of the loads of superblock pl, in that order (scheduling barriers). The
  // loads are spread over the first groups because a wavefront's loads issued together keep it from
  // its MFMAs until the memory pipe has taken them, up to 68 KiB per workgroup.
  auto compute = [&](int slot_off, int pl, int pl_slot, auto mbc, auto ldc) __attribute__((always_inline)) {
    constexpr int MB = decltype(mbc)::value;
    constexpr bool LD = decltype(ldc)::value;
    constexpr int NI = 8 * MB;                 // A fragments (groups) per superblock
    constexpr int PD = 3;
    constexpr int NU = C::LOADS + 4, LPG = (2 * NU + NI - 1) / NI;   // loads per group
    const char* slot = lds_c + slot_off;
    const char* lb = slot + 8192 * MB + wave * C::BWAVE;
    u32x4 q[NB][2];
    u32x2 hq[NB][2];
    uint32_t sw[NB][2];   // the converted scale/bias of the superblock's two groups
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int t = 2 * nb + half;
      sw[nb][0] = reinterpret_cast<const uint32_t*>(lb + C::NT * C::CB + t * 128)[2 * r16 + hh];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        if (FMT == FMT_INT3) {   // the source lane's three words
          const uint32_t* w3 = reinterpret_cast<const uint32_t*>(lb + t * C::CB) + 3 * (lg0 + 16 * g);
          q[nb][g] = u32x4{w3[0], w3[1], w3[2], 0u};
        } else {
          q[nb][g] = reinterpret_cast<const u32x4*>(lb + t * C::CB)[lg0 + 16 * g];
        }
        if (FMT == FMT_INT6)
          hq[nb][g] = reinterpret_cast<const u32x2*>(lb + C::NT * (C::CB + 128) + t * 512)[lg0 + 16 * g];
      }
    }
    DeqSb dsb[NB];
    // both lanes of a row need both groups' scale and bias: lane half hh converts group hh's, and the
    // halves swap
    auto sb_conv = [&](int grp) __attribute__((always_inline)) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if (grp == 0) {
          const uint32_t own = deq_conv(sw[nb][0], rex[nb]);
          const auto both = __builtin_amdgcn_permlane32_swap(own, own, false, false);
          sw[nb][0] = both[0];
          sw[nb][1] = both[1];
        }
        dsb[nb] = deq_sb(sw[nb][grp]);
      }
    };
    auto deq_unit = [&](int n, int u, u32x4* bfo) __attribute__((always_inline)) {
      const int nb = u >> 2, j = u & 3, s1 = n >> 2, c = n & 3, s = 2 * s1 + (c & 1);
      const u32x4& w = q[nb][c >> 1];
      if constexpr (FMT == FMT_INT6)
        bfo[nb][j] = deq_pair6(w[s], s1 ? hq[nb][c >> 1].y : hq[nb][c >> 1].x, c & 1, j, dsb[nb]);
      else if constexpr (FMT == FMT_INT3)
        bfo[nb][j] = deq_pair3(w.x, w.y, w.z, 4 * s + j, dsb[nb]);
      else
        bfo[nb][j] = deq_pair(w[s], j, dsb[nb]);
    };
    u32x4 bf[2][NB];
    u32x4 A[NI];
    auto load_a = [&](int m) __attribute__((always_inline)) {
      const int n = m / MB, i = m % MB;
      A[m] = *reinterpret_cast<const u32x4*>(slot + la[n & 3] + 8192 * i + 2048 * (n >> 2));
    };
#pragma unroll
    for (int m = 0; m < PD; ++m) load_a(m);
    sb_conv(0);
#pragma unroll
    for (int u = 0; u < 4 * NB; ++u) deq_unit(0, u, bf[0]);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      if (n == 3) sb_conv(1);      // group 1 feeds steps 4 to 7
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int m = n * MB + i;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[i][nb] = mfma32_f16(A[m], bf[n & 1][nb], acc[i][nb]);
        if (m + PD < NI) load_a(m + PD);
        if (n < 7) {
#pragma unroll
          for (int u = i * 4 * NB / MB; u < (i + 1) * 4 * NB / MB; ++u) deq_unit(n + 1, u, bf[(n + 1) & 1]);
        }
        if constexpr (LD) {
#pragma unroll
          for (int u = m * LPG; u < (m + 1) * LPG && u < NU; ++u) issue(pl, pl_slot, u, mbc);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  auto run = [&](auto mbc) __attribute__((always_inline)) {
    constexpr int MB = decltype(mbc)::value;
    constexpr int NS = C::slots(MB), SLOT = C::slot(MB), AHEAD = NS - 1;
    // wait until at most the loads of `sbs` superblocks are outstanding
    auto wait_but = [&](auto sbs) __attribute__((always_inline)) {
      constexpr int S = decltype(sbs)::value;
      if (a_on) wait_vmcnt<S * (C::LOADS + 4)>(); else wait_vmcnt<S * C::LOADS>();
    };
    const int n0 = min(AHEAD, nsb);
    for (int p = 0; p < n0; ++p)
#pragma unroll
      for (int u = 0; u < C::LOADS + 4; ++u) issue(p, p * SLOT, u, mbc);
    if (n0 == AHEAD) wait_but(std::integral_constant<int, AHEAD - 1>{}); else wait_vmcnt<0>();
    lg_barrier();
    int cur = 0, nxt = AHEAD * SLOT;   // slots of superblock p and of p + AHEAD
    auto step = [&](int& off) __attribute__((always_inline)) { off = (off == (NS - 1) * SLOT) ? 0 : off + SLOT; };
    int p = 0;
    for (; p + AHEAD < nsb; ++p) {
      compute(cur, p + AHEAD, nxt, mbc, std::true_type{});
      wait_but(std::integral_constant<int, AHEAD - 1>{});
      lg_barrier();
      step(cur);
      step(nxt);
    }
    for (; p < nsb; ++p) {
      compute(cur, 0, 0, mbc, std::false_type{});
      wait_vmcnt<0>();
      lg_barrier();
      step(cur);
    }
  };
  switch (mb_act) {
    case 1: run(std::integral_constant<int, 1>{}); break;
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    default: run(std::integral_constant<int, 4>{}); break;
  }

  // epilogue: lane holds C[row 8 (j / 4) + 4 (lane / 32) + j % 4][col lane % 32] of each 32x32 block
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i >= mb_act) break;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int mr = 32 * i + 8 * (j >> 2) + 4 * hh + (j & 3);
      const float rs = (mr < m_cnt) ? row_tab[mr] : -1.0f;
      const bool ok = rs >= 0.f;   // (rows whose activation row is invalid are written as zeros)
      // undo both power-of-two scalings (activation row, weight row): exact
      auto val = [&](int nb) { return ok ? ldexpf(acc[i][nb][j] * rs, -rex[nb]) : 0.f; };
      if (EPI == EPI_SWIGLU && NB == 1) {
        const float v = val(0);
        const float up = __shfl_xor(v, 16);   // the up tile's row, 16 lanes on
        if (mr < m_cnt && half == 0) store_out<EPI>(a, m0 + mr, 128 * cb + 16 * wave + r16, v, up);
      } else if (mr < m_cnt) {
        if (EPI == EPI_SWIGLU) {
          store_out<EPI>(a, m0 + mr, 256 * cb + 32 * wave + r32, val(0), val(NB - 1));
        } else {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            store_out<EPI>(a, m0 + mr, (256 * cb + 32 * wave) * NB + 32 * nb + r32, val(nb), 0.f);
        }
      }
    }
  }
}

// ============================================================================ bf16 weights
// Workgroup tile: 128 sorted positions x 256 weight rows (SwiGLU: 128 gate + 128 up rows -> 128 h
// columns), one 128-deep k superblock per iteration. Wavefront w owns all 128 positions (8 m-blocks of
// 16) and two 16-row weight tiles (SwiGLU: gate tile w and its up tile). Activations go global -> LDS
// two superblocks ahead, three slots ([m-block][step][64 lanes] x 16 B; wavefront w loads m-block w,
// lane l fetching row l%16's 8-k chunk that MFMA lane l consumes); the weight fragments are read
// into registers one superblock ahead. A partly filled tile computes only its first 2, 4 or 8 m-blocks.
constexpr int kLgNBuf = 3;
constexpr size_t kLgLdsBytes = kLgNBuf * kPfABytes + 512;   // 96.5 KiB, the last 512 B the rows' validity

struct LgStage {
  u32x4 q[2][4];   // 2 tiles x 4 steps of B fragments
};

template <int EPI>
__global__ void __launch_bounds__(kPfThreads) qmm_large_kernel(QmmArgs a) {
  extern __shared__ u32x4 lds[];
  char* lds_c = reinterpret_cast<char*>(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int e, m0, m_cnt;
  // (the tile order of prefill_kernel, 256-row weight blocks)
  const int nbk = a.n_rows / 256;
  const int G = (nbk >= 32) ? 1 : 32 / nbk;
  const int wi = blockIdx.x, xcd = wi & 7, kx = wi >> 3;
  const int gk = kx / (G * nbk), rk = kx - gk * (G * nbk);
  const int mt = (gk * 8 + xcd) * G + rk / nbk;
  const int cb = rk % nbk;
  const int mrows = (a.dense_mtile > 0 && !a.offsets && !a.tile_map) ? a.dense_mtile : kLargeMTile;
  if (mt >= a.mtiles || !resolve_mtile(a, mt, mrows, e, m0, m_cnt)) return;
  const int64_t ebase = static_cast<int64_t>(e) * (a.n_rows / 16);
  const int nsb = a.K / 128;
  const int mb_act = __builtin_amdgcn_readfirstlane((m_cnt + 15) >> 4);   // 1..8

  // activation source: lane -> row lane%16 of m-block `wave`, k-chunk 4s + lane/16 of step s (rows past
  // the tile and invalid rows as in prefill_kernel)
  const bool a_on = wave < mb_act;
  const int arow_r = 16 * wave + (lane & 15);
  const int64_t arow = (arow_r < m_cnt) ? act_row(a, m0 + arow_r) : -1;
  const char* arow_ptr = reinterpret_cast<const char*>(a.act + (arow >= 0 ? arow : 0) * static_cast<int64_t>(a.K)) +
                         16 * (lane >> 4);
  const uint32_t lds_base = lds_offset(lds);
  // wavefront w's lanes 0-15 publish which rows of m-block w have data, for the epilogue
  int* row_ok = reinterpret_cast<int*>(lds_c + kLgNBuf * kPfABytes);
  if (a_on && lane < 16) row_ok[arow_r] = arow >= 0;
  const u32x4* wp[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int tl = (EPI == EPI_SWIGLU) ? (t == 0 ? 8 * cb + wave : a.n_rows / 32 + 8 * cb + wave)
                                       : 16 * cb + 2 * wave + t;
    wp[t] = static_cast<const u32x4*>(a.codes) + (ebase + tl) * (a.K / 32) * 64 + lane;
  }
  auto issue = [&](int p) __attribute__((always_inline)) {
    if (!a_on) return;
    const char* src = arow_ptr + 256 * p;
    const uint32_t dst = lds_base + (p % kLgNBuf) * kPfABytes + wave * 4 * 1024;
#pragma unroll
    for (int s = 0; s < 4; ++s) dma16(src + 64 * s, dst + s * 1024);
  };
  f32x4_t acc[8][2];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // One superblock: four 32-k MFMA steps of MB slots; slot i issues the two MFMAs of m-block i and the
  // read of its A fragment for step s+1, in that order (scheduling barriers).
  auto compute = [&](int p, const LgStage& gb, auto mbc) __attribute__((always_inline)) {
    constexpr int MB = decltype(mbc)::value;
    const u32x4* la = reinterpret_cast<const u32x4*>(lds_c + (p % kLgNBuf) * kPfABytes) + lane;
    u32x4 A[2][MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) A[0][i] = la[256 * i];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = s & 1;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[i][t] = mfma16(as_bf16x8(A[c][i]), as_bf16x8(gb.q[t][s]), acc[i][t]);
        if (s < 3) A[c ^ 1][i] = la[256 * i + 64 * (s + 1)];
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  LgStage gbf[2];
  auto load_bf = [&](int p, LgStage& g) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < 4; ++s) g.q[t][s] = wp[t][(4 * p + s) * 64];
  };
  // Before the barrier that publishes superblock p+1, a wavefront waits until only its loads of p+2
  // remain outstanding.
  auto run = [&](auto mbc) __attribute__((always_inline)) {
    auto wait_next = [&](bool far) __attribute__((always_inline)) {
      if (a_on && far) wait_vmcnt<4>(); else wait_vmcnt<0>();
    };
    issue(0);
    if (nsb > 1) issue(1);
    load_bf(0, gbf[0]);
    wait_next(nsb > 1);
    lg_barrier();
    auto iter = [&](int p, const LgStage& cur, LgStage& nxt) __attribute__((always_inline)) {
      const bool far = p + 2 < nsb;
      if (far) issue(p + 2);
      load_bf(p + 1, nxt);
      compute(p, cur, mbc);
      wait_next(far);
      lg_barrier();
    };
    int p = 0;
    for (; p + 2 < nsb; p += 2) {
      iter(p, gbf[0], gbf[1]);
      iter(p + 1, gbf[1], gbf[0]);
    }
    if (p + 1 < nsb) {
      iter(p, gbf[0], gbf[1]);
      compute(p + 1, gbf[1], mbc);
    } else {
      compute(p, gbf[0], mbc);
    }
  };
  if (mb_act <= 2) run(std::integral_constant<int, 2>{});
  else if (mb_act <= 4) run(std::integral_constant<int, 4>{});
  else run(std::integral_constant<int, 8>{});

  // epilogue: lane holds C[row 4(lane/16) + j][col lane%16] of each 16x16 block
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (i >= mb_act) break;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int mr = 16 * i + 4 * (lane >> 4) + j;
      if (mr >= m_cnt) continue;
      // rows whose activation row is invalid read as zeros (their A data was row 0's)
      const bool ok = row_ok[mr] != 0;
      auto val = [&](int t) { return ok ? acc[i][t][j] : 0.f; };
      if (EPI == EPI_SWIGLU) {
        store_out<EPI>(a, m0 + mr, 128 * cb + 16 * wave + (lane & 15), val(0), val(1));
      } else {
#pragma unroll
        for (int t = 0; t < 2; ++t)
          store_out<EPI>(a, m0 + mr, 256 * cb + 32 * wave + 16 * t + (lane & 15), val(t), 0.f);
      }
    }
  }
}

// ============================================================================ router logits
// Logits of batches above the decode sizes, short of those that fill the chip with qmm_large_kernel's tiles:
// 16 MB tokens x 64 weight rows per workgroup, a 128-deep k superblock per iteration, two 16x16 blocks per
// wavefront (weight tile w % 4, m-blocks 2 (w / 4) and the next), tokens and weights through an LDS ring of
// [16-row block][step] x 1 KiB: a weight tile's fragments as they are stored; of a token block 64 bytes of each
// row, loaded by four neighbouring lanes, 16-byte chunk c at c ^ (row / 4 % 4), which spreads the fragment
// reads over all banks.
//
// Every logit is one accumulator over all of K in k order, which is qmm_large_kernel's sum: the expert ids of a
// prompt depend on neither the kernel that a batch size takes nor K's split over wavefronts, whose sums
// differ by up to 8e-6 at c2 and move a token across a tie of its last expert now and then.
//
// What bounds it is latency, K / 128 rounds of a barrier, fragment reads and dependent MFMAs with the loads NS - 1
// superblocks ahead. us, the large kernel before, now: 2048 x 256 391 tokens 25 / 9.1, 2048 29 / 9.8; 4096 x 512 300
// 45 / 15, 1000 46 / 16, 2000 48 / 21; 7168 x 256 800 76 / 24, 2300 108 / 43. (32-token tiles with six slots: the same,
// and 144 KiB that no other workgroup can share. Lanes that load 16 bytes of 16 rows each: 2300 49.)
template <int MB>
struct RouterCfg {
  static constexpr int WAVES = 2 * MB;                       // MB = 2 or 4
  static constexpr int SLOT = (MB + 4) * 4096;               // one superblock: MB token blocks, 4 weight tiles
  static constexpr int NS = (MB == 2) ? 3 : 4;
  static constexpr int LOADS = 2 + 16 / WAVES;               // per wavefront and superblock
  static constexpr size_t LDS = static_cast<size_t>(NS) * SLOT;   // 72 or 128 KiB
};

template <int MB>
__global__ void __launch_bounds__(64 * RouterCfg<MB>::WAVES) router_logits_kernel(QmmArgs a, int n_tok, int n_rb, int n_wg) {
  using C = RouterCfg<MB>;
  extern __shared__ u32x4 lds[];
  const char* lds_c = reinterpret_cast<const char*>(lds);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // (each XCD takes a run of tiles, a token block's weight blocks together: its L2 reads its share of x once)
  const int per = (n_wg + 7) / 8;
  const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per || id >= n_wg) return;
  const int tb = id / n_rb, rb = id % n_rb;
  const int rows = static_cast<int>(a.dense_rows);
  const int nsb = a.K / 128;
  // loads: two steps of token block ab, and 16 / WAVES steps of weight tile w % 4. Tokens past the end read row 0
  // (never stored).
  const int ab = (MB == 2) ? wave >> 1 : wave & 3, as = 2 * ((MB == 2) ? wave & 1 : wave >> 2);
  const int ws = (16 / C::WAVES) * (wave >> 2);
  const int t = 16 * MB * tb + 16 * ab + (lane >> 2);
  const char* xp = reinterpret_cast<const char*>(a.act + (t < rows ? t : 0) * static_cast<int64_t>(a.K)) +
                   16 * ((lane & 3) ^ ((lane >> 4) & 3));
  const char* wp = static_cast<const char*>(a.codes) + (4 * rb + (wave & 3)) * static_cast<int64_t>(a.K / 32) * 1024;
  const uint32_t lds_base = lds_offset(lds);
  auto issue = [&](int p) __attribute__((always_inline)) {
    const uint32_t dst = lds_base + p % C::NS * C::SLOT;
#pragma unroll
    for (int j = 0; j < 2; ++j) dma16(xp + 256 * p + 64 * (as + j), dst + (4 * ab + as + j) * 1024);
#pragma unroll
    for (int j = 0; j < 16 / C::WAVES; ++j)
      dma16s(wp + (4 * static_cast<int64_t>(p) + ws + j) * 1024, 16 * lane, dst + (4 * (MB + (wave & 3)) + ws + j) * 1024);
  };
  const int n0 = min(C::NS - 1, nsb);
  for (int p = 0; p < n0; ++p) issue(p);
  const int mb = 2 * (wave >> 2);
  const int xo = 4 * (lane & 15) + ((lane >> 4) ^ ((lane >> 2) & 3));   // the lane's fragment in a token block's step
  f32x4_t acc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int p = 0; p < nsb; ++p) {
    // this wavefront's loads of superblock p have landed (those of the NS - 2 after it may be in flight); the
    // barrier publishes p and retires p - 1, whose slot the loads of p + NS - 1 take
    if (p + C::NS - 2 < nsb) wait_vmcnt<(C::NS - 2) * C::LOADS>(); else wait_vmcnt<0>();
    lg_barrier();
    if (p + C::NS - 1 < nsb) issue(p + C::NS - 1);
    const u32x4* sl = reinterpret_cast<const u32x4*>(lds_c + p % C::NS * C::SLOT);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bf16x8_t B = as_bf16x8(sl[256 * (MB + (wave & 3)) + 64 * s + lane]);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = mfma16(as_bf16x8(sl[256 * (mb + i) + 64 * s + xo]), B, acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 16 * (MB * tb + mb + i) + 4 * (lane >> 4) + j;
      if (row < rows) store_out<EPI_F32>(a, row, 64 * rb + 16 * (wave & 3) + (lane & 15), acc[i][j], 0.f);
    }
}

template <int MB>
static int launch_router_k(const QmmArgs& a, hipStream_t stream) {
  using C = RouterCfg<MB>;
  const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(router_logits_kernel<MB>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(C::LDS));
  if (err != hipSuccess) return fail(std::string("router logits: LDS attribute: ") + hipGetErrorString(err));
  const int64_t n_tok = (a.dense_rows + 16 * MB - 1) / (16 * MB), n_rb = a.n_rows / 64, n_wg = n_tok * n_rb;
  if (n_wg > (int64_t(1) << 30)) return fail("router logits: product too large for one launch");
  router_logits_kernel<MB><<<dim3(static_cast<unsigned>((n_wg + 7) / 8 * 8)), 64 * C::WAVES, C::LDS, stream>>>(
      a, static_cast<int>(n_tok), static_cast<int>(n_rb), static_cast<int>(n_wg));
  return check_launch("router logits");
}

int launch_router_logits(const QmmArgs& a, hipStream_t stream) {
  if (a.offsets || a.tile_map || a.dense_rows <= 0 || a.dense_rows > (int64_t(1) << 30) || a.act_stride || a.norm_w)
    return fail("router logits: one dense bf16 segment");
  if (a.K <= 0 || a.K % 128 || a.n_rows <= 0 || a.n_rows % 64)
    return fail("router logits: K % 128 == 0 and weight rows % 64 == 0 required");
  // 32-token tiles while they are at most one workgroup per CU, 64-token ones above, where the smaller ones would
  // read a third more. us, 32 against 64 tokens: 2048 x 256 391 9.1 / 12, 2048 9.8 / 12, 3000 12.9 / 11.6; 4096 x 512 1000
  // 16.5 / 18, 1500 23 / 20; 7168 x 256 800 24 / 28, 1500 27 / 31, 2300 45 / 43.
  const bool two = (a.dense_rows + 31) / 32 * (a.n_rows / 64) <= 256;
  return two ? launch_router_k<2>(a, stream) : launch_router_k<4>(a, stream);
}

// ============================================================================ launcher
// 1-D grid in the XCD-grouped order the kernels decode: m-tiles padded to whole groups of 8 XCDs x G
// m-tiles; workgroups past `mtiles` exit at once. The kernels' dynamic LDS is above the default
// per-kernel limit; set it for the current device.
static int launch_tiles(void (*kernel)(QmmArgs), const QmmArgs& a, int block_rows, size_t lds_bytes, int64_t mtiles,
                        hipStream_t stream) {
  const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes));
  if (err != hipSuccess) return fail(std::string("qmm(large): LDS attribute: ") + hipGetErrorString(err));
  const int nbk = a.n_rows / block_rows;
  const int G = (nbk >= 32) ? 1 : 32 / nbk;
  const int64_t mpad = (mtiles + 8 * G - 1) / (8 * G) * (8 * G);
  QmmArgs b = a;
  b.mtiles = static_cast<int>(mtiles);
  kernel<<<dim3(static_cast<unsigned>(mpad * nbk)), kPfThreads, lds_bytes, stream>>>(b);
  return 0;
}

template <int FMT, int EPI>
static int launch_prefill(const QmmArgs& a, int64_t mtiles, hipStream_t stream) {
  // 512-row weight blocks (SwiGLU: 256-row gate and up halves; a second activation: blocks on one side
  // of its split), so that an A fragment feeds two MFMAs. int6's 1.5 KiB superblocks leave no room
  // for the second slot of 512 rows.
  if constexpr (FMT != FMT_INT6) {
    if (a.n_rows % 512 == 0 && (!a.act16_hi || a.split_tile % 32 == 0))
      return launch_tiles(prefill_kernel<FMT, EPI, 2>, a, 512, PfCfg<FMT, 2>::LDS, mtiles, stream);
  }
  return launch_tiles(prefill_kernel<FMT, EPI, 1>, a, 256, PfCfg<FMT, 1>::LDS, mtiles, stream);
}

int launch_large(const QmmArgs& a, int fmt, int epi, int64_t mtiles, hipStream_t stream) {
  if (epi == EPI_SWIGLU && !prefill_reach(fmt, a.n_rows, a.K))
    return fail("qmm(large): gate and up tiles more than 4 GiB apart (the small regime takes them)");
#define QMOE_LARGE(F)                                                                  \
  (epi == EPI_SWIGLU ? launch_prefill<F, EPI_SWIGLU>(a, mtiles, stream)                \
   : epi == EPI_BF16 ? launch_prefill<F, EPI_BF16>(a, mtiles, stream)                  \
                     : launch_prefill<F, EPI_F32>(a, mtiles, stream))
  if (fmt == FMT_INT4) return QMOE_LARGE(FMT_INT4);
  if (fmt == FMT_INT3) return QMOE_LARGE(FMT_INT3);
  if (fmt == FMT_INT6) return QMOE_LARGE(FMT_INT6);
#undef QMOE_LARGE
  if (epi == EPI_SWIGLU) return launch_tiles(qmm_large_kernel<EPI_SWIGLU>, a, 256, kLgLdsBytes, mtiles, stream);
  if (epi == EPI_BF16) return launch_tiles(qmm_large_kernel<EPI_BF16>, a, 256, kLgLdsBytes, mtiles, stream);
  return launch_tiles(qmm_large_kernel<EPI_F32>, a, 256, kLgLdsBytes, mtiles, stream);
}

}  // namespace qmoe
