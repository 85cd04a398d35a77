// Single-stream attention kernel for every 16-bit head size (gfx950): NW
// waves x 32 query rows per tile (8 waves and 256 rows for D = 96 and 128;
// for D = 64 the dual map, 4 waves of 64 rows (two 32-row halves that share
// every LDS operand) and two work-groups per CU, and, for comparisons, 8 waves
// or 12 waves and 384 rows; for D = 192 and 256 the wide map, 4 waves and 128
// rows, one wave per SIMD with O in AGPRs and K and V in two-stage rings, and
// for D = 192 by default the dual-wide map, the wide map with 64 rows per wave
// as two 32-row halves and 256-row tiles; and for D = 64 and 128 the half map,
// 4 waves of 32 rows on 128-row tiles, two work-groups per CU, for frames of
// 127 to 254 rows and launches too small for 256-row tiles),
// each wave issuing S = K Q^T, the softmax and O += V^T P^T of consecutive
// 32-key sub-blocks as one instruction stream
// (the key loop is hand-scheduled assembly generated by gen_stream_asm.py into
// lvsa_attn_stream_body.inc, with the asm operand lists; its header comment
// has the schedule, the register map and the hazard rules).  This file holds
// the C++ around it: the work item, the pointers and per-lane constants the
// loop reads (passed in the registers the loop expects), the epilogue, and
// the work-queue loop of the persistent launch.
//
// The loop handles plan descriptors "none" and "two-part" only; lvsa_attn_fwd
// sends geometries that can produce generic descriptors (query frames below
// 255 rows, 127 for the 128-row tiles of the wide and half maps, or key frames
// below 64 rows) to attn_fwd_pp_kernel / attn_fwd_kernel, and accepts 384-row tiles
// only for query frames of at least 383 rows (256-row tiles at D = 192, which
// only the dual-wide map runs, for at least 255).
#pragma once
#include "lvsa_attn_kernels.h"
#include "lvsa_attn_stream_body.inc"

namespace lvsa {
namespace {

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x6 __attribute__((ext_vector_type(6)));
typedef unsigned u32x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x12 __attribute__((ext_vector_type(12)));
typedef unsigned u32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x32 __attribute__((ext_vector_type(32)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

template <int N>
struct U32Vec;
template <>
struct U32Vec<2> { typedef u32x2 type; };
template <>
struct U32Vec<4> { typedef u32x4 type; };
template <>
struct U32Vec<6> { typedef u32x6 type; };
template <>
struct U32Vec<8> { typedef u32x8 type; };
template <>
struct U32Vec<12> { typedef u32x12 type; };
template <>
struct U32Vec<16> { typedef u32x16 type; };
template <>
struct U32Vec<32> { typedef u32x32 type; };

// Q at D = 96, 192 and 256 (24, 48 and 64 registers) goes to the asm as two
// operands: 24 registers have no inline-asm operand class, and the wider
// ones are split at 32.
template <int LO, int HI>
struct U32Split {
  typename U32Vec<LO>::type lo;
  typename U32Vec<HI>::type hi;
};
template <>
struct U32Vec<24> { typedef U32Split<16, 8> type; };
template <>
struct U32Vec<48> { typedef U32Split<32, 16> type; };
template <>
struct U32Vec<64> { typedef U32Split<32, 32> type; };

// Q of the dual-wide map (D = 192, two 32-row halves: 96 registers): half 0
// in VGPRs, half 1 in AGPRs, each as a 32- and a 16-register operand.
struct U32DualWide {
  u32x32 lo;
  u32x16 hi;
  u32x32 alo;
  u32x16 ahi;
};
template <>
struct U32Vec<96> { typedef U32DualWide type; };

template <class V>
__device__ __forceinline__ void vset(V& v, int i, uint32_t x) { v[i] = x; }
__device__ __forceinline__ void vset(U32DualWide& v, int i, uint32_t x) {
  if (i < 32) v.lo[i] = x;
  else if (i < 48) v.hi[i - 32] = x;
  else if (i < 80) v.alo[i - 48] = x;
  else v.ahi[i - 80] = x;
}
template <int LO, int HI>
__device__ __forceinline__ void vset(U32Split<LO, HI>& v, int i, uint32_t x) {
  if (i < LO) v.lo[i] = x;
  else v.hi[i - LO] = x;
}

// One work item (a query tile of 32 * NW rows of one head, 64 * NW with two
// 32-row halves per wave, or a chunk of a text tile): Q to registers, the
// generated key loop over the item's plan entries with the K/V ring at LDS
// address lds0, the normalised O (or the text partial) and the LSE to memory.
// DW selects the dual-wide map of D = 192 (4 waves of 64 rows on the wide
// map's rings, 256-row tiles), HALF the half map of D = 64 and 128 (4 waves of
// 32 rows, 128-row tiles, two work-groups per CU).  KG = 2 (half map): two
// groups of 4 waves take the first and the second half of the entries, each
// with a ring of its own, and are merged by log-sum-exp through LDS.
template <int D, int NW, typename E, bool DW = false, bool HALF = false, int KG = 1>
__device__ __forceinline__ void stream_item(const AttnParams& p, const WorkItem& it, uint32_t lds0) {
  static_assert(((D == 128 || D == 96) && NW == 8) || (D == 64 && (NW == 8 || NW == 12 || NW == 4)) ||
                    ((D == 192 || D == 256) && NW == 4) || (D == 128 && NW == 4 && HALF),
                "the generated loops exist for D = 128 and 96 with 8 waves, D = 64 with 4, 8 or 12, "
                "D = 192 and 256 with 4 and D = 128 with 4 (the half map)");
  static_assert(!HALF || ((D == 64 || D == 128) && NW == 4), "the half map is D = 64 or 128 with 4 waves");
  static_assert(!DW || (D == 192 && NW == 4), "the dual-wide map is D = 192 with 4 waves");
  using Op = Ops<E>;
  constexpr bool kWide = NW == 4 && D >= 192;   // one wave per SIMD, O in AGPRs
  constexpr bool kRing2 = NW == 4 && D >= 128;  // K and V rings of two stages
  // 64 rows per wave (two 32-row halves): D = 64 with two work-groups per CU,
  // and the dual-wide map
  constexpr bool kDual = (NW == 4 && D == 64 && !HALF) || DW;
  constexpr int NR = kDual ? 2 : 1;             // 32-row halves per wave
  constexpr int BM = 32 * NR * NW;              // query rows per tile
  // LDS layout: D = 96 rows on the D = 128 pitch, D = 192 rows on the D = 256 pitch
  constexpr int DL = D == 96 ? 128 : D == 192 ? 256 : D;
  constexpr int RB = 2 * DL;              // bytes per K/V row in LDS
  constexpr int TILE = kBN * RB;          // one K or V block
  constexpr int NT = D / 32;
  constexpr int NQK = D / 16;

  const int lane = threadIdx.x & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = KG == 1 ? wave_id : wave_id % NW;   // row wave
  const int kg = KG == 1 ? 0 : wave_id / NW;           // key group
  const int h = lane >> 5;
  const int i32 = lane & 31;

  const int tile = it.tile, head = it.head, batch = it.batch;
  const bool text = it.text;
  const int hk = head / p.group;

  const char* qbase;
  char* obase;
  int64_t qrs, ors;
  int nrows;
  int64_t r0;
  float* lse;
  if (!text) {
    qbase = p.q + 2 * (batch * p.q_str[0] + head * p.q_str[2]);
    obase = p.o + 2 * (batch * p.o_str[0] + head * p.o_str[2]);
    qrs = 2 * p.q_str[1];
    ors = 2 * p.o_str[1];
    nrows = p.n_q;
    r0 = (int64_t)tile * BM;
    lse = p.lse ? p.lse + ((int64_t)batch * p.H + head) * p.n_q : nullptr;
    if (it.vhalf >= 0) video_partial_dst<D>(p, it, BM, r0, obase, ors, lse);
  } else {
    qbase = p.qt + 2 * (batch * p.qt_str[0] + head * p.qt_str[2]);
    obase = p.ot + 2 * (batch * p.ot_str[0] + head * p.ot_str[2]);
    qrs = 2 * p.qt_str[1];
    ors = 2 * p.ot_str[1];
    nrows = p.n_tq;
    r0 = (int64_t)(tile - p.n_vt) * BM;
    lse = p.lse_t ? p.lse_t + ((int64_t)batch * p.H + head) * p.n_tq : nullptr;
    if (p.text_chunks > 1) text_partial_dst<D>(p, it, obase, ors, lse);
  }
  const bool partial = (text && p.text_chunks > 1) || it.vhalf >= 0;
  int e0, e1;
  item_entries(p, it, e0, e1);
  const uint32_t lds_item = lds0;
  int ahead = 0;                       // blocks that group 0 takes more than this one
  if constexpr (KG == 2) {
    const int n0 = (e1 - e0 + 1) / 2;
    ahead = kg == 0 ? 0 : n0 - (e1 - e0 - n0);
    if (kg == 0) e1 = e0 + n0;
    else e0 += n0;
    lds0 += (uint32_t)(kg * 2 * (kRing2 ? 2 : kPPStages) * TILE);
  }
  const int n = e1 - e0;

  // Q fragments (B operand of S^T = K Q^T): row i32 of each 32-row half of
  // this wave, d = 16c + 8h .. +7 (two halves: half r at 4 NQK r ..).
  const int64_t my_row = r0 + 32 * NR * wave + i32;
  typename U32Vec<4 * NQK * NR>::type qv;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int64_t row = my_row + 32 * r;
    const int64_t qr = row < nrows ? row : (int64_t)nrows - 1;
    const char* qp = qbase + qr * qrs + 16 * h;
#pragma unroll
    for (int c = 0; c < NQK; ++c) {
      const u32x4 t = *reinterpret_cast<const u32x4*>(qp + 32 * c);
      vset(qv, 4 * NQK * r + 4 * c, t[0]);
      vset(qv, 4 * NQK * r + 4 * c + 1, t[1]);
      vset(qv, 4 * NQK * r + 4 * c + 2, t[2]);
      vset(qv, 4 * NQK * r + 4 * c + 3, t[3]);
    }
  }

  // LDS read offsets: K operand of k-step c (row i32, 16-byte chunk 2c + h,
  // swizzled); V^T operands of d-tile dt (rows rowA and rowA + 8, read with
  // ds_read_b64_tr_b16).  V tiles start at 4 * TILE.
  typename U32Vec<NQK>::type koff;
  typename U32Vec<2 * NT>::type voff;
  {
    const int sw_k = swz<DL>(i32 & 15);
#pragma unroll
    for (int c = 0; c < NQK; ++c) koff[c] = lds0 + i32 * RB + ((((2 * c + h) ^ sw_k)) << 4);
    const int g16 = lane & 15;
    const int rowA = 4 * h + (g16 >> 2);
    const int sw_a = swz<DL>(rowA), sw_b = swz<DL>(rowA + 8);
    const int dgrp = (lane >> 4) & 1;
#pragma unroll
    for (int dt = 0; dt < NT; ++dt) {
      const int chunk = 4 * dt + 2 * dgrp + ((lane & 3) >> 1);
      const int inb = (lane & 1) * 8;
      constexpr int VB = (kRing2 ? 2 : kPPStages) * TILE;   // V stages follow the K stages
      voff[dt] = lds0 + VB + rowA * RB + ((chunk ^ sw_a) << 4) + inb;
      voff[NT + dt] = lds0 + VB + (rowA + 8) * RB + ((chunk ^ sw_b) << 4) + inb;
    }
  }
  // Copy geometry: instruction ii of the wave's K (V) copies fills LDS KiB
  // 8*ii + cw of the block, cw = wave % 8, i.e. (D = 128) rows 32*ii + 4*cw +
  // lane/16 at physical chunk lane%16, the row & 15 of which does not depend
  // on ii, or (D = 64, 8 waves: one instruction) rows 8*cw + lane/8 at
  // physical chunk lane%8.  The dual map's 4 waves fill KiB 4*ii + cw (rows
  // 32*ii + 8*cw + lane/8: two instructions per tensor).  With 12 waves, waves
  // 8-11 repeat the copies of waves 0-3 (same bytes to the same LDS
  // addresses), so every wave runs the same loop.
  // Wide map (4 waves, 512-byte rows): copy ii of wave w fills LDS KiB
  // 4*ii + w of a block, rows 8*ii + 2*w + lane/32 at physical chunk lane%32;
  // rows 16*(ii >> 1) go in the copy's soffset, the rest in the lane offset,
  // whose swizzle depends on the parity of ii: one (row, chunk) pair each.
  // Chunks past a row's data (D = 96: 12-15, D = 192: 24-31) are copied from
  // the lane offset 0x7FFF0000 plus the block's soffset (the host keeps
  // sources below 2^31 bytes, so the sum stays below 2^32).  For a source
  // shorter than that offset the copy lies past the buffer's range and
  // writes zeros without touching memory; for a longer one it reads bytes of
  // the source into those chunks.  Either way no LDS read touches them.
  const int cw = wave & 7;
  typename U32Vec<kWide ? 4 : 2>::type dma;
  {
    constexpr int NCH = RB / 16;          // 16-byte chunks per row
    constexpr uint32_t NDATA = 2 * D / 16;   // chunks of a row that hold data
#pragma unroll
    for (int par = 0; par < (kWide ? 2 : 1); ++par) {
      const uint32_t row = kWide ? (uint32_t)(8 * par + 2 * cw + lane / NCH) : (uint32_t)(cw * (1024 / RB) + lane / NCH);
      const uint32_t chunk = (uint32_t)((lane % NCH) ^ swz<DL>((int)(row & 15)));
      dma[2 * par] = row;
      dma[2 * par + 1] = chunk >= NDATA ? 0x7FFF0000u : chunk * 16;
    }
  }
  // A operand of the row-sum MFMAs (16x16x32, when the loop computes row sums
  // on the matrix core): ones in lanes 0 and 32 (row 0, k-groups 0 and 2) and
  // lanes 20 and 52 (row 4, k-groups 1 and 3), zero elsewhere.
  u32x4 ones;
  {
    const uint32_t one = std::is_same<E, __bf16>::value ? 0x3f803f80u : 0x3c003c00u;
    const uint32_t x = (lane == 0 || lane == 20 || lane == 32 || lane == 52) ? one : 0u;
    ones = u32x4{x, x, x, x};
  }
  u32x4 misc;                        // tile row, 4*h, -inf, mask temp
  misc[0] = (uint32_t)(32 * NR * wave + i32);   // tile row (the dual map: of half 0; half 1 is 32 below)
  // the half map's tile may be the second half of a plan tile of 2 * BM rows
  if constexpr (HALF) misc[0] += text ? 0u : (uint32_t)(BM * (tile & p.plan_shift));
  misc[1] = (uint32_t)(4 * h);
  misc[2] = 0xff800000u;
  misc[3] = 0u;

  // Scalar operands: entries of the item, block count, scale; K/V bases of
  // both sources; row strides, source lengths, the wave's LDS copy base.
  const char* kb0 = p.k + 2 * (batch * p.k_str[0] + hk * p.k_str[2]);
  const char* vb0 = p.v + 2 * (batch * p.v_str[0] + hk * p.v_str[2]);
  const char* kb1 = p.n_x ? p.kx + 2 * (batch * p.kx_str[0] + hk * p.kx_str[2]) : kb0;
  const char* vb1 = p.n_x ? p.vx + 2 * (batch * p.vx_str[0] + hk * p.vx_str[2]) : vb0;
  auto lo32 = [](const void* ptr) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uint64_t)ptr); };
  auto hi32 = [](const void* ptr) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)ptr >> 32));
  };
  const uint2* ep = p.entries + e0;
  u32x4 sa;
  sa[0] = lo32(ep);
  sa[1] = hi32(ep);
  sa[2] = (uint32_t)__builtin_amdgcn_readfirstlane(n);
  sa[3] = __builtin_bit_cast(uint32_t, p.scale_log2);
  u32x8 sb;
  sb[0] = lo32(kb0);
  sb[1] = hi32(kb0);
  sb[2] = lo32(vb0);
  sb[3] = hi32(vb0);
  sb[4] = lo32(kb1);
  sb[5] = hi32(kb1);
  sb[6] = lo32(vb1);
  sb[7] = hi32(vb1);
  u32x8 sc;
  sc[0] = (uint32_t)(2 * p.k_str[1]);
  sc[1] = (uint32_t)(2 * p.v_str[1]);
  sc[2] = (uint32_t)(2 * p.kx_str[1]);
  sc[3] = (uint32_t)(2 * p.vx_str[1]);
  sc[4] = (uint32_t)p.n_k;
  sc[5] = (uint32_t)p.n_x;
  sc[6] = (uint32_t)wave;
  sc[7] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + 1024u * (uint32_t)cw));

  floatx16 o0 = floatx16{0}, o1 = floatx16{0}, o2 = floatx16{0}, o3 = floatx16{0};
  floatx16 o4 = floatx16{0}, o5 = floatx16{0}, o6 = floatx16{0}, o7 = floatx16{0};
  floatx16 o8 = floatx16{0}, o9 = floatx16{0}, o10 = floatx16{0}, o11 = floatx16{0};
  // running max (log2 units) and this lane's row sum; the dual map: (m0, m1, l0, l1)
  typename std::conditional<kDual, floatx4, floatx2>::type ml;
  if constexpr (kDual) ml = floatx4{-1e30f, -1e30f, 0.f, 0.f};
  else ml = floatx2{-1e30f, 0.f};

  if (n > 0) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 is written by the copies
    constexpr bool bf = std::is_same<E, __bf16>::value;
    if constexpr (HALF && D == 128 && bf) {
      asm volatile(LVSA_STREAM128W4H_LOOP_BF16
                   : LVSA_STREAM128W4H_OUTPUTS(o0, o1, o2, o3, ml, misc)
                   : LVSA_STREAM128W4H_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM128W4H_CLOBBERS);
    } else if constexpr (HALF && D == 128) {
      asm volatile(LVSA_STREAM128W4H_LOOP_F16
                   : LVSA_STREAM128W4H_OUTPUTS(o0, o1, o2, o3, ml, misc)
                   : LVSA_STREAM128W4H_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM128W4H_CLOBBERS);
    } else if constexpr (HALF && bf) {
      asm volatile(LVSA_STREAM64W4H_LOOP_BF16
                   : LVSA_STREAM64W4H_OUTPUTS(o0, o1, ml, misc)
                   : LVSA_STREAM64W4H_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64W4H_CLOBBERS);
    } else if constexpr (HALF) {
      asm volatile(LVSA_STREAM64W4H_LOOP_F16
                   : LVSA_STREAM64W4H_OUTPUTS(o0, o1, ml, misc)
                   : LVSA_STREAM64W4H_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64W4H_CLOBBERS);
    } else if constexpr (D == 128 && bf) {
      asm volatile(LVSA_STREAM128_LOOP_BF16
                   : LVSA_STREAM128_OUTPUTS(o0, o1, o2, o3, ml, misc)
                   : LVSA_STREAM128_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM128_CLOBBERS);
    } else if constexpr (D == 128) {
      asm volatile(LVSA_STREAM128_LOOP_F16
                   : LVSA_STREAM128_OUTPUTS(o0, o1, o2, o3, ml, misc)
                   : LVSA_STREAM128_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM128_CLOBBERS);
    } else if constexpr (D == 96 && bf) {
      asm volatile(LVSA_STREAM96_LOOP_BF16
                   : LVSA_STREAM96_OUTPUTS(o0, o1, o2, ml, misc)
                   : LVSA_STREAM96_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM96_CLOBBERS);
    } else if constexpr (D == 96) {
      asm volatile(LVSA_STREAM96_LOOP_F16
                   : LVSA_STREAM96_OUTPUTS(o0, o1, o2, ml, misc)
                   : LVSA_STREAM96_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM96_CLOBBERS);
    } else if constexpr (D == 256 && bf) {
      asm volatile(LVSA_STREAM256W4_LOOP_BF16
                   : LVSA_STREAM256W4_OUTPUTS(o0, o1, o2, o3, o4, o5, o6, o7, ml, misc)
                   : LVSA_STREAM256W4_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM256W4_CLOBBERS);
    } else if constexpr (D == 256) {
      asm volatile(LVSA_STREAM256W4_LOOP_F16
                   : LVSA_STREAM256W4_OUTPUTS(o0, o1, o2, o3, o4, o5, o6, o7, ml, misc)
                   : LVSA_STREAM256W4_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM256W4_CLOBBERS);
    } else if constexpr (DW && bf) {
      asm volatile(LVSA_STREAM192W4D_LOOP_BF16
                   : LVSA_STREAM192W4D_OUTPUTS(o0, o1, o2, o3, o4, o5, o6, o7, o8, o9, o10, o11, ml, misc)
                   : LVSA_STREAM192W4D_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM192W4D_CLOBBERS);
    } else if constexpr (DW) {
      asm volatile(LVSA_STREAM192W4D_LOOP_F16
                   : LVSA_STREAM192W4D_OUTPUTS(o0, o1, o2, o3, o4, o5, o6, o7, o8, o9, o10, o11, ml, misc)
                   : LVSA_STREAM192W4D_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM192W4D_CLOBBERS);
    } else if constexpr (D == 192 && bf) {
      asm volatile(LVSA_STREAM192W4_LOOP_BF16
                   : LVSA_STREAM192W4_OUTPUTS(o0, o1, o2, o3, o4, o5, ml, misc)
                   : LVSA_STREAM192W4_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM192W4_CLOBBERS);
    } else if constexpr (D == 192) {
      asm volatile(LVSA_STREAM192W4_LOOP_F16
                   : LVSA_STREAM192W4_OUTPUTS(o0, o1, o2, o3, o4, o5, ml, misc)
                   : LVSA_STREAM192W4_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM192W4_CLOBBERS);
    } else if constexpr (kDual && bf) {
      asm volatile(LVSA_STREAM64W4_LOOP_BF16
                   : LVSA_STREAM64W4_OUTPUTS(o0, o1, o2, o3, ml, misc)
                   : LVSA_STREAM64W4_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64W4_CLOBBERS);
    } else if constexpr (kDual) {
      asm volatile(LVSA_STREAM64W4_LOOP_F16
                   : LVSA_STREAM64W4_OUTPUTS(o0, o1, o2, o3, ml, misc)
                   : LVSA_STREAM64W4_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64W4_CLOBBERS);
    } else if constexpr (NW == 12 && bf) {
      asm volatile(LVSA_STREAM64W12_LOOP_BF16
                   : LVSA_STREAM64W12_OUTPUTS(o0, o1, ml, misc)
                   : LVSA_STREAM64W12_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64W12_CLOBBERS);
    } else if constexpr (NW == 12) {
      asm volatile(LVSA_STREAM64W12_LOOP_F16
                   : LVSA_STREAM64W12_OUTPUTS(o0, o1, ml, misc)
                   : LVSA_STREAM64W12_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64W12_CLOBBERS);
    } else if constexpr (bf) {
      asm volatile(LVSA_STREAM64_LOOP_BF16
                   : LVSA_STREAM64_OUTPUTS(o0, o1, ml, misc)
                   : LVSA_STREAM64_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64_CLOBBERS);
    } else {
      asm volatile(LVSA_STREAM64_LOOP_F16
                   : LVSA_STREAM64_OUTPUTS(o0, o1, ml, misc)
                   : LVSA_STREAM64_INPUTS(qv, koff, voff, dma, sa, sb, sc, ones)
                   : LVSA_STREAM64_CLOBBERS);
    }
#pragma clang diagnostic pop
  }
  if constexpr (KG == 2) {
    // The key loop passes a barrier per block, and one more before the drain
    // of a two-stage ring; a group of fewer blocks (one fewer at most) makes
    // up for the rest here.
    const int rest = ahead == 0 ? 0 : ahead + ((kRing2 && n == 0) ? 1 : 0);
    for (int b = 0; b < rest; ++b) wg_barrier();
    constexpr int W = 16 * NT + 2;     // registers a lane hands over
    auto* x = (__attribute__((address_space(3))) float*)lds_item + wave * W * 64 + lane;
    const float l_own = sum_halves(ml[1]);
    floatx16 own[4] = {o0, o1, o2, o3};
    __syncthreads();                   // both groups have left their rings
    if (kg == 1) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) x[(16 * t + i) * 64] = own[t][i];
      x[16 * NT * 64] = ml[0];
      x[(16 * NT + 1) * 64] = l_own;
    }
    __syncthreads();
    if (kg == 1) return;
    const float m1 = x[16 * NT * 64], l1 = x[(16 * NT + 1) * 64];
    const float m = vmax(ml[0], m1);
    const float a0 = __builtin_amdgcn_exp2f(ml[0] - m), a1 = __builtin_amdgcn_exp2f(m1 - m);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) own[t][i] = a0 * own[t][i] + a1 * x[(16 * t + i) * 64];
    o0 = own[0];
    o1 = own[1];
    o2 = own[2];
    o3 = own[3];
    ml[0] = m;
    // the epilogue adds both lane halves
    ml[1] = h == 0 ? a0 * l_own + a1 * l1 : 0.f;
  }

  // Epilogue, per 32-row half: combine the row sum of both lane halves,
  // normalise, store.
  const floatx16 oall[12] = {o0, o1, o2, o3, o4, o5, o6, o7, o8, o9, o10, o11};
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const floatx16* oacc = oall + NT * r;
    const int64_t row = my_row + 32 * r;
    const float m_run = ml[r];
    const float l_tot = sum_halves(ml[NR + r]);
    if (row < nrows && partial) {
      store_text_partial<NT>(obase + row * ors, lse + 2 * row, h, oacc, m_run, l_tot);
    } else if (row < nrows) {
      const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
      char* op = obase + row * ors;
#pragma unroll
      for (int dt = 0; dt < NT; ++dt) {
#pragma unroll
        for (int rq = 0; rq < 4; rq += 2) {
          // A lane holds d = 32 dt + 8 rq + 4 h .. + 3 and the same 8 further;
          // the two lanes of a row trade so that each stores 16 contiguous
          // bytes.  A small launch's tiles all store at once, so half as many
          // stores show: 24 x 130 + 37 text tokens 51.6 -> 50.0 us, 9 x 256
          // 31.9 -> 30.7, 33 x 256 142.4 -> 138.5 (12 heads, D = 128).  A
          // second trade (v_permlane16_swap) for 64 bytes per row was within
          // 0.3%.
          uint32_t a[2], b[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            a[k] = (uint32_t)Op::bits(oacc[dt][4 * rq + 2 * k] * inv) |
                   ((uint32_t)Op::bits(oacc[dt][4 * rq + 2 * k + 1] * inv) << 16);
            b[k] = (uint32_t)Op::bits(oacc[dt][4 * rq + 4 + 2 * k] * inv) |
                   ((uint32_t)Op::bits(oacc[dt][4 * rq + 5 + 2 * k] * inv) << 16);
            float fa = __builtin_bit_cast(float, a[k]), fb = __builtin_bit_cast(float, b[k]);
            swap_halves(fa, fb);
            a[k] = __builtin_bit_cast(uint32_t, fa);
            b[k] = __builtin_bit_cast(uint32_t, fb);
          }
          *reinterpret_cast<u32x4*>(op + 2 * (32 * dt + 8 * rq + 8 * h)) = u32x4{a[0], a[1], b[0], b[1]};
        }
      }
      if (lse && h == 0) {
        lse[row] = l_tot > 0.f ? (m_run + __log2f(l_tot)) * 0.69314718055994530942f : -INFINITY;
      }
    }
  }
}

// Without work queues, work-group b runs item map_work(b).  With them
// (p.queues), each of the p.grid work-groups takes items until every queue is
// empty (queue_next); thread 0 takes the item and the barrier hands it to the
// other waves.  The barrier after an item keeps the next item's first copies
// out of the LDS ring until every wave has left the key loop.  The dual map
// (D = 64, 4 waves) runs two work-groups per CU: 256 VGPRs per wave and a
// 64 KiB ring each; so does the half map.  DW: the dual-wide map of D = 192,
// HALF: the half map, KG: its key groups (stream_item).
template <int D, int NW, typename E, bool DW = false, bool HALF = false, int KG = 1>
__global__ __launch_bounds__(64 * NW * KG, (NW == 4 && D <= 128) ? 2 : 1) void attn_fwd_stream_kernel(AttnParams p) {
  // one K or V block (D = 96 on the D = 128 pitch, D = 192 on the D = 256 pitch)
  constexpr int TILE = kBN * 2 * (D == 96 ? 128 : D == 192 ? 256 : D);
  // K and V stages: four each, two each in the wide map (4 waves, D = 192 and
  // 256) and the half map of D = 128
  __shared__ __attribute__((aligned(1024))) char smem_raw[KG * 2 * ((NW == 4 && D >= 128) ? 2 : kPPStages) * TILE];
  __shared__ int next_item;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char*)smem_raw;
  int qx = 0, dry = 0;                    // thread 0: queue being drained, queues found empty
  if (p.queues && threadIdx.x == 0) qx = xcd_id();
  for (bool first = true;; first = false) {
    WorkItem it;
    if (p.queues) {
      if (threadIdx.x == 0) next_item = queue_next(p, qx, dry);
      __syncthreads();
      const int nx = __builtin_amdgcn_readfirstlane(next_item);
      if (nx < 0) break;
      it = queue_item(p, nx & (kXcds - 1), nx >> 3);
    } else {
      if (!first) break;
      it = map_work(p);
      if (it.tile < 0) break;
    }
    stream_item<D, NW, E, DW, HALF, KG>(p, it, lds0);   // one call site: one copy of the key loop
    __syncthreads();
  }
}

}  // namespace
}  // namespace lvsa
