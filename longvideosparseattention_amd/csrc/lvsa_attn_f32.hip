// fp32 attention for fp32 callers (gfx950).
//
// The reference's lvsa_sdpa computes in the caller's dtype
// (lvsa/sparse_attention.py:670, 689-704): an fp32 caller gets fp32 scores,
// softmax and P.V.  Two kernels walk the same block plan as the 16-bit ones
// (128-row tiles, 64-key blocks, the same mask descriptors):
//
// attn_fwd_f32_kernel   both contractions on v_mfma_f32_32x32x2_f32.  It runs
//   calls without the scratch of the other one.
//
// attn_fwd_split_kernel   every fp32 operand as a sum of two fp16 numbers
//   (x = hi + lo, each rounded to nearest: 22 bits of x, and x scaled by a
//   power of two so that neither leaves fp16's range), and each product as
//   hi hi + hi lo + lo hi on v_mfma_f32_32x32x16_f16 with fp32 accumulation.
//   The fp16 matrix rate is 16 times the fp32 one, so three such products
//   cost 3/16 of the fp32 MFMAs; and an MFMA adds 16 products per rounding of
//   the accumulator instead of 2, which is where the fp32 kernel loses most
//   of its accuracy, so the result is closer to the exact one (below).
//   split_f32_kernel splits K and V once per call into the scratch, in the
//   order in which the MFMAs read their operands, so the attention kernel
//   only copies them to LDS.  Q is split when a tile is loaded, P in the
//   softmax.  One power of two serves a block of K or V (a row of Q), so
//   numbers below 2^-16 of its largest lose bits one by one.  Tiles that meet
//   a block or row with more than a few of them (kSmallExp), infinity, a
//   non-finite result, an overflowing score or V blocks too far apart are
//   computed again by the fp32 loop, so such inputs give what they gave there.
//
// Error against float64 (relative 2-norm) on N(0, 1) inputs, split and fp32
// MFMAs: 3.9e-7 and 8.9e-7 at 9 x 256 tokens, 12 heads, D = 128; 1.2e-6 and
// 2.0e-6 at 13 x 1350 + 226 text tokens, 6 heads, D = 64.
#include "lvsa_attn_kernels.h"

namespace lvsa {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(4))) int32_t* const_i32;
typedef const __attribute__((address_space(4))) uint32_t* const_u32;

// The tile of a work item: its rows of Q and O, and its plan entries.
struct Tile {
  const char* qbase;
  char* obase;
  int64_t qrs, ors;
  int nrows;
  int64_t r0;
  float* lse;
  bool text, partial;
  int e0, e1;
};

template <int D>
__device__ __forceinline__ Tile f32_tile(const AttnParams& p, const WorkItem& it) {
  Tile t;
  t.text = it.text;
  if (!it.text) {
    t.qbase = p.q + 4 * (it.batch * p.q_str[0] + it.head * p.q_str[2]);
    t.obase = p.o + 4 * (it.batch * p.o_str[0] + it.head * p.o_str[2]);
    t.qrs = 4 * p.q_str[1];
    t.ors = 4 * p.o_str[1];
    t.nrows = p.n_q;
    t.r0 = (int64_t)it.tile * kBM;
    t.lse = p.lse ? p.lse + ((int64_t)it.batch * p.H + it.head) * p.n_q : nullptr;
    if (it.vhalf >= 0) video_partial_dst<D>(p, it, kBM, t.r0, t.obase, t.ors, t.lse);
  } else {
    t.qbase = p.qt + 4 * (it.batch * p.qt_str[0] + it.head * p.qt_str[2]);
    t.obase = p.ot + 4 * (it.batch * p.ot_str[0] + it.head * p.ot_str[2]);
    t.qrs = 4 * p.qt_str[1];
    t.ors = 4 * p.ot_str[1];
    t.nrows = p.n_tq;
    t.r0 = (int64_t)(it.tile - p.n_vt) * kBM;
    t.lse = p.lse_t ? p.lse_t + ((int64_t)it.batch * p.H + it.head) * p.n_tq : nullptr;
    if (p.text_chunks > 1) text_partial_dst<D>(p, it, t.obase, t.ors, t.lse);
  }
  t.partial = (it.text && p.text_chunks > 1) || it.vhalf >= 0;
  item_entries(p, it, t.e0, t.e1);
  return t;
}

// O (unnormalised), running max (log2 units) and row sum of this lane's row
// to memory: normalised with the LSE, or as the partial of a text chunk.
template <int NT>
__device__ __forceinline__ void store_f32(const Tile& t, int64_t my_row, int h, const floatx16* oacc, float m_run,
                                          float l_tot) {
  if (my_row >= t.nrows) return;
  if (t.partial) {
    store_text_partial<NT>(t.obase + my_row * t.ors, t.lse + 2 * my_row, h, oacc, m_run, l_tot);
    return;
  }
  const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
  char* op = t.obase + my_row * t.ors;
#pragma unroll
  for (int dt = 0; dt < NT; ++dt) {
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const int d0 = 32 * dt + 8 * rq + 4 * h;
      *reinterpret_cast<floatx4*>(op + 4 * d0) =
          floatx4{oacc[dt][4 * rq] * inv, oacc[dt][4 * rq + 1] * inv, oacc[dt][4 * rq + 2] * inv,
                  oacc[dt][4 * rq + 3] * inv};
    }
  }
  if (t.lse && h == 0) t.lse[my_row] = l_tot > 0.f ? (m_run + log2f(l_tot)) * 0.69314718055994530942f : -INFINITY;
}

// One tile on the fp32 MFMAs, by the first four of THREADS / 64 waves (the
// others help to stage K and V).  Exact online softmax: the running max moves
// with every block that raises it.  Per wave (32 query rows) and key block:
//   S^T = K Q^T   A = K[key][d] (lane l: key l%32 of a 32-key half, d from
//                 a float4 at 8g + 4(l/32)), B = Q (registers), the four
//                 components of the float4 as four k-steps;
//   O^T += V^T P^T  k-step c of key half kh pairs keys 32kh + 8(c/4) + c%4
//                 and +4 (lane halves), i.e. the keys whose P this lane
//                 already holds in accumulator register c: B = that register,
//                 A = V[key][32dt + l%32] (one LDS dword per lane).
// K and V blocks are staged through padded LDS rows (D + 4 floats) at ks and
// vs by plain vector loads, one barrier pair per block.
template <int D, int THREADS>
__device__ __forceinline__ void f32_item(const AttnParams& p, const WorkItem& it, const Tile& t, float* ks, float* vs,
                                         const uint32_t* relw) {
  constexpr int PITCH = D + 4;   // floats per LDS row
  constexpr int NG = D / 8;      // float4 pairs of S's contraction
  constexpr int NT = D / 32;     // 32-wide d tiles of O
  constexpr int C4 = D / 4;      // float4 per K/V row

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5;
  const int i32 = lane & 31;
  const int hk = it.head / p.group;
  const bool active = wave < kWaves;

  const char* kb0 = p.k + 4 * (it.batch * p.k_str[0] + hk * p.k_str[2]);
  const char* vb0 = p.v + 4 * (it.batch * p.v_str[0] + hk * p.v_str[2]);
  const char* kb1 = p.n_x ? p.kx + 4 * (it.batch * p.kx_str[0] + hk * p.kx_str[2]) : kb0;
  const char* vb1 = p.n_x ? p.vx + 4 * (it.batch * p.vx_str[0] + hk * p.vx_str[2]) : vb0;

  // Q of row i32: components d = 8g + 4h .. +3 in q[4g ..].
  const int64_t my_row = t.r0 + 32 * wave + i32;
  float q[D / 2];
  {
    const int64_t qr = my_row < t.nrows ? my_row : (int64_t)t.nrows - 1;
    const char* qp = t.qbase + qr * t.qrs + 16 * h;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(qp + 32 * g);
      q[4 * g] = x[0];
      q[4 * g + 1] = x[1];
      q[4 * g + 2] = x[2];
      q[4 * g + 3] = x[3];
    }
  }

  floatx16 oacc[NT];
#pragma unroll
  for (int dt = 0; dt < NT; ++dt) oacc[dt] = floatx16{0};
  float m_run = -1e30f;   // running max of s * scale * log2(e)
  float l_run = 0.f;      // this lane's share of the row sum
  const float cs = p.scale_log2;
  const int my_tile_row = 32 * wave + i32;

  for (int e = t.e0; e < t.e1; ++e) {
    const uint2 ent = p.entries[e];
    const uint32_t cx = ent.x, cy = ent.y;
    const bool extra = (cx >> 31) != 0;
    const int64_t nsrc = extra ? p.n_x : p.n_k;
    int64_t k0 = (int64_t)(cx & 0x7fffffffu) * kBN;
    if (k0 >= nsrc) k0 = 0;   // never produced by the plan; keeps every load in bounds
    const char* kb = extra ? kb1 : kb0;
    const char* vb = extra ? vb1 : vb0;
    const int64_t krs = 4 * (extra ? p.kx_str[1] : p.k_str[1]);
    const int64_t vrs = 4 * (extra ? p.vx_str[1] : p.v_str[1]);

    __syncthreads();   // the previous block's LDS reads are done
    for (int idx = tid; idx < kBN * C4; idx += THREADS) {
      const int row = idx / C4, c = idx - row * C4;
      int64_t key = k0 + row;
      key = key < nsrc ? key : nsrc - 1;   // rows past the source end are masked by the descriptor
      *reinterpret_cast<floatx4*>(&ks[row * PITCH + 4 * c]) = *reinterpret_cast<const floatx4*>(kb + key * krs + 16 * c);
      *reinterpret_cast<floatx4*>(&vs[row * PITCH + 4 * c]) = *reinterpret_cast<const floatx4*>(vb + key * vrs + 16 * c);
    }
    __syncthreads();
    if (!active) continue;

    floatx16 s0 = floatx16{0}, s1 = floatx16{0};
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const floatx4 a0 = *reinterpret_cast<const floatx4*>(&ks[i32 * PITCH + 8 * g + 4 * h]);
      const floatx4 a1 = *reinterpret_cast<const floatx4*>(&ks[(32 + i32) * PITCH + 8 * g + 4 * h]);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[c], q[4 * g + c], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[c], q[4 * g + c], s1, 0, 0, 0);
      }
    }

    if ((cy & 3u) != kKindNone) {
      const uint32_t keep = block_keep_bits(p, cx, cy, my_tile_row, my_row, t.nrows, h, relw);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s0[r] = keep_or_ninf(s0[r], keep, r);
        s1[r] = keep_or_ninf(s1[r], keep, r + 16);
      }
    }

    // Exact online softmax: the row max over both lanes of the row.
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fmaxf(s0[r], s1[r]));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx * cs);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int dt = 0; dt < NT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s0[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[r], cs, -m_run));
      s1[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s1[r], cs, -m_run));
      l_run += s0[r] + s1[r];
    }

#pragma unroll
    for (int dt = 0; dt < NT; ++dt) {
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const int key = 8 * (c >> 2) + 4 * h + (c & 3);
        const float a0 = vs[key * PITCH + 32 * dt + i32];
        const float a1 = vs[(32 + key) * PITCH + 32 * dt + i32];
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, s0[c], oacc[dt], 0, 0, 0);
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, s1[c], oacc[dt], 0, 0, 0);
      }
    }
  }
  if (active) store_f32<NT>(t, my_row, h, oacc, m_run, l_run + __shfl_xor(l_run, 32));
}

// LDS of one tile on the fp32 MFMAs: K and V rows.
template <int D>
constexpr int kF32Lds = 2 * kBN * (D + 4) * 4;

template <int D>
__global__ __launch_bounds__(kThreads, D <= 128 ? 2 : 1) void attn_fwd_f32_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) float lds[kF32Lds<D> / 4];
  __shared__ uint32_t relw[kBM * kRelPitch];
  const WorkItem it = map_work(p);
  if (it.tile < 0) return;
  const Tile t = f32_tile<D>(p, it);
  // published by the first block's barrier
  if (p.rel_lds && !it.text) load_rel_rows<kBM>(p, relw, t.r0, t.nrows, threadIdx.x, kThreads);
  f32_item<D, kThreads>(p, it, t, lds, lds + kBN * (D + 4), relw);
}

// ───────────────────────── split into two fp16 numbers ─────────────────────────
//
// Scratch: one slot per (batch, K/V head, key block of 64 rows, K or V), the
// blocks of the frame-structured source first and those of the extra rows
// after them.  A slot holds the hi and then the lo numbers of its block as
// D / 8 operand fragments of 1 KiB each (lane l reads 16 bytes at 16 l):
//   K: fragment half * (D / 16) + c, lane (i, h): key 32 half + i,
//      d = 16 c + 8 h .. + 7;
//   V: fragment st * (D / 32) + dt, lane (i, h): d = 32 dt + i, keys
//      16 st + 8 (j / 4) + 4 h + j % 4, j = 0 .. 7 (the keys whose P the lane
//      of row i already holds).
// After the slots, one int per slot: the block's exponent e, x = (hi + lo) 2^e
// with the largest |hi| in [2^14, 2^15] (kZeroBlock: all zero, kWideBlock: not
// for the split).  Rows past the source's end are zeros.
constexpr int kZeroBlock = INT32_MIN;
constexpr int kWideBlock = INT32_MIN + 1;
constexpr int kSplitExp = 14;     // exponent of the largest scaled number
// Scaled numbers from 2^-2 on keep 22 bits: lo's last bit is 2^-24 there.
// Smaller ones are off by up to 2^-25 whatever their size, which shows where a
// row or channel holds little else: an outlier in another row of the block
// (one that the tile's rows may not even attend) or in another channel.  Of
// N(0, 1) numbers 5 in 10^5 are that small.
constexpr int kSmallExp = -2;

__host__ __device__ constexpr int64_t split_slot_bytes(int D) { return 4LL * kBN * D; }

__device__ __forceinline__ float pow2i(int e) { return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23); }

// hi and lo of eight scaled numbers.
__device__ __forceinline__ void split8(const float* x, halfx8& hi, halfx8& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    hi[j] = (_Float16)x[j];
    lo[j] = (_Float16)(x[j] - (float)hi[j]);
  }
}

// The same of eight numbers times the power of two sc, a pair of them in four
// instructions: v_fma_mixlo and v_fma_mixhi each for hi and for lo.  The empty
// asm keeps the compiler from packed conversions, which leave the products to
// instructions of their own and form hi a second time for lo (seven).  The
// kernel's waves wait for issue half of the time (VALU 55% and MFMA 53% busy at
// 13 frames of 1350 tokens, 226 text tokens, 6 heads, D = 64): with the row max
// by v_maximum3, 966 -> 911 us there and 91.2 -> 87.7 at 9 x 256 tokens, 12
// heads, D = 128, bit for bit.
__device__ __forceinline__ void split8(const float* x, float sc, halfx8& hi, halfx8& lo) {
  auto keep = [](auto& y) __attribute__((always_inline)) { asm("" : "+v"(y)); };
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    _Float16 h0 = (_Float16)(x[j] * sc);
    keep(h0);
    halfx2 t = halfx2{h0, (_Float16)(x[j + 1] * sc)};
    keep(t);
    _Float16 l0 = (_Float16)__builtin_fmaf(x[j], sc, -(float)t[0]);
    keep(l0);
    hi[j] = t[0];
    hi[j + 1] = t[1];
    lo[j] = l0;
    lo[j + 1] = (_Float16)__builtin_fmaf(x[j + 1], sc, -(float)t[1]);
  }
}

// Exponent to scale a group of numbers by, from the largest of their |x| (0
// and infinity included: the latter stays infinite).  Bounded so that the
// scale and its inverse are normal numbers.
__device__ __forceinline__ int split_exponent(float amax) {
  const int e = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFF) - 127;
  return (e < -112 ? -112 : e) - kSplitExp;
}

// |x| as an integer in its order, zero as the largest: one v_lshl_add.
__device__ __forceinline__ uint32_t size_key(float x) { return (__builtin_bit_cast(uint32_t, x) << 1) - 1u; }
// Nonzero numbers to be scaled by 2^-e are small if their size_key is below this.
__device__ __forceinline__ uint32_t small_key(int e) { return size_key(ldexpf(1.f, e + kSmallExp)); }

// Too many small numbers in a share of a row or channel: more than two and
// more than a quarter of its `n` nonzero ones.
__device__ __forceinline__ bool mostly_small(int small, int n) { return small > 2 && 4 * small > n; }

// Whether a wave's part x of a block (lane (i, h): NF fragments of 8 numbers)
// holds rows or channels of mostly small numbers, or is mostly small as a
// whole.  The numbers j of a fragment over the 32 lanes i are one channel of a
// K block and one row of a V block; a lane's own numbers are one row of K
// (over all fragments, by_lane) and one channel of V in each fragment.  Run
// after the stores and only by waves with a small number (a tenth of them on
// N(0, 1) inputs), it adds 0.7 us to the 12.0 of 9 x 256 tokens, 12 heads, D =
// 128, and 0.8 to the 18.6 of 13 x 1350 + 226 tokens, 6 heads, D = 64.
template <int NF>
__device__ __forceinline__ bool wide_part(const float (&x)[NF][8], uint32_t below, float own_max, bool by_lane) {
  // two small numbers in all cannot be too many (the usual case)
  int few = 0;
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) few += size_key(x[i][j]) < below;
  if (__popcll(__ballot(few > 0)) <= 2 && !__ballot(few > 1) && __popcll(__ballot(own_max > 0.f)) > 8) return false;
  bool wide = false;
  int own = 0, own_small = 0, all = 0, all_small = 0;
#pragma unroll
  for (int i = 0; i < NF; ++i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool nz = x[i][j] != 0.f, sm = size_key(x[i][j]) < below;
      const uint64_t n = __ballot(nz), m = __ballot(sm);
      const int n0 = __popc((uint32_t)n), n1 = __popc((uint32_t)(n >> 32));
      const int m0 = __popc((uint32_t)m), m1 = __popc((uint32_t)(m >> 32));
      wide |= mostly_small(m0, n0) || mostly_small(m1, n1);
      all += n0 + n1;
      all_small += m0 + m1;
      own += nz;
      own_small += sm;
    }
    if (!by_lane || i == NF - 1) {
      wide |= mostly_small(own_small, own);
      own = own_small = 0;
    }
  }
  return wide || 4 * all_small > all;
}

// One slot.  HBM bound: reads the block once and writes as many bytes; the
// conversions are a few instructions per number.
template <int D>
__device__ __forceinline__ void split_slot(const AttnParams& p, int slot, float* wmax) {
  constexpr int NF = D / 32;      // fragments per wave
  constexpr int ND = D / 16, NT = D / 32;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = lane >> 5, i32 = lane & 31;
  const int nkc = (p.n_k + kBN - 1) / kBN, nbt = nkc + (p.n_x + kBN - 1) / kBN;
  const bool is_v = slot & 1;
  int r = slot >> 1;
  const int blk = r % nbt;
  r /= nbt;
  const int hk = r % p.Hkv, batch = r / p.Hkv;
  const bool extra = blk >= nkc;
  const int nsrc = extra ? p.n_x : p.n_k;
  const int k0 = (extra ? blk - nkc : blk) * kBN;
  const char* base = extra ? (is_v ? p.vx : p.kx) : (is_v ? p.v : p.k);
  const int64_t* str = extra ? (is_v ? p.vx_str : p.kx_str) : (is_v ? p.v_str : p.k_str);
  base += 4 * (batch * str[0] + hk * str[2]);
  const int64_t rs = 4 * str[1];

  float x[NF][8];
  float amax = 0.f;
  uint32_t least = ~0u;           // size_key of the smallest nonzero number
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const int f = wave * NF + i;
    if (!is_v) {
      const int key = k0 + 32 * (f / ND) + i32, d = 16 * (f % ND) + 8 * h;
      floatx4 a = floatx4{0.f, 0.f, 0.f, 0.f}, b = a;
      if (key < nsrc) {
        const char* src = base + key * rs + 4 * d;
        a = *reinterpret_cast<const floatx4*>(src);
        b = *reinterpret_cast<const floatx4*>(src + 16);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[i][j] = a[j];
        x[i][4 + j] = b[j];
      }
    } else {
      const int d = 32 * (f % NT) + i32;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = k0 + 16 * (f / NT) + 8 * (j >> 2) + 4 * h + (j & 3);
        x[i][j] = key < nsrc ? *reinterpret_cast<const float*>(base + key * rs + 4 * d) : 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      amax = fmaxf(amax, fabsf(x[i][j]));
      const uint32_t key = size_key(x[i][j]);
      least = least < key ? least : key;
    }
  }
  const float own_max = amax;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
  if (lane == 0) wmax[wave] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  const int e = split_exponent(amax);
  const float sc = pow2i(-e);
  char* dst = p.split + (int64_t)slot * split_slot_bytes(D) + lane * 16;
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = x[i][j] * sc;
    halfx8 hi, lo;
    split8(y, hi, lo);
    char* d = dst + (wave * NF + i) * 1024;
    *reinterpret_cast<halfx8*>(d) = hi;
    *reinterpret_cast<halfx8*>(d + (D / 8) * 1024) = lo;
  }
  // while the stores are under way
  const uint32_t below = small_key(e);
  bool wide = amax == INFINITY;   // the block's other numbers would be scaled to 0; a NaN spoils only its own
  if (__ballot(least < below)) wide |= wide_part<NF>(x, below, own_max, !is_v);
  wide = __syncthreads_or(wide);
  if (threadIdx.x == 0) p.split_exp[slot] = amax == 0.f ? kZeroBlock : wide ? kWideBlock : e;
}

template <int D>
__global__ __launch_bounds__(kThreads) void split_f32_kernel(AttnParams p) {
  __shared__ float wmax[kWaves];
  split_slot<D>(p, blockIdx.x, wmax);
}

// Whether a tile can list the block of a slot: it holds rows of a key frame in
// `seen` (a relation row), or extra rows, which every tile lists.
__device__ __forceinline__ bool slot_seen(const AttnParams& p, int slot, const uint32_t* seen) {
  const int nkc = (p.n_k + kBN - 1) / kBN, nbt = nkc + (p.n_x + kBN - 1) / kBN;
  const int blk = (slot >> 1) % nbt;
  if (blk >= nkc) return true;
  const uint32_t k0 = (uint32_t)blk * kBN, k1 = k0 + kBN < (uint32_t)p.n_k ? k0 + kBN : (uint32_t)p.n_k;
  const uint32_t f0 = p.kf0 + (p.ko + k0) / (uint32_t)p.C, f1 = p.kf0 + (p.ko + k1 - 1) / (uint32_t)p.C;
  bool any = false;
  for (uint32_t f = f0; f <= f1 && (f >> 5) < (uint32_t)p.words; ++f) any |= (seen[f >> 5] >> (f & 31)) & 1u;
  return any;
}

// The same for calls of fewer query rows than keys, which may attend few of
// them: only the blocks that a tile can list.  A work-group takes every
// gridDim-th slot and tests 256 of them at a time, a thread each.  One tile
// that attends 2 of 8,000 blocks (12 heads, D = 128) takes 25 us on the fp32
// MFMAs, 2,643 with every block split and 34 so; 6 of 800 blocks 62, 293 and
// 35; 16 tiles of 10 of 800 121, 307 and 95.
template <int D>
__global__ __launch_bounds__(kThreads) void split_seen_f32_kernel(AttnParams p) {
  __shared__ float wmax[kWaves];
  __shared__ uint32_t seen[kSeenWords];
  __shared__ uint64_t todo[kWaves];
  const int tid = threadIdx.x;
  for (int w = tid; w < p.words; w += kThreads) seen[w] = 0;
  __syncthreads();
  const int rows = (int)((p.qo + (uint32_t)(p.n_q - 1)) / (uint32_t)p.R) + 1;
  for (int i = tid; i < rows * p.words; i += kThreads) {
    const uint32_t x = p.rel[(int64_t)p.qf0 * p.words + i];
    if (x) atomicOr(&seen[i % p.words], x);
  }
  __syncthreads();
  for (int64_t s0 = blockIdx.x; s0 < p.split_slots; s0 += (int64_t)gridDim.x * kThreads) {
    const int64_t mine = s0 + (int64_t)gridDim.x * tid;
    const uint64_t on = __ballot(mine < p.split_slots && slot_seen(p, (int)mine, seen));
    if ((tid & 63) == 0) todo[tid >> 6] = on;
    __syncthreads();
    for (int w = 0; w < kWaves; ++w) {
      for (uint64_t m = todo[w]; m; m &= m - 1)
        split_slot<D>(p, (int)(s0 + (int64_t)gridDim.x * (64 * w + __builtin_ctzll(m))), wmax);
    }
    __syncthreads();   // `todo` has been read
  }
}

// KG groups of four waves take the tile's key blocks in turn (group g blocks
// g, g + KG, ...), each with K and V buffers of its own in LDS, and are merged
// by log-sum-exp through LDS at the end.
template <int D, int KG>
__global__ __launch_bounds__(kThreads * KG, D >= 192 ? 1 : KG == 2 ? 2 : D == 64 ? 3 : 2)
void attn_fwd_split_kernel(AttnParams p) {
  constexpr int ND = D / 16;                       // MFMA k-steps of S
  constexpr int NT = D / 32;                       // 32-wide d tiles of O
  constexpr int NFR = D / 8;                       // fragments of a block's hi (lo) numbers
  constexpr int TILE = 2 * NFR * 1024;             // bytes of one K or V block
  constexpr int NIW = TILE / 1024 / kWaves;        // 1 KiB copies per wave and block
  constexpr int LA = 3;                            // operands read this many MFMAs ahead
  constexpr int LDS = KG * 2 * TILE > kF32Lds<D> ? KG * 2 * TILE : kF32Lds<D>;
  static_assert(KG == 1 || (KG - 1) * kWaves * (NT * 16 + 3) * 256 <= LDS, "the merge must fit the buffers");
  __shared__ __attribute__((aligned(1024))) char smem_raw[LDS];
  __shared__ uint32_t relw[kBM * kRelPitch];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / kWaves, rw = wave % kWaves;   // key group, row wave
  const int h = lane >> 5;
  const int i32 = lane & 31;
  lds_char* ks = (lds_char*)smem_raw + kg * 2 * TILE;
  lds_char* vs = ks + TILE;

  const WorkItem it = map_work(p);
  if (it.tile < 0) return;
  const Tile t = f32_tile<D>(p, it);
  const int64_t my_row = t.r0 + 32 * rw + i32;
  const int my_tile_row = 32 * rw + i32;
  if (p.rel_lds && !t.text) load_rel_rows<kBM>(p, relw, t.r0, t.nrows, threadIdx.x, kThreads * KG);

  const int nkc = (p.n_k + kBN - 1) / kBN, nbt = nkc + (p.n_x + kBN - 1) / kBN;
  const int64_t slot0 = ((int64_t)it.batch * p.Hkv + it.head / p.group) * nbt;
  const const_u32 entries = (const_u32)(uintptr_t)p.entries;
  const const_i32 exps = (const_i32)(uintptr_t)p.split_exp;
  // slot of the K block of an entry (its V block is the next slot)
  auto slot_of = [&](uint32_t cx) __attribute__((always_inline)) {
    int b = (int)(cx & 0x7fffffffu) + ((cx >> 31) ? nkc : 0);
    if (b >= nbt) b = 0;   // never produced by the plan; keeps every copy in bounds
    return 2 * (slot0 + b);
  };
  auto copy = [&](int64_t slot, lds_char* dst) __attribute__((always_inline)) {
    const char* src = p.split + slot * split_slot_bytes(D) + rw * NIW * 1024;
#pragma unroll
    for (int i = 0; i < NIW; ++i) dma16_async(src + i * 1024, lane * 16, dst + (rw * NIW + i) * 1024);
  };
  auto frag = [&](const lds_char* b, int f) __attribute__((always_inline)) {
    return *reinterpret_cast<const __attribute__((address_space(3))) halfx8*>(b + f * 1024 + lane * 16);
  };

  int e = t.e0 + kg;
  uint2 ent = uint2{0, 0};
  int64_t slot = 0;
  if (e < t.e1) {
    ent = uint2{entries[2 * (int64_t)e], entries[2 * (int64_t)e + 1]};
    slot = slot_of(ent.x);
    copy(slot, ks);
  }

  // Q of row i32, scaled by the row's power of two: d = 16c + 8h .. + 7.
  halfx8 qh[ND], ql[ND];
  int eq;                       // Q = (hi + lo) 2^eq
  bool redo = false;            // the tile leaves the split's range
  {
    const int64_t qr = my_row < t.nrows ? my_row : (int64_t)t.nrows - 1;
    const char* qp = t.qbase + qr * t.qrs + 32 * h;
    float q[ND][8];
    float amax = 0.f;
    uint32_t least = ~0u;
#pragma unroll
    for (int c = 0; c < ND; ++c) {
      const floatx4 a = *reinterpret_cast<const floatx4*>(qp + 64 * c);
      const floatx4 b = *reinterpret_cast<const floatx4*>(qp + 64 * c + 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        q[c][j] = a[j];
        q[c][4 + j] = b[j];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        amax = fmaxf(amax, fabsf(q[c][j]));
        const uint32_t key = size_key(q[c][j]);
        least = least < key ? least : key;
      }
    }
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    eq = split_exponent(amax);
    const float sc = pow2i(-eq);
    const uint32_t below = small_key(eq);
    if (__ballot(least < below)) {
      int n = 0, small = 0;
#pragma unroll
      for (int c = 0; c < ND; ++c) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          n += q[c][j] != 0.f;
          small += size_key(q[c][j]) < below;
        }
      }
      n += __shfl_xor(n, 32);
      small += __shfl_xor(small, 32);
      redo = 4 * small > n;
    }
#pragma unroll
    for (int c = 0; c < ND; ++c) {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[c][j] *= sc;
      split8(q[c], qh[c], ql[c]);
    }
  }

  floatx16 oacc[NT];            // sum of P V 2^(kPExp - vexp)
#pragma unroll
  for (int dt = 0; dt < NT; ++dt) oacc[dt] = floatx16{0};
  float m_run = -1e30f;         // running max of s * scale * log2(e)
  float l_run = 0.f;            // this lane's share of the row sum
  constexpr int kNoV = -200;
  int vexp = kNoV;              // exponent of oacc (uniform): the largest of the V blocks so far
  // P is split times 2^12: the running max moves once a block's max exceeds
  // it by more than 3, so that stays within 2^15, and fp16 holds P's lo part
  // down to 2^-37 of the largest P.  (Scaled after the exponential: 12 added
  // to its argument would round the argument to 4 bits less.)
  constexpr int kPExp = 12;
  constexpr float kMaxLag = 3.f;
  // P of a V block 2^lag below the largest is split times 2^(12 - lag), so that
  // it adds to oacc at its scale.  A lag of 15 still leaves rows that attend
  // only such blocks closer to float64 than the fp32 loop does (20 x 192
  // tokens, D = 128: 3.8e-7 and 8.0e-7).
  constexpr int kMaxVLag = 15, kMaxRise = 64;

  const int rounds = (t.e1 - t.e0 + KG - 1) / KG;
  // Two groups run half a round apart (one barrier), so that on each SIMD one
  // wave's P V meets the other's scores and softmax.
  if constexpr (KG == 2) {
    if (kg == 1) __syncthreads();
  }
  for (int r = 0; r < rounds; ++r) {
    const bool have = e < t.e1;
    wait_vm0();
    __syncthreads();            // K has landed for every wave; V's buffer is free again
    halfx8 ph[4], pl[4];
    const int64_t cur = slot;
    if (have) {
      copy(cur + 1, vs);
      const uint2 now = ent;
      const int kexp = exps[cur], ve = exps[cur + 1];
      // S^T of both key halves: the small products (hi lo, lo hi) first, so
      // only the D / 16 hi hi MFMAs round at the size of S
      floatx16 s[2] = {floatx16{0}, floatx16{0}};
      __builtin_amdgcn_s_setprio(1);
      {
        halfx8 a[4 * ND];
        // operands 0 .. 4 ND - 1: (lo, hi) of both halves per k-step, then hi again (b)
        auto operand = [&](int i) __attribute__((always_inline)) {
          const int c = i >> 2, half = i & 1;
          return frag(ks, ((i & 2) ? 0 : NFR) + half * ND + c);
        };
        constexpr int NO = 4 * ND;
#pragma unroll
        for (int i = -LA; i < NO; ++i) {
          if (i + LA < NO) {
            a[i + LA] = operand(i + LA);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
          }
          if (i >= 0) {
            s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], (i & 2) ? ql[i >> 2] : qh[i >> 2], s[i & 1], 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
          }
        }
        halfx8 b[2 * ND];
#pragma unroll
        for (int i = -LA; i < 2 * ND; ++i) {
          if (i + LA < 2 * ND) {
            // D = 64 has the registers to keep K's hi operands (13 x 1350 +
            // 226 tokens, 6 heads: 907 -> 894 us)
            if constexpr (D == 64) {
              b[i + LA] = a[4 * ((i + LA) >> 1) + 2 + ((i + LA) & 1)];
            } else {
              b[i + LA] = frag(ks, ((i + LA) & 1) * ND + ((i + LA) >> 1));
              __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
          }
          if (i >= 0) {
            s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[i], qh[i >> 1], s[i & 1], 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          }
        }
      }
      __builtin_amdgcn_s_setprio(0);
      if ((now.y & 3u) != kKindNone) {
        const uint32_t keep = block_keep_bits(p, now.x, now.y, my_tile_row, my_row, t.nrows, h, relw);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[0][i] = keep_or_ninf(s[0][i], keep, i);
          s[1][i] = keep_or_ninf(s[1][i], keep, i + 16);
        }
      }
      float mc[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float m = vmax(vmax(s[0][4 * c], s[0][4 * c + 1]), s[0][4 * c + 2]);
        m = vmax(vmax(m, s[0][4 * c + 3]), s[1][4 * c]);
        m = vmax(vmax(m, s[1][4 * c + 1]), s[1][4 * c + 2]);
        mc[c] = vmax(m, s[1][4 * c + 3]);
      }
      float mx = vmax(vmax(vmax(mc[0], mc[1]), mc[2]), mc[3]);
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      // the fp32 loop takes the tile: no further blocks here
      if (kexp == kWideBlock || ve == kWideBlock) {
        redo = true;
        e = t.e1;
      }
      // An all-zero K block's scores are zero whatever the exponent.
      const int es = eq + (kexp <= kWideBlock ? 0 : kexp);
      const float cs = ldexpf(p.scale_log2, es);
      const float top = ldexpf(mx, es);       // the fp32 score
      redo |= top == INFINITY;                // overflows there, not here
      const float mxs = top * p.scale_log2;
      int lag = 0;              // V of this block is 2^-lag of oacc's scale
      float down = 1.f;         // what oacc is scaled by for this block's V
      if (ve > kWideBlock) {
        if (ve > vexp) {
          // further down, oacc would leave fp32's range itself
          redo |= vexp != kNoV && ve - vexp > kMaxRise;
          down = vexp - ve < -126 ? 0.f : pow2i(vexp - ve);
          vexp = ve;
        }
        lag = vexp - ve;
        if (lag > kMaxVLag) {
          redo = true;
          lag = kMaxVLag;
        }
      }
      if (__builtin_amdgcn_ballot_w64(mxs > m_run + kMaxLag) || down != 1.f) {
        const float m_new = fmaxf(m_run, mxs);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < NT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha * down;
        m_run = m_new;
      }
      const float ps = pow2i(kPExp - lag);
      float ls[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          x[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[st >> 1][8 * (st & 1) + j], cs, -m_run));
          ls[j & 3] = st == 0 && j < 4 ? x[j] : ls[j & 3] + x[j];
        }
        split8(x, ps, ph[st], pl[st]);
      }
      l_run += (ls[0] + ls[1]) + (ls[2] + ls[3]);
    }
    e += KG;
    const bool more = e < t.e1;
    if (more) {
      ent = uint2{entries[2 * (int64_t)e], entries[2 * (int64_t)e + 1]};
      slot = slot_of(ent.x);
    }
    wait_vm0();
    __syncthreads();            // V has landed for every wave; K's buffer is free again
    if (more) copy(slot, ks);
    if (have) {
      halfx8 vh[NFR], vl[NFR];
      constexpr int LP = 1;     // operand pairs read ahead of their three MFMAs
#pragma unroll
      for (int f = -LP; f < NFR; ++f) {
        if (f + LP < NFR) {
          vh[f + LP] = frag(vs, f + LP);
          vl[f + LP] = frag(vs, NFR + f + LP);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        if (f >= 0) {
          const int st = f / NT, dt = f % NT;
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl[f], ph[st], oacc[dt], 0, 0, 0);
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[f], pl[st], oacc[dt], 0, 0, 0);
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[f], ph[st], oacc[dt], 0, 0, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
        }
      }
    }
  }
  if constexpr (KG == 2) {
    if (kg == 0) __syncthreads();
  }

  // Merge the groups: m, l and O at their true scale.
  const float vscale = vexp < -126 ? 0.f : pow2i(vexp);   // -200: no V block but zeros
#pragma unroll
  for (int dt = 0; dt < NT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = oacc[dt][i] * pow2i(-kPExp) * vscale;
  float l_tot = l_run + __shfl_xor(l_run, 32);
  if constexpr (KG > 1) {
    auto* x = (__attribute__((address_space(3))) float*)smem_raw;
    constexpr int W = NT * 16 + 2;
    __syncthreads();            // the last block's LDS reads are done
    if (kg > 0) {
      auto* o = x + ((kg - 1) * kWaves + rw) * W * 64 + lane;
#pragma unroll
      for (int dt = 0; dt < NT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[(dt * 16 + i) * 64] = oacc[dt][i];
      o[NT * 16 * 64] = m_run;
      o[(NT * 16 + 1) * 64] = l_tot;
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int g = 1; g < KG; ++g) {
        const auto* o = x + ((g - 1) * kWaves + rw) * W * 64 + lane;
        const float m1 = o[NT * 16 * 64], l1 = o[(NT * 16 + 1) * 64];
        const float m_new = fmaxf(m_run, m1);
        const float a0 = __builtin_amdgcn_exp2f(m_run - m_new), a1 = __builtin_amdgcn_exp2f(m1 - m_new);
        l_tot = a0 * l_tot + a1 * l1;
        m_run = m_new;
#pragma unroll
        for (int dt = 0; dt < NT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[dt][i] = a0 * oacc[dt][i] + a1 * o[(dt * 16 + i) * 64];
      }
    }
  }
  // Anything non-finite: an input was, or a product left the range.  x - x is
  // 0 for finite x and NaN otherwise.
  float bad = l_tot - l_tot;
#pragma unroll
  for (int dt = 0; dt < NT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) bad += oacc[dt][i] - oacc[dt][i];
  redo |= kg == 0 && !(bad == 0.f);
  if (__builtin_expect(__syncthreads_or(redo), 0)) {
    float* f = (float*)smem_raw;
    f32_item<D, kThreads * KG>(p, it, t, f, f + kBN * (D + 4), relw);
    return;
  }
  if (kg == 0) store_f32<NT>(t, my_row, h, oacc, m_run, l_tot);
}

template <int D>
int launch_f32_d(const AttnParams& p, int cus, hipStream_t stream) {
  const dim3 grid(p.grid);
  if (!p.split) {
    hipLaunchKernelGGL(attn_fwd_f32_kernel<D>, grid, dim3(kThreads), 0, stream, p);
    return launch_status("lvsa_attn_fwd (fp32)");
  }
  if (p.split_seen) {
    const int groups = 8 * (cus > 0 ? cus : 1);
    hipLaunchKernelGGL(split_seen_f32_kernel<D>, dim3(p.split_slots < groups ? p.split_slots : groups), dim3(kThreads),
                       0, stream, p);
  } else {
    hipLaunchKernelGGL(split_f32_kernel<D>, dim3(p.split_slots), dim3(kThreads), 0, stream, p);
  }
  const int rc = launch_status("lvsa_attn_fwd (fp32 split)");
  if (rc != LVSA_OK) return rc;
  if constexpr (D <= 128) {
    if (p.total_work <= cus) {
      hipLaunchKernelGGL((attn_fwd_split_kernel<D, 2>), grid, dim3(2 * kThreads), 0, stream, p);
      return launch_status("lvsa_attn_fwd (fp32)");
    }
  }
  hipLaunchKernelGGL((attn_fwd_split_kernel<D, 1>), grid, dim3(kThreads), 0, stream, p);
  return launch_status("lvsa_attn_fwd (fp32)");
}

}  // namespace

int64_t f32_split_bytes(int64_t slots, int D) { return slots * (split_slot_bytes(D) + 4); }

int launch_f32(const AttnParams& p, int D, int cus, hipStream_t stream) {
  switch (D) {
    case 64: return launch_f32_d<64>(p, cus, stream);
    case 96: return launch_f32_d<96>(p, cus, stream);
    case 128: return launch_f32_d<128>(p, cus, stream);
    case 192: return launch_f32_d<192>(p, cus, stream);
    default: return launch_f32_d<256>(p, cus, stream);
  }
}

}  // namespace lvsa
