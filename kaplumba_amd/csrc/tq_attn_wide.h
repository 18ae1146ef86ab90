// Many query rows per kv head (prefill chunks, wide verify) outside the
// packed d = 128 causal case of tq_attn_tile.h: a partial kernel of the
// general path (tq_attn_general.h) on the matrix cores.  One body serves
//   packed MSE caches of any bit widths, plain f16 and plain bf16 caches,
//   head dims padded to 32 KS (keys) and 16 CT (values),
//   causal rows, ragged windows and array masks.
// A workgroup is 8 waves of 16 RT query rows of one kv head over one slab of
// its tokens.  Each SUB-token step decodes (or copies) K and V into LDS once,
// as MFMA operands, and every wave reads them from there.
//
// LDS holds one K and one V slot; a step has two phases, each closed by a
// barrier:
//   A  scores and softmax of step i from the K slot; V of step i into the V slot
//   B  O += P V of step i from the V slot; K of step i + 1 into the K slot
// so decode work always runs beside matrix products of the other slot.  The
// four lead waves decode first, the four trailing ones (their SIMD partners)
// last, so that one wave's decode meets the other's products.  Every thread
// loads the packed words (or 16-byte pieces) of its own units one whole step
// ahead, into registers; nothing is staged in between.
//
// What bounds it: matrix products, LDS reads (an operand is read once per
// 16 RT rows) and softmax add up at two waves per SIMD.  SUB is 64 where the
// slots fit, 32 at the widest packed heads.  RT is 2 up to KS = 4 and 1 beyond:
// packed queries and outputs take 8 RT (KS + CT/2) registers, 128 of 256 at KS = 4
// and 8.  (KS = 2 leaves room by that count, but packed kernels of RT 3 and 4 spill
// 16 to 308 bytes there.)  The compiler's totals: 200 (KS 2, one weight piece), 224
// (KS 8), 256 and 100 bytes of scratch (KS 4, two pieces), 214 (KS 4, plain bf16).
//
// Measured, append and attention of one layer, against the kernel that took
// the call before: 512 queries x 8192 tokens under a 4096-key boolean window,
// d = 128, 3 bits: 2815 -> 176 us (vector kernel); 2 x 500 queries x 4097
// tokens, d = 64, K3/V4: 243 -> 129 us, and 512 queries x 4096 tokens, d = 256,
// K4/V2, dense: 538 -> 152 us (attn_mfma_kernel: decodes per 16 or 4 rows);
// 512 queries x 8192 plain bf16 tokens, d = 128: 345 -> 168 us
// (attn_plain_kernel: reads K/V per 16 rows).  Partial kernels alone, in a trace:
// 163, 120, 120 and 167 us.
//
// Weight pieces WP.  1: f16 weights, as the other packed kernels.  More where
// the general vector kernel held weights in f32: f16 hi + lo (2; under a power
// of two that keeps the lo parts normal), bf16 hi + mid + lo (3); plain bf16
// layers always take hi + lo (2), as attn_plain_kernel.  Scores: packed keys
// K_hi Q_hi + K_hi Q_lo + K_lo Q_hi (f32-class); plain keys are exact in
// their type and so are the queries, which share it: one product.
//
// Masked tokens keep the other kernels' rules (-FLT_MAX scores, uniform rows
// where everything is masked); a block only walks the tokens that some row of
// it sees: up to the last causal limit, and between the first and last key
// that gen_mask_range_kernel found kept, its splits sharing that range evenly.
#pragma once

#include <type_traits>

#include "tq_attn_general.h"
#include "tq_attn_mfma.h"
#include "tq_attn_slots.h"
#include "tq_attn_small.h"

namespace tq {

enum WideSrc { kWidePacked = 0, kWideF16 = 1, kWideBf16 = 2 };

constexpr int kWideNW = 8;
constexpr int kWideThreads = 64 * kWideNW;

// The smallest built (key steps of 32, value blocks of 16) that holds the
// dims; false where none does.
inline bool wide_dims(int Dk, int Dv, int& ks, int& ct) {
  const int sizes[5][2] = {{2, 4}, {3, 6}, {4, 8}, {6, 8}, {8, 16}};
  for (const auto& z : sizes)
    if (Dk <= 32 * z[0] && Dv <= 16 * z[1]) {
      ks = z[0];
      ct = z[1];
      return true;
    }
  return false;
}

// 16-row tiles per wave and query rows per workgroup at ks key steps
constexpr int wide_rt(int ks) { return ks <= 4 ? 2 : 1; }
constexpr int wide_block_rows(int ks) { return 16 * wide_rt(ks) * kWideNW; }

template <int KS, int CT, int RT, int SRC, int WP>
struct WideShape {
  static constexpr bool PACKED = SRC == kWidePacked;
  static constexpr int DKP = 32 * KS;
  static constexpr int DVP = 16 * CT;
  static constexpr int SUB = PACKED && DKP + DVP > 256 ? 32 : 64;  // tokens per step
  static constexpr int H = SUB / 32;                               // 32-token halves per step
  static constexpr int PARTS = PACKED ? 2 : 1;                     // hi / lo operand parts
  static constexpr int ROWS = 16 * RT * kWideNW;                   // query rows per workgroup
  static constexpr int KROW = 2 * DKP + 16;   // bytes per key row (f16, padded)
  static constexpr int VCT = H * 1024 + 32;   // bytes per 16-column value block; + 32: blocks of one
                                              // token's row start in different banks
  static constexpr int KTAB = 0;
  static constexpr int VTAB = KTAB + (PACKED ? 16384 : 0);  // pair tables: up to 256 keys x 8 or 64 x 32 entries
  static constexpr int KHI = VTAB + (PACKED ? 16384 : 0);
  static constexpr int KLO = KHI + SUB * KROW;
  static constexpr int VHI = KHI + PARTS * SUB * KROW;
  static constexpr int VLO = VHI + CT * VCT;
  static constexpr int NRM = VHI + PARTS * CT * VCT;  // SUB key norms, SUB value norms
  static constexpr int RNG = NRM + (PACKED ? SUB * 8 : 0);
  static constexpr int BYTES = RNG + kWideNW * 8;
  static constexpr int KU = SUB * DKP / 8 / kWideThreads + (SUB * DKP / 8 % kWideThreads != 0);  // units of 8 coordinates per thread
  static constexpr int VU = SUB * DVP / 8 / kWideThreads + (SUB * DVP / 8 % kWideThreads != 0);
  static constexpr int RW = PACKED ? 2 : 4;  // registers per loaded unit
  static_assert(BYTES <= 160 * 1024, "wide kernel LDS");
  static_assert(KHI % 16 == 0 && VHI % 16 == 0 && VCT % 16 == 0 && NRM % 16 == 0, "16-byte LDS pieces");
  static_assert(SUB * DKP / 8 % 64 == 0 && SUB * DVP / 8 % 64 == 0, "whole waves of units");
};

// The general path kept f32 weights: more pieces, and array masks.
template <int SRC, int WP>
constexpr bool wide_general() {
  return WP == (SRC == kWideBf16 ? 3 : 2);
}

template <int SRC>
__device__ __forceinline__ f32x4_t mfma_wide(u32x4_t a, u32x4_t b, f32x4_t c) {
  typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
  if constexpr (SRC == kWideBf16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, a), __builtin_bit_cast(bf8_t, b), c, 0, 0, 0);
  else
    return mfma_f16(a, b, c);
}

// Eight mask bytes (nonzero = keep) of keys tok .. tok + 7 of one mask row:
// one 8-byte load where keys are adjacent, else one load per key; keys at or
// past n (the window's end) are not read and count as kept.
__device__ __forceinline__ uint2 wide_mask_bytes(const uint8_t* row, int64_t st, int tok, int n) {
  if (st == 1 && tok + 8 <= n) {
    uint2 v;
    __builtin_memcpy(&v, row + tok, 8);
    return v;
  }
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t k = tok + j < n ? (row[(tok + j) * st] != 0 ? 1u : 0u) : 1u;
    w[j >> 2] |= k << (8 * (j & 3));
  }
  return make_uint2(w[0], w[1]);
}

// Two halves of a plain value operand, those that are infinite or NaN as zeros.
template <int SRC>
__device__ __forceinline__ uint32_t wide_finite2(uint32_t x) {
  constexpr uint32_t ulp = SRC == kWideBf16 ? 0x00800080u : 0x04000400u;  // one exponent step
  const uint32_t m = ((x & 0x7fff7fffu) + ulp) & 0x80008000u;             // bit 15 where all exponent bits are set
  return x & ~(m | (m - (m >> 15)));
}

// z + 0 x of two halves: z, or NaN where a half is infinite or NaN.
template <int SRC>
__device__ __forceinline__ float wide_times0(uint32_t x, float z) {
  if constexpr (SRC == kWideBf16) {
    typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2_t, x), bf2_t{}, z, false);
  } else {
    typedef _Float16 f2_t __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f2_t, x), f2_t{}, z, false);
  }
}

template <int SRC>
__device__ __forceinline__ u32x4_t wide_finite(u32x4_t x) {
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = wide_finite2<SRC>(x[j]);
  return x;
}

// An additive mask entry in log2 units; finite entries stay finite.
__device__ __forceinline__ float wide_mask_add(const GenParams& p, int64_t off) {
  float m;
  if (p.mask_kind == TQ_MASK_ADD_F32)
    m = static_cast<const float*>(p.mask)[off];
  else if (p.mask_kind == TQ_MASK_ADD_F16)
    m = f16_bits_to_f32(static_cast<const uint16_t*>(p.mask)[off]);
  else
    m = bf16_bits_to_f32(static_cast<const uint16_t*>(p.mask)[off]);
  const float t = m * 1.4426950408889634f;
  return (t == -INFINITY && m != -INFINITY) ? -FLT_MAX : t;
}

// Scores grow by up to 2^kWideLazy past a row's reference maximum before it moves.
constexpr float kWideLazy = 7.f;
constexpr float kWideTop = 32768.f;  // bound of scaled weights, whole in f16

// Row state of the online softmax, one row per 16-lane column (lanes n + 16 g):
// m reference maximum (log2 units), l this lane's share of the sum, vsc the power
// of two that the weights p * n_t of packed values carry as f16 pieces (plain: p).
//
// Where the weights are f32-class (wide_general), vsc follows the row's own: it
// drops when one passes 2^15 under it and rises with the maximum (what O holds
// shrinks then).  A token of huge norm that the row masks or hardly weighs (a
// padded or corrupt one) so costs the others no bits; a scale by the norms lost
// all of them from 2^30 on.  One-piece weights keep the tuned kernels' rule, one
// scale for all rows, of the largest norm met (a scale a row: prefill of d = 64,
// which keeps every token of its window, 128.0 -> 131.4 us).
struct WideRow {
  float m, l, vsc;
};

__device__ __forceinline__ float wide_row_max(float x) {  // over the row's four lanes
  x = fmaxf(x, xor_lane<16>(x));
  const float2 h = halves(x);
  return fmaxf(h.x, h.y);
}

// The row meets scores of maximum rm (this lane's): moves m where it has to.
// Returns the factor of O.
template <bool PACKED>
__device__ __forceinline__ float wide_row_rise(WideRow& w, float rm) {
  const float r = wide_row_max(rm);
  const float mo = w.m;
  const float mn = r > mo + kWideLazy ? fmaxf(mo, r) : mo;
  const float am = mo == mn ? 1.f : (mo == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mo - mn));
  w.l *= am;
  w.m = mn;
  float f = am;
  if constexpr (PACKED) {
    if (am == 0.f) {  // nothing is held any more (so far only masked keys, or far below)
      w.vsc = 0x1p126f;
    } else if (am < 1.f) {  // the whole part of the shrinkage goes to vsc, up to 2^126
      int e = 0;
      frexpf(w.vsc, &e);
      const int up = min(static_cast<int>(mn - mo), 127 - e);
      w.vsc = ldexpf(w.vsc, up);
      f = ldexpf(am, up);
    }
  }
  return f;
}

// The row's weights (or norms) reach wm (this lane's): where that passes top under
// vsc, brings it to 2^WEXP.  Returns the factor of O.
template <int WEXP>
__device__ __forceinline__ float wide_row_drop(WideRow& w, float wm, float top) {
  const float x = wide_row_max(wm);
  float f = 1.f;
  if (x * w.vsc > top) {
    int e = 0;
    frexpf(x, &e);
    const float v = ldexpf(1.f, max(WEXP - e, -120));
    f = v / w.vsc;
    w.vsc = v;
  }
  return f;
}

// A lane's coordinates 32 s + 8 g .. + 7 of a rotated query row in f32 (src: its
// first), as hi and lo f16 parts under the row's scale, which is returned; a row
// that is not live, and steps past DkP, are zeros.
template <int KS>
__device__ __forceinline__ float wide_split_row(const float* src, int DkP, bool row_live, u32x4_t (&qh)[KS], u32x4_t (&ql)[KS]) {
  float v[KS][8];
  float mx = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const bool in = 32 * s < DkP;  // uniform: whole steps past the row are zero
    const float4 a = *reinterpret_cast<const float4*>(src + (in ? 32 * s : 0));
    const float4 c = *reinterpret_cast<const float4*>(src + (in ? 32 * s : 0) + 4);
    const bool live = in && row_live;
    v[s][0] = live ? a.x : 0.f, v[s][1] = live ? a.y : 0.f, v[s][2] = live ? a.z : 0.f, v[s][3] = live ? a.w : 0.f;
    v[s][4] = live ? c.x : 0.f, v[s][5] = live ? c.y : 0.f, v[s][6] = live ? c.z : 0.f, v[s][7] = live ? c.w : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[s][e]));
  }
  const float sq = f16_query_scale(wide_row_max(mx));
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t h0, l0, h1, l1;
      split_f16(v[s][2 * e] * sq, h0, l0);
      split_f16(v[s][2 * e + 1] * sq, h1, l1);
      qh[s][e] = h0 | (h1 << 16);
      ql[s][e] = l0 | (l1 << 16);
    }
  return sq;
}

// Pair tables of both codebooks: entry (a | b << bits) = (hi c_a | hi c_b << 16,
// lo c_a | lo c_b << 16) of the codebook scaled by a power of two (largest magnitude
// in [2^12, 2^13)), 2^esh bytes of copies each.  Called by all NT threads; TMP: 128
// bytes that nothing else uses.  Returns the keys' scale.
template <int NT, int KTAB, int VTAB, int TMP>
__device__ __forceinline__ float wide_pair_tables(unsigned char* lds, const GenParams& p, int kesh, int vesh, int tid, float& sv) {
  float* cbl = reinterpret_cast<float*>(lds + TMP);
  const int kb = p.kbits, vb = p.vbits;
  if (tid < (1 << kb)) cbl[tid] = p.kcb[tid];
  if (tid < (1 << vb)) cbl[16 + tid] = p.vcb[tid];
  lds_barrier();
  auto table = [&](const float* cb, int bits, int esh, int at) {
    float mx = 0.f;
    for (int i = 0; i < (1 << bits); ++i) mx = fmaxf(mx, fabsf(cb[i]));
    const float sc = f16_split_scale(mx);
    for (int e = tid; e < ((1 << (2 * bits + esh)) >> 3); e += NT) {
      const int key = e >> (esh - 3);
      uint32_t h0, l0, h1, l1;
      split_f16(cb[key & ((1 << bits) - 1)] * sc, h0, l0);
      split_f16(cb[key >> bits] * sc, h1, l1);
      *reinterpret_cast<uint2*>(lds + at + e * 8) = make_uint2(h0 | (h1 << 16), l0 | (l1 << 16));
    }
    return sc;
  };
  const float sk = table(cbl, kb, kesh, KTAB);
  sv = table(cbl + 16, vb, vesh, VTAB);
  lds_barrier();
  return sk;
}

template <int KS, int CT, int RT, int SRC, int WP>
__global__ __launch_bounds__(kWideThreads) void gen_wide_kernel(GenParams p, int n_blocks) {
  using S = WideShape<KS, CT, RT, SRC, WP>;
  constexpr bool PACKED = S::PACKED;
  constexpr bool GEN = wide_general<SRC, WP>();
  constexpr int SUB = S::SUB, H = S::H;
  constexpr float kLazy = kWideLazy;
  constexpr int kWExp = (SRC != kWideBf16 && WP > 1) ? (PACKED ? 4 : 8) : 0;  // the largest weights carry 2^kWExp
  __shared__ __align__(16) unsigned char lds[S::BYTES];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15;
  const int g = lane >> 4;
  // workgroup ids go to the 8 XCDs in turn: with a multiple of 8 (sequence,
  // kv head) pairs, pair h runs on XCD h % 8 (its K/V enter one L2 once)
  int pair, wi;
  {
    const int id = blockIdx.x;
    const int per = n_blocks * p.n_splits;
    if ((p.B * p.Hkv) % 8 == 0) {
      const int k = id >> 3;
      pair = (k / per) * 8 + (id & 7);
      wi = k % per;
    } else {
      pair = id / per;
      wi = id % per;
    }
  }
  const int split = wi % p.n_splits;
  const int rb = wi / p.n_splits;
  const int gk = pair % p.Hkv;
  const int b = pair / p.Hkv;
  const int RL = p.R * p.L;
  const int row_w0 = rb * S::ROWS + 16 * RT * wave;  // first kv-head row of this wave
  const bool wave_live = row_w0 < RL;
  const int64_t grp0 = (static_cast<int64_t>(b) * p.Hkv + gk) * p.n_rg;  // 8-row groups of this head

  int64_t start;
  int len;
  {
    int64_t end = p.seq_lens ? static_cast<int64_t>(p.seq_lens[b]) : p.T;
    end = end > p.T ? p.T : (end < 0 ? 0 : end);
    int64_t s0 = p.seq_starts ? static_cast<int64_t>(p.seq_starts[b]) : 0;
    s0 = s0 < 0 ? 0 : (s0 > end ? end : s0);
    start = s0;
    len = static_cast<int>(end - s0);
  }

  // ---- rows of this wave: causal limits, mask rows, the keys they see
  bool row_ok[RT];
  int lim[RT];        // causal: tokens t <= lim (relative to the window) are visible
  int64_t mrow[GEN ? RT : 1];
  int wlo = INT32_MAX, whi = 0, lim_min = INT32_MAX;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int rr_lane = row_w0 + 16 * rt + n;
    row_ok[rt] = rr_lane < RL;
    const int rr = row_ok[rt] ? rr_lane : 0;
    const int r = rr / p.L;
    const int l = rr - r * p.L;
    lim[rt] = p.causal ? len - p.L + l : INT32_MAX;
    int lo = 0, hi = p.causal && lim[rt] >= 0 && p.mask_kind == TQ_MASK_NONE ? lim[rt] + 1 : len;
    if constexpr (GEN) {
      mrow[rt] = b * p.m_sb + gk * p.m_sg + r * p.m_sr + l * p.m_sl + start * p.m_st;
      if (p.mrange) {
        const int2 mr = p.mrange[b * p.mr_sb + gk * p.mr_sg + r * p.mr_sr + l * p.mr_sl];
        lo = mr.x;
        hi = mr.y;
      }
    }
    if (row_ok[rt]) {
      lim_min = min(lim_min, lim[rt]);
      wlo = min(wlo, lo);
      whi = max(whi, hi);
    }
  }
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    lim_min = min(lim_min, __shfl_xor(lim_min, o, 64));
    wlo = min(wlo, __shfl_xor(wlo, o, 64));
    whi = max(whi, __shfl_xor(whi, o, 64));
  }
  lim_min = __builtin_amdgcn_readfirstlane(lim_min);
  wlo = __builtin_amdgcn_readfirstlane(wlo);
  whi = __builtin_amdgcn_readfirstlane(whi);
  int2* rng = reinterpret_cast<int2*>(lds + S::RNG);
  if (lane == 0) rng[wave] = make_int2(wlo, whi);
  __syncthreads();
  int blo = INT32_MAX, bhi = 0;
#pragma unroll
  for (int w = 0; w < kWideNW; ++w) {
    blo = min(blo, rng[w].x);
    bhi = max(bhi, rng[w].y);
  }
  bhi = min(bhi, len);
  blo = min(blo, bhi);
  blo = __builtin_amdgcn_readfirstlane(blo);
  bhi = __builtin_amdgcn_readfirstlane(bhi);
  // the block's tokens in n_splits even pieces of whole 32-token halves
  const int piece = ((bhi - blo + p.n_splits - 1) / p.n_splits + 31) / 32 * 32;
  const int64_t tb64 = blo + static_cast<int64_t>(split) * piece;
  if (tb64 >= bhi) {  // no tokens: a neutral partial per row (the merge skips it)
    for (int r = tid; r < S::ROWS; r += kWideThreads) {
      const int rr = rb * S::ROWS + r;
      if (rr >= RL) continue;
      float* pm = p.pml + ((grp0 + rr / 8) * p.n_splits + split) * 16 + (rr % 8) * 2;
      pm[0] = -INFINITY;
      pm[1] = 0.f;
    }
    return;
  }
  const int t_begin = static_cast<int>(tb64);
  const int t_end = min(bhi, t_begin + piece);
  const int ntiles = (t_end - t_begin + SUB - 1) / SUB;
  const int64_t rowbase = (static_cast<int64_t>(b) * p.Hkv + gk) * p.cap + start;

  // ---- loads of this thread's units: unit e = tid + 512 u covers 8
  // coordinates of token e / (dims / 8).  A token past the split's end reads
  // the last one instead (its score is masked below).
  const char* const kbase = static_cast<const char*>(p.k) + rowbase * (PACKED ? p.kpw * 4 : p.Dk * 2);
  const char* const vbase = static_cast<const char*>(p.v) + rowbase * (PACKED ? p.vpw * 4 : p.Dv * 2);
  const int kstride = PACKED ? p.kpw * 4 : p.Dk * 2;
  const int vstride = PACKED ? p.vpw * 4 : p.Dv * 2;
  const int kb = p.kbits, vb = p.vbits;
  uint32_t kreg[S::KU][S::RW], vreg[S::VU][S::RW];
  float nreg = 0.f;
  auto unit_load = [&](const char* base, int stride, int bits, int pw, int dim, int c8, int tok, uint32_t (&r)[S::RW]) {
    const char* row = base + static_cast<int64_t>(min(tok, t_end - 1)) * stride;
    if constexpr (PACKED) {
      // the unit's 8 * bits bits start in word w0 and end in w0 or w0 + 1
      // (3 bits); padding units stay inside the row
      const int w0 = min((8 * bits * c8) >> 5, pw - 1);
      const uint32_t* rw = reinterpret_cast<const uint32_t*>(row);
      r[0] = rw[w0];
      r[1] = rw[min(w0 + 1, pw - 1)];
    } else {
      uint4 x = make_uint4(0u, 0u, 0u, 0u);
      if (8 * c8 < dim) x = reinterpret_cast<const uint4*>(row)[c8];
      r[0] = x.x;
      r[1] = x.y;
      r[2] = x.z;
      r[3] = x.w;
    }
  };
  constexpr int KC8 = S::DKP / 8, VC8 = S::DVP / 8;
  auto load_k = [&](int i) {
    const int t0 = t_begin + i * SUB;
#pragma unroll
    for (int u = 0; u < S::KU; ++u) {
      const int e = tid + u * kWideThreads;
      if (e < SUB * KC8) unit_load(kbase, kstride, kb, p.kpw, p.Dk, e % KC8, t0 + e / KC8, kreg[u]);
    }
    if constexpr (PACKED) {
      if (tid < 2 * SUB) {  // key norms, then value norms
        const int64_t at = rowbase + min(t0 + (tid & (SUB - 1)), t_end - 1);
        nreg = load_norm(tid < SUB ? p.kn : p.vn, p.norm_dtype, at);
      }
    }
  };
  auto load_v = [&](int i) {
    const int t0 = t_begin + i * SUB;
#pragma unroll
    for (int u = 0; u < S::VU; ++u) {
      const int e = tid + u * kWideThreads;
      if (e < SUB * VC8) unit_load(vbase, vstride, vb, p.vpw, p.Dv, e % VC8, t0 + e / VC8, vreg[u]);
    }
  };
  load_k(0);
  load_v(0);

  // ---- query rows: lane (row n, g) holds coordinates 32 s + 8 g .. + 7.
  // Packed keys: hi and lo parts of q_rot * sq, sq a power of two that brings
  // the row's largest magnitude into [2^12, 2^13); from wide_qprep_kernel, or
  // (dense rotation) formed here from the f32 rows of the rotation kernel.
  u32x4_t qh[RT][KS], ql[PACKED ? RT : 1][PACKED ? KS : 1];
  float qmul[RT];  // MFMA units -> score units (log2)
  {
    const int64_t pair_row0 = static_cast<int64_t>(pair) * RL;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int rr = row_ok[rt] ? row_w0 + 16 * rt + n : 0;
      bool rows32 = false;
      if constexpr (PACKED) rows32 = p.q_rows32 != 0;
      if (rows32) {
        if constexpr (PACKED) {
          const float sq =
              wide_split_row<KS>(p.qrot + (pair_row0 + rr) * p.DkP + 8 * g, p.DkP, row_ok[rt], qh[rt], ql[rt]);
          qmul[rt] = sq;
        }
      } else {
        const u32x4_t* src = reinterpret_cast<const u32x4_t*>(p.qhl) + (pair_row0 + rr) * (4 * KS * S::PARTS) + g;
        const u32x4_t z = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          qh[rt][s] = src[4 * s];
          qh[rt][s] = row_ok[rt] ? qh[rt][s] : z;
          if constexpr (PACKED) {
            ql[rt][s] = src[4 * KS + 4 * s];
            ql[rt][s] = row_ok[rt] ? ql[rt][s] : z;
          }
        }
        qmul[rt] = PACKED ? p.qsq[pair_row0 + rr] : 1.4426950408889634f;
      }
    }
  }

  // ---- pair tables
  float sv = 1.f;
  const int kesh = kb == 4 ? 6 : 8, vesh = vb == 4 ? 6 : 8;  // log2 of an entry's bytes over its copies
  if constexpr (PACKED) {
    const float sk = wide_pair_tables<kWideThreads, S::KTAB, S::VTAB, S::KHI>(lds, p, kesh, vesh, tid, sv);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) qmul[rt] = 1.4426950408889634f / (sk * qmul[rt]);
  }
  const uint32_t ktab = S::KTAB + (lane & ((1 << (kesh - 3)) - 1)) * 8;
  const uint32_t vtab = S::VTAB + (lane & ((1 << (vesh - 3)) - 1)) * 8;

  // 8 coordinates of a unit as hi and lo parts (packed) or as stored
  auto unit_parts = [&](const uint32_t (&r)[S::RW], int bits, int c8, uint32_t tab, int esh, uint4& hi, uint4& lo) {
    if constexpr (PACKED) {
      const uint32_t x = __builtin_amdgcn_alignbit(r[1], r[0], (8 * bits * c8) & 31);
      const uint32_t kmask = (1u << (2 * bits)) - 1u;
      uint2 e[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) e[m] = lds_at<uint2>(lds, tab + (((x >> (2 * m * bits)) & kmask) << esh));
      hi = make_uint4(e[0].x, e[1].x, e[2].x, e[3].x);
      lo = make_uint4(e[0].y, e[1].y, e[2].y, e[3].y);
    } else {
      hi = make_uint4(r[0], r[1], r[2], r[3]);
    }
  };
  auto put_k = [&]() {
#pragma unroll
    for (int u = 0; u < S::KU; ++u) {
      const int e = tid + u * kWideThreads;
      if (e < SUB * KC8) {
        const int t = e / KC8, c8 = e % KC8;
        uint4 hi, lo;
        unit_parts(kreg[u], kb, c8, ktab, kesh, hi, lo);
        unsigned char* d = lds + S::KHI + ((t & ~31) + tile_kslot(t & 31)) * S::KROW + c8 * 16;
        *reinterpret_cast<uint4*>(d) = hi;
        if constexpr (PACKED) *reinterpret_cast<uint4*>(d + (S::KLO - S::KHI)) = lo;
      }
    }
    if constexpr (PACKED)
      if (tid < 2 * SUB) reinterpret_cast<float*>(lds + S::NRM)[tid] = nreg;
  };
  auto put_v = [&](auto careful, int i) {
#pragma unroll
    for (int u = 0; u < S::VU; ++u) {
      const int e = tid + u * kWideThreads;
      if (e < SUB * VC8) {
        const int t = e / VC8, c8 = e % VC8;
        uint4 hi, lo;
        unit_parts(vreg[u], vb, c8, vtab, vesh, hi, lo);
        if constexpr (careful)  // the split's last token again, at weight 0
          if (t_begin + i * SUB + t >= t_end) hi = make_uint4(0u, 0u, 0u, 0u);
        unsigned char* d = lds + S::VHI + (c8 >> 1) * S::VCT + (t >> 5) * 1024 + tile_vslot(t & 31) * 32 + (c8 & 1) * 16;
        *reinterpret_cast<uint4*>(d) = hi;
        if constexpr (PACKED) *reinterpret_cast<uint4*>(d + (S::VLO - S::VHI)) = lo;
      }
    }
  };

  f32x4_t O[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) O[rt][ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  WideRow row[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) row[rt] = WideRow{-INFINITY, 0.f, PACKED ? 0x1p126f : static_cast<float>(1 << kWExp)};

  constexpr float kOneTop = static_cast<float>(1 << kWExp);
  float vlim = 0.f;  // one-piece weights: norms up to here need no new scale

  const uint32_t ka = S::KHI + n * S::KROW + 16 * g;
  uint32_t vtr[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) vtr[h] = S::VHI + tile_vslot(8 * g + 4 * h + (n >> 2)) * 32 + (n & 3) * 8;
  typedef __attribute__((address_space(3))) unsigned char lds_u8;
  typedef short s16x4v __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4v lds_s16x4;
  lds_u8* const l3 = (lds_u8*)lds;
  auto read_tr = [&](uint32_t off) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(l3 + off)));
  };

  // S^T of half hf of the step in the K slot
  auto scores = [&](int hf, f32x4_t (&C)[RT][2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t at = ka + (32 * hf + 16 * h) * S::KROW;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) C[rt][h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4_t ah = lds_at<u32x4_t>(lds, at + 64 * s);
        if constexpr (PACKED) {
          const u32x4_t al = lds_at<u32x4_t>(lds, at + (S::KLO - S::KHI) + 64 * s);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            C[rt][h] = mfma_wide<SRC>(ah, qh[rt][s], C[rt][h]);
            C[rt][h] = mfma_wide<SRC>(ah, ql[rt][s], C[rt][h]);
            C[rt][h] = mfma_wide<SRC>(al, qh[rt][s], C[rt][h]);
          }
        } else {
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) C[rt][h] = mfma_wide<SRC>(ah, qh[rt][s], C[rt][h]);
        }
      }
    }
  };

  // O rows 4 g + k of this lane take the factor of row 4 g + k
  float fac[RT];
  bool pending = false;  // wave-uniform: fac applies between the step's halves
  auto rescale = [&](const float (&f)[RT]) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float ar[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) ar[k] = __shfl(f[rt], 4 * g + k, 64);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int k = 0; k < 4; ++k) O[rt][ct][k] *= ar[k];
    }
  };

  // softmax of half hf: tokens t0 + 8 g + j of this lane; the weights as A operands
  auto softmax = [&](int t0, int hf, const f32x4_t (&C)[RT][2], const uint2 (&mk)[RT], u32x4_t (&A)[RT][WP]) {
    float knv[8], vnv[8];
    float vm = 0.f;
    if constexpr (PACKED) {
      const float* kn = reinterpret_cast<const float*>(lds + S::NRM) + 32 * hf + 8 * g;
      *reinterpret_cast<float4*>(knv) = *reinterpret_cast<const float4*>(kn);
      *reinterpret_cast<float4*>(knv + 4) = *reinterpret_cast<const float4*>(kn + 4);
      *reinterpret_cast<float4*>(vnv) = *reinterpret_cast<const float4*>(kn + SUB);
      *reinterpret_cast<float4*>(vnv + 4) = *reinterpret_cast<const float4*>(kn + SUB + 4);
#pragma unroll
      for (int j = 0; j < 8; ++j) vm = fmaxf(vm, vnv[j]);
    }
    // y = n_t <q, c> in MFMA units of the row; x = y * qmul in log2 units
    float y[RT][8];
    bool grow = PACKED && !GEN && vm > vlim;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float ym = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        y[rt][j] = own_reg(C[rt][j >> 2][j & 3]);
        if constexpr (PACKED) y[rt][j] *= knv[j];
        ym = fmaxf(ym, y[rt][j]);
      }
      grow |= ym * qmul[rt] > row[rt].m + kLazy;
          }
    bool special = t0 + 32 > t_end || t0 + 31 > lim_min;  // wave-uniform
    if constexpr (GEN) {
      if (p.mask_kind == TQ_MASK_BOOL) {
        bool all = true;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) all &= mk[rt].x == 0x01010101u && mk[rt].y == 0x01010101u;
        special |= __any(all ? 0 : 1) != 0;
      } else if (p.mask_kind != TQ_MASK_NONE) {
        special = true;
      }
    }
    float pe[RT][8];
    bool moved = false;
    // the step's first half rescales O at once; its second half only after the
    // first half's products, which still carry the old scale
    auto scale_moved = [&]() {
      if (hf == 0)
        rescale(fac);
      else
        pending = true;
    };
    if (special || __any(grow ? 1 : 0)) {
      // slow path: masks, a new reference maximum
      float rm[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int j = 0; j < 8; ++j) y[rt][j] *= qmul[rt];
        if (special) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int tok = t0 + 8 * g + j;
            if (tok > lim[rt]) y[rt][j] = -FLT_MAX;
            if constexpr (GEN) {
              if (p.mask_kind == TQ_MASK_BOOL) {
                if ((((j < 4 ? mk[rt].x : mk[rt].y) >> (8 * (j & 3))) & 0xffu) == 0u) y[rt][j] = -FLT_MAX;
              } else if (p.mask_kind != TQ_MASK_NONE) {
                if (tok < t_end) y[rt][j] += wide_mask_add(p, mrow[rt] + tok * p.m_st);
              }
            }
            if (tok >= t_end) y[rt][j] = -INFINITY;
          }
        }
        rm[rt] = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) rm[rt] = fmaxf(rm[rt], y[rt][j]);
      }
      bool up = false;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) up |= rm[rt] > row[rt].m + kLazy;
      if constexpr (PACKED && !GEN) up |= vm > vlim;
      if (__any(up ? 1 : 0)) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) fac[rt] = wide_row_rise<PACKED && GEN>(row[rt], rm[rt]);
        if constexpr (PACKED && !GEN) {
          const float f = wide_row_drop<kWExp>(row[0], wave_max(vm), kOneTop);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            fac[rt] *= f;
            row[rt].vsc = row[0].vsc;
          }
          vlim = kOneTop / row[0].vsc;
        }
        if constexpr (PACKED && GEN)
          moved = true;
        else
          scale_moved();
      }
      // masked keys (-FLT_MAX) weigh 1 while their whole row is masked
      // (m = -FLT_MAX), else 0; keys past the end (-inf) always 0
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          pe[rt][j] = row[rt].m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(y[rt][j] - row[rt].m);
    } else {
      // every score within 2^7 of a finite reference maximum
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const float nm = -row[rt].m;
#pragma unroll
        for (int j = 0; j < 8; ++j) pe[rt][j] = __builtin_amdgcn_exp2f(__builtin_fmaf(y[rt][j], qmul[rt], nm));
      }
    }
    float vs[8];  // one scale for all rows: with n_t in one factor
#pragma unroll
    for (int j = 0; j < 8; ++j) vs[j] = PACKED && !GEN ? vnv[j] * row[0].vsc : row[0].vsc;
    if constexpr (PACKED && GEN) {
      // no weight passes 2^15 while the norms, times the 2^7 that a score may
      // stand above its reference, do not: one compare a row
      bool near = false;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) near |= vm * row[rt].vsc > kWideTop / 128.f;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          row[rt].l += pe[rt][j];
          pe[rt][j] *= vnv[j];
        }
      if (__any(near ? 1 : 0)) {
        float wm[RT];
        bool over = false;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          wm[rt] = 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) wm[rt] = fmaxf(wm[rt], pe[rt][j]);
          over |= wm[rt] * row[rt].vsc > kWideTop;
        }
        if (__any(over ? 1 : 0)) {
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            const float f = wide_row_drop<kWExp>(row[rt], wm[rt], kWideTop);
            fac[rt] = moved ? fac[rt] * f : f;
          }
          moved = true;
        }
      }
      if (moved) scale_moved();
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (!(PACKED && GEN)) row[rt].l += pe[rt][j];
        w[j] = pe[rt][j];
        if constexpr (PACKED || kWExp != 0) w[j] *= PACKED && GEN ? row[rt].vsc : vs[j];
        // in a register of its own: the product folded into the f16 conversion
        // rounds once, and the low part would belong to another high part
        if constexpr (WP > 1) w[j] = own_reg(w[j]);
      }
#pragma unroll
      for (int q = 0; q < WP; ++q) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (SRC == kWideBf16) {
            const uint32_t a = f32_to_bf16_bits(w[2 * j]), c = f32_to_bf16_bits(w[2 * j + 1]);
            A[rt][q][j] = a | (c << 16);
            if (q + 1 < WP) {
              w[2 * j] -= bf16_bits_to_f32(static_cast<uint16_t>(a));
              w[2 * j + 1] -= bf16_bits_to_f32(static_cast<uint16_t>(c));
            }
          } else {
            const uint32_t a = pack_f16x2(w[2 * j], w[2 * j + 1]);
            A[rt][q][j] = a;
            if (q + 1 < WP) {
              w[2 * j] -= f16_bits_to_f32(static_cast<uint16_t>(a));
              w[2 * j + 1] -= f16_bits_to_f32(static_cast<uint16_t>(a >> 16));
            }
          }
        }
      }
    }
  };

  // O += P V of half hf of the step in the V slot
  auto pv = [&](auto careful, int hf, const u32x4_t (&A)[RT][WP]) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const uint32_t off = ct * S::VCT + hf * 1024;
      const uint2 h0 = read_tr(vtr[0] + off);
      const uint2 h1 = read_tr(vtr[1] + off);
      const u32x4_t bh = {h0.x, h0.y, h1.x, h1.y};
      u32x4_t bf = bh;  // of the weights' low pieces
      if constexpr (careful) bf = wide_finite<SRC>(bh);
      if constexpr (PACKED) {
        const uint2 g0 = read_tr(vtr[0] + off + (S::VLO - S::VHI));
        const uint2 g1 = read_tr(vtr[1] + off + (S::VLO - S::VHI));
        const u32x4_t bl = {g0.x, g0.y, g1.x, g1.y};
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          O[rt][ct] = mfma_wide<SRC>(A[rt][0], bh, O[rt][ct]);
          O[rt][ct] = mfma_wide<SRC>(A[rt][0], bl, O[rt][ct]);
          if constexpr (WP > 1) O[rt][ct] = mfma_wide<SRC>(A[rt][1], bh, O[rt][ct]);
        }
      } else {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int q = 0; q < WP; ++q) O[rt][ct] = mfma_wide<SRC>(A[rt][q], q > 0 ? bf : bh, O[rt][ct]);
      }
    }
  };

  // ---- the walk over the split's tokens: K of step 0 in its slot, K of step 1 and
  // V of step 0 loading
  const bool lead = wave < kWideNW / 2;
  auto walk = [&](auto careful) __attribute__((always_inline)) {
    put_k();
    if (ntiles > 1) load_k(1);
    lds_barrier();
#pragma unroll 1
    for (int i = 0; i < ntiles; ++i) {
      const int t0 = t_begin + i * SUB;
      const bool act = wave_live && t0 < whi && t0 + SUB > wlo;  // some row of the wave sees a token
      u32x4_t A[H][RT][WP];
      if (lead) {
        put_v(careful, i);
        if (i + 1 < ntiles) load_v(i + 1);
      }
      if (act) {
#pragma unroll
        for (int hf = 0; hf < H; ++hf) {
          uint2 mk[RT];
          if constexpr (GEN) {
            if (p.mask_kind == TQ_MASK_BOOL) {
#pragma unroll
              for (int rt = 0; rt < RT; ++rt)
                mk[rt] = wide_mask_bytes(static_cast<const uint8_t*>(p.mask) + mrow[rt], p.m_st, t0 + 32 * hf + 8 * g, len);
            }
          }
          f32x4_t C[RT][2];
          scores(hf, C);
          softmax(t0 + 32 * hf, hf, C, mk, A[hf]);
        }
      }
      if (!lead) {
        put_v(careful, i);
        if (i + 1 < ntiles) load_v(i + 1);
      }
      lds_barrier();
      if (lead && i + 1 < ntiles) {
        put_k();
        if (i + 2 < ntiles) load_k(i + 2);
      }
      if (act) {
#pragma unroll
        for (int hf = 0; hf < H; ++hf) {
          if (hf > 0 && pending) {
            rescale(fac);
            pending = false;
          }
          pv(careful, hf, A[hf]);
        }
      }
      if (!lead && i + 1 < ntiles) {
        put_k();
        if (i + 2 < ntiles) load_k(i + 2);
      }
      lds_barrier();
    }
  };
  walk(std::false_type{});
  if constexpr (GEN && !PACKED) {
    // An infinite value times the weights' low pieces, which may be negative or 0,
    // is a NaN where its product with the weight itself (the vector kernel's) is
    // infinite.  A block with a NaN in its result walks its tokens once more, the
    // low pieces against finite values only; no other block pays for it.
    bool nan = false;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int k = 0; k < 4; ++k) nan |= O[rt][ct][k] != O[rt][ct][k];
    const bool any = __any(nan ? 1 : 0);
    if (lane == 0) rng[wave].x = any ? 1 : 0;  // (the ranges have been read)
    lds_barrier();
    int again = 0;
#pragma unroll
    for (int w = 0; w < kWideNW; ++w) again |= rng[w].x;
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(again) != 0, 0)) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        row[rt] = WideRow{-INFINITY, 0.f, static_cast<float>(1 << kWExp)};
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) O[rt][ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      load_k(0);
      load_v(0);
      walk(std::true_type{});
    }
  }
  // ---- partials: (o, m, l) per row, o = O / (vsc sv) (packed: in the rotated value basis)
  if (!wave_live) return;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float lr = row[rt].l + xor_lane<16>(row[rt].l);
    {
      const float2 h = halves(lr);
      lr = h.x + h.y;
    }
    const int rr = row_w0 + 16 * rt + n;
    if (g == 0 && row_ok[rt]) {
      float* pm = p.pml + ((grp0 + rr / 8) * p.n_splits + split) * 16 + (rr % 8) * 2;
      pm[0] = row[rt].m * 0.6931471805599453f;  // natural-log units
      pm[1] = lr;
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float osc = (PACKED && GEN ? __shfl(1.f / row[rt].vsc, 4 * g + k, 64) : 1.f / row[0].vsc) / sv;
      const int rr = row_w0 + 16 * rt + 4 * g + k;
      if (rr >= RL) continue;
      float* po = p.po + (((grp0 + rr / 8) * p.n_splits + split) * 8 + rr % 8) * static_cast<int64_t>(p.Dv);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        if (16 * ct + n < p.Dv) po[16 * ct + n] = O[rt][ct][k] * osc;
    }
}

}  // namespace tq
