// Few query rows per kv head (decode, verify, short chunks) outside the tuned
// kernels: a partial kernel of the general path (tq_attn_general.h) on the matrix
// cores, for head dims up to 256, packed MSE caches of any widths and plain f16 /
// bf16 caches, causal rows, ragged windows and array masks.
//
// A workgroup takes 16 query rows of one kv head and a slab of its tokens; each
// of its 8 waves walks every eighth 32-token sub-chunk alone, without barriers:
//   * keys straight into A operands: lane (token, g) looks the pair table up with
//     the 8 coordinates 32 s + 8 g of its token (or loads them, plain caches);
//   * values through a wave-private LDS tile of 64 columns, written as decoded
//     and read back transposed (ds_read_b64_tr_b16) as B operands;
//   * the words of the next sub-chunk load while this one is worked on.
// The waves' partials meet in LDS at the end.  Softmax, masks, weight pieces and
// query operands as in tq_attn_wide.h.  Bound by the vector work of the lookups
// (about 18 instructions per 8 coordinates) at two waves per SIMD; short caches
// by the launches around it.
//
// Measured, one attention call, GQA 4 over 8 kv heads, against the vector kernel
// (8 rows a workgroup, f32 multiply-adds): d = 96, 4 bits, 8 sequences x 6000
// tokens 112 -> 38 us, 16384 tokens 268 -> 64; one sequence x 1024 tokens 32 ->
// 19; plain bf16 d = 96 8 x 6000 154 -> 35; a 512-key window over 8 x 6000 tokens
// of d = 128 110 -> 22, d = 256 216 -> 41.  Packed keys of more than 128
// coordinates spill (48 bytes at KS 6, 576 at KS 8; plain KS 8 80 to 128).
#pragma once

#include "tq_attn_wide.h"

namespace tq {

constexpr int kNarrowRows = 16;  // query rows per workgroup

template <int KS, int CT, int SRC>
struct NarrowShape {
  static constexpr bool PACKED = SRC == kWidePacked;
  static constexpr int NW = 8;
  static constexpr int NT = 64 * NW;
  static constexpr int DVP = 16 * CT;
  static constexpr int PARTS = PACKED ? 2 : 1;
  static constexpr int CC = CT < 4 ? CT : 4;    // 16-column blocks of values in LDS at a time
  static constexpr int VCT = 1024 + 32;         // bytes per block (see WideShape)
  static constexpr int VBYTES = PARTS * CC * VCT;
  static constexpr int WAVE = VBYTES + (PACKED ? 256 : 0);  // one wave's tile and norms
  static constexpr int KTAB = 0;
  static constexpr int VTAB = KTAB + (PACKED ? 16384 : 0);
  static constexpr int TILE = VTAB + (PACKED ? 16384 : 0);
  static constexpr int LOOP = TILE + NW * WAVE;
  // after the loop: every wave's o [16][DVP] f32, then (m, l) [NW][16][2]
  static constexpr int OML = NW * 16 * DVP * 4;
  static constexpr int POST = OML + NW * 16 * 8;
  static constexpr int BYTES = LOOP > POST ? LOOP : POST;
  static constexpr int KU = 2 * KS;  // key units per lane: two 16-token tiles
  static constexpr int VU = CT;      // value units per lane: 32 tokens x 2 CT pieces / 64
  static constexpr int RW = PACKED ? 2 : 4;
  static_assert(BYTES <= 160 * 1024 && VCT % 16 == 0 && WAVE % 16 == 0, "narrow kernel LDS");
};

template <int KS, int CT, int SRC>
__global__ __launch_bounds__(512) void gen_narrow_kernel(GenParams p, int n_groups) {
  using S = NarrowShape<KS, CT, SRC>;
  constexpr bool PACKED = S::PACKED;
  constexpr int WP = SRC == kWideBf16 ? 3 : 2;
  constexpr float kLazy = kWideLazy;
  constexpr int kWExp = SRC != kWideBf16 ? 8 : 0;  // the largest weights carry 2^kWExp
  constexpr int SUB = 32;
  __shared__ __align__(16) unsigned char lds[S::BYTES];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15;
  const int g = lane >> 4;
  const int split = blockIdx.x % p.n_splits;
  const int rb = blockIdx.x / p.n_splits % n_groups;
  const int pair = blockIdx.x / (p.n_splits * n_groups);
  const int gk = pair % p.Hkv;
  const int b = pair / p.Hkv;
  const int RL = p.R * p.L;
  const int row0 = rb * kNarrowRows;
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
  // ---- rows (lane n: row row0 + n; every wave holds all of them)
  const bool row_ok = row0 + n < RL;
  const int rr = row_ok ? row0 + n : 0;
  const int rq = rr / p.L;
  const int lq = rr - rq * p.L;
  const int lim = p.causal ? len - p.L + lq : INT32_MAX;  // causal: tokens t <= lim are visible
  const int64_t mrow = b * p.m_sb + gk * p.m_sg + rq * p.m_sr + lq * p.m_sl + start * p.m_st;
  int lim_min = row_ok ? lim : INT32_MAX;
  int blo = INT32_MAX, bhi = 0;
  {
    int lo = 0, hi = p.causal && lim >= 0 && p.mask_kind == TQ_MASK_NONE ? lim + 1 : len;
    if (p.mrange) {
      const int2 mr = p.mrange[b * p.mr_sb + gk * p.mr_sg + rq * p.mr_sr + lq * p.mr_sl];
      lo = mr.x;
      hi = mr.y;
    }
    if (row_ok) {
      blo = lo;
      bhi = hi;
    }
  }
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    lim_min = min(lim_min, __shfl_xor(lim_min, o, 64));
    blo = min(blo, __shfl_xor(blo, o, 64));
    bhi = max(bhi, __shfl_xor(bhi, o, 64));
  }
  lim_min = __builtin_amdgcn_readfirstlane(lim_min);
  bhi = min(__builtin_amdgcn_readfirstlane(bhi), len);
  blo = min(__builtin_amdgcn_readfirstlane(blo), bhi);
  const int piece = ((bhi - blo + p.n_splits - 1) / p.n_splits + SUB - 1) / SUB * SUB;
  const int64_t tb64 = blo + static_cast<int64_t>(split) * piece;
  if (tb64 >= bhi) {  // no tokens: a neutral partial per row (the merge skips it)
    if (tid < kNarrowRows && row0 + tid < RL) {
      const int r = row0 + tid;
      float* pm = p.pml + ((grp0 + r / 8) * p.n_splits + split) * 16 + (r % 8) * 2;
      pm[0] = -INFINITY;
      pm[1] = 0.f;
    }
    return;
  }
  const int t_begin = static_cast<int>(tb64);
  const int t_end = min(bhi, t_begin + piece);
  const int nsub = (t_end - t_begin + SUB - 1) / SUB;
  const int64_t rowbase = (static_cast<int64_t>(b) * p.Hkv + gk) * p.cap + start;
  const char* const kbase = static_cast<const char*>(p.k) + rowbase * (PACKED ? p.kpw * 4 : p.Dk * 2);
  const char* const vbase = static_cast<const char*>(p.v) + rowbase * (PACKED ? p.vpw * 4 : p.Dv * 2);
  const int kstride = PACKED ? p.kpw * 4 : p.Dk * 2;
  const int vstride = PACKED ? p.vpw * 4 : p.Dv * 2;
  const int kb = p.kbits, vb = p.vbits;

  // ---- loads: the 8 coordinates c8 of a token as the words that hold them, or
  // as stored (zeros past the dim).  A token past the slab reads its last one.
  auto unit_load = [&](const char* base, int stride, int bits, int pw, int dim, int c8, int tok, uint32_t (&r)[S::RW]) {
    const char* row = base + static_cast<int64_t>(min(tok, t_end - 1)) * stride;
    if constexpr (PACKED) {
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
  // key tile h, lane row n: token 8 (n / 4) + 4 h + n % 4, so lane (row n, g) of
  // the scores ends with tokens 8 g .. 8 g + 7
  const int ktok = 8 * (n >> 2) + (n & 3);
  uint32_t kreg[S::KU][S::RW], vreg[S::VU][S::RW];
  float nreg = 0.f;
  // plain rows of more than 128 columns: values load after the scores of their own
  // sub-chunk, where the keys' registers are free (one ahead they spill)
  constexpr bool LATE_V = !PACKED && CT > 8;
  auto load_v = [&](int i) {
    const int t0 = t_begin + i * SUB;
    // value unit u: piece u of 64 lanes (token lane / 2, half lane % 2 of block u)
#pragma unroll
    for (int u = 0; u < S::VU; ++u) unit_load(vbase, vstride, vb, p.vpw, p.Dv, 2 * u + (lane & 1), t0 + (lane >> 1), vreg[u]);
  };
  auto load = [&](int i) {
    const int t0 = t_begin + i * SUB;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) unit_load(kbase, kstride, kb, p.kpw, p.Dk, 4 * s + g, t0 + ktok + 4 * h, kreg[2 * s + h]);
    if constexpr (PACKED) {
      const int64_t at = rowbase + min(t0 + (lane & 31), t_end - 1);
      nreg = load_norm(lane < 32 ? p.kn : p.vn, p.norm_dtype, at);
    }
    if constexpr (!LATE_V) load_v(i);
  };
  if (wave < nsub) load(wave);

  // ---- query rows as B operands (every wave the same): see gen_wide_kernel
  u32x4_t qh[KS], ql[PACKED ? KS : 1];
  float qmul = 1.4426950408889634f;  // MFMA units -> score units (log2)
  {
    const int64_t qrow = static_cast<int64_t>(pair) * RL + rr;
    if (PACKED && p.q_rows32) {
      float sq = 1.f;
      if constexpr (PACKED) sq = wide_split_row<KS>(p.qrot + qrow * p.DkP + 8 * g, p.DkP, row_ok, qh, ql);
      qmul = sq;
    } else {
      const u32x4_t* src = reinterpret_cast<const u32x4_t*>(p.qhl) + qrow * (4 * KS * S::PARTS) + g;
      const u32x4_t z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        qh[s] = src[4 * s];
        qh[s] = row_ok ? qh[s] : z;
        if constexpr (PACKED) {
          ql[s] = src[4 * KS + 4 * s];
          ql[s] = row_ok ? ql[s] : z;
        }
      }
      if constexpr (PACKED) qmul = p.qsq[qrow];
    }
  }

  // ---- pair tables (as gen_wide_kernel)
  float sv = 1.f;
  const int kesh = kb == 4 ? 6 : 8, vesh = vb == 4 ? 6 : 8;
  if constexpr (PACKED) {
    const float sk = wide_pair_tables<S::NT, S::KTAB, S::VTAB, S::TILE>(lds, p, kesh, vesh, tid, sv);
    qmul = 1.4426950408889634f / (sk * qmul);
  }
  const uint32_t ktab = S::KTAB + (lane & ((1 << (kesh - 3)) - 1)) * 8;
  const uint32_t vtab = S::VTAB + (lane & ((1 << (vesh - 3)) - 1)) * 8;
  auto unit_parts = [&](const uint32_t (&r)[S::RW], int bits, int c8, uint32_t tab, int esh, u32x4_t& hi, u32x4_t& lo) {
    if constexpr (PACKED) {
      const uint32_t x = __builtin_amdgcn_alignbit(r[1], r[0], (8 * bits * c8) & 31);
      const uint32_t kmask = (1u << (2 * bits)) - 1u;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const uint2 e = lds_at<uint2>(lds, tab + (((x >> (2 * m * bits)) & kmask) << esh));
        hi[m] = e.x;
        lo[m] = e.y;
      }
    } else {
      hi = u32x4_t{r[0], r[1], r[2], r[3]};
    }
  };

  f32x4_t O[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) O[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  WideRow row = {-INFINITY, 0.f, PACKED ? 0x1p126f : static_cast<float>(1 << kWExp)};
  unsigned char* const tile = lds + S::TILE + wave * S::WAVE;
  const uint32_t tile_off = S::TILE + wave * S::WAVE;
  uint32_t vtr[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) vtr[h] = tile_off + tile_vslot(8 * g + 4 * h + (n >> 2)) * 32 + (n & 3) * 8;
  typedef __attribute__((address_space(3))) unsigned char lds_u8;
  typedef short s16x4v __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4v lds_s16x4;
  lds_u8* const l3 = (lds_u8*)lds;
  auto read_tr = [&](uint32_t off) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(l3 + off)));
  };
  unsigned char* const vdst = tile + tile_vslot(lane >> 1) * 32 + (lane & 1) * 16;

#pragma unroll 1
  for (int i = wave; i < nsub; i += S::NW) {
    const int t0 = t_begin + i * SUB;
    uint2 mk = make_uint2(0x01010101u, 0x01010101u);
    if (p.mask_kind == TQ_MASK_BOOL)
      mk = wide_mask_bytes(static_cast<const uint8_t*>(p.mask) + mrow, p.m_st, t0 + 8 * g, len);
    float knv[8], vnv[8];
    if constexpr (PACKED) {
      float* nt = reinterpret_cast<float*>(tile + S::VBYTES);
      nt[lane] = nreg;
      wave_sync();
      *reinterpret_cast<float4*>(knv) = *reinterpret_cast<const float4*>(nt + 8 * g);
      *reinterpret_cast<float4*>(knv + 4) = *reinterpret_cast<const float4*>(nt + 8 * g + 4);
      *reinterpret_cast<float4*>(vnv) = *reinterpret_cast<const float4*>(nt + 32 + 8 * g);
      *reinterpret_cast<float4*>(vnv + 4) = *reinterpret_cast<const float4*>(nt + 32 + 8 * g + 4);
    }
    // ---- scores S^T = K Q^T, tiles h of 16 tokens
    f32x4_t C[2];
    C[0] = C[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4_t ah, al;
        unit_parts(kreg[2 * s + h], kb, 4 * s + g, ktab, kesh, ah, al);
        C[h] = mfma_wide<SRC>(ah, qh[s], C[h]);
        if constexpr (PACKED) {
          C[h] = mfma_wide<SRC>(ah, ql[s], C[h]);
          C[h] = mfma_wide<SRC>(al, qh[s], C[h]);
        }
      }
    if constexpr (LATE_V) load_v(i);
    // ---- softmax: tokens t0 + 8 g + j of this lane's row
    float y[8];
    float ym = -INFINITY;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      y[j] = own_reg(C[j >> 2][j & 3]);
      if constexpr (PACKED) y[j] *= knv[j];
      y[j] *= qmul;
      ym = fmaxf(ym, y[j]);
    }
    const bool special = t0 + SUB > t_end || t0 + SUB - 1 > lim_min || p.mask_kind != TQ_MASK_NONE;  // wave-uniform
    if (special) {
      ym = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int tok = t0 + 8 * g + j;
        if (tok > lim) y[j] = -FLT_MAX;
        if (p.mask_kind == TQ_MASK_BOOL) {
          if ((((j < 4 ? mk.x : mk.y) >> (8 * (j & 3))) & 0xffu) == 0u) y[j] = -FLT_MAX;
        } else if (p.mask_kind != TQ_MASK_NONE) {
          if (tok < t_end) y[j] += wide_mask_add(p, mrow + tok * p.m_st);
        }
        if (tok >= t_end) y[j] = -INFINITY;
        ym = fmaxf(ym, y[j]);
      }
    }
    float fo = 1.f;  // factor of the row's O
    bool moved = __any(ym > row.m + kLazy ? 1 : 0);
    if (moved) fo = wide_row_rise<PACKED>(row, ym);
    float w[8];
    float wm = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float pe = row.m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(y[j] - row.m);
      row.l += pe;
      w[j] = PACKED ? pe * vnv[j] : pe;
      wm = fmaxf(wm, w[j]);
    }
    if constexpr (PACKED) {
      if (__any(wm * row.vsc > kWideTop ? 1 : 0)) {
        fo *= wide_row_drop<kWExp>(row, wm, kWideTop);
        moved = true;
      }
    }
    if (moved) {
      float ar[4];  // O rows 4 g + k of this lane take the factor of row 4 g + k
#pragma unroll
      for (int k = 0; k < 4; ++k) ar[k] = __shfl(fo, 4 * g + k, 64);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int k = 0; k < 4; ++k) O[ct][k] *= ar[k];
    }
    u32x4_t A[WP];
    {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        // in a register of its own: the product folded into the f16 conversion
        // rounds once, and the low part would belong to another high part
        w[j] = own_reg(w[j] * row.vsc);
      }
#pragma unroll
      for (int q = 0; q < WP; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (SRC == kWideBf16) {
            const uint32_t a = f32_to_bf16_bits(w[2 * j]), c = f32_to_bf16_bits(w[2 * j + 1]);
            A[q][j] = a | (c << 16);
            w[2 * j] -= bf16_bits_to_f32(static_cast<uint16_t>(a));
            w[2 * j + 1] -= bf16_bits_to_f32(static_cast<uint16_t>(c));
          } else {
            const uint32_t a = pack_f16x2(w[2 * j], w[2 * j + 1]);
            A[q][j] = a;
            w[2 * j] -= f16_bits_to_f32(static_cast<uint16_t>(a));
            w[2 * j + 1] -= f16_bits_to_f32(static_cast<uint16_t>(a >> 16));
          }
        }
    }
    // ---- O += P V, CC blocks of 16 columns at a time through the wave's tile.
    // Infinite values (and NaN) meet the weight itself only, as in gen_wide_kernel:
    // a sub-chunk that holds any gives its low pieces finite values.
    bool careful = false;
    if constexpr (!PACKED) {
      float z = 0.f;  // NaN from the first infinity or NaN on
#pragma unroll
      for (int u = 0; u < S::VU; ++u)
#pragma unroll
        for (int w = 0; w < 4; ++w) z = wide_times0<SRC>(vreg[u][w], z);
      careful = __any(z != z ? 1 : 0);
    }
#pragma unroll
    for (int c0 = 0; c0 < CT; c0 += S::CC) {
      wave_sync();  // the tile's last readers are behind
#pragma unroll
      for (int c = 0; c < S::CC; ++c) {
        if (c0 + c >= CT) continue;
        u32x4_t hi, lo;
        unit_parts(vreg[c0 + c], vb, 2 * (c0 + c) + (lane & 1), vtab, vesh, hi, lo);
        if constexpr (!PACKED)  // the slab's last token again, at weight 0
          if (careful && t0 + (lane >> 1) >= t_end) hi = u32x4_t{0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4_t*>(vdst + c * S::VCT) = hi;
        if constexpr (PACKED) *reinterpret_cast<u32x4_t*>(vdst + (S::CC + c) * S::VCT) = lo;
      }
      if (c0 + S::CC >= CT && i + S::NW < nsub) load(i + S::NW);  // registers are free from here on
      wave_sync();
#pragma unroll
      for (int c = 0; c < S::CC; ++c) {
        if (c0 + c >= CT) continue;
        const uint2 h0 = read_tr(vtr[0] + c * S::VCT);
        const uint2 h1 = read_tr(vtr[1] + c * S::VCT);
        const u32x4_t bh = {h0.x, h0.y, h1.x, h1.y};
        u32x4_t bf = bh;  // of the weights' low pieces
        if constexpr (!PACKED)
          if (careful) bf = wide_finite<SRC>(bh);
        if constexpr (PACKED) {
          const uint2 g0 = read_tr(vtr[0] + (S::CC + c) * S::VCT);
          const uint2 g1 = read_tr(vtr[1] + (S::CC + c) * S::VCT);
          const u32x4_t bl = {g0.x, g0.y, g1.x, g1.y};
          O[c0 + c] = mfma_wide<SRC>(A[0], bh, O[c0 + c]);
          O[c0 + c] = mfma_wide<SRC>(A[0], bl, O[c0 + c]);
          O[c0 + c] = mfma_wide<SRC>(A[1], bh, O[c0 + c]);
        } else {
#pragma unroll
          for (int q = 0; q < WP; ++q) O[c0 + c] = mfma_wide<SRC>(A[q], q > 0 ? bf : bh, O[c0 + c]);
        }
      }
    }
  }

  // ---- the waves' partials meet in LDS: o scaled to the value basis, (m, l)
  float lr = row.l + xor_lane<16>(row.l);
  {
    const float2 h = halves(lr);
    lr = h.x + h.y;
  }
  float osc[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) osc[k] = __shfl(1.f / row.vsc, 4 * g + k, 64) / sv;
  __syncthreads();
  float* s_o = reinterpret_cast<float*>(lds) + wave * 16 * S::DVP;
  float2* s_ml = reinterpret_cast<float2*>(lds + S::OML);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int k = 0; k < 4; ++k) s_o[(4 * g + k) * S::DVP + 16 * ct + n] = O[ct][k] * osc[k];
  if (g == 0) s_ml[wave * 16 + n] = make_float2(row.m, lr);
  __syncthreads();
  const int rows = min(kNarrowRows, RL - row0);
  for (int e = tid; e < rows * S::DVP; e += S::NT) {
    const int r = e / S::DVP;
    const int d = e % S::DVP;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < S::NW; ++w) mx = fmaxf(mx, s_ml[w * 16 + r].x);
    float o = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < S::NW; ++w) {
      const float2 ml = s_ml[w * 16 + r];
      const float f = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - mx);
      l += f * ml.y;
      o += f * reinterpret_cast<const float*>(lds)[(w * 16 + r) * S::DVP + d];
    }
    const int row = row0 + r;
    const int64_t at = (grp0 + row / 8) * p.n_splits + split;
    if (d < p.Dv) p.po[(at * 8 + row % 8) * p.Dv + d] = o;
    if (d == 0) {
      float* pm = p.pml + at * 16 + (row % 8) * 2;
      pm[0] = mx * 0.6931471805599453f;  // natural-log units
      pm[1] = l;
    }
  }
}

}  // namespace tq
