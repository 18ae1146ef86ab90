// What runs ahead of the wide kernel (tq_attn_wide.h): its query operands and
// the keys each mask row keeps.  Included by tq_attn_general.hip.
#pragma once

#include "tq_attn_wide.h"

namespace tq {

// Query rows for the wide kernel: words of 8 halves, word w holding
// coordinates 8 w .. + 7, zeros past Dk.  Packed keys: q_rot times sq, a power
// of two that brings the row's largest magnitude into [2^12, 2^13), as 4 KS
// hi words then 4 KS lo words; q_rot = H(s * q_s) / sqrt(Dk) (kWideQHad, Dk = 64,
// 128 or 256; other rotations reach the wide kernel as f32 rows).  Plain keys
// (kWideQPlain): q_s as it is, in the type it shares with the cache.
// q_s = round_qdtype(q * scale).
// 16 lanes per row, lane j words j and j + 16, so the butterflies run over
// coordinate bits 0-2 in registers, 3-6 across the lanes of a DPP row and 7
// between a lane's two words.
constexpr int kWideQpThreads = 256;
enum WideQ { kWideQPlain = 0, kWideQHad = 1 };

template <int MODE>
__global__ __launch_bounds__(kWideQpThreads) void wide_qprep_kernel(GenParams p, int rows, int words) {
  const int row = blockIdx.x * (kWideQpThreads / 16) + (threadIdx.x >> 4);
  const int j = threadIdx.x & 15;
  if (row >= rows) return;  // whole 16-lane groups
  float v[2][8];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) v[u][e] = 0.f;
  {
    const int l = row % p.L;
    const int bh = row / p.L;
    const int64_t qo = static_cast<int64_t>(bh / p.Hq) * p.q_sb + static_cast<int64_t>(bh % p.Hq) * p.q_sh + l * p.q_sl;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int w = j + 16 * u;
      if (8 * w >= p.Dk) continue;
      if (p.q_dtype == TQ_DTYPE_F32) {
        const float* src = static_cast<const float*>(p.q) + qo + 8 * w;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] = src[e] * p.scale_q;
      } else {
        const uint16_t* src = static_cast<const uint16_t*>(p.q) + qo + 8 * w;
        const bool bf = p.q_dtype == TQ_DTYPE_BF16;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = (bf ? bf16_bits_to_f32(src[e]) : f16_bits_to_f32(src[e])) * p.scale_q;
          v[u][e] = bf ? round_to<TQ_DTYPE_BF16>(x) : round_to<TQ_DTYPE_F16>(x);
        }
      }
      if constexpr (MODE == kWideQHad) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] *= p.krot[8 * w + e];
      }
    }
  }
  if constexpr (MODE == kWideQHad) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int hb = 1; hb < 8; hb <<= 1)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if ((e & hb) == 0) {
            const float a = v[u][e], c = v[u][e + hb];
            v[u][e] = a + c;
            v[u][e + hb] = a - c;
          }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float x = v[u][e];
        float o = xor_lane<1>(x);
        x = (j & 1) ? o - x : x + o;
        o = xor_lane<2>(x);
        x = (j & 2) ? o - x : x + o;
        o = xor_lane<4>(x);
        x = (j & 4) ? o - x : x + o;
        if (p.Dk > 64) {
          o = xor_lane<8>(x);
          x = (j & 8) ? o - x : x + o;
        }
        v[u][e] = x;
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = v[0][e], c = v[1][e];
      v[0][e] = (p.Dk > 128 ? a + c : a) * p.rscale_k;
      v[1][e] = p.Dk > 128 ? (a - c) * p.rscale_k : 0.f;
    }
  }
  u32x4_t* dst = reinterpret_cast<u32x4_t*>(p.qhl) + static_cast<int64_t>(row) * words * (MODE == kWideQPlain ? 1 : 2);
  if constexpr (MODE == kWideQPlain) {
    const bool bf = p.q_dtype == TQ_DTYPE_BF16;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int w = j + 16 * u;
      if (w >= words) continue;
      u32x4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t a = bf ? f32_to_bf16_bits(v[u][2 * e]) : f32_to_f16_bits(v[u][2 * e]);
        const uint32_t c = bf ? f32_to_bf16_bits(v[u][2 * e + 1]) : f32_to_f16_bits(v[u][2 * e + 1]);
        o[e] = a | (c << 16);
      }
      dst[w] = o;
    }
  } else {
    float mx = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (j + 16 * u >= words) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[u][e]));
    }
    mx = row16_max(mx);
    const float sq = f16_query_scale(mx);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int w = j + 16 * u;
      if (w >= words) continue;
      u32x4_t h, l;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t h0, l0, h1, l1;
        split_f16(v[u][2 * e] * sq, h0, l0);
        split_f16(v[u][2 * e + 1] * sq, h1, l1);
        h[e] = h0 | (h1 << 16);
        l[e] = l0 | (l1 << 16);
      }
      dst[w] = h;
      dst[words + w] = l;
    }
    if (j == 0) p.qsq[row] = sq;
  }
}

// Keys that each mask row keeps: (first, last + 1) relative to the window.
// A row that keeps none gets the whole window (its weights are uniform); an
// additive entry is dropped only at -inf (a row of nothing else gets an empty
// range: its output is zero either way).  One workgroup per distinct mask row
// (row = ((b * ng + g) * nr + r) * L + l over the axes the mask varies along).
__global__ __launch_bounds__(256) void gen_mask_range_kernel(GenParams p, int ng, int nr, int nl) {
  __shared__ int s_lo[4], s_hi[4];
  const int row = blockIdx.x;
  const int l = row % nl;
  const int r = row / nl % nr;
  const int gk = row / (nl * nr) % ng;
  const int b = row / (nl * nr * ng);
  int64_t end = p.seq_lens ? static_cast<int64_t>(p.seq_lens[b]) : p.T;
  end = end > p.T ? p.T : (end < 0 ? 0 : end);
  int64_t start = p.seq_starts ? static_cast<int64_t>(p.seq_starts[b]) : 0;
  start = start < 0 ? 0 : (start > end ? end : start);
  const int len = static_cast<int>(end - start);
  const int64_t base = b * p.m_sb + gk * p.m_sg + r * p.m_sr + l * p.m_sl + start * p.m_st;
  int lo = INT32_MAX, hi = 0;
  if (p.mask_kind == TQ_MASK_BOOL && p.m_st == 1) {
    // 16 bytes per lane from the first aligned address on, the ends by single bytes
    const uint8_t* row8 = static_cast<const uint8_t*>(p.mask) + base;
    const int head = min(len, static_cast<int>(-reinterpret_cast<intptr_t>(row8) & 15));
    const int body = (len - head) / 16;
    auto one = [&](int t) {
      if (row8[t]) {
        lo = min(lo, t);
        hi = max(hi, t + 1);
      }
    };
    if (static_cast<int>(threadIdx.x) < head) one(threadIdx.x);
    for (int k = threadIdx.x; k < body; k += 256) {
      const uint4 v = reinterpret_cast<const uint4*>(row8 + head)[k];
      if ((v.x | v.y | v.z | v.w) != 0u) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if ((w[e >> 2] >> (8 * (e & 3))) & 0xffu) {
            lo = min(lo, head + 16 * k + e);
            hi = max(hi, head + 16 * k + e + 1);
          }
      }
    }
    const int tail = head + 16 * body;
    if (tail + static_cast<int>(threadIdx.x) < len && threadIdx.x < 16) one(tail + threadIdx.x);
  } else {
    for (int t = threadIdx.x; t < len; t += 256) {
      const int64_t off = base + t * p.m_st;
      const bool keep = p.mask_kind == TQ_MASK_BOOL ? static_cast<const uint8_t*>(p.mask)[off] != 0
                                                    : wide_mask_add(p, off) != -INFINITY;
      if (keep) {
        lo = min(lo, t);
        hi = max(hi, t + 1);
      }
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    s_lo[threadIdx.x >> 6] = lo;
    s_hi[threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      lo = min(lo, s_lo[w]);
      hi = max(hi, s_hi[w]);
    }
    if (hi == 0 && p.mask_kind == TQ_MASK_BOOL) {
      lo = 0;
      hi = len;
    }
    p.mrange[row] = make_int2(lo, hi);
  }
}

}  // namespace tq
