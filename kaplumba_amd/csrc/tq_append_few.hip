// Dense-rotation append at dims that are multiples of 8 up to 256, but not 64, 128
// or 256 (those take tq_append_dense.hip at every size: its sums run in another
// order, and a vector's words must not depend on how many are appended with it),
// on v_mfma_f32_16x16x32_bf16, keys and values in one launch.
//
// Semantics and arithmetic as tq_append_dense.hip: y * max(n, eps) = x @ R^T from
// bf16 pieces that sum to the f32 operands (R three; x one for bf16, two for
// f16, three for f32), products whose orders add up to more than 2 skipped,
// sums in f32; indices by strict compares against mid * max(n, eps).  Norms
// take the shared tree, the dim zero-padded to whole 32-element groups, so they
// are bit-exact.
//
// A workgroup takes 16 vectors and 64 coordinates (whole words at every width)
// of one side.  Each of 4 waves owns 16 coordinates and splits their rows of R
// straight into B fragments: no LDS, one round trip of loads; the norm is
// formed by every wave.  Indices meet in LDS for the packing.
//
// Ties.  Sums in another order than the vector kernel's (tq_append_general.hip)
// may put a coordinate within some ulps of a midpoint on its other side.  Where a
// coordinate lies within the bound of both kernels' rounding of a threshold
// (tie_units), its index comes from the vector kernel's own arithmetic (IEEE
// division, four fused chains), so the two agree bit for bit: one coordinate in
// 5400 at d = 96, 4 bits (2100 at d = 192), a branch that one wave in 21 (9) takes.
#include "tq_append.h"
#include "tq_pieces.h"

namespace tq {
namespace {

__device__ __forceinline__ float halves_add(float x) {  // x of lanes l and l ^ 32
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __fadd_rn(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

constexpr int kFewThreads = 256;
constexpr int kFewCoords = 64;              // coordinates per workgroup
constexpr int kFewMaxDim = 256;
constexpr int kFewIdxRow = kFewCoords + 4;  // bytes per vector's indices in LDS

// How far the two kernels' sums of one coordinate can lie apart, in units of
// 2^-24 |x| |R_i| (sum_k |x_k R_ik| <= |x| |R_i|).  Vector kernel: D / 4 fused adds a
// chain, the two adds of the chains and the division, one unit each.  Here: a
// product rounds by up to 4 units of its accumulator and terms (3.7 the largest over
// 5e5 random and one-signed ones, and the terms count once in all), so 4 per step
// of the main chain and 4; the other chains, 2^-8 of it, one; two adds, the
// threshold's product and the skipped terms one each.
constexpr float tie_units(int D, int steps) { return D / 4 + 3 + 4 * steps + 4 + 1 + 4; }

// Orders a wave's own LDS accesses (the LDS serves a wave in order).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// KS: 32-element steps that hold the dim (a multiple of 8)
template <int KS, int XDT>
__global__ __launch_bounds__(kFewThreads) void append_few_kernel(AppendArgs ka, AppendArgs va, int D, int kbits, int vbits,
                                                                int n_vec) {
  constexpr int NX = XDT == TQ_DTYPE_BF16 ? 1 : (XDT == TQ_DTYPE_F16 ? 2 : 3);
  __shared__ __align__(16) uint8_t s_idx[16 * kFewIdxRow];
  __shared__ uint8_t s_tie[kFewThreads / 64][256];  // per wave: vector << 4 | coordinate
  const bool key = blockIdx.z == 0;
  const AppendArgs a = select_args(key, ka, va);
  const int bits = key ? kbits : vbits;
  const int nmid = (1 << bits) - 1;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15;
  const int g = lane >> 4;

  // ---- loads: this wave's rows of R (coordinates past D read the last row and
  // are not stored), then the 16 vectors (past the end: the last one, not
  // stored).  D % 8 == 0, so whole 8-element pieces lie inside D or past it.
  const int s0 = blockIdx.y * kFewCoords;  // the workgroup's first coordinate
  const int coord = s0 + 16 * wave + n;
  float4 rv[KS][2];
  {
    const float* row = a.rot + static_cast<int64_t>(min(coord, D - 1)) * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int k = min(32 * s + 8 * g, D - 8);
      rv[s][0] = *reinterpret_cast<const float4*>(row + k);
      rv[s][1] = *reinterpret_cast<const float4*>(row + k + 4);
    }
  }
  const int vec = min(static_cast<int>(blockIdx.x) * 16 + n, n_vec - 1);
  const int l = vec % a.L;
  const int bh = vec / a.L;
  const int64_t xoff = static_cast<int64_t>(bh / a.H) * a.sb + static_cast<int64_t>(bh % a.H) * a.sh + l * a.sl;
  const int64_t out_row = static_cast<int64_t>(bh) * a.cap + a.offset + l;
  u32x4_t xr[KS][XDT == TQ_DTYPE_F32 ? 2 : 1];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int k = min(32 * s + 8 * g, D - 8);
    if constexpr (XDT == TQ_DTYPE_F32) {
      const u32x4_t* src = reinterpret_cast<const u32x4_t*>(static_cast<const float*>(a.x) + xoff + k);
      xr[s][0] = src[0];
      xr[s][1] = src[1];
    } else {
      xr[s][0] = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.x) + xoff + k);
    }
  }
  float mid[15];
#pragma unroll
  for (int m = 0; m < 15; ++m) mid[m] = a.mid[min(m, nmid - 1)];

  // ---- pieces of x and the norm.  Lane (vector n, g) holds elements 32 s + 8 g
  // + e: the tree's folds at 16 and 8 run across lanes 32 and 16 apart, those at
  // 4, 2, 1 in registers, group sums pairwise.
  u32x4_t xp[KS][NX];
  float gs[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) gs[q] = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    float v[8];
    const bool in = 32 * s + 8 * g < D;
#pragma unroll
    for (int h = 0; h < (XDT == TQ_DTYPE_F32 ? 2 : 1); ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) xr[s][h][e] = in ? xr[s][h][e] : 0u;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (XDT == TQ_DTYPE_F32) {
        v[e] = __uint_as_float(xr[s][e >> 2][e & 3]);
      } else {
        const uint16_t u = static_cast<uint16_t>(xr[s][0][e >> 1] >> (16 * (e & 1)));
        v[e] = XDT == TQ_DTYPE_F16 ? f16_bits_to_f32(u) : bf16_bits_to_f32(u);
      }
    }
    if constexpr (XDT == TQ_DTYPE_BF16)
      xp[s][0] = xr[s][0];
    else
      split8<NX>(v, xp[s]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float q = halves_add(__fmul_rn(v[e], v[e]));
      q = __fadd_rn(q, xor_lane<16>(q));
      v[e] = q;
    }
#pragma unroll
    for (int w = 4; w >= 1; w >>= 1)
#pragma unroll
      for (int e = 0; e < w; ++e) v[e] = __fadd_rn(v[e], v[e + w]);
    gs[s] = v[0];
  }
#pragma unroll
  for (int w = 1; w < 8; w <<= 1)
#pragma unroll
    for (int q = 0; q < 8; q += 2 * w) gs[q] = __fadd_rn(gs[q], gs[q + w]);  // groups past the dim add exact zeros
  const float nrm = sqrt_rn(gs[0]);
  const float den = fmaxf(nrm, kNormEps);
  if (blockIdx.y == 0 && wave == 0 && g == 0 && static_cast<int>(blockIdx.x) * 16 + n < n_vec) {
    if (a.norm_dtype == TQ_DTYPE_F16)
      static_cast<uint16_t*>(a.norms)[out_row] = f32_to_f16_bits(nrm);
    else
      static_cast<float*>(a.norms)[out_row] = nrm;
  }
  float dj[4];  // of result rows 4 g + j
#pragma unroll
  for (int j = 0; j < 4; ++j) dj[j] = __shfl(den, 4 * g + j, 64);

  // ---- products and indices: lane (coordinate n, g) holds vectors 4 g + j
  float r2 = 0.f;  // squared length of this lane's row of R
  f32x4_t acc[3];  // one chain per order of the piece products
#pragma unroll
  for (int p = 0; p < 3; ++p) acc[p] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const float4 r0 = rv[s][0], r1 = rv[s][1];
    const float r[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) r2 = __builtin_fmaf(r[e], r[e], r2);
    u32x4_t w[3];
    split8<3>(r, w);
#pragma unroll
    for (int p = 2; p >= 0; --p)
#pragma unroll
      for (int q = NX - 1; q >= 0; --q)
        if (q + p <= 2) acc[q + p] = mfma_bf16(xp[s][q], w[p], acc[q + p]);
  }
  // |x . R_i| sums to at most |x| |R_i|; clamped tail pieces only add to r2
  r2 += xor_lane<16>(r2);
  r2 = halves_add(r2);
  const float margin = tie_units(D, KS) * 0x1p-24f * __builtin_amdgcn_sqrtf(r2);
  uint32_t idx[4] = {0u, 0u, 0u, 0u};
  float y[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) y[j] = __fadd_rn(__fadd_rn(acc[2][j], acc[1][j]), acc[0][j]);
  // (a norm past f32's range has no threshold to compare with)
  bool tie[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) tie[j] = dj[j] == INFINITY;
#pragma unroll
  for (int m = 0; m < 15; ++m) {
    if (m >= nmid) break;  // uniform
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = y[j] - __fmul_rn(mid[m], dj[j]);
      idx[j] += d > 0.f ? 1u : 0u;
      tie[j] |= fabsf(d) <= margin * dj[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) s_idx[(4 * g + j) * kFewIdxRow + 16 * wave + n] = static_cast<uint8_t>(idx[j]);
  if (__any(tie[0] | tie[1] | tie[2] | tie[3])) {
    // the wave's ties as a list, then sixteen lanes a tie: four to each chain of the
    // vector kernel, a quarter of its elements each, loaded and divided side by
    // side and added in order (the chain goes from quarter to quarter, which sit
    // one lane bit apart)
    int ties = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint64_t set = __ballot(tie[j] ? 1 : 0);
      const int at = ties + __builtin_popcountll(set & ((uint64_t(1) << lane) - 1));
      if (tie[j]) s_tie[wave][at] = static_cast<uint8_t>((4 * g + j) << 4 | n);
      ties += __builtin_popcountll(set);
    }
    wave_lds_order();
    const int slot = (lane >> 2) & 3;
    const int quarter = slot ^ (slot >> 1);
    const int per = (D / 4 + 3) / 4;  // elements of a quarter, at most 2 KS
    const int k0 = quarter * per;
#pragma unroll 1
    for (int t0 = 0; t0 < ties; t0 += 4) {
      const int code = s_tie[wave][min(t0 + (lane >> 4), ties - 1)];
      const int tv = code >> 4;
      const int tn = code & 15;
      const int gv = min(static_cast<int>(blockIdx.x) * 16 + tv, n_vec - 1);
      const int bh = gv / a.L;
      const int64_t tx = static_cast<int64_t>(bh / a.H) * a.sb + static_cast<int64_t>(bh % a.H) * a.sh +
                         (gv - bh * a.L) * a.sl + (lane & 3);
      const float* row = a.rot + static_cast<int64_t>(min(s0 + 16 * wave + tn, D - 1)) * D + (lane & 3);
      const float td = __shfl(den, tv, 64);
      float u[2 * KS], r[2 * KS];
#pragma unroll
      for (int e = 0; e < 2 * KS; ++e) {
        const int k = min(4 * (k0 + e), D - 4);
        u[e] = load_elem<XDT>(a.x, tx + k);
        r[e] = row[k];
      }
#pragma unroll
      for (int e = 0; e < 2 * KS; ++e) u[e] = __fdiv_rn(u[e], td);
      float c = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q > 0) {
          const float from = (q & 1) ? xor_lane<4>(c) : xor_lane<8>(c);
          c = quarter == q ? from : c;
        }
        if (quarter == q) {
#pragma unroll
          for (int e = 0; e < 2 * KS; ++e)
            if (e < per && 4 * (k0 + e) < D) c = __builtin_fmaf(u[e], r[e], c);
        }
      }
      c = __fadd_rn(c, xor_lane<1>(c));
      const float ty = __fadd_rn(c, xor_lane<2>(c));
      uint32_t ti = 0;
#pragma unroll
      for (int m = 0; m < 15; ++m)
        if (m < nmid) ti += ty > mid[m] ? 1u : 0u;
      if ((lane & 3) == 0 && quarter == 3) s_idx[tv * kFewIdxRow + 16 * wave + tn] = static_cast<uint8_t>(ti);
    }
  }
  __syncthreads();

  // ---- pack: thread (vector, word); LSB-first, zeros past the last coordinate
  const int pw = (D * bits + 31) / 32;
  const int v = tid >> 4;
  const int w = tid & 15;                     // word of the slice: 2 bits of them
  const int pword = blockIdx.y * 2 * bits + w;
  const int gv = static_cast<int>(blockIdx.x) * 16 + v;
  if (w < 2 * bits && pword < pw && gv < n_vec) {
    const uint8_t* row = s_idx + v * kFewIdxRow;
    const int dl = D - s0;  // coordinates of the slice that exist
    uint32_t word = 0;
    if (bits == 3) {
      const int ca = 32 * w / 3, cb = min(min(dl, kFewCoords) - 1, (32 * w + 31) / 3);
      for (int c = ca; c <= cb; ++c) {
        const int sh = 3 * c - 32 * w;  // negative for a field straddling the word's start
        const uint32_t q = row[c];
        word |= sh >= 0 ? q << sh : q >> -sh;
      }
    } else {
      // 32 / bits coordinates per word, four bytes at a time
      const int per = 32 / bits;
      for (int c = 0; c < per; c += 4) {
        if (per * w + c >= dl) break;
        const uint32_t q = *reinterpret_cast<const uint32_t*>(row + per * w + c);
        const uint32_t f = (q & 0xffu) | ((q >> 8 & 0xffu) << bits) | ((q >> 16 & 0xffu) << (2 * bits)) | ((q >> 24) << (3 * bits));
        word |= f << (c * bits);
      }
    }
    const int vl = gv % a.L;
    const int vbh = gv / a.L;
    a.packed[(static_cast<int64_t>(vbh) * a.cap + a.offset + vl) * pw + pword] = word;
  }
}

template <int KS>
int launch_few(const AppendArgs& k, const AppendArgs& v, int sides, int dim, int kbits, int vbits, int x_dtype,
               hipStream_t st) {
  const int n_vec = k.B * k.H * k.L;
  const dim3 grid(static_cast<unsigned>((n_vec + 15) / 16), static_cast<unsigned>((dim + kFewCoords - 1) / kFewCoords),
                  static_cast<unsigned>(sides));
  switch (x_dtype) {
    case TQ_DTYPE_F32:
      hipLaunchKernelGGL((append_few_kernel<KS, TQ_DTYPE_F32>), grid, dim3(kFewThreads), 0, st, k, v, dim, kbits, vbits, n_vec);
      break;
    case TQ_DTYPE_F16:
      hipLaunchKernelGGL((append_few_kernel<KS, TQ_DTYPE_F16>), grid, dim3(kFewThreads), 0, st, k, v, dim, kbits, vbits, n_vec);
      break;
    default:
      hipLaunchKernelGGL((append_few_kernel<KS, TQ_DTYPE_BF16>), grid, dim3(kFewThreads), 0, st, k, v, dim, kbits, vbits, n_vec);
      break;
  }
  return check_launch("append_few_kernel");
}

}  // namespace

// Every count of vectors: K + V, 8 heads, bf16, 3 bits, us in the vector kernel ->
// here, ties included (one adds 1 us to a launch, 2.5-5 with four lanes a tie):
// d = 96 26 -> 4.9 for 8 vectors a side, 33 -> 12.0 for 4096; d = 192 43 -> 6.2 and
// 77 -> 23.3.
bool append_few_path(int64_t n_vec, int dim) {
  return dim % 8 == 0 && dim >= 8 && dim <= kFewMaxDim && dim != 64 && dim != 128 && dim != 256 &&
         n_vec < (int64_t(1) << 31) - 16;
}

int launch_append_few(const AppendArgs& k, const AppendArgs& v, int sides, int dim, int kbits, int vbits, int x_dtype,
                      hipStream_t st) {
  switch ((dim + 31) / 32) {
    case 1:
    case 2: return launch_few<2>(k, v, sides, dim, kbits, vbits, x_dtype, st);
    case 3: return launch_few<3>(k, v, sides, dim, kbits, vbits, x_dtype, st);
    case 4: return launch_few<4>(k, v, sides, dim, kbits, vbits, x_dtype, st);
    case 5:
    case 6: return launch_few<6>(k, v, sides, dim, kbits, vbits, x_dtype, st);
    default: return launch_few<8>(k, v, sides, dim, kbits, vbits, x_dtype, st);
  }
}

}  // namespace tq
