// y = x . M for many rows x and one dense rotation matrix M (R_K of the
// queries, R_V^-1 of merged outputs) on v_mfma_f32_16x16x32_bf16.
//
// f32-class products: M and f32 rows go into three bf16 pieces (24
// significand bits), f16 queries into two, bf16 queries into one; all pieces
// of an entry sum to it exactly, products whose orders add up to more than 2
// are below f32 resolution and skipped, sums run in f32, in one chain per order:
// a matrix product may round its accumulator by up to 4 units of 2^-24 of the
// sum of magnitudes (measured), and the main chain so meets one of them per 32
// terms instead of up to six.  Error of a reconstruction at d = 64 / 256 with all
// orders in one chain 0.9e-7 / 2.2e-7, so 0.5e-7 / 0.8e-7; f32 chains of d terms
// 1.5e-7 / 2.9e-7.
//
// rotate_kernel: a workgroup takes 128 rows and 64 columns.  It splits its 64
// columns of M once into LDS, in B-fragment order (conflict-free 16-byte
// reads); each of 8 waves keeps the pieces of its 16 rows in registers as A
// fragments.  Bound by LDS reads (one fragment per 16 rows) and the split.
// rotate_few_kernel: for few rows a workgroup takes 16 rows and 64 columns, a
// wave one 16-column tile whose pieces it splits straight into registers: no
// LDS, one round trip of loads.  Latency-bound.
#include <algorithm>

#include "tq_pieces.h"
#include "tq_rotate.h"

namespace tq {
namespace {

// The product's sum from its chains, one per order of the pieces' product: the
// main chain is rounded once per step only.
__device__ __forceinline__ f32x4_t sum_orders(f32x4_t o0, f32x4_t o1, f32x4_t o2) {
  f32x4_t y;
#pragma unroll
  for (int j = 0; j < 4; ++j) y[j] = __fadd_rn(__fadd_rn(o2[j], o1[j]), o0[j]);
  return y;
}

constexpr int kFromF32Rows = -1;  // XT: contiguous f32 rows; else the queries' TQ_DTYPE_*

// The pieces of one A fragment set: lane (row n, g) of the 16 rows from r0 on
// holds entries 32 s + 8 g .. + 7 (a row past the end reads the last one).
// VEC: every load is a 16-byte piece (queries: x_vec; f32 rows always), so the
// body is straight-line code.
template <int KS, int XT, bool VEC>
struct RowPieces {
  static constexpr bool QUERY = XT != kFromF32Rows;
  static constexpr int NX = XT == TQ_DTYPE_BF16 ? 1 : (XT == TQ_DTYPE_F16 ? 2 : 3);  // pieces of x
  float v[KS][8];

  __device__ __forceinline__ void load(const RotateArgs& a, int r0, int n, int g) {
    const int row = min(r0 + n, a.rows - 1);
    const int K = a.k;
    if constexpr (QUERY) {
      const int l = row % a.L;
      const int bh = row / a.L;
      const int64_t qo = static_cast<int64_t>(bh / a.Hq) * a.x_sb + static_cast<int64_t>(bh % a.Hq) * a.x_sh + l * a.x_sl;
      if constexpr (VEC && XT == TQ_DTYPE_F32) {
        const float* xr = static_cast<const float*>(a.x) + qo;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            *reinterpret_cast<float4*>(v[s] + 4 * h) =
                *reinterpret_cast<const float4*>(xr + min(32 * s + 8 * g + 4 * h, K - 4));
      } else if constexpr (VEC) {
        uint4 h[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s)
          h[s] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.x) + qo + min(32 * s + 8 * g, K - 8));
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const uint32_t w[4] = {h[s].x, h[s].y, h[s].z, h[s].w};
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint16_t u = static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)));
            v[s][e] = XT == TQ_DTYPE_F16 ? f16_bits_to_f32(u) : bf16_bits_to_f32(u);
          }
        }
      } else {
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int e = 0; e < 8; ++e) v[s][e] = load_elem<XT>(a.x, qo + min(32 * s + 8 * g + e, K - 1));
      }
    } else {
      const float* xr = static_cast<const float*>(a.x) + static_cast<int64_t>(row) * K;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h)  // K % 4 == 0: whole float4 pieces
          *reinterpret_cast<float4*>(v[s] + 4 * h) =
              *reinterpret_cast<const float4*>(xr + min(32 * s + 8 * g + 4 * h, K - 4));
    }
  }

  __device__ __forceinline__ void split(const RotateArgs& a, int g, u32x4_t (&xp)[KS][NX]) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if constexpr (QUERY) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[s][e] *= a.scale;
          if constexpr (XT == TQ_DTYPE_F16) v[s][e] = round_to<TQ_DTYPE_F16>(v[s][e]);
        }
      }
      if (32 * s + 32 > a.k) {  // uniform: the row ends in this step or before it
#pragma unroll
        for (int e = 0; e < 8; ++e) v[s][e] = 32 * s + 8 * g + e < a.k ? v[s][e] : 0.f;
      }
      split8<NX>(v[s], xp[s]);  // bf16 queries: one piece, which is their rounding to bf16
    }
  }
};

// Eight entries of M for one B-fragment lane: column col, entries k0 .. k0 + 7
// (clamped into the matrix; zeroed by fragment_zero).
template <bool QUERY, bool VEC>
__device__ __forceinline__ void fragment_load(const RotateArgs& a, int col, int k0, float (&m)[8]) {
  const int colc = min(col, a.n - 1);
  if constexpr (QUERY && VEC) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      *reinterpret_cast<float4*>(m + 4 * h) =
          *reinterpret_cast<const float4*>(a.mat + static_cast<int64_t>(colc) * a.k + min(k0 + 4 * h, a.k - 4));
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = min(k0 + e, a.k - 1);
      m[e] = QUERY ? a.mat[static_cast<int64_t>(colc) * a.k + k] : a.mat[static_cast<int64_t>(k) * a.n + colc];
    }
  }
}

__device__ __forceinline__ void fragment_zero(const RotateArgs& a, int col, int k0, float (&m)[8]) {
  if (__all(k0 + 8 <= a.k && col < a.n)) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) m[e] = (k0 + e < a.k && col < a.n) ? m[e] : 0.f;
}

// Lane (column col + 16 t, g) holds rows r0 + 4 g + j of tile t.  Queries go to
// f32 rows, every column below out_stride (those past n are zero, as M's are there).
template <int ODT, int NT>
__device__ __forceinline__ void store_typed(const RotateArgs& a, int r0, int g, int col, int ncols, const f32x4_t (&y)[NT]) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = r0 + 4 * g + j;
      if (r < a.rows && col + 16 * t < ncols)
        store_elem<ODT>(a.out, static_cast<int64_t>(r) * a.out_stride + col + 16 * t, y[t][j]);
    }
}

template <bool QUERY, int NT>
__device__ __forceinline__ void store_tiles(const RotateArgs& a, int r0, int g, int col, const f32x4_t (&y)[NT]) {
  if constexpr (QUERY) {
    store_typed<TQ_DTYPE_F32, NT>(a, r0, g, col, a.out_stride, y);
  } else {
    switch (a.out_dtype) {
      case TQ_DTYPE_F32: store_typed<TQ_DTYPE_F32, NT>(a, r0, g, col, a.n, y); break;
      case TQ_DTYPE_F16: store_typed<TQ_DTYPE_F16, NT>(a, r0, g, col, a.n, y); break;
      default: store_typed<TQ_DTYPE_BF16, NT>(a, r0, g, col, a.n, y); break;
    }
  }
}

constexpr int kRotateRows = kTileRows128;  // rows per rotate_kernel workgroup

template <int KS, int XT>
__global__ __launch_bounds__(512) void rotate_kernel(RotateArgs a) {
  using X = RowPieces<KS, XT, true>;
  __shared__ u32x4_t s_m[3 * 4 * KS * 64];  // [piece][16-column tile][k step][lane]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int n = lane & 15;
  const int g = lane >> 4;
  const int c0 = blockIdx.y * 64;
  const int r0 = blockIdx.x * kRotateRows + 16 * (tid >> 6);
  // fragment (tile t, step s, lane): column c0 + 16 t + lane % 16, entries
  // 32 s + 8 (lane / 16) .. + 7; every load is issued before the first use
  constexpr int FR = 4 * KS * 64;
  constexpr int FPT = (FR + 511) / 512;
  float m[FPT][8];
#pragma unroll
  for (int i = 0; i < FPT; ++i) {
    const int f = min(tid + 512 * i, FR - 1);
    fragment_load<X::QUERY, true>(a, c0 + 16 * (f / (64 * KS)) + (f & 15), 32 * ((f >> 6) % KS) + 8 * ((f >> 4) & 3), m[i]);
  }
  X x;
  x.load(a, r0, n, g);
#pragma unroll
  for (int i = 0; i < FPT; ++i) {
    const int f = tid + 512 * i;
    if (FR % 512 != 0 && f >= FR) break;  // whole waves
    fragment_zero(a, c0 + 16 * (f / (64 * KS)) + (f & 15), 32 * ((f >> 6) % KS) + 8 * ((f >> 4) & 3), m[i]);
    u32x4_t w[3];
    split8<3>(m[i], w);
#pragma unroll
    for (int p = 0; p < 3; ++p) s_m[p * FR + f] = w[p];
  }
  u32x4_t xp[KS][X::NX];
  x.split(a, g, xp);
  __syncthreads();

  f32x4_t acc[3][4];
#pragma unroll
  for (int o = 0; o < 3; ++o)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[o][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int mp = 2; mp >= 0; --mp)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const u32x4_t b = s_m[mp * FR + (t * KS + s) * 64 + lane];
#pragma unroll
        for (int q = X::NX - 1; q >= 0; --q)
          if (q + mp <= 2) acc[q + mp][t] = mfma_bf16(xp[s][q], b, acc[q + mp][t]);
      }
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[0][t] = sum_orders(acc[0][t], acc[1][t], acc[2][t]);
  store_tiles<X::QUERY, 4>(a, r0, g, c0 + n, acc[0]);
}

template <int KS, int XT, bool VEC>
__global__ __launch_bounds__(256) void rotate_few_kernel(RotateArgs a) {
  using X = RowPieces<KS, XT, VEC>;
  const int lane = threadIdx.x & 63;
  const int n = lane & 15;
  const int g = lane >> 4;
  const int col = blockIdx.y * 64 + 16 * (threadIdx.x >> 6) + n;
  const int r0 = blockIdx.x * 16;
  if (blockIdx.y * 64 + 16 * static_cast<int>(threadIdx.x >> 6) >= (X::QUERY ? a.out_stride : a.n)) return;
  float m[KS][8];
#pragma unroll
  for (int s = 0; s < KS; ++s) fragment_load<X::QUERY, VEC>(a, col, 32 * s + 8 * g, m[s]);
  X x;
  x.load(a, r0, n, g);
  u32x4_t xp[KS][X::NX];
  x.split(a, g, xp);
  f32x4_t acc[3];
#pragma unroll
  for (int p = 0; p < 3; ++p) acc[p] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    fragment_zero(a, col, 32 * s + 8 * g, m[s]);
    u32x4_t w[3];
    split8<3>(m[s], w);
#pragma unroll
    for (int p = 2; p >= 0; --p)
#pragma unroll
      for (int q = X::NX - 1; q >= 0; --q)
        if (q + p <= 2) acc[q + p] = mfma_bf16(xp[s][q], w[p], acc[q + p]);
  }
  const f32x4_t y[1] = {sum_orders(acc[0], acc[1], acc[2])};
  store_tiles<X::QUERY, 1>(a, r0, g, col, y);
}

template <int KS, int XT>
int launch_ks(const RotateArgs& a, hipStream_t st) {
  const int cols = XT == kFromF32Rows ? a.n : a.out_stride;
  const unsigned gy = static_cast<unsigned>((cols + 63) / 64);
  // 128 rows per workgroup where that still gives one to most CUs
  const unsigned gx = static_cast<unsigned>(tiles_of(a.rows));
  const bool vec = XT == kFromF32Rows || a.x_vec;
  if (vec && static_cast<int64_t>(gx) * gy >= device_cu_count() / 2)
    hipLaunchKernelGGL((rotate_kernel<KS, XT>), dim3(gx, gy), dim3(512), 0, st, a);
  else if (vec)
    hipLaunchKernelGGL((rotate_few_kernel<KS, XT, true>), dim3(static_cast<unsigned>((a.rows + 15) / 16), gy), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((rotate_few_kernel<KS, XT, false>), dim3(static_cast<unsigned>((a.rows + 15) / 16), gy), dim3(256), 0, st, a);
  return check_launch("rotate_kernel");
}

template <int XT>
int launch_any(const RotateArgs& a, hipStream_t st) {
  if (a.rows <= 0) return TQ_OK;
  if (a.rows > kMaxTiledRows || a.k < 4 || a.n < 1 || a.k > kRotateMaxDim || a.n > kRotateMaxDim || a.out_stride > kRotateMaxDim)
    return fail(TQ_ERR_UNSUPPORTED, "rotate: %d rows, %d x %d", a.rows, a.k, a.n);
  switch ((a.k + 31) / 32) {
    case 1:
    case 2: return launch_ks<2, XT>(a, st);
    case 3: return launch_ks<3, XT>(a, st);
    case 4: return launch_ks<4, XT>(a, st);
    case 5:
    case 6: return launch_ks<6, XT>(a, st);
    default: return launch_ks<8, XT>(a, st);
  }
}

// Dequantize with the dense rotation: rotate_kernel's products with the rows
// decoded from packed indices (the three pieces of every codebook level in an
// LDS table), scaled by the vector's norm.  A workgroup walks 128-vector tiles
// with one split of its 64 columns of R.
template <int KS>
__global__ __launch_bounds__(512) void dequant_dense_kernel(DequantGeneralArgs a, int n_vec) {
  __shared__ u32x4_t s_m[3 * 4 * KS * 64];  // [piece][16-column tile][k step][lane]
  __shared__ uint2 s_cb[16];                // pieces 0 | 1 << 16, 2 of a level
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int n = lane & 15;
  const int g = lane >> 4;
  const int c0 = blockIdx.y * 64;
  const int D = a.D;
  RotateArgs ra{};
  ra.k = ra.n = D;
  ra.mat = a.rot;
  constexpr int FR = 4 * KS * 64;
  constexpr int FPT = (FR + 511) / 512;
  float m[FPT][8];
#pragma unroll
  for (int i = 0; i < FPT; ++i) {
    const int f = min(tid + 512 * i, FR - 1);
    fragment_load<false, true>(ra, c0 + 16 * (f / (64 * KS)) + (f & 15), 32 * ((f >> 6) % KS) + 8 * ((f >> 4) & 3), m[i]);
  }
  if (tid < (1 << a.bits)) {
    float v[8] = {a.cb[tid], 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    u32x4_t w[3];
    split8<3>(v, w);
    s_cb[tid] = make_uint2((w[0][0] & 0xffffu) | (w[1][0] << 16), w[2][0] & 0xffffu);
  }
#pragma unroll
  for (int i = 0; i < FPT; ++i) {
    const int f = tid + 512 * i;
    if (FR % 512 != 0 && f >= FR) break;  // whole waves
    fragment_zero(ra, c0 + 16 * (f / (64 * KS)) + (f & 15), 32 * ((f >> 6) % KS) + 8 * ((f >> 4) & 3), m[i]);
    u32x4_t w[3];
    split8<3>(m[i], w);
#pragma unroll
    for (int p = 0; p < 3; ++p) s_m[p * FR + f] = w[p];
  }
  __syncthreads();
  const int bits = a.bits;
  const int sh = (8 * g * bits) & 31;
  const uint32_t mask = (1u << bits) - 1u;
  walk_tiles(n_vec, blockIdx.x, gridDim.x, [&](int tile0) {
    const int r0 = tile0 + 16 * (tid >> 6);
    if (r0 >= n_vec) return;  // a wave past the end
    // the fragments stay in LDS: hoisted out of the loop they spill
    asm volatile("" ::: "memory");
    // lane (vector n, g): coordinates 32 s + 8 g .. + 7, 8 * bits bits from word
    // s * bits + (8 g bits) / 32 on; words past the row's last are not read
    // (their coordinates meet zero rows of R)
    const int vec = min(r0 + n, n_vec - 1);
    const int bh = vec / a.T;
    const uint32_t* row = a.packed + (static_cast<int64_t>(bh) * a.cap + (vec - bh * a.T)) * a.PW;
    uint32_t x[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int w = s * bits + ((8 * g * bits) >> 5);
      x[s] = __builtin_amdgcn_alignbit(row[min(w + 1, a.PW - 1)], row[min(w, a.PW - 1)], sh);
    }
    float nrm[4];
    int vj[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      vj[j] = r0 + 4 * g + j;
      const int v = min(vj[j], n_vec - 1);
      const int vbh = v / a.T;
      nrm[j] = load_norm(a.norms, a.norm_dtype, static_cast<int64_t>(vbh) * a.cap + (v - vbh * a.T));
    }
    f32x4_t acc[3][4];
#pragma unroll
    for (int o = 0; o < 3; ++o)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[o][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4_t xp[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint2 u = s_cb[(x[s] >> (2 * e * bits)) & mask];
        const uint2 v = s_cb[(x[s] >> ((2 * e + 1) * bits)) & mask];
        xp[0][e] = __builtin_amdgcn_perm(v.x, u.x, 0x05040100u);
        xp[1][e] = __builtin_amdgcn_perm(v.x, u.x, 0x07060302u);
        xp[2][e] = __builtin_amdgcn_perm(v.y, u.y, 0x05040100u);
      }
#pragma unroll
      for (int mp = 2; mp >= 0; --mp)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const u32x4_t b = s_m[mp * FR + (t * KS + s) * 64 + lane];
#pragma unroll
          for (int q = 2; q >= 0; --q)
            if (q + mp <= 2) acc[q + mp][t] = mfma_bf16(xp[q], b, acc[q + mp][t]);
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int col = c0 + 16 * t + n;
      const f32x4_t y = sum_orders(acc[0][t], acc[1][t], acc[2][t]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (vj[j] < n_vec && col < D) a.out[static_cast<int64_t>(vj[j]) * D + col] = nrm[j] * y[j];
    }
  });
}

template <int KS>
int launch_dequant_ks(const DequantGeneralArgs& a, int n, hipStream_t st) {
  const int gy = (a.D + 63) / 64;
  const int gx = std::min(tiles_of(n), std::max(1, 2 * device_cu_count() / gy));
  hipLaunchKernelGGL(dequant_dense_kernel<KS>, dim3(static_cast<unsigned>(gx), static_cast<unsigned>(gy)), dim3(512), 0, st, a, n);
  return check_launch("dequant_dense_kernel");
}

}  // namespace

int launch_dequant_dense(const DequantGeneralArgs& a, int n, hipStream_t st) {
  switch ((a.D + 31) / 32) {
    case 1:
    case 2: return launch_dequant_ks<2>(a, n, st);
    case 3: return launch_dequant_ks<3>(a, n, st);
    case 4: return launch_dequant_ks<4>(a, n, st);
    case 5:
    case 6: return launch_dequant_ks<6>(a, n, st);
    default: return launch_dequant_ks<8>(a, n, st);
  }
}

int launch_rotate_queries(const RotateArgs& a, hipStream_t st) {
  switch (a.x_dtype) {
    case TQ_DTYPE_F32: return launch_any<TQ_DTYPE_F32>(a, st);
    case TQ_DTYPE_F16: return launch_any<TQ_DTYPE_F16>(a, st);
    default: return launch_any<TQ_DTYPE_BF16>(a, st);
  }
}

int launch_rotate_rows(const RotateArgs& a, hipStream_t st) { return launch_any<kFromF32Rows>(a, st); }

}  // namespace tq
