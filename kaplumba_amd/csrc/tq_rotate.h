// Dense rotations of many f32 or query rows on the matrix cores.
#pragma once

#include "tq_append.h"
#include "tq_common.h"
#include "tq_tiles.h"

namespace tq {

struct RotateArgs {
  // input rows: queries (element strides over (b, h, l), rounded after the
  // scale) or contiguous f32 rows of k values
  const void* x;
  int64_t x_sb, x_sh, x_sl;
  int x_dtype;  // TQ_DTYPE_*, queries only
  int Hq, L;
  int x_vec;          // queries: rows start 16-byte aligned and k fills 16-byte pieces (mat's rows too)
  float scale;
  int rows, k, n;     // y[rows, n] = x[rows, k] . M
  const float* mat;   // queries: row i of mat (k entries) gives y_i; f32 rows: y_i = sum_d x_d mat[d, i]
  void* out;          // queries: f32; f32 rows: out_dtype
  int out_dtype;
  int out_stride;     // elements per output row; queries: columns n .. out_stride - 1 are zeroed
};

constexpr int kRotateMaxDim = 256;

// At most kMaxTiledRows rows or vectors.
// q_rot = round_qdtype(q * scale) @ mat^T into f32 rows (k = n <= 256)
int launch_rotate_queries(const RotateArgs& a, hipStream_t st);
// out = x @ mat for f32 rows x (k = n <= 256, a multiple of 4, rows and x 16-byte aligned)
int launch_rotate_rows(const RotateArgs& a, hipStream_t st);

// out[vec] = norm * (codebook[idx] @ R) for n packed vectors of any dim up to 256
constexpr int kDequantDenseMin = 2048;
int launch_dequant_dense(const DequantGeneralArgs& a, int n, hipStream_t st);

}  // namespace tq
