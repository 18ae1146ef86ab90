// Launch of one instantiation of the wide kernel (included by tq_attn_wide_*.hip).
#pragma once

#include "tq_attn_narrow.h"
#include "tq_attn_wide.h"

namespace tq {

template <int KS, int CT, int SRC, int WP>
int launch_wide(const GenParams& p, hipStream_t st) {
  constexpr int RT = wide_rt(KS);
  const int rows = wide_block_rows(KS);
  const int n_blocks = (p.R * p.L + rows - 1) / rows;
  const int64_t wgs = static_cast<int64_t>(p.B) * p.Hkv * n_blocks * p.n_splits;
  if (wgs > INT32_MAX) return fail(TQ_ERR_UNSUPPORTED, "attention: %lld wide workgroups", static_cast<long long>(wgs));
  hipLaunchKernelGGL((gen_wide_kernel<KS, CT, RT, SRC, WP>), dim3(static_cast<unsigned>(wgs)), dim3(kWideThreads), 0,
                     st, p, n_blocks);
  return check_launch("gen_wide_kernel");
}

template <int SRC, int WP>
int launch_wide_any(const GenParams& p, hipStream_t st) {
  int ks = 0, ct = 0;
  if (!wide_dims(p.Dk, p.Dv, ks, ct))
    return fail(TQ_ERR_UNSUPPORTED, "attention: no wide kernel for head dims k %d / v %d", p.Dk, p.Dv);
  switch (ks) {
    case 2: return launch_wide<2, 4, SRC, WP>(p, st);
    case 3: return launch_wide<3, 6, SRC, WP>(p, st);
    case 4: return launch_wide<4, 8, SRC, WP>(p, st);
    case 6: return launch_wide<6, 8, SRC, WP>(p, st);
    default: return launch_wide<8, 16, SRC, WP>(p, st);
  }
}

// The shapes that the tuned kernels' f16 / bf16 hi + lo weights serve: one dim of 64, 128 or 256.
template <int SRC, int WP>
int launch_wide_pow2(const GenParams& p, hipStream_t st) {
  switch (p.Dk) {
    case 64: return launch_wide<2, 4, SRC, WP>(p, st);
    case 128: return launch_wide<4, 8, SRC, WP>(p, st);
    default: return launch_wide<8, 16, SRC, WP>(p, st);
  }
}

template <int KS, int CT, int SRC>
int launch_narrow(const GenParams& p, hipStream_t st) {
  const int groups = (p.R * p.L + kNarrowRows - 1) / kNarrowRows;
  const int64_t wgs = static_cast<int64_t>(p.B) * p.Hkv * groups * p.n_splits;
  if (wgs > INT32_MAX) return fail(TQ_ERR_UNSUPPORTED, "attention: %lld narrow workgroups", static_cast<long long>(wgs));
  hipLaunchKernelGGL((gen_narrow_kernel<KS, CT, SRC>), dim3(static_cast<unsigned>(wgs)), dim3(512), 0, st, p, groups);
  return check_launch("gen_narrow_kernel");
}

template <int SRC>
int launch_narrow_any(const GenParams& p, hipStream_t st) {
  int ks = 0, ct = 0;
  if (!wide_dims(p.Dk, p.Dv, ks, ct))
    return fail(TQ_ERR_UNSUPPORTED, "attention: no narrow kernel for head dims k %d / v %d", p.Dk, p.Dv);
  switch (ks) {
    case 2: return launch_narrow<2, 4, SRC>(p, st);
    case 3: return launch_narrow<3, 6, SRC>(p, st);
    case 4: return launch_narrow<4, 8, SRC>(p, st);
    case 6: return launch_narrow<6, 8, SRC>(p, st);
    default: return launch_narrow<8, 16, SRC>(p, st);
  }
}

}  // namespace tq
