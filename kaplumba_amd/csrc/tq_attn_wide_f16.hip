// Wide- and narrow-kernel launches over plain f16 caches.
#include "tq_attn_wide_launch.h"

namespace tq {

int launch_wide_f16(const GenParams& p, bool f32_weights, hipStream_t st) {
  return f32_weights ? launch_wide_any<kWideF16, 2>(p, st) : launch_wide_pow2<kWideF16, 1>(p, st);
}

int launch_narrow_f16(const GenParams& p, hipStream_t st) { return launch_narrow_any<kWideF16>(p, st); }

}  // namespace tq
