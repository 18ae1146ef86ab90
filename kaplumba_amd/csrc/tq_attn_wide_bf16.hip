// Wide- and narrow-kernel launches over plain bf16 caches.
#include "tq_attn_wide_launch.h"

namespace tq {

int launch_wide_bf16(const GenParams& p, bool f32_weights, hipStream_t st) {
  return f32_weights ? launch_wide_any<kWideBf16, 3>(p, st) : launch_wide_pow2<kWideBf16, 2>(p, st);
}

int launch_narrow_bf16(const GenParams& p, hipStream_t st) { return launch_narrow_any<kWideBf16>(p, st); }

}  // namespace tq
