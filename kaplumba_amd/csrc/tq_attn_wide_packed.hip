// Wide- and narrow-kernel launches over packed MSE caches.
#include "tq_attn_wide_launch.h"

namespace tq {

int launch_wide_packed(const GenParams& p, bool f32_weights, hipStream_t st) {
  if (f32_weights) return launch_wide_any<kWidePacked, 2>(p, st);
  return p.Dk == 64 ? launch_wide<2, 4, kWidePacked, 1>(p, st) : launch_wide<8, 16, kWidePacked, 1>(p, st);
}

int launch_narrow_packed(const GenParams& p, hipStream_t st) { return launch_narrow_any<kWidePacked>(p, st); }

}  // namespace tq
