// kernels_pow2_f32_short.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f32_64(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 64, 16, 8>(p, src, dst);
}
int pow2_f32_128(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 128, 16, 8>(p, src, dst);
}
int pow2_f32_256(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 256, 16, 8>(p, src, dst);
}

}  // namespace pfk
