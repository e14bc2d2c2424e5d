// kernels_pow2_f32_2048.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f32_2048(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 2048, 8, 16>(p, src, dst);
}

}  // namespace pfk
