// kernels_pow2_f32_1024.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f32_1024(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 1024, 16, 16>(p, src, dst);
}

}  // namespace pfk
