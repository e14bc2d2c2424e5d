// kernels_pow2_f32_512.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f32_512(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 512, 16, 16>(p, src, dst);
}

}  // namespace pfk
