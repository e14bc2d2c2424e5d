// kernels_pow2_f32_4096.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f32_4096(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 4096, 4, 16>(p, src, dst);
}

}  // namespace pfk
