// kernels_pow2_f64_512.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f64_512(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 512, 8, 8>(p, src, dst);
}

}  // namespace pfk
