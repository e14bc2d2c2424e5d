// kernels_pow2_f64_1024.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f64_1024(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 1024, 8, 16>(p, src, dst);
}

}  // namespace pfk
