// kernels_pow2_f64_short.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f64_64(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 64, 8, 8>(p, src, dst);
}
int pow2_f64_128(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 128, 8, 8>(p, src, dst);
}
int pow2_f64_256(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 256, 8, 8>(p, src, dst);
}

}  // namespace pfk
