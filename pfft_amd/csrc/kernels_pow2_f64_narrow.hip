// kernels_pow2_f64_narrow.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f64n_64(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 64, 4, 8, false>(p, src, dst);
}
int pow2_f64n_128(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 128, 4, 8, false>(p, src, dst);
}
int pow2_f64n_256(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 256, 4, 8, false>(p, src, dst);
}
int pow2_f64n_512(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 512, 4, 8, false>(p, src, dst);
}
int pow2_f64n_1024(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 1024, 4, 16, false>(p, src, dst);
}
int pow2_f64n_2048(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 2048, 2, 16, false>(p, src, dst);
}
int pow2_f64n_4096(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<double, 4096, 1, 16, false>(p, src, dst);
}

}  // namespace pfk
