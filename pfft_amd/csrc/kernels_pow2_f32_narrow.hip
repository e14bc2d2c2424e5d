// kernels_pow2_f32_narrow.hip -- instantiations of pow2_tile.hpp.
#include "pow2_tile.hpp"
#include "pow2_launch.hpp"

namespace pfk {

int pow2_f32n_64(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 64, 8, 8, false>(p, src, dst);
}
int pow2_f32n_128(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 128, 8, 8, false>(p, src, dst);
}
int pow2_f32n_256(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 256, 8, 8, false>(p, src, dst);
}
int pow2_f32n_512(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 512, 8, 8, false>(p, src, dst);
}
int pow2_f32n_1024(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 1024, 8, 16, false>(p, src, dst);
}
int pow2_f32n_2048(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 2048, 4, 16, false>(p, src, dst);
}
int pow2_f32n_4096(const pfk_pass *p, const void *src, void *dst) {
  return launch_nf<float, 4096, 2, 16, false>(p, src, dst);
}

}  // namespace pfk
