// kernels_mixed_r2r_f32.hip -- instantiations of mixed_launch.hpp.
#include "mixed_launch.hpp"

namespace pfk {

int launch_mixed_r2r_f32(const pfk_pass *p, const MixGeo &g, int nt, size_t lds,
                         const void *src, void *dst) {
  return launch_mixed_r2r_t<float>(p, g, nt, lds, src, dst);
}

}  // namespace pfk
