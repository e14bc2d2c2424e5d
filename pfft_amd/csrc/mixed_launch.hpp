// mixed_launch.hpp -- kernel and launcher of the mixed-radix pass, instantiated
// per precision.
#pragma once
#include "mixed_tile.hpp"

namespace pfk {

// Resident workgroups walk the tiles: workgroup b takes tiles b, b + grid, ...
// 512 threads at most, and registers for 16 waves per CU.
template <typename T, int KIND, bool BIG>
__global__ void __launch_bounds__(512, 4)
k_mixed(const pfk_pass P, const MixGeo G, const int64_t ntiles, const int64_t nlines,
        const int last, const T *__restrict__ src, T *__restrict__ dst) {
  extern __shared__ unsigned char mix_smem[];
  stamp_begin(P, blockIdx.x);
  mix_table<T>(P, G, mix_smem);
  int odd = 0;
  for (int64_t id = blockIdx.x; id < ntiles; id += gridDim.x, odd ^= 1) {
    const int64_t tile = P.xcd_remap ? xcd_remap(id, ntiles) : id;
    mixed_tile<T, KIND, BIG>(P, G, tile * G.C, nlines, odd, src, dst, mix_smem);
  }
  stamp_end(P, walk_left(last));
}

// Launch with nt threads and `lds` bytes of LDS per workgroup.
template <typename T, int KIND, bool BIG>
static int launch_mixed_k(const pfk_pass *p, const MixGeo &g, int nt, size_t lds,
                          const void *src, void *dst) {
  static size_t granted = 65536;   // dynamic LDS the kernel may use
  if (lds > granted) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_mixed<T, KIND, BIG>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             160 * 1024);
    if (e != hipSuccess) { set_error("pfk_launch_pass(mixed LDS)", e); return -1; }
    granted = 160 * 1024;
  }
  int64_t lines = g.text;
  for (int i = 0; i < p->nb; i++) lines *= p->bext[i];
  const int64_t ntiles = (lines + g.C - 1) / g.C;
  if (ntiles <= 0) return 0;
  // resident workgroups: by LDS and by waves (128 VGPRs: 16 per CU)
  static int ncu = 0;
  if (!ncu) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        ncu < 8)
      ncu = 8;
  }
  int64_t per_cu = (int64_t)(160 * 1024 / lds), by_waves = 16 / (nt / 64);
  if (by_waves < per_cu) per_cu = by_waves;
  if (per_cu < 1) per_cu = 1;
  const int64_t res = per_cu * (ncu / 8) * 8, grid = ntiles < res ? ntiles : res;
  hipLaunchKernelGGL((k_mixed<T, KIND, BIG>), dim3((unsigned)grid), dim3(nt), lds, g_stream, *p, g,
                     ntiles, lines, (int)((ntiles - 1) % grid), (const T *)src, (T *)dst);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("pfk_launch_pass(mixed)", e); return -1; }
  return 0;
}

template <typename T>
[[maybe_unused]] static int launch_mixed_t(const pfk_pass *p, const MixGeo &g, int nt, size_t lds,
                          const void *src, void *dst) {
  switch (p->kind) {
    case PFK_C2C:
      return g.big ? launch_mixed_k<T, PFK_C2C, true>(p, g, nt, lds, src, dst)
                   : launch_mixed_k<T, PFK_C2C, false>(p, g, nt, lds, src, dst);
    case PFK_R2C:
      return g.big ? launch_mixed_k<T, PFK_R2C, true>(p, g, nt, lds, src, dst)
                   : launch_mixed_k<T, PFK_R2C, false>(p, g, nt, lds, src, dst);
    default:
      return g.big ? launch_mixed_k<T, PFK_C2R, true>(p, g, nt, lds, src, dst)
                   : launch_mixed_k<T, PFK_C2R, false>(p, g, nt, lds, src, dst);
  }
}

template <typename T>
[[maybe_unused]] static int launch_mixed_r2r_t(const pfk_pass *p, const MixGeo &g, int nt, size_t lds,
                              const void *src, void *dst) {
#define PFK_CASE(K) \
  case K: return launch_mixed_k<T, mix_kind_r2r(K), false>(p, g, nt, lds, src, dst)
  switch (p->r2r) {
    PFK_CASE(PFK_DHT);
    PFK_CASE(PFK_REDFT00);
    PFK_CASE(PFK_REDFT01);
    PFK_CASE(PFK_REDFT10);
    PFK_CASE(PFK_REDFT11);
    PFK_CASE(PFK_RODFT00);
    PFK_CASE(PFK_RODFT01);
    PFK_CASE(PFK_RODFT10);
    PFK_CASE(PFK_RODFT11);
    default: return 1;
  }
#undef PFK_CASE
}

}  // namespace pfk
