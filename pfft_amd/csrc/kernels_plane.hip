// kernels_plane.hip -- geometry and launches of the plane pass (plane_tile.hpp).
#include "plane_tile.hpp"

namespace pfk {

// Resident workgroups walk the planes.
template <typename T>
__global__ void __launch_bounds__(1024)
k_plane(const pfk_pass P, const PlaneGeo G, const int64_t nplanes, const int last,
        const T *__restrict__ src, T *__restrict__ dst) {
  extern __shared__ unsigned char plane_smem[];
  stamp_begin(P, blockIdx.x);
  bool tables = true;
  for (int64_t id = blockIdx.x; id < nplanes; id += gridDim.x, tables = false) {
    int64_t u = id, s = 0, d = 0;
    for (int i = 0; i < P.nb; ++i) {
      const int64_t k = u % P.bext[i];
      u /= P.bext[i];
      s += k * P.bsin[i];
      d += k * P.bsout[i];
    }
    plane_tile<T>(G, P.sign, src + 2 * s, dst + 2 * d, P.twm, G.twc, tables, plane_smem);
  }
  stamp_end(P, walk_left(last));
}

static size_t plane_lds(const pfk_pass *p, PlaneGeo *g) {
  g->n1 = (int)p->pl->n;
  g->n2 = (int)p->nf;
  g->pitch = g->n2 + ((g->n2 - 1) >> 4) + 1;
  int L = 1;
  g->ntw1 = g->ntw2 = 0;
  for (int s = 0; s < p->mix_n; s++) {
    if (s) g->ntw1 += (p->mix_rad[s] - 1) * L;
    L *= p->mix_rad[s];
  }
  L = 1;
  for (int s = 0; s < p->pl->mix_n; s++) {
    if (s) g->ntw2 += (p->pl->mix_rad[s] - 1) * L;
    L *= p->pl->mix_rad[s];
  }
  return (size_t)(g->ntw1 + g->ntw2 + g->n1 * g->pitch) * (p->prec == PFK_F64 ? 16 : 8);
}

int plane_threads(const pfk_pass *p) {
  PlaneGeo g;
  const int w = (int)((16 * plane_lds(p, &g) + 160 * 1024 - 1) / (160 * 1024));
  return 64 * (w < 1 ? 1 : w > 16 ? 16 : w);
}

int plane_geo(const pfk_pass *p, int nt, PlaneGeo *g, size_t *lds) {
  if (p->pl->n < 2 || p->nf < 2 || p->pl->n > 1024 || p->nf > 1024 || !p->twm || !p->pl->twm ||
      p->mix_n < 1 || p->pl->mix_n < 1 || p->mix_n + p->pl->mix_n > PFK_PLANE_MAXST)
    return 1;
  *lds = plane_lds(p, g);
  // Larger planes leave a CU one workgroup, whose load, stages and store follow
  // one another (384 uneven complex64 transforms: 1093 us at 110 KiB, 1118 at
  // 150, 1210 at 72, 1430 without planes).
  if (*lds > 110 * 1024) return 1;
  g->nst = p->mix_n + p->pl->mix_n;
  g->nrow = p->mix_n;
  g->s1 = p->pl->sin;
  g->d1 = p->pl->sout;
  g->twc = p->pl->twm;
  g->keep_ld = (p->cache & PFK_KEEP_SRC) != 0;
  g->keep_st = (p->cache & PFK_KEEP_DST) != 0;
  int L = 1, tw = 0;
  for (int s = 0; s < g->nst; s++) {
    const bool col = s >= p->mix_n;
    if (s == p->mix_n) { L = 1; tw = g->ntw1; }
    const int n = col ? g->n1 : g->n2, lines = col ? g->n2 : g->n1;
    const int R = col ? p->pl->mix_rad[s - p->mix_n] : p->mix_rad[s];
    if (R > 16) return 1;
    PlaneStage *t = &g->st[s];
    t->R = R;
    t->nb = n / R;
    t->L = L;
    t->tw = tw;
    t->col = col;
    const int cap = nt * (R >= 16 ? 1 : 16 / R);   // butterflies the threads hold
    if (cap < t->nb) return 1;
    const int chunks = (lines + cap / t->nb - 1) / (cap / t->nb);
    t->lines = (lines + chunks - 1) / chunks;
    t->mdiv = recip(col ? t->lines : t->nb);
    t->mlen = recip(L);
    if (L > 1) tw += (R - 1) * L;
    L *= R;
  }
  return 0;
}

template <typename T>
static int launch_plane_t(const pfk_pass *p, const PlaneGeo &g, int nt, size_t lds,
                          const void *src, void *dst) {
  static size_t granted = 65536;
  static int ncu = 0;
  if (lds > granted) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_plane<T>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             160 * 1024);
    if (e != hipSuccess) { set_error("pfk_launch_pass(plane LDS)", e); return 1; }
    granted = 160 * 1024;
  }
  if (!ncu) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        ncu < 1)
      ncu = 1;
  }
  int64_t planes = 1;
  for (int i = 0; i < p->nb; i++) planes *= p->bext[i];
  if (planes <= 0) return 0;
  int64_t per = (int64_t)(160 * 1024 / lds);
  if (per > 16 / (nt / 64)) per = 16 / (nt / 64);
  const int64_t res = per * ncu, grid = planes < res ? planes : res;
  hipLaunchKernelGGL(k_plane<T>, dim3((unsigned)grid), dim3(nt), lds, g_stream, *p, g, planes,
                     (int)((planes - 1) % grid), (const T *)src, (T *)dst);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("pfk_launch_pass(plane)", e); return 1; }
  return 0;
}

int launch_plane(const pfk_pass *p, const void *src, void *dst) {
  PlaneGeo g;
  size_t lds;
  const int nt = plane_threads(p);
  if (plane_geo(p, nt, &g, &lds)) { set_error_msg("pfk: bad plane pass"); return 1; }
  return p->prec == PFK_F64 ? launch_plane_t<double>(p, g, nt, lds, src, dst)
                            : launch_plane_t<float>(p, g, nt, lds, src, dst);
}

}  // namespace pfk

extern "C" size_t pfk_plane_covers(const pfk_pass *p) {
  pfk::PlaneGeo g;
  size_t lds = 0;
  if (pfk_init() || pfk::g_generic_only) return 0;
  return pfk::plane_geo(p, pfk::plane_threads(p), &g, &lds) ? 0 : lds;
}
