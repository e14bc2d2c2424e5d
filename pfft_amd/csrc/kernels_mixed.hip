// kernels_mixed.hip -- launch geometry of the mixed-radix kernel
// (mixed_tile.hpp).
#include "mixed_tile.hpp"

namespace pfk {

int launch_mixed_f64(const pfk_pass *p, const MixGeo &g, int nt, size_t lds, const void *src,
                     void *dst);
int launch_mixed_f32(const pfk_pass *p, const MixGeo &g, int nt, size_t lds, const void *src,
                     void *dst);
int launch_mixed_r2r_f64(const pfk_pass *p, const MixGeo &g, int nt, size_t lds,
                         const void *src, void *dst);
int launch_mixed_r2r_f32(const pfk_pass *p, const MixGeo &g, int nt, size_t lds,
                         const void *src, void *dst);

static size_t mix_lds(const MixGeo *g, size_t esz) {
  return (size_t)g->C * (32 + (size_t)(g->big + 1) * g->pitch * esz) + (size_t)g->ntw * esz;
}

static bool even_strides(const pfk_pass *p, bool in) {
  if ((in ? p->tsin : p->tsout) & 1) return false;
  for (int i = 0; i < p->nb; i++)
    if ((in ? p->bsin[i] : p->bsout[i]) & 1) return false;
  return true;
}

// Launch geometry of a covered pass; returns the workgroup size, 0 if the
// line does not fit.
static int mixed_geo(const pfk_pass *p, MixGeo *g, const void *src, const void *dst) {
  const bool f64 = p->prec == PFK_F64;
  const size_t esz = f64 ? 16 : 8;
  const bool r2r = p->kind == PFK_R2R;
  const int nf = !r2r ? (int)p->nf
                 : pfk_r2r_mode(p->r2r) == 0 ? (int)(pfk_r2r_inner_len(p->r2r, p->n) / 2)
                                             : (int)(p->n / 2);
  g->m = nf;
  int L = 1, off = 0;
  g->nst = p->mix_n;
  g->big = 0;
  for (int s = 0; s < p->mix_n; s++) {
    const int R = p->mix_rad[s];
    g->rad[s] = R;
    g->nb[s] = nf / R;
    g->len[s] = L;
    g->off[s] = off;
    if (s) off += (R - 1) * L;
    g->offr[s] = off;
    if (R > 16) {
      off += R;
      g->big = 1;
    }
    g->mpair[s] = recip((int64_t)((R + 1) / 2) * (nf / R));
    g->mnb[s] = recip(nf / R);
    g->mlen[s] = recip(L);
    L *= R;
  }
  const bool real = p->kind != PFK_C2C, even = !(p->n & 1);
  int rows = (p->kind == PFK_C2R && even) ? nf + 1 : nf;   // complex slots of a line
  if (r2r && pfk_r2r_mode(p->r2r) == 1) rows = nf + 1;   // r2r_put
  const size_t ua = 2 * (f64 ? sizeof(double) : sizeof(float));
  g->lm_ld = p->sin == 1;
  g->lm_st = p->sout == 1;
  g->plain = !real && p->nin == nf && p->nout == nf && !p->zin && !p->zout && !p->imod.on &&
             !p->omod.on;
  g->vec = 0;
  if (p->kind == PFK_R2C && even)
    g->vec = p->sin == 1 && p->nin == p->n && !p->zin && !p->imod.on && even_strides(p, true) &&
             (uintptr_t)src % ua == 0;
  if (p->kind == PFK_C2R && even)
    g->vec = p->sout == 1 && p->nout == p->n && !p->zout && !p->omod.on &&
             even_strides(p, false) && (uintptr_t)dst % ua == 0;
  g->ntw = off;
  g->mload = recip(r2r ? p->n : rows);
  g->mstore = recip(r2r && pfk_r2r_mode(p->r2r) == 0 ? nf + 1 : p->nout);
  g->mrow = recip(nf);
  g->keep_ld = (p->cache & PFK_KEEP_SRC) != 0;
  g->keep_st = (p->cache & PFK_KEEP_DST) != 0;
  // Lines per tile.  Where a side runs across the lines: one 128-byte segment
  // of them (half of it moved 360x300x250 complex128 column passes from 189 /
  // 221 to 270 / 258 us, twice changed nothing).  Where both sides run along
  // the lines no width is needed and small tiles interleave better: 16 KiB for
  // real and complex64 lines (250-point complex64 97 us against 104 at 32 KiB,
  // r2c of 250 117 against 131), 32 KiB for complex128 (178 against 184).
  // Halved while the tile exceeds 80 KiB (two workgroups per CU) or 512 threads,
  // and, down to the segment (two lines along the lines), while the pass has
  // fewer than two tiles per CU.  A matrix-core stage takes 8 lines at least.
  // r2r tiles go below the segment, to 4 lines, while the pass has fewer than two
  // tiles per CU: such a pass is bound by what one workgroup does to one tile
  // (single-precision plans, three launches a pass / segments / 4 lines: 1024x128x2
  // 83 / 79 / 61 us with kinds up to 1.23 times the three launches, 128x128x8 94 /
  // 81 / 56, 64x64x64 85 / 62 / 45; 8 lines 70, 65, 45).
  int64_t lines = p->text;
  for (int i = 0; i < p->nb; i++) lines *= p->bext[i];
  const int cmin = g->big ? 8 : 1;
  const int seg = (int)(128 / esz) * (r2r ? 2 : 1);   // lines of a 128-byte segment
  const int cseg = (g->lm_ld && g->lm_st) ? (g->big ? 8 : 2) : seg;
  const size_t tile = real || !f64 || !(g->lm_ld && g->lm_st) ? 16384 : 32768;
  int C = (g->lm_ld && g->lm_st) ? 1 : seg;
  while (C < 64 && (size_t)(2 * C) * rows * esz <= tile) C *= 2;
  if (C < cmin) C = cmin;
  while (C > cseg && lines < 512 * (int64_t)C) C /= 2;
  bool few = false;
  for (;; C /= 2) {
    // row pitch of 2 slots modulo the 256 bytes of a bank cycle, so that 8 (16)
    // lines x 2 positions spread over all banks; consecutive positions do anyway,
    // and a first stage along the lines has an odd radix where there is one
    // (pfk_mix_factorize), so its stores do too
    const int cyc = (int)(256 / esz);
    int pitch = rows;
    while (C > 1 && pitch % cyc != 2) pitch++;
    g->C = C;
    g->pitch = pitch;
    g->logC = __builtin_ctz(C);
    int nt = C;
    if (g->big) nt = nf * C / 4 < 256 ? nf * C / 4 : 256;
    if (nt < C) nt = C;
    for (int s = 0; s < g->nst; s++) {
      if (g->rad[s] > 16) continue;
      const int per = g->rad[s] >= 16 ? 1 : 16 / g->rad[s];
      const int need = (g->nb[s] * C + per - 1) / per;
      if (need > nt) nt = need;
    }
    nt = (nt + 63) / 64 * 64;
    const size_t lds = mix_lds(g, esz);
    // r2r: threads beyond the butterflies for the steps before and after the
    // transform, up to 16 waves a CU at the tile's LDS
    const int nt16 = 64 * (int)((16 * lds + 160 * 1024 - 1) / (160 * 1024));
    if (r2r && nt < nt16 && nt16 <= 512) nt = nt16;
    // rows of tiles where rounding them up wastes at most 1/10
    const int64_t up = (p->text + C - 1) / C * C;
    g->text = (up - p->text) * 10 <= p->text ? up : p->text;
    // r2r lines too long for half a segment, or with matrix-core stages, keep the
    // three launches
    if (r2r && g->big) return 0;
    if (r2r && !(g->lm_ld && g->lm_st) && C < seg / 2 && !few) return 0;
    if ((nt <= 512 && lds <= 80 * 1024) || (C == cmin && nt <= 512 && lds <= 158 * 1024)) {
      if (!r2r || C <= 4 || lines >= 512 * (int64_t)C) return nt;
      few = true;
      continue;
    }
    if (C == cmin) return 0;
  }
}

int mixed_covers(const pfk_pass *p) {
  if (!p->twm || p->mix_n < 1 || p->n1 || p->dec_in || p->dec_out || p->twn) return 0;
  if (p->kind == PFK_R2R) {
    if (p->r2r_path != 1) return 0;
  } else if (p->kind != PFK_C2C && p->kind != PFK_R2C && p->kind != PFK_C2R) {
    return 0;
  }
  if (p->kind == PFK_C2C && p->hw) return 0;
  MixGeo g;
  return mixed_geo(p, &g, nullptr, nullptr) > 0;
}

int launch_mixed(const pfk_pass *p, const void *src, void *dst) {
  if (!mixed_covers(p)) return 1;
  MixGeo g;
  const int nt = mixed_geo(p, &g, src, dst);
  if (p->kind == PFK_R2R)
    return p->prec == PFK_F64 ? launch_mixed_r2r_f64(p, g, nt, mix_lds(&g, 16), src, dst)
                              : launch_mixed_r2r_f32(p, g, nt, mix_lds(&g, 8), src, dst);
  return p->prec == PFK_F64 ? launch_mixed_f64(p, g, nt, mix_lds(&g, 16), src, dst)
                            : launch_mixed_f32(p, g, nt, mix_lds(&g, 8), src, dst);
}

}  // namespace pfk
