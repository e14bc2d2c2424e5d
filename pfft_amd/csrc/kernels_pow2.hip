// kernels_pow2.hip -- dispatch of the power-of-two pass kernels (pow2_tile.hpp).
// Each length is instantiated in a translation unit of its precision and
// length range (kernels_pow2_f64_*.hip, kernels_pow2_f32_*.hip), so that they
// compile in parallel.
#include "pfk_internal.hpp"
#include "pow2_launch.hpp"

namespace pfk {

// A pass with every input and output position present and no modulation
// or adjoint weights runs the plain (PL) instantiations.
bool pass_plain(const pfk_pass *p) {
  if (p->zin || p->zout || p->imod.on || p->omod.on || p->hw || p->twn) return false;
  if (p->kind == PFK_C2C) return p->nin == p->nf && p->nout == p->nf;
  if (p->kind == PFK_R2C) return p->nin == p->n && p->nout == p->nf + 1;
  if (p->kind == PFK_C2R) return p->nin == p->nf + 1 && p->nout == p->n;
  return false;
}

// Tile width C (consecutive lines per workgroup) gives 128-byte segments:
// C = 8 for 16-byte FP64 complex, C = 16 for 8-byte FP32 complex (C = 4 / 8
// at the longest lengths, where the tile would exceed 128 KiB of LDS).
// E = 16 elements per thread from NF = 1024 on keeps the workgroup at
// <= 1024 threads; complex64 takes E = 16 from NF = 512 (512 threads in
// two radix-16 stages and a radix-2 one, 95-117 VGPRs without spills, two
// workgroups per CU: its column passes of the 512^3 pair 207-212 -> 200 us
// against E = 8 at 1024 threads).
static int launch_pow2_f64(const pfk_pass *p, const void *src, void *dst) {
  switch (p->nf) {
    case 64: return pow2_f64_64(p, src, dst);
    case 128: return pow2_f64_128(p, src, dst);
    case 256: return pow2_f64_256(p, src, dst);
    case 512: return pow2_f64_512(p, src, dst);
    case 1024: return pow2_f64_1024(p, src, dst);
    case 2048: return pow2_f64_2048(p, src, dst);
    case 4096: return pow2_f64_4096(p, src, dst);
    default: return 1;
  }
}

// alternative (narrower) tiles: half the lines per workgroup, half the LDS
static int launch_pow2_f64n(const pfk_pass *p, const void *src, void *dst) {
  switch (p->nf) {
    case 64: return pow2_f64n_64(p, src, dst);
    case 128: return pow2_f64n_128(p, src, dst);
    case 256: return pow2_f64n_256(p, src, dst);
    case 512: return pow2_f64n_512(p, src, dst);
    case 1024: return pow2_f64n_1024(p, src, dst);
    case 2048: return pow2_f64n_2048(p, src, dst);
    case 4096: return pow2_f64n_4096(p, src, dst);
    default: return 1;
  }
}

static int launch_pow2_f32(const pfk_pass *p, const void *src, void *dst) {
  switch (p->nf) {
    case 64: return pow2_f32_64(p, src, dst);
    case 128: return pow2_f32_128(p, src, dst);
    case 256: return pow2_f32_256(p, src, dst);
    case 512: return pow2_f32_512(p, src, dst);
    case 1024: return pow2_f32_1024(p, src, dst);
    case 2048: return pow2_f32_2048(p, src, dst);
    case 4096: return pow2_f32_4096(p, src, dst);
    default: return 1;
  }
}

static int launch_pow2_f32n(const pfk_pass *p, const void *src, void *dst) {
  switch (p->nf) {
    case 64: return pow2_f32n_64(p, src, dst);
    case 128: return pow2_f32n_128(p, src, dst);
    case 256: return pow2_f32n_256(p, src, dst);
    case 512: return pow2_f32n_512(p, src, dst);
    case 1024: return pow2_f32n_1024(p, src, dst);
    case 2048: return pow2_f32n_2048(p, src, dst);
    case 4096: return pow2_f32n_4096(p, src, dst);
    default: return 1;
  }
}

int fast_covers(const pfk_pass *p) {
  if (p->n1 || p->dec_in || p->dec_out) return 0;   // long lines, decimated steps
  if (p->twn && (p->kind != PFK_C2C || (p->variant & ~4))) return 0;   // default tiles only
  if (p->kind != PFK_C2C && p->kind != PFK_R2C && p->kind != PFK_C2R) return 0;
  const int64_t nf = p->nf;
  if (nf < 64 || nf > 4096 || (nf & (nf - 1))) return 0;
  if (p->kind == PFK_R2C) {
    // real input: contiguous, not embedded
    if (p->n != 2 * nf || p->sin != 1 || p->zin != 0 || p->nin != p->n) return 0;
    if (p->hw == 1) return 0;
  }
  if (p->kind == PFK_C2R) {
    if (p->n != 2 * nf || p->sout != 1 || p->zout != 0 || p->nout != p->n) return 0;
    if (p->hw == 2) return 0;
  }
  if (p->kind == PFK_C2C && p->hw) return 0;
  return 1;
}

int launch_fast(const pfk_pass *p, const void *src, void *dst) {
  if (g_generic_only || p->variant == 1 || !fast_covers(p)) return 1;
  if ((p->variant & 3) == 2)
    return (p->prec == PFK_F64) ? launch_pow2_f64n(p, src, dst)
                                : launch_pow2_f32n(p, src, dst);
  return (p->prec == PFK_F64) ? launch_pow2_f64(p, src, dst) : launch_pow2_f32(p, src, dst);
}

}  // namespace pfk

extern "C" int pfk_pass_plain(const pfk_pass *p) { return pfk::pass_plain(p) ? 1 : 0; }

extern "C" int pfk_pass_kernels(const pfk_pass *p) {
  if (pfk::g_generic_only) return 0;
  int m = 0;
  if (pfk::mfma_covers(p)) m |= PFK_HAS_MFMA;
  if (pfk::fast_covers(p)) m |= PFK_HAS_POW2;
  if (pfk::small_covers(p)) m |= PFK_HAS_SMALL;
  if (pfk::mixed_covers(p)) m |= PFK_HAS_MIXED;
  return m;
}
