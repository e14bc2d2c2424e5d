// pow2_launch.hpp -- launchers of the power-of-two pass kernels, one per
// length, precision and tile width (n: half the lines per workgroup).
#pragma once
#include "pfk_internal.hpp"

namespace pfk {

bool pass_plain(const pfk_pass *p);

int pow2_f64_64(const pfk_pass *p, const void *src, void *dst);
int pow2_f64_128(const pfk_pass *p, const void *src, void *dst);
int pow2_f64_256(const pfk_pass *p, const void *src, void *dst);
int pow2_f64_512(const pfk_pass *p, const void *src, void *dst);
int pow2_f64_1024(const pfk_pass *p, const void *src, void *dst);
int pow2_f64_2048(const pfk_pass *p, const void *src, void *dst);
int pow2_f64_4096(const pfk_pass *p, const void *src, void *dst);
int pow2_f32_64(const pfk_pass *p, const void *src, void *dst);
int pow2_f32_128(const pfk_pass *p, const void *src, void *dst);
int pow2_f32_256(const pfk_pass *p, const void *src, void *dst);
int pow2_f32_512(const pfk_pass *p, const void *src, void *dst);
int pow2_f32_1024(const pfk_pass *p, const void *src, void *dst);
int pow2_f32_2048(const pfk_pass *p, const void *src, void *dst);
int pow2_f32_4096(const pfk_pass *p, const void *src, void *dst);
int pow2_f64n_64(const pfk_pass *p, const void *src, void *dst);
int pow2_f64n_128(const pfk_pass *p, const void *src, void *dst);
int pow2_f64n_256(const pfk_pass *p, const void *src, void *dst);
int pow2_f64n_512(const pfk_pass *p, const void *src, void *dst);
int pow2_f64n_1024(const pfk_pass *p, const void *src, void *dst);
int pow2_f64n_2048(const pfk_pass *p, const void *src, void *dst);
int pow2_f64n_4096(const pfk_pass *p, const void *src, void *dst);
int pow2_f32n_64(const pfk_pass *p, const void *src, void *dst);
int pow2_f32n_128(const pfk_pass *p, const void *src, void *dst);
int pow2_f32n_256(const pfk_pass *p, const void *src, void *dst);
int pow2_f32n_512(const pfk_pass *p, const void *src, void *dst);
int pow2_f32n_1024(const pfk_pass *p, const void *src, void *dst);
int pow2_f32n_2048(const pfk_pass *p, const void *src, void *dst);
int pow2_f32n_4096(const pfk_pass *p, const void *src, void *dst);

}  // namespace pfk
