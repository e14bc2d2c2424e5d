// dft_regs.hpp -- in-place DFTs of 2 to 16 complex values held in registers.
#pragma once
#include "pass_access.hpp"

namespace pfk {

template <typename T>
__device__ __forceinline__ C2<T> cadd(C2<T> a, C2<T> b) { return C2<T>{a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ C2<T> csub(C2<T> a, C2<T> b) { return C2<T>{a.x - b.x, a.y - b.y}; }
// multiply by SIGN*i
template <int SIGN, typename T>
__device__ __forceinline__ C2<T> mul_si(C2<T> a) {
  return SIGN < 0 ? C2<T>{a.y, -a.x} : C2<T>{-a.y, a.x};
}

template <int SIGN, typename T>
__device__ __forceinline__ void dft2(C2<T> &a, C2<T> &b) {
  const C2<T> s = cadd(a, b), d = csub(a, b);
  a = s;
  b = d;
}

// in-place DFT-4 of (a0,a1,a2,a3) with W4 = SIGN*i
template <int SIGN, typename T>
__device__ __forceinline__ void dft4(C2<T> &a0, C2<T> &a1, C2<T> &a2, C2<T> &a3) {
  const C2<T> c0 = cadd(a0, a2), c1 = csub(a0, a2);
  const C2<T> c2 = cadd(a1, a3), c3 = mul_si<SIGN>(csub(a1, a3));
  a0 = cadd(c0, c2);
  a2 = csub(c0, c2);
  a1 = cadd(c1, c3);
  a3 = csub(c1, c3);
}

// in-place DFT-8 of v[0..7] (natural order in and out)
template <int SIGN, typename T>
__device__ __forceinline__ void dft8(C2<T> *v) {
  C2<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
  C2<T> o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  dft4<SIGN>(e0, e1, e2, e3);
  dft4<SIGN>(o0, o1, o2, o3);
  const T s = (T)0.70710678118654752440084436210484903928L;
  // W8^1 = s(1 + SIGN i), W8^2 = SIGN i, W8^3 = s(-1 + SIGN i)
  const C2<T> t1{s * (o1.x - (SIGN) * o1.y), s * (o1.y + (SIGN) * o1.x)};
  const C2<T> t2 = mul_si<SIGN>(o2);
  const C2<T> t3{s * (-o3.x - (SIGN) * o3.y), s * (-o3.y + (SIGN) * o3.x)};
  v[0] = cadd(e0, o0);
  v[4] = csub(e0, o0);
  v[1] = cadd(e1, t1);
  v[5] = csub(e1, t1);
  v[2] = cadd(e2, t2);
  v[6] = csub(e2, t2);
  v[3] = cadd(e3, t3);
  v[7] = csub(e3, t3);
}

// in-place DFT-16 of v[0..15] as 4x4: DFT-4 over stride-4 groups, twiddle
// W16^(r*q), DFT-4 across groups
template <int SIGN, typename T>
__device__ __forceinline__ void dft16(C2<T> *v) {
#pragma unroll
  for (int r = 0; r < 4; ++r) dft4<SIGN>(v[r], v[r + 4], v[r + 8], v[r + 12]);
  // v[r + 4q] now holds sub-DFT output q of group r; multiply by W16^(r*q)
  const T c1 = (T)0.92387953251128675612818318939678828682L;  // cos(pi/8)
  const T s1 = (T)0.38268343236508977172845998403039886676L;  // sin(pi/8)
  const T h = (T)0.70710678118654752440084436210484903928L;
  const T S = (T)SIGN;
  // W16^1 = c1 + S i s1, W16^2 = h + S i h, W16^3 = s1 + S i c1,
  // W16^4 = S i, W16^6 = -h + S i h, W16^9 = -c1 - S i s1
  const C2<T> w1{c1, S * s1}, w2{h, S * h}, w3{s1, S * c1};
  const C2<T> w6{-h, S * h}, w9{-c1, -S * s1};
  v[5] = cmul(v[5], w1);
  v[9] = cmul(v[9], w2);
  v[13] = cmul(v[13], w3);
  v[6] = cmul(v[6], w2);
  v[10] = mul_si<SIGN>(v[10]);
  v[14] = cmul(v[14], w6);
  v[7] = cmul(v[7], w3);
  v[11] = cmul(v[11], w6);
  v[15] = cmul(v[15], w9);
#pragma unroll
  for (int q = 0; q < 4; ++q) dft4<SIGN>(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
  // output k = q + 4*s sits in v[4q + s]: transpose the 4x4 index
  C2<T> o[16];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int t = 0; t < 4; ++t) o[q + 4 * t] = v[4 * q + t];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = o[k];
}

// cos and sin of 2 pi m / R, m = 1 .. (R-1)/2
template <int R>
struct OddC;
template <>
struct OddC<3> {
  static constexpr double c[1] = {-0.50000000000000000000};
  static constexpr double s[1] = {0.86602540378443859659};
};
template <>
struct OddC<5> {
  static constexpr double c[2] = {0.30901699437494745126, -0.80901699437494745126};
  static constexpr double s[2] = {0.95105651629515353118, 0.58778525229247313710};
};
template <>
struct OddC<7> {
  static constexpr double c[3] = {0.62348980185873348336, -0.22252093395631439288, -0.90096886790241914600};
  static constexpr double s[3] = {0.78183148246802980363, 0.97492791218182361934, 0.43388373911755812040};
};
template <>
struct OddC<9> {
  static constexpr double c[4] = {0.76604444311897801345, 0.17364817766693035894, -0.50000000000000000000, -0.93969262078590842791};
  static constexpr double s[4] = {0.64278760968653936292, 0.98480775301220802032, 0.86602540378443859659, 0.34202014332566871291};
};
template <>
struct OddC<11> {
  static constexpr double c[5] = {0.84125353283118120551, 0.41541501300188643508, -0.14231483827328514358, -0.65486073394528510061, -0.95949297361449736865};
  static constexpr double s[5] = {0.54064081745559755543, 0.90963199535451833011, 0.98982144188093268422, 0.75574957435425826890, 0.28173255684142967104};
};
template <>
struct OddC<13> {
  static constexpr double c[6] = {0.88545602565320991051, 0.56806474673115581187, 0.12053668025532304764, -0.35460488704253562142, -0.74851074817110108128, -0.97094181742605201180};
  static constexpr double s[6] = {0.46472317204376856203, 0.82298386589365635224, 0.99270887409805397272, 0.93501624268541483342, 0.66312265824079519305, 0.23931566428755776665};
};

// in-place DFT of an odd length: outputs q and R-q share the sums
// C_q = x_0 + sum_r cos(2 pi q r/R) (x_r + x_(R-r)) and
// S_q = sum_r sin(2 pi q r/R) (x_r - x_(R-r)), r <= (R-1)/2, a quarter of the
// multiplications of the direct sum.  For 3 and 5 the sine terms are added to
// C_q one by one, which rounds less often (9 in this form and not as 3 x 3 for
// the same reason: 162 points in float err by 9.6e-8 against 1.09e-7, summed
// directly by 9.5e-8).
template <int R, int SIGN, typename T>
__device__ __forceinline__ void dft_odd(C2<T> *v) {
  constexpr int H = (R - 1) / 2;
  C2<T> a[H], b[H];
  C2<T> sum = v[0];
#pragma unroll
  for (int r = 1; r <= H; ++r) {
    a[r - 1] = cadd(v[r], v[R - r]);
    b[r - 1] = csub(v[r], v[R - r]);
    sum = cadd(sum, a[r - 1]);
  }
#pragma unroll
  for (int q = 1; q <= H; ++q) {
    C2<T> C = v[0];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      const int m = q * r % R, mm = m > H ? R - m : m;
      if (mm == 0) {
        C = cadd(C, a[r - 1]);
      } else {
        const T c = (T)OddC<R>::c[mm - 1];
        C.x += c * a[r - 1].x;
        C.y += c * a[r - 1].y;
      }
    }
    C2<T> p = C, n = C, S{0, 0};
    bool any = false;
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      const int m = q * r % R, mm = m > H ? R - m : m;
      if (mm == 0) continue;
      const T s = (T)(m > H ? -OddC<R>::s[mm - 1] : OddC<R>::s[mm - 1]) * (T)SIGN;
      if (R <= 5) {
        p.x -= s * b[r - 1].y;
        p.y += s * b[r - 1].x;
        n.x += s * b[r - 1].y;
        n.y -= s * b[r - 1].x;
      } else if (!any) {
        S = C2<T>{s * b[r - 1].x, s * b[r - 1].y};
        any = true;
      } else {
        S.x += s * b[r - 1].x;
        S.y += s * b[r - 1].y;
      }
    }
    v[q] = R <= 5 ? p : C2<T>{C.x - S.y, C.y + S.x};
    v[R - q] = R <= 5 ? n : C2<T>{C.x + S.y, C.y - S.x};
  }
  v[0] = sum;
}

template <int R, int SIGN, typename T>
__device__ __forceinline__ void dft_any(C2<T> *v);

// in-place DFT of R1 * R2, coprime (Good-Thomas: both index maps are
// permutations, no twiddles)
template <int R1, int R2, int SIGN, typename T>
__device__ __forceinline__ void dft_coprime(C2<T> *v) {
  constexpr int R = R1 * R2;
  C2<T> x[R2][R1];
#pragma unroll
  for (int i = 0; i < R2; ++i) {
#pragma unroll
    for (int j = 0; j < R1; ++j) x[i][j] = v[(R2 * j + R1 * i) % R];
    dft_any<R1, SIGN>(x[i]);
  }
  // output k has k = j (mod R1), k = i (mod R2)
#pragma unroll
  for (int j = 0; j < R1; ++j) {
    C2<T> y[R2];
#pragma unroll
    for (int i = 0; i < R2; ++i) y[i] = x[i][j];
    dft_any<R2, SIGN>(y);
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (k % R1 == j) v[k] = y[k % R2];
  }
}

// in-place DFT of 2 to 16 values, natural order in and out
template <int R, int SIGN, typename T>
__device__ __forceinline__ void dft_any(C2<T> *v) {
  if constexpr (R == 2) dft2<SIGN>(v[0], v[1]);
  else if constexpr (R == 4) dft4<SIGN>(v[0], v[1], v[2], v[3]);
  else if constexpr (R == 8) dft8<SIGN>(v);
  else if constexpr (R == 16) dft16<SIGN>(v);
  else if constexpr (R == 6) dft_coprime<2, 3, SIGN>(v);
  else if constexpr (R == 10) dft_coprime<2, 5, SIGN>(v);
  else if constexpr (R == 12) dft_coprime<4, 3, SIGN>(v);
  else if constexpr (R == 14) dft_coprime<2, 7, SIGN>(v);
  else if constexpr (R == 15) dft_coprime<3, 5, SIGN>(v);
  else dft_odd<R, SIGN>(v);
}

}  // namespace pfk
