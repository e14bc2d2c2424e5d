// mixed_tile.hpp -- pass computation of one tile of lines for any length whose
// prime factors fit the codelets (2..13, composite radices to 16) or the
// matrix cores (larger primes).
//
// Work split.  A workgroup transforms C lines held in LDS, [line][position].
// A stage of radix R is NB = nf/R butterflies per line; a thread takes whole
// butterflies (at most 16 values): it reads them into registers, multiplies the
// twiddles, transforms them with a straight-line codelet and writes them back
// (Stockham: output (b-k)*R + k + q*L of butterfly b, k = b mod L).  The first
// stage reads global memory instead of LDS and the last stage writes it, so a
// line of s stages makes s-1 trips through LDS.  Which lanes take which
// butterflies is free in every stage: on a side whose lines are contiguous
// consecutive lanes take consecutive butterflies of a line, else consecutive
// lines, so both sides coalesce whatever the layout.
//
// Twiddles come from a table in stage order, [stage][r][k], which a workgroup
// copies to LDS once and uses for all its tiles (read through the vector L1
// instead, the stages of a 360x300x250 complex128 transform took 15% longer).
// Only the forward table exists: a backward transform conjugates its input and
// its output.
//
// Primes above 13 (one stage each, radix R): with x_0 apart, the pair sums
// A_r = x_r + x_(R-r) and differences B_r = x_r - x_(R-r), r <= (R-1)/2, give
//   Y_q     = x_0 + sum_r cos(2 pi q r/R) A_r - i sum_r sin(2 pi q r/R) B_r,
//   Y_(R-q) = the same with + i,
// two dense real products over r for all lines and both components: matrix
// core work (16x16x4 tiles: 16 outputs q by 8 lines x {re, im} by 4 r).
//
// Bound: the HBM sweep, at 3.7-5.1 TB/s (0.7-1.5 for the general kernel, whose
// stages sum each output over its radix with a division per element).
// Forward+backward pairs, general kernel -> this one: c2c 360x300x250
// complex128 4.26 -> 1.28 ms, r2c 210x196x330 complex64 908 -> 210 us, c2c
// 29x27x31 complex128 142 -> 96 us.  Without any stage arithmetic and
// exchanges the first of these takes 1.07 ms.  Registers (128) and LDS leave
// 16 waves per CU in flight.
#pragma once
#include "dft_regs.hpp"

namespace pfk {

// Launch geometry of a mixed-radix pass, filled on the host (mixed_geo).
struct MixGeo {
  int C, logC, pitch;      // lines per tile, LDS row pitch in complex slots
  int nst;                 // stages
  int plain;               // every position present, no modulation or weights
  int lm_ld, lm_st;        // lanes along the lines on the load / store side
  int vec;                 // real side readable as aligned complex pairs
  int ntw;                 // entries of the stage table
  int big;                 // 1: some stage runs on the matrix cores (a second tile in LDS)
  int keep_ld, keep_st;    // ordinary instead of streaming accesses
  int64_t text;            // tile extent the lines are numbered by (mix_lines)
  int rad[PFK_MIX_MAXST], nb[PFK_MIX_MAXST], len[PFK_MIX_MAXST], off[PFK_MIX_MAXST];
  uint32_t mnb[PFK_MIX_MAXST], mlen[PFK_MIX_MAXST];   // reciprocals of nb, len
  int offr[PFK_MIX_MAXST];  // W_R table of a matrix-core stage
  uint32_t mload, mstore;  // reciprocals of the staged load / store loop lengths
  uint32_t mpair[PFK_MIX_MAXST], mrow;   // ... of the pair-sum loop, of nf
};

// i / d for i * d < 2^32 with m = ceil(2^32 / d) (m = 0: d = 1)
__device__ __forceinline__ int div_m(int i, uint32_t m) {
  return m ? (int)__umulhi((uint32_t)i, m) : i;
}

template <typename T>
struct MixCtx {
  const pfk_pass &P;
  const MixGeo &G;
  int nl;                    // lines of this tile (the last one may be ragged)
  const int64_t *so, *dof;   // LDS: source / destination offset of each line
  const T *src;
  T *dst;
  const C2<T> *tw;           // LDS: stage table
  C2<T> *lds, *lds2;         // the tile, the second one (G.big)
  T cj;   // -1 conjugates the input and the output of the forward transform
};

__device__ __forceinline__ int mix_slot(const MixGeo &G, int c, int p) {
  return c * G.pitch + p;
}

// 16 elements per thread and stage, whole butterflies
template <int R>
constexpr int mix_items() { return R >= 16 ? 1 : 16 / R; }

// element p of line c as the stages see it (complex; r2c even: the packed
// pair; odd real lines as complex).  C2R even lines do not come here (their
// half spectrum is staged).
template <typename T, int KIND>
__device__ __forceinline__ C2<T> mix_load(const MixCtx<T> &X, const int c, const int p) {
  const pfk_pass &P = X.P;
  const int64_t line = X.so[c < X.nl ? c : 0];
  C2<T> v;
  if constexpr (KIND == PFK_C2C) {
    const C2<T> *s = reinterpret_cast<const C2<T> *>(X.src) + line;
    const int j = p - (int)P.zin;
    const bool ok = j >= 0 && j < (int)P.nin;
    v = s[(int64_t)(ok ? j : 0) * P.sin];
    const T f = msign<T>(P.imod, j);
    v = ok ? C2<T>{v.x * f, v.y * f} : C2<T>{0, 0};
  } else if constexpr (KIND == PFK_R2C) {
    const T *s = X.src + line;
    const bool even = !(P.n & 1);
    const int j = (even ? 2 * p : p) - (int)P.zin, nin = (int)P.nin;
    const bool ok0 = j >= 0 && j < nin, ok1 = even && j + 1 >= 0 && j + 1 < nin;
    const T a = s[(int64_t)(ok0 ? j : 0) * P.sin];
    const T b = s[(int64_t)(ok1 ? j + 1 : 0) * P.sin];
    v.x = ok0 ? a * msign<T>(P.imod, j) : (T)0;
    v.y = ok1 ? b * msign<T>(P.imod, j + 1) : (T)0;
  } else {   // odd c2r: Hermitian extension of the half spectrum
    const C2<T> *s = reinterpret_cast<const C2<T> *>(X.src) + line;
    const int n = (int)P.n;
    const bool up = 2 * p > n;
    const int k = up ? n - p : p, j = k - (int)P.zin;
    const bool ok = j >= 0 && j < (int)P.nin;
    v = s[(int64_t)(ok ? j : 0) * P.sin];
    T f = msign<T>(P.imod, j);
    if (P.hw == 1 && k != 0) f *= (T)0.5;
    v.x = ok ? v.x * f : (T)0;
    v.y = (ok && k != 0) ? (up ? -v.y : v.y) * f : (T)0;
  }
  v.y *= X.cj;
  return v;
}

// output p of line c (not the even r2c combine)
template <typename T, int KIND>
__device__ __forceinline__ void mix_store(const MixCtx<T> &X, const int c, const int p,
                                          C2<T> v) {
  const pfk_pass &P = X.P;
  if (c >= X.nl) return;
  const int64_t line = X.dof[c];
  v.y *= X.cj;
  if constexpr (KIND == PFK_C2R) {
    T *d = X.dst + line;
    const bool even = !(P.n & 1);
    const int j = (even ? 2 * p : p) - (int)P.zout, nout = (int)P.nout;
    if (j >= 0 && j < nout) d[(int64_t)j * P.sout] = v.x * msign<T>(P.omod, j);
    if (even && j + 1 >= 0 && j + 1 < nout)
      d[(int64_t)(j + 1) * P.sout] = v.y * msign<T>(P.omod, j + 1);
  } else {
    C2<T> *d = reinterpret_cast<C2<T> *>(X.dst) + line;
    const int j = p - (int)P.zout;
    if (j < 0 || j >= (int)P.nout) return;
    T f = msign<T>(P.omod, j);
    if (KIND == PFK_R2C && P.hw == 2 && p != 0) f *= (T)2;   // odd n: no Nyquist
    d[(int64_t)j * P.sout] = C2<T>{v.x * f, v.y * f};
  }
}

// Z_k = E_k + i O_k of an even c2r line from its staged half spectrum
// (E = X_k + conj X_(h-k), O = (X_k - conj X_(h-k)) W_n^k)
template <typename T>
__device__ __forceinline__ C2<T> c2r_pack(const MixCtx<T> &X, const int c, const int k) {
  const int h = (int)X.P.nf;
  const C2<T> a = X.lds[mix_slot(X.G, c, k)], b = X.lds[mix_slot(X.G, c, h - k)];
  C2<T> z;
  if (k == 0) {
    z = C2<T>{a.x + b.x, a.x - b.x};
  } else {
    const C2<T> E{a.x + b.x, a.y - b.y};
    const C2<T> O =
        cmul(C2<T>{a.x - b.x, a.y + b.y}, reinterpret_cast<const C2<T> *>(X.P.rtw)[k]);
    z = C2<T>{E.x - O.y, E.y + O.x};
  }
  z.y *= X.cj;
  return z;
}

// one stage of a codelet radix
template <typename T, int KIND, int R>
__device__ __forceinline__ void mix_stage(const MixCtx<T> &X, const int s) {
  constexpr int I = mix_items<R>();
  const MixGeo &G = X.G;
  const bool first = s == 0, last = s == G.nst - 1;
  const bool packed = KIND == PFK_C2R && !(X.P.n & 1);   // first stage reads LDS too
  const bool z_lds = KIND == PFK_R2C && !(X.P.n & 1);    // last stage writes LDS too
  const int NB = G.nb[s], L = G.len[s], items = NB * G.C;
  const bool lm = first ? G.lm_ld : G.lm_st;
  const C2<T> *tw = X.tw + G.off[s];
  C2<T> v[I][R];
  int cs[I], bs[I], ks[I];
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int it0 = (int)threadIdx.x + i * (int)blockDim.x;
    const int it = it0 < items ? it0 : 0;
    if (lm) {
      cs[i] = div_m(it, G.mnb[s]);
      bs[i] = it - cs[i] * NB;
    } else {
      cs[i] = it & (G.C - 1);
      bs[i] = it >> G.logC;
    }
    ks[i] = last ? bs[i] : bs[i] - div_m(bs[i], G.mlen[s]) * L;
    if (it0 >= items) cs[i] = G.C;   // no store (below and in mix_store: c >= nl)
  }
  if (first && !packed && KIND != PFK_C2R && (G.plain || G.vec)) {
    // every position present, no modulation: one address per butterfly and a
    // uniform step
    const int64_t sin = KIND == PFK_C2C ? X.P.sin : 1, step = NB * sin;
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int64_t line = X.so[cs[i] < X.nl ? cs[i] : 0];
      const C2<T> *a = (KIND == PFK_C2C ? reinterpret_cast<const C2<T> *>(X.src) + line
                                        : reinterpret_cast<const C2<T> *>(X.src + line)) +
                       bs[i] * sin;
      if (G.keep_ld) {
#pragma unroll
        for (int r = 0; r < R; ++r) v[i][r] = a[r * step];
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) v[i][r] = ld_stream(a + r * step);
      }
    }
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r].y *= X.cj;
  } else if (first && !packed) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = mix_load<T, KIND>(X, cs[i], bs[i] + r * NB);
  } else if (first) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int r = 0; r < R; ++r)
        v[i][r] = c2r_pack(X, cs[i] < G.C ? cs[i] : 0, bs[i] + r * NB);
  } else {
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int c = cs[i] < G.C ? cs[i] : 0;
      v[i][0] = X.lds[mix_slot(G, c, bs[i])];
#pragma unroll
      for (int r = 1; r < R; ++r)
        v[i][r] = cmul(X.lds[mix_slot(G, c, bs[i] + r * NB)], tw[(r - 1) * L + ks[i]]);
    }
  }
#pragma unroll
  for (int i = 0; i < I; ++i) dft_any<R, -1>(v[i]);
  if (last && !z_lds && KIND != PFK_R2C && (G.plain || G.vec)) {
        const int64_t sout = KIND == PFK_C2C ? X.P.sout : 1, step = NB * sout;
#pragma unroll
    for (int i = 0; i < I; ++i) {
      if (cs[i] >= X.nl) continue;
      const int64_t line = X.dof[cs[i]];
      C2<T> *a = (KIND == PFK_C2C ? reinterpret_cast<C2<T> *>(X.dst) + line
                                  : reinterpret_cast<C2<T> *>(X.dst + line)) +
                 bs[i] * sout;
#pragma unroll
      for (int q = 0; q < R; ++q) v[i][q].y *= X.cj;
      st_batch<R>(G.keep_st, v[i], [&](int q) { return a + q * step; });
    }
    return;
  }
  if (last && !z_lds) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int q = 0; q < R; ++q) mix_store<T, KIND>(X, cs[i], bs[i] + q * NB, v[i][q]);
    return;
  }
  if (!first || packed) lds_barrier();   // every thread has read its inputs
#pragma unroll
  for (int i = 0; i < I; ++i)
    if (cs[i] < G.C) {
      const int o = (bs[i] - ks[i]) * R + ks[i];
#pragma unroll
      for (int q = 0; q < R; ++q) X.lds[mix_slot(G, cs[i], o + q * L)] = v[i][q];
    }
  lds_barrier();
}

__device__ __forceinline__ void mfma16(double a, double b,
                                       double __attribute__((ext_vector_type(4))) &c) {
  c = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void mfma16(float a, float b,
                                       float __attribute__((ext_vector_type(4))) &c) {
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// one stage of a prime radix above 13 on the matrix cores (C a multiple of 8)
template <typename T, int KIND>
__device__ __forceinline__ void mix_big(const MixCtx<T> &X, const int s) {
  typedef T v4 __attribute__((ext_vector_type(4)));
  const MixGeo &G = X.G;
  const bool first = s == 0, last = s == G.nst - 1;
  const bool packed = KIND == PFK_C2R && !(X.P.n & 1);
  const bool z_lds = KIND == PFK_R2C && !(X.P.n & 1);
  const int R = G.rad[s], NB = G.nb[s], L = G.len[s], H = (R - 1) / 2, NT = blockDim.x;
  const C2<T> *tw = X.tw + G.off[s], *tr = X.tw + G.offr[s];
  // pair sums A_r at position r*NB + b, differences B_r at (R-r)*NB + b of the
  // second tile, U pairs per thread at a time
  constexpr int U = 4;
  const int cnt = (H + 1) * NB, total = G.C * cnt;
  const bool lm = first && !packed && G.lm_ld;
  for (int i0 = threadIdx.x; i0 < total; i0 += U * NT) {
    C2<T> x[U], y[U];
    int cc[U], pp[U], mm[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u * NT < total ? i0 + u * NT : i0;
      if (lm) {
        cc[u] = div_m(i, G.mpair[s]);
        pp[u] = i - cc[u] * cnt;
      } else {
        cc[u] = i & (G.C - 1);
        pp[u] = i >> G.logC;
      }
      const int r = div_m(pp[u], G.mnb[s]), b = pp[u] - r * NB;
      mm[u] = r ? (R - r) * NB + b : pp[u];
      if (first && !packed) {
        x[u] = mix_load<T, KIND>(X, cc[u], pp[u]);
        y[u] = mix_load<T, KIND>(X, cc[u], mm[u]);
      } else if (first) {
        x[u] = c2r_pack(X, cc[u], pp[u]);
        y[u] = c2r_pack(X, cc[u], mm[u]);
      } else {
        const int k = b - div_m(b, G.mlen[s]) * L;
        x[u] = X.lds[mix_slot(G, cc[u], pp[u])];
        y[u] = X.lds[mix_slot(G, cc[u], mm[u])];
        if (r) {
          x[u] = cmul(x[u], tw[(r - 1) * L + k]);
          y[u] = cmul(y[u], tw[(R - r - 1) * L + k]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool dc = pp[u] == mm[u];
      const C2<T> a = dc ? x[u] : cadd(x[u], y[u]);
      X.lds2[mix_slot(G, cc[u], pp[u])] = a;
      if (!dc) X.lds2[mix_slot(G, cc[u], mm[u])] = csub(x[u], y[u]);
    }
  }
  lds_barrier();
  // Y_q and Y_(R-q), q <= H: a wave takes one butterfly of 8 lines and 16
  // values of q.  Operand columns are (line, re/im); the table operand is
  // W_R^(q r mod R), its index advanced by 4 q per step of 4 r.
  const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4, part = col >> 3;
  const int MT = (H + 16) / 16, LG = G.C >> 3, units = NB * LG * MT;
  for (int un = threadIdx.x >> 6; un < units; un += NT >> 6) {
    const int mt = un % MT, v = un / MT, g = v % LG, b = v / LG;
    const int c = g * 8 + (col & 7), q = mt * 16 + col;
    const T *row = reinterpret_cast<const T *>(X.lds2 + mix_slot(G, c, b)) + part;
    v4 ac = {0, 0, 0, 0}, as = {0, 0, 0, 0};
    int m = (q * (1 + kq)) % R;
    const int dm = (4 * q) % R;
    for (int r0 = 1; r0 <= H; r0 += 4) {
      const int r = r0 + kq;
      const bool ok = r <= H;
      const int rr = ok ? r : H;
      const C2<T> w = tr[m];
      const T ba = row[2 * (rr * NB)], bb = row[2 * ((R - rr) * NB)];
      mfma16(ok ? w.x : (T)0, ba, ac);
      mfma16(ok ? w.y : (T)0, bb, as);
      m += dm;
      m = m >= R ? m - R : m;
    }
    const T x0 = row[0];
    const int k = b - div_m(b, G.mlen[s]) * L, o = (b - k) * R + k;
    T *d0 = reinterpret_cast<T *>(X.lds + mix_slot(G, c, o)) + part;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // i S': the other component of S' (lane ^ 8), negated for the real part
      const T t = __shfl_xor((T)as[i], 8);
      const T e = x0 + ac[i], f = part ? t : -t;
      const int qo = mt * 16 + (sizeof(T) == 8 ? 4 * i + kq : 4 * kq + i);
      if (qo <= H) {
        d0[2 * (qo * L)] = qo ? e + f : e;
        if (qo) d0[2 * ((R - qo) * L)] = e - f;
      }
    }
  }
  lds_barrier();
  if (!last || z_lds) return;
  const int nf = (int)X.P.nf;
  for (int i = threadIdx.x; i < G.C * nf; i += NT) {
    const int c = G.lm_st ? div_m(i, G.mrow) : i & (G.C - 1);
    const int p = G.lm_st ? i - c * nf : i >> G.logC;
    mix_store<T, KIND>(X, c, p, X.lds[mix_slot(G, c, p)]);
  }
}

// Source and destination offsets of the tile's lines.  The pass's lines are
// numbered tile index fastest, then the batch indices.  `text` is the tile
// extent rounded up to whole tiles where that wastes little (the tiles of
// every row then start on the row's own 128-byte segments), else the extent
// itself (tiles run across rows and only the last one is ragged).
__device__ __forceinline__ void mix_lines(const pfk_pass &P, const int C, const int64_t text,
                                          const int64_t line0, const int nl, int64_t *so,
                                          int64_t *dof) {
  const int c = threadIdx.x;
  if (c < C) {
    int64_t l = line0 + (c < nl ? c : 0), s, d;
    if (line0 + C < ((int64_t)1 << 32) && text < ((int64_t)1 << 32)) {
      uint32_t u = (uint32_t)l, t = u % (uint32_t)text;
      u /= (uint32_t)text;
      s = (int64_t)t * P.tsin;
      d = (int64_t)t * P.tsout;
      for (int i = 0; i < P.nb; ++i) {
        const uint32_t e = (uint32_t)P.bext[i], k = u % e;   // at most the line count
        u /= e;
        s += (int64_t)k * P.bsin[i];
        d += (int64_t)k * P.bsout[i];
      }
    } else {
      const int64_t t = l % text;
      l /= text;
      s = t * P.tsin;
      d = t * P.tsout;
      for (int i = 0; i < P.nb; ++i) {
        const int64_t k = l % P.bext[i];
        l /= P.bext[i];
        s += k * P.bsin[i];
        d += k * P.bsout[i];
      }
    }
    so[c] = s;
    dof[c] = d;
  }
  lds_barrier();
}

// LDS of a workgroup: the stage table, two sets of line offsets (a tile's are
// written while the previous tile's are still read) and the tile.
template <typename T>
__device__ __forceinline__ C2<T> *mix_table(const pfk_pass &P, const MixGeo &G,
                                            unsigned char *smem) {
  C2<T> *tw = reinterpret_cast<C2<T> *>(smem);
  for (int i = threadIdx.x; i < G.ntw; i += blockDim.x)
    tw[i] = reinterpret_cast<const C2<T> *>(P.twm)[i];
  return tw;
}

// The pass on the tile of lines line0 .. line0 + G.C - 1 (of nlines, numbered
// by G.text); `odd` alternates between a workgroup's consecutive tiles.  BIG:
// with matrix-core stages (their registers stay out of the other kernels:
// 360x300x250 complex128 pair 1.30 ms without them, 1.37 with).
template <typename T, int KIND, bool BIG>
__device__ __forceinline__ void mixed_tile(const pfk_pass &P, const MixGeo &G,
                                           const int64_t line0, const int64_t nlines,
                                           const int odd, const T *__restrict__ src,
                                           T *__restrict__ dst, unsigned char *smem) {
  C2<T> *tw = reinterpret_cast<C2<T> *>(smem);
  int64_t *off0 = reinterpret_cast<int64_t *>(tw + G.ntw);
  int64_t *so = off0 + odd * 2 * G.C, *dof = so + G.C;
  int64_t left = nlines - line0;
  if (G.text != P.text) left = P.text - line0 % G.text;
  const int nl = left < G.C ? (int)left : G.C;
  mix_lines(P, G.C, G.text, line0, nl, so, dof);
  MixCtx<T> X{P, G, nl, so, dof, src, dst, tw, reinterpret_cast<C2<T> *>(off0 + 4 * G.C),
              reinterpret_cast<C2<T> *>(off0 + 4 * G.C) + (BIG ? G.C * G.pitch : 0), P.sign < 0 ? (T)1 : (T)-1};
  const bool even = !(P.n & 1);
  const int h = (int)P.nf;
  if (KIND == PFK_C2R && even) {
    // the half spectrum of every line into LDS (embed, modulation, adjoint
    // weights), 128 bytes of loads in flight per thread
    constexpr int U = sizeof(T) == 8 ? 8 : 16;
    const int cnt = h + 1, total = G.C * cnt, NT = blockDim.x;
    for (int b = threadIdx.x; b < total; b += U * NT) {
      C2<T> v[U];
      int cc[U], kk[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = b + u * NT < total ? b + u * NT : b;
        if (G.lm_ld) {
          cc[u] = div_m(i, G.mload);
          kk[u] = i - cc[u] * cnt;
        } else {
          cc[u] = i & (G.C - 1);
          kk[u] = i >> G.logC;
        }
        const int j = kk[u] - (int)P.zin;
        const bool ok = j >= 0 && j < (int)P.nin;
        v[u] = (reinterpret_cast<const C2<T> *>(src) +
                so[cc[u]])[(int64_t)(ok ? j : 0) * P.sin];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = kk[u] - (int)P.zin;
        const bool ok = j >= 0 && j < (int)P.nin;
        T f = ok ? msign<T>(P.imod, j) : (T)0;
        if (P.hw == 1 && kk[u] != 0 && kk[u] != h) f *= (T)0.5;
        X.lds[mix_slot(G, cc[u], kk[u])] = ok ? C2<T>{v[u].x * f, v[u].y * f} : C2<T>{0, 0};
      }
    }
    lds_barrier();
  }
  for (int s = 0; s < G.nst; ++s) {
    switch (G.rad[s]) {
      case 2: mix_stage<T, KIND, 2>(X, s); break;
      case 3: mix_stage<T, KIND, 3>(X, s); break;
      case 4: mix_stage<T, KIND, 4>(X, s); break;
      case 5: mix_stage<T, KIND, 5>(X, s); break;
      case 6: mix_stage<T, KIND, 6>(X, s); break;
      case 7: mix_stage<T, KIND, 7>(X, s); break;
      case 8: mix_stage<T, KIND, 8>(X, s); break;
      case 9: mix_stage<T, KIND, 9>(X, s); break;
      case 10: mix_stage<T, KIND, 10>(X, s); break;
      case 11: mix_stage<T, KIND, 11>(X, s); break;
      case 12: mix_stage<T, KIND, 12>(X, s); break;
      case 13: mix_stage<T, KIND, 13>(X, s); break;
      case 14: mix_stage<T, KIND, 14>(X, s); break;
      case 15: mix_stage<T, KIND, 15>(X, s); break;
      case 16: mix_stage<T, KIND, 16>(X, s); break;
      default:
        if constexpr (BIG) mix_big<T, KIND>(X, s);
        break;
    }
  }
  if (KIND == PFK_R2C && even) {
    // half-spectrum combine: X_k = E_k + W_n^k O_k, U outputs per thread at a
    // time so that their table loads overlap
    constexpr int U = 4;
    const C2<T> *rtw = reinterpret_cast<const C2<T> *>(P.rtw);
    const int cnt = (int)P.nout, total = G.C * cnt, NT = blockDim.x;
    for (int b = threadIdx.x; b < total; b += U * NT) {
      C2<T> w[U];
      int cc[U], kk[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = b + u * NT < total ? b + u * NT : b;
        if (G.lm_st) {
          cc[u] = div_m(i, G.mstore);
          kk[u] = i - cc[u] * cnt + (int)P.zout;
        } else {
          cc[u] = i & (G.C - 1);
          kk[u] = (i >> G.logC) + (int)P.zout;
        }
        w[u] = rtw[kk[u]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = cc[u], k = kk[u], ko = k - (int)P.zout;
        C2<T> x = X.lds[mix_slot(G, c, k == h ? 0 : k)];
        C2<T> y = X.lds[mix_slot(G, c, k == 0 ? 0 : h - k)];
        x.y *= X.cj;
        y.y *= X.cj;
        const C2<T> E{(x.x + y.x) * (T)0.5, (x.y - y.y) * (T)0.5};
        const C2<T> O{(x.y + y.y) * (T)0.5, -(x.x - y.x) * (T)0.5};
        const C2<T> WO = cmul(O, w[u]);
        T f = msign<T>(P.omod, ko);
        if (P.hw == 2 && k != 0 && k != h) f *= (T)2;
        if (b + u * NT < total && c < nl)
          st_elem(G.keep_st, reinterpret_cast<C2<T> *>(dst) + dof[c] + (int64_t)ko * P.sout,
                  C2<T>{(E.x + WO.x) * f, (E.y + WO.y) * f});
      }
    }
  }
}

}  // namespace pfk
