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
// Primes above 13 (one stage each, radix R; up to 587 in complex128 and 1181 in
// complex64, where eight lines in two tiles fill LDS): with x_0 apart, the pair sums
// A_r = x_r + x_(R-r) and differences B_r = x_r - x_(R-r), r <= (R-1)/2, give
//   Y_q     = x_0 + sum_r cos(2 pi q r/R) A_r - i sum_r sin(2 pi q r/R) B_r,
//   Y_(R-q) = the same with + i,
// two dense real products over r for all lines and both components: matrix
// core work (16x16x4 tiles: 16 outputs q by 8 lines x {re, im} by 4 r).
//
// r2r lines of an even inner length (pfk_r2r_inner, path 1) are one launch too:
// the real line is staged in LDS through the kind's permutation (r2r_put), and
// its twiddles and combine (r2r_spectrum, r2r_post) run there.  As launches of
// their own those steps were two further sweeps: 256^3 complex128 DCT-II and
// DCT-III 1218 -> 578 us, 87-96 us a pass.
//
// Bound: the complex passes by waiting, 3.7-5.1 TB/s with 9-14 waves per CU and the
// vector units 25-42% busy (loads, exchanges and stores of a tile follow one
// another; rows that are not whole segments are read up to 1.9 times); the
// single-precision real and the r2r lines by vector instructions, 70% busy, the
// latter at 2.8-3.0 TB/s.  The general kernel, whose stages sum each output over
// its radix with a division per element, runs at 0.7-1.5 TB/s.  Forward+backward
// pairs, general kernel -> this one: c2c 360x300x250 complex128 4.26 -> 1.28 ms,
// r2c 210x196x330 complex64 908 -> 210 us, c2c 29x27x31 complex128 142 -> 96 us.
// Without any stage arithmetic and exchanges the first of these takes 1.07 ms.
// Registers (128) and LDS leave 16 waves per CU in flight.
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
  int m;                   // computed length (P.nf; r2r: the inner one)
  int big;                 // 1: some stage runs on the matrix cores (a second tile in LDS)
  int keep_ld, keep_st;    // ordinary instead of streaming accesses
  int64_t text;            // tile extent the lines are numbered by (mix_lines)
  int rad[PFK_MIX_MAXST], nb[PFK_MIX_MAXST], len[PFK_MIX_MAXST], off[PFK_MIX_MAXST];
  uint32_t mnb[PFK_MIX_MAXST], mlen[PFK_MIX_MAXST];   // reciprocals of nb, len
  int offr[PFK_MIX_MAXST];  // W_R table of a matrix-core stage
  uint32_t mload, mstore;  // reciprocals of the staged load / store loop lengths
  uint32_t mpair[PFK_MIX_MAXST], mrow;   // ... of the pair-sum loop, of nf
};

// KIND of a kernel: PFK_C2C, PFK_R2C, PFK_C2R, or one of the r2r kinds (a kernel
// each: with a switch inside, what the kinds have in common is hoisted above it
// and spilled)
constexpr int mix_kind_r2r(int r2r) { return 16 + r2r; }
constexpr bool mix_r2r(int kind) { return kind >= 16; }
constexpr int mix_r2r_kind(int kind) { return kind - 16; }

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
  int tid;                   // thread index
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

// ---- r2r steps around the inner transform (modes in pfk.h) ----
constexpr int r2r_mode_of(int kind) {   // pfk_r2r_mode
  return kind == PFK_REDFT01 || kind == PFK_RODFT01   ? 1
         : kind == PFK_REDFT11 || kind == PFK_RODFT11 ? 2
                                                      : 0;
}
// Element j of the real line (length n) into its row: where the inner complex
// line of length M (z_q at reals 2q, 2q+1) takes it.
//   mode 0: the reals v_m whose real FFT the kind needs, z_q = (v_2q, v_2q+1);
//   mode 1: (x'_q, x'_(n-q)) at q <= M, x'_n = 0 (r2r_spectrum makes z of it);
//   mode 2: (x'_2q, x'_(n-1-2q)), twiddled when read (mix_staged).
// x' is x, reversed for the RO kinds of modes 1 and 2.
template <int KD, typename T>
__device__ __forceinline__ void r2r_put(T *row, const int n, const int M, const int j,
                                        const T v) {
  if constexpr (KD == PFK_DHT) {
    row[j] = v;
  } else if constexpr (KD == PFK_REDFT10 || KD == PFK_RODFT10) {
    // Makhoul: v_m = x_2m, v_(n-1-m') = x_(2m'+1); DST-II: x_j (-1)^j
    row[(j & 1) ? n - 1 - (j >> 1) : j >> 1] = KD == PFK_RODFT10 && (j & 1) ? -v : v;
  } else if constexpr (KD == PFK_REDFT00) {
    row[j] = v;
    if (j > 0 && j < n - 1) row[2 * (n - 1) - j] = v;
  } else if constexpr (KD == PFK_RODFT00) {   // 0, x_0 .. x_(n-1), 0, -x_(n-1) .. -x_0
    row[j + 1] = v;
    row[2 * (n + 1) - j - 1] = -v;
    if (j == 0) row[0] = row[n + 1] = (T)0;
  } else if constexpr (KD == PFK_REDFT01 || KD == PFK_RODFT01) {
    const int i = KD == PFK_RODFT01 ? n - 1 - j : j;
    if (i <= M) row[2 * i] = v;
    if (i >= M) row[2 * (n - i) + 1] = v;
    if (i == 0) row[1] = (T)0;
  } else {
    const int i = KD == PFK_RODFT11 ? n - 1 - j : j;
    row[(i & 1) ? n - i : i] = v;
  }
}

// mode 1, in place on the staged rows: V_j = e^(i pi j/(2n)) (x'_j - i x'_(n-j)),
// Im of V_0 and V_M dropped as a c2r drops them, then the c2r combine
// z_q = (V_q + conj V_(M-q)) + i W_n^q (V_q - conj V_(M-q)) for q and M - q
template <typename T>
__device__ __forceinline__ void r2r_spectrum(const MixCtx<T> &X) {
  const MixGeo &G = X.G;
  const int M = G.m, total = G.C * (M / 2 + 1), NT = blockDim.x;
  const C2<T> *tw2 = reinterpret_cast<const C2<T> *>(X.P.tw2);
  const C2<T> *rtw = reinterpret_cast<const C2<T> *>(X.P.rtw);
  for (int i = X.tid; i < total; i += NT) {
    const int c = i & (G.C - 1), q = i >> G.logC, r = M - q;
    C2<T> *row = X.lds + mix_slot(G, c, 0);
    const C2<T> xq = row[q], xr = row[r], tq = tw2[q], tr = tw2[r], wq = rtw[q], wr = rtw[r];
    C2<T> a = cmul(C2<T>{tq.x, -tq.y}, C2<T>{xq.x, -xq.y});
    C2<T> b = cmul(C2<T>{tr.x, -tr.y}, C2<T>{xr.x, -xr.y});
    if (q == 0) a.y = b.y = (T)0;
    const C2<T> wd = cmul(wq, C2<T>{a.x - b.x, a.y + b.y});
    row[q] = C2<T>{a.x + b.x - wd.y, a.y - b.y + wd.x};
    if (q > 0 && q < r) {
      const C2<T> we = cmul(wr, C2<T>{b.x - a.x, b.y + a.y});
      row[r] = C2<T>{b.x + a.x - we.y, b.y - a.y + we.x};
    }
  }
  lds_barrier();
}

// the kind's outputs from the inner transform in LDS
template <int KD, typename T>
__device__ __forceinline__ void r2r_post(const MixCtx<T> &X) {
  const pfk_pass &P = X.P;
  const MixGeo &G = X.G;
  const int n = (int)P.n, M = G.m, zout = (int)P.zout, nout = (int)P.nout, NT = blockDim.x;
  constexpr int mode = r2r_mode_of(KD), U = 4;
  const C2<T> *tw2 = reinterpret_cast<const C2<T> *>(P.tw2);
  const C2<T> *rtw = reinterpret_cast<const C2<T> *>(P.rtw);
  auto z = [&](int c, int m) {
    C2<T> v = X.lds[mix_slot(G, c, m)];
    v.y *= X.cj;
    return v;
  };
  auto emit = [&](int c, int kk, T y) {
    const int k = kk - zout;
    if (k >= 0 && k < nout && c < X.nl)
      X.dst[X.dof[c] + (int64_t)k * P.sout] = y * msign<T>(P.omod, k);
  };
  // items: mode 0 the bins m <= M of the real line, each the outputs of m and of
  // its mirror; modes 1 and 2 the kept outputs
  const int cnt = mode == 0 ? M + 1 : nout, total = G.C * cnt;
  for (int b = X.tid; b < total; b += U * NT) {
    int cc[U], mm[U];
    C2<T> w[U], t1[U], t2[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = b + u * NT < total ? b + u * NT : b;
      cc[u] = G.lm_st ? div_m(i, G.mstore) : i & (G.C - 1);
      mm[u] = G.lm_st ? i - cc[u] * cnt : i >> G.logC;
      if constexpr (mode == 0) {
        w[u] = rtw[mm[u]];
        if constexpr (KD == PFK_REDFT10 || KD == PFK_RODFT10) {
          t1[u] = tw2[mm[u]];
          t2[u] = tw2[n - mm[u]];
        }
      } else if constexpr (mode == 2) {
        const int kk = mm[u] + zout;
        t1[u] = tw2[4 * ((kk & 1) ? (n - 1 - kk) / 2 : kk / 2)];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (b + u * NT >= total) break;
      const int c = cc[u], m = mm[u];
      if constexpr (mode == 0) {
        // V_m = E_m + W^m O_m from Z_m and conj Z_(M-m)
        const C2<T> a = z(c, m == M ? 0 : m), b0 = z(c, m == 0 ? 0 : M - m);
        const C2<T> bb{b0.x, -b0.y};
        const C2<T> e{(a.x + bb.x) * (T)0.5, (a.y + bb.y) * (T)0.5};
        const C2<T> o{(a.y - bb.y) * (T)0.5, -(a.x - bb.x) * (T)0.5};
        C2<T> v = cmul(w[u], o);
        v = C2<T>{v.x + e.x, v.y + e.y};
        const bool two = m > 0 && m < M;   // the mirror bin 2M - m has conj V_m
        if constexpr (KD == PFK_DHT) {
          emit(c, m, v.x - v.y);
          if (two) emit(c, n - m, v.x + v.y);
        } else if constexpr (KD == PFK_REDFT10) {
          emit(c, m, 2 * cmul(t1[u], v).x);
          if (two) emit(c, n - m, 2 * cmul(t2[u], C2<T>{v.x, -v.y}).x);
        } else if constexpr (KD == PFK_RODFT10) {   // reversed
          emit(c, n - 1 - m, 2 * cmul(t1[u], v).x);
          if (two) emit(c, m - 1, 2 * cmul(t2[u], C2<T>{v.x, -v.y}).x);
        } else if constexpr (KD == PFK_REDFT00) {
          emit(c, m, v.x);
        } else if (two) {   // RODFT00: n = M - 1 outputs
          emit(c, m - 1, -v.y);
        }
      } else if constexpr (mode == 1) {   // y_2m = v_m, y_(2m+1) = v_(n-1-m), v the real line
        const int kk = m + zout, idx = (kk & 1) ? n - 1 - (kk - 1) / 2 : kk / 2;
        const C2<T> v = z(c, idx / 2);
        const T y = (idx & 1) ? v.y : v.x;
        emit(c, kk, KD == PFK_RODFT01 && (kk & 1) ? -y : y);   // DST-III: (-1)^k
      } else {   // u_j = Z_j W_8n^(4j); y_2j = 2 Re u_j, y_(n-1-2j) = -2 Im u_j
        const int kk = m + zout, j = (kk & 1) ? (n - 1 - kk) / 2 : kk / 2;
        const C2<T> v = cmul(z(c, j), t1[u]);
        const T y = (kk & 1) ? -2 * v.y : 2 * v.x;
        emit(c, kk, KD == PFK_RODFT11 && (kk & 1) ? -y : y);   // DST-IV: (-1)^k
      }
    }
  }
}

// the first stage of these passes reads the staged tile, the last one leaves
// its result there
template <int KIND>
__device__ __forceinline__ bool mix_packed(const pfk_pass &P) {
  return mix_r2r(KIND) || (KIND == PFK_C2R && !(P.n & 1));
}
template <int KIND>
__device__ __forceinline__ bool mix_combined(const pfk_pass &P) {
  return mix_r2r(KIND) || (KIND == PFK_R2C && !(P.n & 1));
}
// element p of a staged line
template <typename T, int KIND>
__device__ __forceinline__ C2<T> mix_staged(const MixCtx<T> &X, const int c, const int p) {
  if constexpr (mix_r2r(KIND)) {
    C2<T> v = X.lds[mix_slot(X.G, c, p)];
    if constexpr (r2r_mode_of(mix_r2r_kind(KIND)) == 2)   // times W_8n^(4p+1)
      v = cmul(v, reinterpret_cast<const C2<T> *>(X.P.tw2)[4 * p + 1]);
    v.y *= X.cj;
    return v;
  } else {
    return c2r_pack(X, c, p);
  }
}

// one stage of a codelet radix
template <typename T, int KIND, int R>
__device__ __forceinline__ void mix_stage(const MixCtx<T> &X, const int s) {
  constexpr int I = mix_items<R>();
  const MixGeo &G = X.G;
  const bool first = s == 0, last = s == G.nst - 1;
  const bool packed = mix_packed<KIND>(X.P), z_lds = mix_combined<KIND>(X.P);
  const int NB = G.nb[s], L = G.len[s], items = NB * G.C;
  const bool lm = first ? G.lm_ld : G.lm_st;
  const C2<T> *tw = X.tw + G.off[s];
  C2<T> v[I][R];
  int cs[I], bs[I], ks[I];
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int it0 = X.tid + i * (int)blockDim.x;
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
  if (first && !packed && KIND != PFK_C2R && !mix_r2r(KIND) && (G.plain || G.vec)) {
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
        v[i][r] = mix_staged<T, KIND>(X, cs[i] < G.C ? cs[i] : 0, bs[i] + r * NB);
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
  const bool packed = mix_packed<KIND>(X.P), z_lds = mix_combined<KIND>(X.P);
  const int R = G.rad[s], NB = G.nb[s], L = G.len[s], H = (R - 1) / 2, NT = blockDim.x;
  const C2<T> *tw = X.tw + G.off[s], *tr = X.tw + G.offr[s];
  // pair sums A_r at position r*NB + b, differences B_r at (R-r)*NB + b of the
  // second tile, U pairs per thread at a time
  constexpr int U = 4;
  const int cnt = (H + 1) * NB, total = G.C * cnt;
  const bool lm = first && !packed && G.lm_ld;
  for (int i0 = X.tid; i0 < total; i0 += U * NT) {
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
        x[u] = mix_staged<T, KIND>(X, cc[u], pp[u]);
        y[u] = mix_staged<T, KIND>(X, cc[u], mm[u]);
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
  const int lane = X.tid & 63, col = lane & 15, kq = lane >> 4, part = col >> 3;
  const int MT = (H + 16) / 16, LG = G.C >> 3, units = NB * LG * MT;
  for (int un = X.tid >> 6; un < units; un += NT >> 6) {
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
  const int nf = G.m;
  for (int i = X.tid; i < G.C * nf; i += NT) {
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
  // r2r: opaque per tile, else what depends on the thread index alone (table
  // entries, addresses) is hoisted out of the tile loop and spilled; the other
  // kinds gain from the hoisting (r2c 210x196x330 complex64 195 us, 206 opaque)
  int tid = threadIdx.x;
  if constexpr (mix_r2r(KIND)) asm volatile("" : "+v"(tid));
  MixCtx<T> X{P, G, nl, so, dof, src, dst, tw, reinterpret_cast<C2<T> *>(off0 + 4 * G.C),
              reinterpret_cast<C2<T> *>(off0 + 4 * G.C) + (BIG ? G.C * G.pitch : 0), tid,
              (mix_r2r(KIND) ? pfk_r2r_mode(P.r2r) != 1 : P.sign < 0) ? (T)1 : (T)-1};
  const bool even = !(P.n & 1);
  const int h = (int)P.nf;
  if (KIND == PFK_C2R && even) {
    // the half spectrum of every line into LDS (embed, modulation, adjoint
    // weights), 128 bytes of loads in flight per thread
    constexpr int U = sizeof(T) == 8 ? 8 : 16;
    const int cnt = h + 1, total = G.C * cnt, NT = blockDim.x;
    for (int b = tid; b < total; b += U * NT) {
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
  if constexpr (mix_r2r(KIND)) {
    // the real lines into their rows, zeros outside the embed
    constexpr int U = 8;
    const int cnt = (int)P.n, total = G.C * cnt, NT = blockDim.x;
    T *rows = reinterpret_cast<T *>(X.lds);
    for (int b = tid; b < total; b += U * NT) {
      T v[U];
      auto at = [&](int u, int &c, int &j) {
        const int i = b + u * NT < total ? b + u * NT : b;
        c = G.lm_ld ? div_m(i, G.mload) : i & (G.C - 1);
        j = G.lm_ld ? i - c * cnt : i >> G.logC;
      };
#pragma unroll
      for (int u = 0; u < U; ++u) {
        int c, j0;
        at(u, c, j0);
        const int j = j0 - (int)P.zin;
        v[u] = src[so[c] + (int64_t)(j >= 0 && j < (int)P.nin ? j : 0) * P.sin];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        int c, j0;
        at(u, c, j0);
        const int j = j0 - (int)P.zin;
        const bool ok = j >= 0 && j < (int)P.nin;
        r2r_put<mix_r2r_kind(KIND)>(rows + 2 * G.pitch * c, cnt, G.m, j0,
                                    ok ? v[u] * msign<T>(P.imod, j) : (T)0);
      }
    }
    lds_barrier();
    if constexpr (r2r_mode_of(mix_r2r_kind(KIND)) == 1) r2r_spectrum(X);
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
  if constexpr (mix_r2r(KIND)) r2r_post<mix_r2r_kind(KIND)>(X);
  if (KIND == PFK_R2C && even) {
    // half-spectrum combine: X_k = E_k + W_n^k O_k, U outputs per thread at a
    // time so that their table loads overlap
    constexpr int U = 4;
    const C2<T> *rtw = reinterpret_cast<const C2<T> *>(P.rtw);
    const int cnt = (int)P.nout, total = G.C * cnt, NT = blockDim.x;
    for (int b = tid; b < total; b += U * NT) {
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
