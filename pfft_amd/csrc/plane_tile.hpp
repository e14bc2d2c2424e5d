// plane_tile.hpp -- two contiguous dimensions of a complex transform in one
// pass: an n1 x n2 plane lives in LDS, its rows (length n2, contiguous in
// memory) are transformed, then its columns, and the plane is stored.
//
// Where a plane fits LDS this replaces two of the sweeps of a 3-d transform by
// one, and one of its launches.  The stages are those of mixed_tile.hpp
// (butterflies of radix 2..16, Stockham order, twiddles in stage order): the
// first row stage reads global memory, the last column stage writes it, both
// in runs along the rows.  A stage whose butterflies exceed what the threads
// hold at once (16 values each) goes through the lines in chunks; a chunk reads
// whole lines before it writes them, and the chunks touch different lines.
//
// Bound: vector instructions in complex64 (77% busy, four stages a sweep); in
// complex128 by waiting as the mixed-radix passes are (43%).  384
// uneven complex64 transforms of sides 24..128 in one batch: 1430 -> 1081 us,
// the plane level at 2.9 TB/s; 300x50x60 complex64 pair 87 -> 72 us.
#pragma once
#include "dft_regs.hpp"

namespace pfk {

#define PFK_PLANE_MAXST 6   /* stages of both dimensions together */

struct PlaneStage {
  int R, nb, L;       // radix, butterflies per line, product of the earlier radices
  int tw;             // twiddles in the LDS table
  int col;            // column stage
  int lines;          // lines per chunk
  uint32_t mdiv;      // row stage: reciprocal of nb; column stage: of `lines`
  uint32_t mlen;      // reciprocal of L
};

struct PlaneGeo {
  int n1, n2, pitch, nst, nrow, ntw1, ntw2;   // nrow: row stages; tables of rows, columns
  int keep_ld, keep_st;
  int64_t s1, d1;     // row strides
  const void *twc;    // stage table of the columns
  PlaneStage st[PFK_PLANE_MAXST];
};

// one slot of padding per 16 positions of a row spreads the row stages' strided
// stores over the banks
__device__ __forceinline__ int plane_slot(const PlaneGeo &G, int row, int x) {
  return row * G.pitch + x + (x >> 4);
}

template <typename T, int R>
__device__ __forceinline__ void plane_stage(const PlaneGeo &G, const int s, const int tid,
                                            const T cj,
                                            const C2<T> *__restrict__ src, C2<T> *__restrict__ dst,
                                            const C2<T> *twl, C2<T> *lds) {
  constexpr int I = R >= 16 ? 1 : 16 / R;
  const PlaneStage &S = G.st[s];
  const bool first = s == 0, last = s == G.nst - 1, col = S.col;
  const int NB = S.nb, L = S.L, W = S.lines, NT = blockDim.x;
  const int total = col ? G.n2 : G.n1;
  const C2<T> *tw = twl + S.tw;
  for (int c0 = 0; c0 < total; c0 += W) {
    const int items = W * NB;
    C2<T> v[I][R];
    int cs[I], bs[I], ks[I];
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int it0 = tid + i * NT, it = it0 < items ? it0 : 0;
      const int hi = div_m(it, S.mdiv), lo = it - hi * (col ? W : NB);
      cs[i] = c0 + (col ? lo : hi);
      bs[i] = col ? hi : lo;
      ks[i] = bs[i] - div_m(bs[i], S.mlen) * L;
      const bool ok = it0 < items && cs[i] < total;
      if (!ok) { cs[i] = c0; bs[i] = 0; ks[i] = -1; }   // reads line c0, writes nothing
    }
    if (first) {
#pragma unroll
      for (int i = 0; i < I; ++i) {
        const C2<T> *a = src + cs[i] * G.s1 + bs[i];
        if (G.keep_ld) {
#pragma unroll
          for (int r = 0; r < R; ++r) v[i][r] = a[r * NB];
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) v[i][r] = ld_stream(a + r * NB);
        }
      }
      if (cj < 0) {
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
          for (int r = 0; r < R; ++r) v[i][r].y = -v[i][r].y;
      }
    } else {
      if (col) {   // one address per butterfly and a uniform step
        const int step = NB * G.pitch;
#pragma unroll
        for (int i = 0; i < I; ++i) {
          const C2<T> *a = lds + plane_slot(G, bs[i], cs[i]);
#pragma unroll
          for (int r = 0; r < R; ++r) v[i][r] = a[r * step];
        }
      } else {
#pragma unroll
        for (int i = 0; i < I; ++i) {
          const C2<T> *a = lds + cs[i] * G.pitch;
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const int p = bs[i] + r * NB;
            v[i][r] = a[p + (p >> 4)];
          }
        }
      }
      if (L > 1) {
#pragma unroll
        for (int i = 0; i < I; ++i) {
          const C2<T> *w = tw + (ks[i] < 0 ? 0 : ks[i]);
#pragma unroll
          for (int r = 1; r < R; ++r) v[i][r] = cmul(v[i][r], w[(r - 1) * L]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < I; ++i) dft_any<R, -1>(v[i]);
    if (last) {   // column stage: position = row of the destination
#pragma unroll
      for (int i = 0; i < I; ++i) {
        if (ks[i] < 0) continue;
        C2<T> *a = dst + bs[i] * G.d1 + cs[i];
        const int64_t step = NB * G.d1;
#pragma unroll
        for (int q = 0; q < R; ++q) {
          v[i][q].y = cj < 0 ? -v[i][q].y : v[i][q].y;
          st_elem(G.keep_st, a + q * step, v[i][q]);
        }
      }
      continue;
    }
    if (!first) lds_barrier();
#pragma unroll
    for (int i = 0; i < I; ++i) {
      if (ks[i] < 0) continue;
      const int o = (bs[i] - ks[i]) * R + ks[i];
      if (col) {
        C2<T> *a = lds + plane_slot(G, o, cs[i]);
        const int step = L * G.pitch;
#pragma unroll
        for (int q = 0; q < R; ++q) a[q * step] = v[i][q];
      } else {
        C2<T> *a = lds + cs[i] * G.pitch;
#pragma unroll
        for (int q = 0; q < R; ++q) {
          const int p = o + q * L;
          a[p + (p >> 4)] = v[i][q];
        }
      }
    }
  }
  lds_barrier();
}

// One plane.  `smem`: tables of the rows and of the columns, then n1 rows of
// `pitch` slots.  Ends with a barrier: LDS may be reused.
template <typename T>
__device__ __forceinline__ void plane_tile(const PlaneGeo &G, const int sign, const T *src,
                                           T *dst, const void *tw_row, const void *tw_col,
                                           const bool tables, unsigned char *smem) {
  C2<T> *twl = reinterpret_cast<C2<T> *>(smem), *lds = twl + G.ntw1 + G.ntw2;
  if (tables) {
    for (int i = threadIdx.x; i < G.ntw1; i += blockDim.x)
      twl[i] = reinterpret_cast<const C2<T> *>(tw_row)[i];
    for (int i = threadIdx.x; i < G.ntw2; i += blockDim.x)
      twl[G.ntw1 + i] = reinterpret_cast<const C2<T> *>(tw_col)[i];
  }
  // opaque per plane: index arithmetic stays in its stage instead of being
  // hoisted out of the plane loop for every radix
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const T cj = sign < 0 ? (T)1 : (T)-1;
  const C2<T> *s = reinterpret_cast<const C2<T> *>(src);
  C2<T> *d = reinterpret_cast<C2<T> *>(dst);
  for (int k = 0; k < G.nst; ++k) {
    switch (G.st[k].R) {
#define PFK_PLANE_R(R) \
  case R: plane_stage<T, R>(G, k, tid, cj, s, d, twl, lds); break;
      PFK_PLANE_R(2) PFK_PLANE_R(3) PFK_PLANE_R(4) PFK_PLANE_R(5) PFK_PLANE_R(6)
      PFK_PLANE_R(7) PFK_PLANE_R(8) PFK_PLANE_R(9) PFK_PLANE_R(10) PFK_PLANE_R(11)
      PFK_PLANE_R(12) PFK_PLANE_R(13) PFK_PLANE_R(14) PFK_PLANE_R(15) PFK_PLANE_R(16)
#undef PFK_PLANE_R
      default: break;
    }
  }
}

// Geometry of a plane pass (pfk_pass.pl) for `nt` threads; 0 if it has one.
int plane_geo(const pfk_pass *p, int nt, PlaneGeo *g, size_t *lds);
// Threads of a plane: by its size, so that a CU holds 16 waves of planes (8
// waves of the largest ones, half as many threads, moved the batch below to
// 1278 us).
int plane_threads(const pfk_pass *p);

}  // namespace pfk
