// pow2_tile.hpp -- register-resident Stockham pass kernels for
// power-of-two lengths 64..4096 on gfx950.
//
// Work split.  One workgroup transforms C lines of length NF (the
// computed complex FFT length).  Each line is handled by T = NF/8
// threads; thread (c, t) holds the 8 elements t + T*m (m = 0..7) of line c
// in registers.  Thread index = t*C + c, so the C lanes with equal t are
// adjacent: every global access by a wave covers 64/C rows of C elements
// (tile dimension contiguous) or C runs of 64/C elements (line contiguous),
// i.e. 128-byte segments for C = 8 and 16-byte complex doubles, whatever the
// load/store layout.
//
// Stages.  NF = 8^a * 2^b: a radix-8 stages and, if b > 0, one final
// radix-2^b stage in which each thread does 8/R butterflies.  With T
// threads per line, the inputs of every stage for thread t are exactly
// positions t + T*m, so only the outputs move: between stages each thread
// writes its outputs to LDS and reads back positions t + T*m.  LDS is laid
// out [position][line] (index p*C + c): the 8 lanes that issue one 16-byte
// access together touch 8 consecutive 16-byte words, so every exchange is
// bank-conflict free without padding.  After the last stage thread t holds
// X[t + T*m] in natural order.
//
// Real transforms (even n, NF = n/2) use the half-length packing:
// r2c loads z_p = x_2p + i x_2p+1, transforms, and unpacks
//   X_k = (Z_k + conj Z_{h-k})/2 - i W^k (Z_k - conj Z_{h-k})/2,  W = e^{sign 2 pi i/n};
// c2r packs Z_k = E_k + i O_k with E_k = X_k + conj X_{h-k},
// O_k = (X_k - conj X_{h-k}) W^k before the transform and stores
// x_2p = Re z_p, x_2p+1 = Im z_p.  The mirror partner Z_{h-k} lives in
// another thread, so both use one extra LDS exchange.
#pragma once
#include <stdlib.h>
#include "pass_access.hpp"
#include "dft_regs.hpp"
#include "pow2_launch.hpp"

namespace pfk {

constexpr int ilog2c(int n) { return n <= 1 ? 0 : 1 + ilog2c(n / 2); }

// One Stockham stage of radix R on the thread's E registers (E = 8 or 16,
// T = NF/E threads per line).  Butterflies b = t + i*T for i < E/R; inputs
// m = i + r*(E/R); twiddle W_NF^(r*k*NF/(L*R)), k = b mod L.  Outputs go to
// register m' = i + q*(E/R) and, unless LAST, their LDS positions to `pos`.
template <typename T, int NF, int E, int R, int L, int SIGN, bool LAST>
__device__ __forceinline__ void stage(C2<T> *v, int *pos, const int t,
                                      const C2<T> *__restrict__ tw) {
  constexpr int TT = NF / E;
  constexpr int NB = E / R;
  constexpr int M = NF / (L * R);
  C2<T> o[E];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int b = t + i * TT;
    const int k = b & (L - 1);
    C2<T> a[R];
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = v[i + r * NB];
    if (L > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) a[r] = cmul(a[r], tw[r * k * M]);
    }
    if (R == 16) dft16<SIGN>(a);
    else if (R == 8) dft8<SIGN>(a);
    else if (R == 4) dft4<SIGN>(a[0], a[1], a[2], a[3]);
    else dft2<SIGN>(a[0], a[1]);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      o[i + q * NB] = a[q];
      if (!LAST) pos[i + q * NB] = (b - k) * R + k + q * L;
    }
  }
#pragma unroll
  for (int m = 0; m < E; ++m) v[m] = o[m];
}

// LDS slot of position p of line c.  Tile-major lane order (consecutive
// lanes = consecutive lines): [position][line], conflict-free without
// padding.  Line-major lane order (consecutive lanes = consecutive
// positions of one line): [line][position] with one slot of padding per 16
// positions, so the radix-8/16 output scatters (position strides 8 and 16)
// spread over the banks, and an odd row pitch, so that the tile-major
// accesses of a staged load or store (consecutive lanes = consecutive
// lines at one position) do too.  The row has room for position NF (the
// Nyquist bin of c2r).
template <int NF>
constexpr int lm_pitch() { return NF + NF / 16 + 1; }
template <int NF, int C, bool LM>
__device__ __forceinline__ int lidx(int p, int c) {
  if constexpr (LM) return c * lm_pitch<NF>() + p + (p >> 4);
  else return p * C + c;
}
template <int NF, int C, bool LM>
constexpr int lds_slots() { return LM ? C * lm_pitch<NF>() : NF * C; }

// In line-major order a line's NF/E lanes are consecutive threads, so with
// at most 64 of them every line lies inside one wavefront, and an exchange
// within lines only reorders data among the lanes of one wave.  A wave's own
// LDS accesses execute in order, so such an exchange needs only the
// compiler to keep them in order (wavefront-scope fences), not a workgroup
// barrier that would hold every wave of the tile.
template <int NF, int E, bool LM>
constexpr bool wave_lines() { return LM && NF / E <= 64; }

template <bool WAVE>
__device__ __forceinline__ void line_sync() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  } else {
    lds_barrier();
  }
}

// Exchange through LDS: write v[m] at position pos[m], read back t + T*m.
template <typename T, int NF, int C, int E, bool LM>
__device__ __forceinline__ void exchange(C2<T> *v, const int *pos, C2<T> *lds, const int t,
                                         const int c) {
  constexpr int TT = NF / E;
#pragma unroll
  for (int m = 0; m < E; ++m) lds[lidx<NF, C, LM>(pos[m], c)] = v[m];
  line_sync<wave_lines<NF, E, LM>()>();
#pragma unroll
  for (int m = 0; m < E; ++m) v[m] = lds[lidx<NF, C, LM>(t + TT * m, c)];
  line_sync<wave_lines<NF, E, LM>()>();
}

// Full length-NF FFT on registers; first stage input = v (positions t+T*m),
// output X[t + T*m] in v[m].  Stages of radix E, then one of radix
// NF / E^A if NF is not a power of E.
template <typename T, int NF, int C, int E, int SIGN, int L, bool LM>
__device__ __forceinline__ void fft_stages(C2<T> *v, int *pos, C2<T> *lds, const int t,
                                           const int c, const C2<T> *__restrict__ tw) {
  constexpr int REM = NF / L;  // remaining length to transform
  if constexpr (REM >= E) {
    constexpr bool LAST = (REM == E);
    stage<T, NF, E, E, L, SIGN, LAST>(v, pos, t, tw);
    if constexpr (!LAST) {
      exchange<T, NF, C, E, LM>(v, pos, lds, t, c);
      fft_stages<T, NF, C, E, SIGN, L * E, LM>(v, pos, lds, t, c, tw);
    }
  } else if constexpr (REM > 1) {
    stage<T, NF, E, REM, L, SIGN, true>(v, pos, t, tw);
  }
}

template <typename T, int NF, int C, int E, int SIGN, bool LM = false>
__device__ __forceinline__ void fft_regs(C2<T> *v, C2<T> *lds, const int t, const int c,
                                         const C2<T> *__restrict__ tw) {
  int pos[E];
  fft_stages<T, NF, C, E, SIGN, 1, LM>(v, pos, lds, t, c, tw);
}

// Exchanges of a length-NF FFT in radix-E stages (stages minus one).
__host__ __device__ constexpr int n_exchanges(int nf, int e) {
  int s = 0, l = 1;
  while (nf / l >= e) { l *= e; ++s; }
  if (nf / l > 1) ++s;
  return s - 1;
}

// Exchange through the line-major LDS layout with a change of lane order:
// v[m] is written at position pos[m] of line cw and read back as position
// tr + T*m of line cr.  WAVE: both sides in line-major order with every line
// inside one wave (no change of order), so wavefront-scope ordering suffices.
template <typename T, int NF, int C, int E, bool WAVE = false>
__device__ __forceinline__ void exchange_x(C2<T> *v, const int *pos, C2<T> *lds, const int cw,
                                           const int tr, const int cr) {
  constexpr int TT = NF / E;
#pragma unroll
  for (int m = 0; m < E; ++m) lds[lidx<NF, C, true>(pos[m], cw)] = v[m];
  line_sync<WAVE>();
#pragma unroll
  for (int m = 0; m < E; ++m) v[m] = lds[lidx<NF, C, true>(tr + TT * m, cr)];
  line_sync<WAVE>();
}

// The FFT of fft_regs with a change of lane order at exchange SW (1-based):
// stages before it run as thread (ta, ca) (position index, line), the
// exchange writes in that order and reads in order (tb, cb), and the later
// stages run as (tb, cb).  K counts the exchanges done.  One of the two
// orders is line-major (the kernels stage tile-major loads or stores), so
// every exchange but the switching one stays within line-major lines.
template <typename T, int NF, int C, int E, int SIGN, int L, int K, int SW>
__device__ __forceinline__ void fft_stages_sw(C2<T> *v, int *pos, C2<T> *lds, const int ta,
                                              const int ca, const int tb, const int cb,
                                              const C2<T> *__restrict__ tw) {
  constexpr int REM = NF / L;
  constexpr bool BEFORE = K < SW;
  const int t = BEFORE ? ta : tb;
  const int c = BEFORE ? ca : cb;
  if constexpr (REM >= E) {
    constexpr bool LAST = (REM == E);
    stage<T, NF, E, E, L, SIGN, LAST>(v, pos, t, tw);
    if constexpr (!LAST) {
      constexpr bool AFTER = K + 1 >= SW;   // the next stage runs as (tb, cb)
      constexpr bool SWITCH = K + 1 == SW;
      exchange_x<T, NF, C, E, !SWITCH && wave_lines<NF, E, true>()>(v, pos, lds, c,
                                                                     AFTER ? tb : ta,
                                                                     AFTER ? cb : ca);
      fft_stages_sw<T, NF, C, E, SIGN, L * E, K + 1, SW>(v, pos, lds, ta, ca, tb, cb, tw);
    }
  } else if constexpr (REM > 1) {
    stage<T, NF, E, REM, L, SIGN, true>(v, pos, t, tw);
  }
}

// Persistent pass kernels.  A fixed grid of resident workgroups walks the
// tiles (workgroup b takes items item0 + b, + G, + 2G, ... below item_end);
// launched with one workgroup per tile instead (G = item_end - item0) the
// same kernel does one tile per workgroup.  While a tile is
// transformed and stored, the loads of the workgroup's next tile are
// already in flight in registers (software pipelining across tiles), so
// HBM stays busy through the compute and LDS phases.  On the last item the
// prefetch degenerates to every lane reading the tile's first element (one
// cached line), which keeps the load sequence free of branches.
//
// Loads are issued unconditionally from clamped in-bounds addresses and
// masked afterwards: a branch between a load and its use would make the
// compiler wait for each load in turn.

// Twiddle tables live in LDS when they fit next to the exchange buffer
// (limit 156 KiB per workgroup): LDS reads count on lgkmcnt, so a twiddle
// read does not wait for the prefetched tile the way a global load would
// (vmcnt completes in order).
template <typename T>
constexpr bool tw_in_lds(int slots, int nf, int extra) {
  return ((size_t)slots + nf + extra) * sizeof(C2<T>) <= 156 * 1024;
}
template <typename T>
__device__ __forceinline__ void stage_table(C2<T> *dst, const C2<T> *src, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) dst[i] = src[i];
}

// c2c: raw loads of elements t + T*m (minus the embed offset) of line c
template <bool KP, typename T, int NF, int C, int E>
__device__ __forceinline__ void load_c2c(const pfk_pass &P, const T *src, const TileCtx &tc,
                                         const bool live, const int c, const int t,
                                         C2<T> *v) {
  constexpr int TT = NF / E;
  const int zin = (int)P.zin, nin = (int)P.nin;
  const C2<T> *s0 = reinterpret_cast<const C2<T> *>(src) + tc.sb;
  const C2<T> *s = (live && c < tc.nl) ? s0 + (int64_t)c * P.tsin : s0;
  const int64_t sin = live ? P.sin : 0;
  ld_batch<KP, E>(P, v, [&](int m) {
    const int j = t + TT * m - zin;
    const bool ok = j >= 0 && j < nin;
    return s + (int64_t)(ok ? j : 0) * sin;
  });
}

// c2c loads of a plain pass (no embed, no modulation): one 64-bit address
// per thread, then constant strides (TT*sin, uniform) between its elements
template <bool KP, typename T, int NF, int C, int E>
__device__ __forceinline__ void load_c2c_pl(const pfk_pass &P, const T *src, const TileCtx &tc,
                                            const bool live, const int c, const int t,
                                            C2<T> *v) {
  constexpr int TT = NF / E;
  const C2<T> *s0 = reinterpret_cast<const C2<T> *>(src) + tc.sb;
  const C2<T> *s = (live && c < tc.nl) ? s0 + (int64_t)c * P.tsin + (int64_t)t * P.sin : s0;
  const int64_t st = live ? (int64_t)TT * P.sin : 0;
  ld_batch<KP, E>(P, v, [&](int m) { return s + m * st; });
}

// Paired-line stores for complex64 tiles whose lines are adjacent in
// memory (tile stride 1), tile-major lane order (line c = 2j + e of the
// tile in lane parity e).  Every 16-byte store covers two adjacent lines at
// one position: lane e = 0 of a pair writes the even element slots m = 0,
// 2, 4, ... of lines 2j and 2j+1, lane e = 1 the odd ones, after one DPP
// lane swap (quad_perm 1,0,3,2: lane ^ 1) per value has handed each lane
// its partner's values.  A wave instruction then moves 128-byte segments
// of 8 positions (the 4 of 8-byte lanes otherwise), the access shape of
// the complex128 tiles.  An odd last line is stored with 8-byte stores.
__device__ __forceinline__ float lane_xor1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}

typedef float pf4 __attribute__((ext_vector_type(4)));

// stores of lines c < tc.nl: pairs as 16-byte stores, an odd last line with
// 8-byte stores
template <bool KP, int NF, int C, int E>
__device__ __forceinline__ void store_c2c_pair(const pfk_pass &P, float *dst, const TileCtx &tc,
                                               const int c, const int t, const C2<float> *v) {
  constexpr int TT = NF / E;
  const int e = c & 1, j = c >> 1;
  C2<float> send[E / 2], recv[E / 2];
#pragma unroll
  for (int i = 0; i < E / 2; ++i) {
    send[i] = e ? v[2 * i] : v[2 * i + 1];
    recv[i] = C2<float>{lane_xor1(send[i].x), lane_xor1(send[i].y)};
  }
  C2<float> *d0 = reinterpret_cast<C2<float> *>(dst) + tc.db;
  if (2 * j + 1 < tc.nl) {
    C2<float> *d = d0 + 2 * j + (int64_t)(t + TT * e) * P.sout;
    const int64_t st = (int64_t)2 * TT * P.sout;
    const bool keep = KP && (P.cache & PFK_KEEP_DST);
#pragma unroll
    for (int i = 0; i < E / 2; ++i) {
      const C2<float> lo = e ? recv[i] : v[2 * i], hi = e ? v[2 * i + 1] : recv[i];
      const pf4 w{lo.x, lo.y, hi.x, hi.y};
      pf4 *q = reinterpret_cast<pf4 *>(d + i * st);
      if (keep) *q = w;
      else __builtin_nontemporal_store(w, q);
    }
  } else if (e == 0 && 2 * j < tc.nl) {
    C2<float> *d = d0 + 2 * j + (int64_t)t * P.sout;
#pragma unroll
    for (int m = 0; m < E; ++m) st_stream(d + (int64_t)TT * m * P.sout, v[m]);
  }
}

// LM: line-major lane order (thread = c*T + t: a wave's lanes run along a
// line), for passes whose lines are contiguous in memory; otherwise
// thread = t*C + c (a wave's lanes run across the tile's lines).
// XS (line-major plain passes only): 1 = the loads, 2 = the stores take the
// tile-major lane order; the FFT switches between the two orders at its
// first (1) or last (2) LDS exchange, so the staging costs no extra pass
// through LDS.  This is for a
// transposing pass whose lines are contiguous on one side and adjacent
// along the tile dimension on the other: complex64 has 8-byte elements,
// so tile-major lanes move 128-byte segments across 16 lines, and
// line-major lanes move 512-byte runs along one line.  Each side is
// accessed in the order that coalesces it.
// TW: output k of tile line c0 + c is multiplied by W_twn^((c0+c)*k) from
// the two-level table tw2 (first step of a long line, pfk.h).
// PL: plain pass (every input and output position present, no
// modulation): no masks or selects, and element addresses advance by a
// uniform stride, which halves the vector instructions spent per element
// outside the butterflies.
template <typename T, int NF, int C, int E, int SIGN, bool LM = false, bool TW = false,
          bool PL = false, int XS = 0, int PAIR = 0, bool KP = false>
__global__ void __launch_bounds__(C *NF / E)
k_c2c_pow2(const pfk_pass P, const int64_t item0, const int64_t item_end, const int64_t ntiles,
           const T *__restrict__ src, T *__restrict__ dst) {
  stamp_begin(P, item0 + blockIdx.x);
  constexpr int TT = NF / E;
  constexpr bool TWL = tw_in_lds<T>(lds_slots<NF, C, LM>(), NF, 0);
  __shared__ C2<T> lds[lds_slots<NF, C, LM>()];
  __shared__ C2<T> twl[TWL ? NF : 1];
  static_assert(XS == 0 || (LM && PL && !TW), "staged loads or stores: line-major plain passes");
  // PAIR: paired-line stores (complex64 plain passes, tile-major side)
  static_assert(PAIR == 0 || (sizeof(T) == 4 && PL && !TW && C % 2 == 0), "paired lines");
  static_assert(!PAIR || !LM || XS == 2, "paired stores need tile-major stores");
  const int tid = threadIdx.x;
  const int c0 = LM ? tid / TT : tid % C, t0 = LM ? tid % TT : tid / C;
  const int cx0 = tid % C, tx0 = tid / C;   // tile-major lane order of staged accesses
  const C2<T> *twg = reinterpret_cast<const C2<T> *>(P.tw);
  if constexpr (TWL) stage_table(twl, twg, NF);
  const C2<T> *tw = TWL ? twl : twg;
  const int zin = (int)P.zin, nin = (int)P.nin, zout = (int)P.zout, nout = (int)P.nout;
  const bool keep = KP && (P.cache & PFK_KEEP_DST);
  int64_t item = item0 + blockIdx.x;
  TileCtx tc = tile_at(P, C, item, ntiles);
  // one step: prefetch the next tile into `nxt`, transform and store `cur`;
  // false after the last item.  Two steps per loop trip alternate the
  // buffers, so no register copy has to wait for the prefetch.
  auto step = [&](C2<T> *cur, C2<T> *nxt) -> bool {
    // lane indices made opaque per step: index arithmetic is recomputed in
    // the loop instead of being hoisted and kept live in registers
    int t = t0, c = c0, tx = tx0, cx = cx0;
    asm volatile("" : "+v"(t), "+v"(c), "+v"(tx), "+v"(cx));
    const int64_t ni = item + gridDim.x;
    const bool more = ni < item_end;
    const TileCtx tn = tile_at(P, C, more ? ni : item, ntiles);
    if constexpr (XS == 1) load_c2c_pl<KP, T, NF, C, E>(P, src, tn, more, cx, tx, nxt);
    else if constexpr (PL) load_c2c_pl<KP, T, NF, C, E>(P, src, tn, more, c, t, nxt);
    else load_c2c<KP, T, NF, C, E>(P, src, tn, more, c, t, nxt);
    const bool valid = c < tc.nl;
    if constexpr (!PL) {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int j = t + TT * m - zin;
        const bool ok = valid && j >= 0 && j < nin;
        const T f = msign<T>(P.imod, j);
        cur[m] = ok ? C2<T>{cur[m].x * f, cur[m].y * f} : C2<T>{0, 0};
      }
    }
    if constexpr (XS == 0) {
      fft_regs<T, NF, C, E, SIGN, LM>(cur, lds, t, c, tw);
    } else {
      // the lane order changes at one of the FFT's own exchanges: the first
      // (tile-major loads, line-major stores) or the last (the reverse)
      static_assert(n_exchanges(NF, E) >= 1, "staged passes need an exchange");
      int pos[E];
      if constexpr (XS == 1)
        fft_stages_sw<T, NF, C, E, SIGN, 1, 0, 1>(cur, pos, lds, tx, cx, t, c, tw);
      else
        fft_stages_sw<T, NF, C, E, SIGN, 1, 0, n_exchanges(NF, E)>(cur, pos, lds, t, c, tx, cx,
                                                                    tw);
    }
    if constexpr (PAIR) {   // tile-major order, paired lines (every lane takes part)
      if constexpr (XS == 2) store_c2c_pair<KP, NF, C, E>(P, dst, tc, cx, tx, cur);
      else store_c2c_pair<KP, NF, C, E>(P, dst, tc, c, t, cur);
    } else if constexpr (XS == 2) {   // registers in tile-major order: tile-major stores
      if (cx < tc.nl) {
        C2<T> *d = reinterpret_cast<C2<T> *>(dst) + tc.db + (int64_t)cx * P.tsout +
                   (int64_t)tx * P.sout;
        const int64_t st = (int64_t)TT * P.sout;
        st_batch<E>(keep, cur, [&](int m) { return d + m * st; });
      }
    } else if (PL && valid) {
      // lines are independent, so a ragged tile's unused lines (garbage in,
      // never stored) cannot affect the stored ones
      C2<T> *d = reinterpret_cast<C2<T> *>(dst) + tc.db + (int64_t)c * P.tsout +
                 (int64_t)t * P.sout;
      const int64_t st = (int64_t)TT * P.sout;
      st_batch<E>(keep, cur, [&](int m) { return d + m * st; });
    } else if (valid) {
      C2<T> *d = reinterpret_cast<C2<T> *>(dst) + tc.db + (int64_t)c * P.tsout;
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int k = t + TT * m - zout;
        if (k >= 0 && k < nout) {
          const T f = msign<T>(P.omod, k);
          C2<T> v{cur[m].x * f, cur[m].y * f};
          if constexpr (TW) {
            const C2<T> *lo = reinterpret_cast<const C2<T> *>(P.tw2);
            const int64_t mm = (tc.c0 + c) * (int64_t)(k + zout);
            v = cmul(v, cmul(lo[mm & 4095], lo[4096 + (mm >> 12)]));
          }
          st_elem(keep, d + (int64_t)k * P.sout, v);
        }
      }
    }
    if (!more) return false;
    // the next tile reuses the LDS exchange buffer (staged lane orders
    // cross waves)
    line_sync<XS == 0 && wave_lines<NF, E, LM>()>();
    item = ni;
    tc = tn;
    return true;
  };
  C2<T> va[E], vb[E];
  if constexpr (XS == 1) load_c2c_pl<KP, T, NF, C, E>(P, src, tc, true, cx0, tx0, va);
  else if constexpr (PL) load_c2c_pl<KP, T, NF, C, E>(P, src, tc, true, c0, t0, va);
  else load_c2c<KP, T, NF, C, E>(P, src, tc, true, c0, t0, va);
  if constexpr (TWL) lds_barrier();
  while (step(va, vb) && step(vb, va)) {
  }
  stamp_end(P, ntiles - 1 - item);
}

// ------------------------------------------------------------------ r2c
// real line of n = 2*NF contiguous samples (sin == 1, no embed) ->
// kept half-spectrum outputs [zout, zout+nout) of the n/2+1.
template <bool KP, typename T, int NF, int C, int E>
__device__ __forceinline__ void load_r2c(const pfk_pass &P, const T *src, const TileCtx &tc,
                                         const bool live, const int c, const int t,
                                         C2<T> *v) {
  constexpr int TT = NF / E;
  const T *s0 = src + tc.sb;
  const C2<T> *s = reinterpret_cast<const C2<T> *>((live && c < tc.nl) ? s0 + (int64_t)c * P.tsin
                                                                     : s0);
  const int step = live ? TT : 0;
  ld_batch<KP, E>(P, v, [&](int m) { return s + (live ? t : 0) + step * m; });
}

template <typename T, int NF, int C, int E, int SIGN, bool PL = false, bool LM = false,
          bool KP = false>
__global__ void __launch_bounds__(C *NF / E)
k_r2c_pow2(const pfk_pass P, const int64_t item0, const int64_t item_end, const int64_t ntiles,
           const T *__restrict__ src, T *__restrict__ dst) {
  stamp_begin(P, item0 + blockIdx.x);
  constexpr int TT = NF / E;
  constexpr int H = NF;  // h = n/2
  constexpr bool TWL = tw_in_lds<T>(lds_slots<NF, C, LM>(), NF, NF);
  __shared__ C2<T> lds[lds_slots<NF, C, LM>()];
  __shared__ C2<T> twl[TWL ? NF : 1], rtwl[TWL ? NF : 1];
  const int tid = threadIdx.x;
  const int c0 = LM ? tid / TT : tid % C, t0 = LM ? tid % TT : tid / C;
  const C2<T> *twg = reinterpret_cast<const C2<T> *>(P.tw);
  const C2<T> *rtwg = reinterpret_cast<const C2<T> *>(P.rtw);
  if constexpr (TWL) {
    stage_table(twl, twg, NF);
    stage_table(rtwl, rtwg, NF);
  }
  const C2<T> *tw = TWL ? twl : twg;
  const C2<T> *rtw = TWL ? rtwl : rtwg;
  const int zout = (int)P.zout, nout = (int)P.nout;
  const bool keep = KP && (P.cache & PFK_KEEP_DST);
  int64_t item = item0 + blockIdx.x;
  TileCtx tc = tile_at(P, C, item, ntiles);
  auto step = [&](C2<T> *cur, C2<T> *nxt) -> bool {
    int t = t0, c = c0;
    asm volatile("" : "+v"(t), "+v"(c));
    const int64_t ni = item + gridDim.x;
    const bool more = ni < item_end;
    const TileCtx tn = tile_at(P, C, more ? ni : item, ntiles);
    load_r2c<KP, T, NF, C, E>(P, src, tn, more, c, t, nxt);
    const bool valid = c < tc.nl;
    if constexpr (!PL) {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int p = t + TT * m;
        const T fx = msign<T>(P.imod, 2 * p), fy = msign<T>(P.imod, 2 * p + 1);
        cur[m] = valid ? C2<T>{cur[m].x * fx, cur[m].y * fy} : C2<T>{0, 0};
      }
    }
    fft_regs<T, NF, C, E, SIGN, LM>(cur, lds, t, c, tw);
    // mirror exchange: Z_{h-k}
#pragma unroll
    for (int m = 0; m < E; ++m) lds[lidx<NF, C, LM>(t + TT * m, c)] = cur[m];
    line_sync<wave_lines<NF, E, LM>()>();
    if (PL && valid) {
      // every output k = t + T*m (and the Nyquist bin, thread t = 0) is kept
      C2<T> *d = reinterpret_cast<C2<T> *>(dst) + tc.db + (int64_t)c * P.tsout;
      C2<T> *dk = d + (int64_t)t * P.sout;
      const int64_t st = (int64_t)TT * P.sout;
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int k = t + TT * m;
        const C2<T> a = cur[m];
        const C2<T> b = lds[lidx<NF, C, LM>((H - k) & (H - 1), c)];
        const C2<T> Ev{(a.x + b.x) * (T)0.5, (a.y - b.y) * (T)0.5};
        const C2<T> O{(a.y + b.y) * (T)0.5, -(a.x - b.x) * (T)0.5};
        const C2<T> WO = cmul(O, rtw[k]);
        st_elem(keep, dk + m * st, C2<T>{Ev.x + WO.x, Ev.y + WO.y});
        if (m == 0 && t == 0)
          st_elem(keep, d + (int64_t)H * P.sout, C2<T>{Ev.x - O.x, Ev.y - O.y});
      }
    } else if (valid) {
      C2<T> *d = reinterpret_cast<C2<T> *>(dst) + tc.db + (int64_t)c * P.tsout;
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int k = t + TT * m;
        const C2<T> a = cur[m];
        const C2<T> b = lds[lidx<NF, C, LM>((H - k) & (H - 1), c)];
        // Ev = (a + conj b)/2, O = -i (a - conj b)/2, X = Ev + W^k O
        const C2<T> Ev{(a.x + b.x) * (T)0.5, (a.y - b.y) * (T)0.5};
        const C2<T> O{(a.y + b.y) * (T)0.5, -(a.x - b.x) * (T)0.5};
        const int ko = k - zout;
        if (ko >= 0 && ko < nout) {
          T f = msign<T>(P.omod, ko);
          if (P.hw == 2 && k != 0) f *= (T)2;
          const C2<T> WO = cmul(O, rtw[k]);
          st_elem(keep, d + (int64_t)ko * P.sout, C2<T>{(Ev.x + WO.x) * f, (Ev.y + WO.y) * f});
        }
        if (k == 0) {  // Nyquist X_h = E_0 - O_0 (W^h = -1)
          const int kn = H - zout;
          if (kn >= 0 && kn < nout) {
            const T f = msign<T>(P.omod, kn);
            d[(int64_t)kn * P.sout] = C2<T>{(Ev.x - O.x) * f, (Ev.y - O.y) * f};
          }
        }
      }
    }
    if (!more) return false;
    line_sync<wave_lines<NF, E, LM>()>();
    item = ni;
    tc = tn;
    return true;
  };
  C2<T> va[E], vb[E];
  load_r2c<KP, T, NF, C, E>(P, src, tc, true, c0, t0, va);
  if constexpr (TWL) lds_barrier();
  while (step(va, vb) && step(vb, va)) {
  }
  stamp_end(P, ntiles - 1 - item);
}

// ------------------------------------------------------------------ c2r
// half spectrum (embedded at zin) -> real line of n = 2*NF contiguous
// samples (sout == 1, no trunc).
template <bool KP, typename T, int NF, int C, int E>
__device__ __forceinline__ void load_c2r(const pfk_pass &P, const T *src, const TileCtx &tc,
                                         const bool live, const int c, const int t, C2<T> *v,
                                         C2<T> &xh) {
  load_c2c<KP, T, NF, C, E>(P, src, tc, live, c, t, v);
  const int jh = NF - (int)P.zin;
  const bool okh = jh >= 0 && jh < (int)P.nin;
  const C2<T> *s0 = reinterpret_cast<const C2<T> *>(src) + tc.sb;
  const C2<T> *s = (live && c < tc.nl) ? s0 + (int64_t)c * P.tsin : s0;
  xh = s[(int64_t)((live && okh) ? jh : 0) * P.sin];
}

// plain half spectrum (all n/2+1 bins, no modulation): loads with uniform
// strides
template <bool KP, typename T, int NF, int C, int E>
__device__ __forceinline__ void load_c2r_pl(const pfk_pass &P, const T *src, const TileCtx &tc,
                                            const bool live, const int c, const int t, C2<T> *v,
                                            C2<T> &xh) {
  load_c2c_pl<KP, T, NF, C, E>(P, src, tc, live, c, t, v);
  const C2<T> *s0 = reinterpret_cast<const C2<T> *>(src) + tc.sb;
  const C2<T> *s = (live && c < tc.nl) ? s0 + (int64_t)c * P.tsin : s0;
  xh = ld_stream(s + (live ? (int64_t)NF * P.sin : 0));
}

template <typename T, int NF, int C, int E, int SIGN, bool PL = false, bool LM = false,
          bool KP = false>
__global__ void __launch_bounds__(C *NF / E)
k_c2r_pow2(const pfk_pass P, const int64_t item0, const int64_t item_end, const int64_t ntiles,
           const T *__restrict__ src, T *__restrict__ dst) {
  stamp_begin(P, item0 + blockIdx.x);
  constexpr int TT = NF / E;
  constexpr int H = NF;
  constexpr int SLOTS = LM ? lds_slots<NF, C, true>() : (NF + 1) * C;   // with the Nyquist bin
  constexpr bool TWL = tw_in_lds<T>(SLOTS, NF, NF);
  __shared__ C2<T> lds[SLOTS];
  __shared__ C2<T> twl[TWL ? NF : 1], rtwl[TWL ? NF : 1];
  const int tid = threadIdx.x;
  const int c0 = LM ? tid / TT : tid % C, t0 = LM ? tid % TT : tid / C;
  const C2<T> *twg = reinterpret_cast<const C2<T> *>(P.tw);
  const C2<T> *rtwg = reinterpret_cast<const C2<T> *>(P.rtw);
  if constexpr (TWL) {
    stage_table(twl, twg, NF);
    stage_table(rtwl, rtwg, NF);
  }
  const C2<T> *tw = TWL ? twl : twg;
  const C2<T> *rtw = TWL ? rtwl : rtwg;
  const int zin = (int)P.zin, nin = (int)P.nin;
  const bool keep = KP && (P.cache & PFK_KEEP_DST);
  int64_t item = item0 + blockIdx.x;
  TileCtx tc = tile_at(P, C, item, ntiles);
  auto step = [&](C2<T> *cur, C2<T> &curh, C2<T> *nxt, C2<T> &nxth) -> bool {
    int t = t0, c = c0;
    asm volatile("" : "+v"(t), "+v"(c));
    const int64_t ni = item + gridDim.x;
    const bool more = ni < item_end;
    const TileCtx tn = tile_at(P, C, more ? ni : item, ntiles);
    if constexpr (PL) load_c2r_pl<KP, T, NF, C, E>(P, src, tn, more, c, t, nxt, nxth);
    else load_c2r<KP, T, NF, C, E>(P, src, tn, more, c, t, nxt, nxth);
    const bool valid = c < tc.nl;
    // X_k, k = t + T*m, and X_h (kept by thread t == 0) into LDS
    if constexpr (PL) {
#pragma unroll
      for (int m = 0; m < E; ++m) lds[lidx<NF, C, LM>(t + TT * m, c)] = cur[m];
      if (t == 0) lds[lidx<NF, C, LM>(H, c)] = C2<T>{curh.x, (T)0};
    } else {
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int k = t + TT * m;
        const int j = k - zin;
        const bool ok = valid && j >= 0 && j < nin;
        T f = msign<T>(P.imod, j);
        if (P.hw == 1 && k != 0) f *= (T)0.5;
        cur[m] = ok ? C2<T>{cur[m].x * f, cur[m].y * f} : C2<T>{0, 0};
        lds[lidx<NF, C, LM>(k, c)] = cur[m];
      }
      if (t == 0) {
        const int jh = H - zin;
        const bool okh = valid && jh >= 0 && jh < nin;
        lds[lidx<NF, C, LM>(H, c)] = okh ? C2<T>{curh.x * msign<T>(P.imod, jh), (T)0} : C2<T>{0, 0};
      }
    }
    line_sync<wave_lines<NF, E, LM>()>();
    // Z_k = E_k + i O_k
#pragma unroll
    for (int m = 0; m < E; ++m) {
      const int k = t + TT * m;
      const C2<T> a = cur[m];
      C2<T> z;
      if (k == 0) {
        const T xhr = lds[lidx<NF, C, LM>(H, c)].x;
        z = C2<T>{a.x + xhr, a.x - xhr};
      } else {
        const C2<T> b = lds[lidx<NF, C, LM>(H - k, c)];
        const C2<T> Ev{a.x + b.x, a.y - b.y};
        const C2<T> O = cmul(C2<T>{a.x - b.x, a.y + b.y}, rtw[k]);
        z = C2<T>{Ev.x - O.y, Ev.y + O.x};
      }
      cur[m] = z;
    }
    line_sync<wave_lines<NF, E, LM>()>();
    fft_regs<T, NF, C, E, SIGN, LM>(cur, lds, t, c, tw);
    if (valid) {
      C2<T> *d = reinterpret_cast<C2<T> *>(dst + tc.db + (int64_t)c * P.tsout);
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const int p = t + TT * m;
        C2<T> x = cur[m];
        if (!PL && P.omod.on) {
          x.x *= msign<T>(P.omod, 2 * p);
          x.y *= msign<T>(P.omod, 2 * p + 1);
        }
        st_elem(keep, d + p, x);
      }
    }
    if (!more) return false;
    line_sync<wave_lines<NF, E, LM>()>();
    item = ni;
    tc = tn;
    return true;
  };
  C2<T> va[E], vb[E], ha, hb;
  if constexpr (PL) load_c2r_pl<KP, T, NF, C, E>(P, src, tc, true, c0, t0, va, ha);
  else load_c2r<KP, T, NF, C, E>(P, src, tc, true, c0, t0, va, ha);
  if constexpr (TWL) lds_barrier();
  while (step(va, ha, vb, hb) && step(vb, hb, va, ha)) {
  }
  stamp_end(P, ntiles - 1 - item);
}

// ------------------------------------------------------------------ dispatch
// Persistent grid: resident workgroups per CU (occupancy of the kernel at
// its LDS size) times the CU count, a multiple of 8 (the XCD count).
template <typename K>
static int64_t persistent_grid(K kernel, int threads) {
  int dev = 0, ncu = 0, occ = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, threads, 0) != hipSuccess ||
      occ < 1)
    occ = 1;
  if (ncu < 8) ncu = 8;
  return (int64_t)occ * (ncu / 8) * 8;
}

// Launches kernel k over `ntiles` items: persistent (grid = resident
// workgroups, `pgrid`) or one workgroup per tile (in chunks of 2^30).
template <typename T>
static int launch_items(void (*k)(pfk_pass, int64_t, int64_t, int64_t, const T *, T *),
                        const pfk_pass *p, int64_t ntiles, int64_t pgrid, bool persistent,
                        int threads, const T *src, T *dst) {
  if (persistent) {
    const int64_t g = ntiles < pgrid ? ntiles : pgrid;
    hipLaunchKernelGGL(k, dim3((unsigned)g), dim3(threads), 0, g_stream, *p, (int64_t)0, ntiles,
                       ntiles, src, dst);
  } else {
    const int64_t chunk = pfk_max_grid(threads);
    for (int64_t base = 0; base < ntiles; base += chunk) {
      const int64_t nblk = (ntiles - base) < chunk ? (ntiles - base) : chunk;
      hipLaunchKernelGGL(k, dim3((unsigned)nblk), dim3(threads), 0, g_stream, *p, base,
                         base + nblk, ntiles, src, dst);
    }
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error("pfk_launch_pass(pow2)", e); return -1; }
  return 0;
}

// Paired-line stores (the PAIR parameter of k_c2c_pow2) on the store side
// (or loads, `in`): lines adjacent in memory (tile stride 1), even element
// strides and a 16-byte-aligned array, so that every pair of lines starts
// on a 16-byte boundary; at least two lines.
static bool pair_side_ok(const pfk_pass *p, bool in, const void *ptr) {
  const int64_t ts = in ? p->tsin : p->tsout, ls = in ? p->sin : p->sout;
  if (p->prec != PFK_F32 || ts != 1 || p->text < 2 || (ls & 1) || ((uintptr_t)ptr & 15))
    return false;
  for (int i = 0; i < p->nb; ++i)
    if ((in ? p->bsin[i] : p->bsout[i]) & 1) return false;
  return true;
}

// Line-major staging of a complex64 c2c pass (the XS parameter of
// k_c2c_pow2): 1 when the lines are contiguous only on the store side and
// adjacent along the tile dimension on the load side, 2 for the reverse.
static int lm_staging(const pfk_pass *p) {
  if (p->sin != 1 && p->tsin == 1 && p->sout == 1) return 1;
  if (p->sin == 1 && p->sout != 1 && p->tsout == 1) return 2;
  return 0;
}

template <typename T>
using pow2_kernel = void (*)(pfk_pass, int64_t, int64_t, int64_t, const T *, T *);

// launch_items of kernel K with its persistent grid (computed once)
template <typename T, pow2_kernel<T> K>
static int launch_one(const pfk_pass *p, int64_t ntiles, int threads, const void *src,
                      void *dst) {
  static int64_t grid = 0;
  if (!grid) grid = persistent_grid(K, threads);
  return launch_items(K, p, ntiles, grid, !(p->variant & 4), threads, (const T *)src, (T *)dst);
}

template <typename T, int NF, int C, int E, int SIGN, bool TWOK, bool PL, bool KP>
static int launch_kind_pl(const pfk_pass *p, int64_t ntiles, const void *src, void *dst) {
  constexpr int NT = C * NF / E;
#define PFK_LAUNCH_C2C(LM, TW, PLAIN, XS, PAIR) \
  launch_one<T, k_c2c_pow2<T, NF, C, E, SIGN, LM, TW, PLAIN, XS, PAIR, KP>>(p, ntiles, NT, src, dst)
#define PFK_LAUNCH_REAL(K, LM) \
  launch_one<T, K<T, NF, C, E, SIGN, PL, LM, KP>>(p, ntiles, NT, src, dst)
  if (p->kind == PFK_C2C && p->twn) {
    if constexpr (TWOK && !PL && !KP) return PFK_LAUNCH_C2C(false, true, false, 0, 0);
    return 1;
  }
  // line-major lane order (variant bit 8): complex64, and complex128 on
  // plain passes
  constexpr bool LMOK = sizeof(T) == 4 || PL;
  const bool lm = LMOK && (p->variant & 8);
  if (p->kind == PFK_C2C) {
    if constexpr (LMOK) {
      if (lm) {
        const int xs = PL ? lm_staging(p) : 0;
        if constexpr (PL && sizeof(T) == 4) {
          // paired-line stores on the tile side of a transposing pass (512-point
          // complex64 lines: 5.10 -> 5.27 TB/s); paired loads measured no
          // faster there and slower on passes that are tile-adjacent on both
          // sides (5.0 -> 4.7 TB/s), so those keep 8-byte lanes
          if (xs == 2 && pair_side_ok(p, false, dst))
            return PFK_LAUNCH_C2C(true, false, true, 2, 1);
        }
        if constexpr (PL) {
          if (xs == 1) return PFK_LAUNCH_C2C(true, false, true, 1, 0);
          if (xs == 2) return PFK_LAUNCH_C2C(true, false, true, 2, 0);
        }
        return PFK_LAUNCH_C2C(true, false, PL, 0, 0);
      }
    }
    return PFK_LAUNCH_C2C(false, false, PL, 0, 0);
  }
  const bool r2c = p->kind == PFK_R2C;
  if constexpr (LMOK) {
    if (lm) return r2c ? PFK_LAUNCH_REAL(k_r2c_pow2, true) : PFK_LAUNCH_REAL(k_c2r_pow2, true);
  }
  return r2c ? PFK_LAUNCH_REAL(k_r2c_pow2, false) : PFK_LAUNCH_REAL(k_c2r_pow2, false);
#undef PFK_LAUNCH_C2C
#undef PFK_LAUNCH_REAL
}

// the plain and the cache-keeping instantiations exist for the default tiles
// only; a step of a long line streams
template <typename T, int NF, int C, int E, int SIGN, bool TWOK>
static int launch_kind(const pfk_pass *p, int64_t ntiles, const void *src, void *dst) {
  if constexpr (TWOK) {
    const bool pl = pass_plain(p);
    if (p->cache && !p->twn)
      return pl ? launch_kind_pl<T, NF, C, E, SIGN, true, true, true>(p, ntiles, src, dst)
                : launch_kind_pl<T, NF, C, E, SIGN, true, false, true>(p, ntiles, src, dst);
    if (pl) return launch_kind_pl<T, NF, C, E, SIGN, true, true, false>(p, ntiles, src, dst);
  }
  return launch_kind_pl<T, NF, C, E, SIGN, TWOK, false, false>(p, ntiles, src, dst);
}

// TWOK: the table also instantiates the twiddled first step of long lines
template <typename T, int NF, int C, int E, bool TWOK = true>
static int launch_nf(const pfk_pass *p, const void *src, void *dst) {
  int64_t ntiles = (p->text + C - 1) / C;
  for (int i = 0; i < p->nb; ++i) ntiles *= p->bext[i];
  if (ntiles <= 0) return 0;
  return p->sign < 0 ? launch_kind<T, NF, C, E, -1, TWOK>(p, ntiles, src, dst)
                     : launch_kind<T, NF, C, E, +1, TWOK>(p, ntiles, src, dst);
}


}  // namespace pfk
