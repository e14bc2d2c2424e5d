// pass_access.hpp -- global accesses, index modulation and tile decoding
// shared by the register-resident pass kernels.
#pragma once
#include "pfk_internal.hpp"

namespace pfk {

template <typename T>
using C2 = cpx<T>;

// Global accesses.  Streaming (nontemporal) accesses leave nothing behind in
// the 256 MB memory-side cache, kept ones do: an array that the next pass or
// the next chunk of the plan touches again while it is still there is kept
// (pfk_pass.cache), everything else is streamed.  The kernels' KP
// instantiations choose at run time; the others stream without looking (the
// choice alone cost passes that stream 1%: 512^3 complex128 pair 2.29 -> 2.31
// ms).
template <typename T>
__device__ __forceinline__ C2<T> ld_stream(const C2<T> *p) {
  typedef T v2 __attribute__((ext_vector_type(2)));
  const v2 v = __builtin_nontemporal_load(reinterpret_cast<const v2 *>(p));
  return C2<T>{v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void st_stream(C2<T> *p, C2<T> v) {
  typedef T v2 __attribute__((ext_vector_type(2)));
  v2 w;
  w.x = v.x;
  w.y = v.y;
  __builtin_nontemporal_store(w, reinterpret_cast<v2 *>(p));
}
// loads v[m] = *at(m), m < N, kept or streamed: one uniform branch around the
// whole batch of loads
template <bool KP, int N, typename T, typename At>
__device__ __forceinline__ void ld_batch(const pfk_pass &P, C2<T> *v, At at) {
  if (KP && (P.cache & PFK_KEEP_SRC)) {
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = *at(m);
  } else {
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = ld_stream(at(m));
  }
}
template <typename T>
__device__ __forceinline__ void st_elem(const bool keep, C2<T> *p, C2<T> v) {
  if (keep) *p = v;
  else st_stream(p, v);
}
// stores *at(m) = v[m], m < N
template <int N, typename T, typename At>
__device__ __forceinline__ void st_batch(const bool keep, const C2<T> *v, At at) {
  if (keep) {
#pragma unroll
    for (int m = 0; m < N; ++m) *at(m) = v[m];
  } else {
#pragma unroll
    for (int m = 0; m < N; ++m) st_stream(at(m), v[m]);
  }
}

// +-1 modulation factor of index j, computed with selects only: a branch
// here would sit between a load and its use and make the compiler wait for
// every load before issuing the next one.
template <typename T>
__device__ __forceinline__ T msign(const pfk_mod &m, int64_t j) {
  const int64_t t = j + m.start;
  const int s = (m.on && t < m.half) ? ((t & 1) ? -m.extra : m.extra) : 1;
  return (T)s;
}

// i / d for i * d < 2^32, with m = recip(d) (m = 0: d = 1)
__device__ __forceinline__ int div_m(int i, uint32_t m) {
  return m ? (int)__umulhi((uint32_t)i, m) : i;
}
static inline uint32_t recip(int64_t d) {   // ceil(2^32 / d)
  return d <= 1 ? 0 : (uint32_t)((((uint64_t)1 << 32) + (uint64_t)d - 1) / (uint64_t)d);
}

struct TileCtx {
  int64_t sb, db;
  int64_t c0;   // first line of the tile along the tile dimension
  int nl;
};

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  With remap on, XCD x runs a contiguous range of tiles in order, so
// tiles that share cache lines at their edges run on the same L2 close in
// time.  The map is a bijection on [0, n) for any n; item i runs on XCD
// i mod 8 because the persistent grid is a multiple of 8.
__device__ __forceinline__ int64_t xcd_remap(int64_t b, int64_t n) {
  const int64_t q = n >> 3, r = n & 7;
  const int64_t x = b & 7, j = b >> 3;
  return x * q + (x < r ? x : r) + j;
}

// Tile of work item `item` (0 <= item < ntiles).  Tile counts below 2^32
// (every practical pass) decode with 32-bit divisions, several times
// shorter than the 64-bit chain.
__device__ __forceinline__ TileCtx tile_at(const pfk_pass &P, int C, int64_t item,
                                           int64_t ntiles) {
  const int64_t ntt = (P.text + C - 1) / C;
  const int64_t tileid = P.xcd_remap ? xcd_remap(item, ntiles) : item;
  int64_t tt, sb = 0, db = 0;
  if (ntiles <= (int64_t)0xFFFFFFFFu) {
    uint32_t id = (uint32_t)tileid;
    const uint32_t n32 = (uint32_t)ntt;
    tt = id % n32;
    id /= n32;
    for (int i = 0; i < P.nb; ++i) {
      const uint32_t e = (uint32_t)P.bext[i];
      const uint32_t d = id % e;
      id /= e;
      sb += (int64_t)d * P.bsin[i];
      db += (int64_t)d * P.bsout[i];
    }
  } else {
    tt = tileid % ntt;
    int64_t bflat = tileid / ntt;
    for (int i = 0; i < P.nb; ++i) {
      const int64_t e = P.bext[i];
      const int64_t d = bflat % e;
      bflat /= e;
      sb += d * P.bsin[i];
      db += d * P.bsout[i];
    }
  }
  const int64_t c0 = tt * C;
  TileCtx r;
  r.c0 = c0;
  r.nl = (int)((P.text - c0) < C ? (P.text - c0) : C);
  r.sb = sb + c0 * P.tsin;
  r.db = db + c0 * P.tsout;
  return r;
}

}  // namespace pfk
