// pfk_internal.hpp -- shared definitions of the HIP translation units.
#pragma once
#include <hip/hip_runtime.h>
#include "pfk.h"

namespace pfk {

template <typename T>
struct alignas(2 * sizeof(T)) cpx {
  T x, y;
};

template <typename T>
__device__ __forceinline__ cpx<T> cmul(cpx<T> a, cpx<T> b) {
  return cpx<T>{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}

// Workgroup barrier ordering LDS accesses only.  The pass kernels share
// nothing through global memory inside a launch, so a barrier need not wait
// for outstanding global stores (or prefetched loads, which complete in
// order with them) the way __syncthreads() does.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Times of a pass (pfk_pass.stamp): its start from the workgroup whose first
// work item is item 0 of the pass, its end from the workgroups whose last item
// is among the last PFK_STAMP_ENDS of the pass (`left` items follow it).  In a
// walk b, b + grid, ... those are not the last workgroups of the grid: with
// items left over after the full rounds, the low-numbered ones run them, and
// the others end up to a round earlier.  Every lane stores: a test of the
// thread index would keep it in a register to the end, one more than the 128
// that leave the 512-point complex128 kernels 16 waves per CU (512^3 pair 2.28
// -> 2.38 ms).
__device__ __forceinline__ void stamp_begin(const pfk_pass &P, const int64_t first) {
  if (P.stamp && first == 0) *P.stamp = wall_clock64();
}
__device__ __forceinline__ void stamp_end(const pfk_pass &P, const int64_t left) {
  if (P.stamp_end && left < PFK_STAMP_ENDS) P.stamp_end[left] = wall_clock64();
}

// `left` of this workgroup in a walk whose last item workgroup `last` runs.  From
// the block index rather than the walk's counter, whose life to the end of the
// kernel cost the mixed-radix kernel a spilled register (100^3 complex128 47.9 ->
// 49.5 us).
__device__ __forceinline__ int64_t walk_left(const int last) {
  const int left = last - (int)blockIdx.x;
  return left < 0 ? left + (int)gridDim.x : left;
}

extern hipStream_t g_stream;
extern int g_generic_only;   // PFFT_AMD_GENERIC_ONLY=1: route every pass to the general kernel
extern int g_max_lds;
void set_error(const char *what, hipError_t e);
void set_error_msg(const char *msg);

// Specialised kernels: return 0 if the pass was launched, nonzero if the
// pass shape is not covered (the caller then uses the general kernel).
int launch_fast(const pfk_pass *p, const void *src, void *dst);
int launch_generic(const pfk_pass *p, const void *src, void *dst);
int launch_mfma(const pfk_pass *p, const void *src, void *dst);
int launch_mfma_chain(const pfk_pass *p, const void *src, void *dst);
int launch_small(const pfk_pass *p, const void *src, void *dst);
int launch_plane(const pfk_pass *p, const void *src, void *dst);
int launch_mixed(const pfk_pass *p, const void *src, void *dst);
int mixed_covers(const pfk_pass *p);  // 1 if launch_mixed has a kernel for the shape
int fast_covers(const pfk_pass *p);   // 1 if launch_fast has a kernel for the shape
int mfma_covers(const pfk_pass *p);   // 1 if launch_mfma has a kernel for the shape
int mfma_chain_covers(const pfk_pass *p);   // plain 256..1024-point passes (chained MFMA)
int small_covers(const pfk_pass *p);  // 1 if launch_small has a kernel for the shape

}  // namespace pfk
