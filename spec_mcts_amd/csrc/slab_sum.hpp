// Sums over the K-slice slabs a Q4_0 matmul kernel leaves (q40_matmul.hpp), in slice order, in fp32.
#pragma once

#include "q40_matmul.hpp"

namespace smh {

// The numbers of slabs that the kernels below are instantiated for are 1 .. 6, 8, 10, 12 and 16, which are nearly all that the plans of 7B, 13B,
// 34B and 70B shapes come to (7, 9, 11 and 13 .. 15 at a few row counts): the next one takes those in between, from this one up.
__host__ __device__ constexpr int least_slabs(int KS) { return KS <= 6 ? KS : KS <= 12 ? KS - 1 : 13; }
// Elements idx .. of `ks` slabs on their way, KS or a few less (past the last one that one again, for slab_add to leave out): T is float,
// f2 or f4 (idx a multiple of 2 or 4).  Kernels that live by this are instantiated by KS: with a condition on each load the compiler moves
// what it has between registers in between, and waits for it first (two or three trips to memory one behind the other instead of
// one).  In turn: eight steps of 100 branches (7B) 31.85 -> 31.30 ms, 37 branches 2986 -> 2942 us a step, 512-row prefill 8.64 -> 8.46 ms,
// 10 branches of three 70B layers 537 -> 528 us.
template <typename T, int KS>
__device__ __forceinline__ void slab_load(const void *partial, long idx, long slab_stride, int ks, T (&v)[KS]) {
    const float *p = reinterpret_cast<const float *>(partial) + idx;
#pragma unroll
    for (int s = 0; s < KS; ++s) v[s] = *reinterpret_cast<const T *>(p + (s < least_slabs(KS) ? s : min(s, ks - 1)) * slab_stride);
}
// ... added in slice order.
template <typename T, int KS>
__device__ __forceinline__ T slab_add(const T (&v)[KS], int ks) {
    float zero = 0.f;
    asm("" : "+v"(zero));                                    // (a zero that the compiler knows it adds where the first slab is loaded, and waits there)
    T tot = T{} + zero;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const T next = tot + v[s];
        tot = s < least_slabs(KS) || s < ks ? next : tot;
    }
    return tot;
}
// Four consecutive elements of `ksplit` slabs, added.
__device__ __forceinline__ f4 slab_sum4(const void *partial, long idx, long slab_stride, int ksplit) {
    const float *p = reinterpret_cast<const float *>(partial) + idx;
    f4 v[SMH_MAX_KSPLIT];
#pragma unroll
    for (int s = 0; s < SMH_MAX_KSPLIT; ++s) v[s] = (s < ksplit) ? *reinterpret_cast<const f4 *>(p + s * slab_stride) : f4{0.f, 0.f, 0.f, 0.f};
    return slab_add(v, SMH_MAX_KSPLIT);
}

}  // namespace smh
