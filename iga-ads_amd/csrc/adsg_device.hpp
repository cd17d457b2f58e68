// Device helpers shared by the element-loop kernels (adsg_rhs.hip, adsg_rhs_march.hip) and the segmented
// line sweeps (adsg_seg.inc).
#pragma once

#include <hip/hip_runtime.h>

#include "adsg_kernels.hpp"

namespace adsg {

namespace {

constexpr int kXcds = 8;  // MI355X: 8 accelerator complex dies, 32 CUs each

// block b (dispatched to XCD b % 8) -> tile index, a bijection of [0, n) that gives every
// XCD a contiguous range of tiles
__device__ __forceinline__ int xcd_contiguous(int b, int n) {
    const int per = n / kXcds, rem = n % kXcds;
    const int x = b % kXcds, i = b / kXcds;
    return x < rem ? x * (per + 1) + i : rem * (per + 1) + (x - rem) * per + i;
}

// A read of read-only, wave-uniform data through the constant address space: always a
// scalar load, also after instructions the compiler must treat as memory writes.
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p) {
    using CT = const __attribute__((address_space(4))) T*;
    return *(CT)(p);
}

// Orders a wave's LDS writes before its later LDS reads by other lanes of the same wave (LDS
// operations of one wave complete in issue order; the fences keep the compiler from moving
// accesses across): a transpose inside one wave needs no workgroup barrier.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// index of a spilled entry in the spill arrays: array delta = dx + 2 dy + 4 dz, position
// (cx, cy, cz) in its extents
template <typename T>
__device__ __forceinline__ long spill_index(const rhs_params<T>& prm, int dx, int dy, int dz, int cx, int cy,
                                            int cz) {
    const int delta = dx + 2 * dy + 4 * dz;
    long off = 0;
#pragma unroll
    for (int j = 1; j < 8; ++j)
        if (delta == j) off = prm.spill_off[j];  // selects: no dynamic index into the argument
    const long ex = dx ? prm.spill_ext[0][1] : prm.spill_ext[0][0];
    const long ey = dy ? prm.spill_ext[1][1] : prm.spill_ext[1][0];
    return off + cx + ex * (cy + ey * cz);
}

}  // namespace

}  // namespace adsg
