// Reductions over a wave64 by data-parallel primitives, and an LDS-only
// barrier: what the pivot searches of the panel factorisations use.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vx {

// Maximum over the wave of values that are no NaN, at least 0 (v_max_f64
// itself: fmax would quiet its operands first).
template <int CTRL>
__device__ __forceinline__ double dpp_max(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(v), "v"(__hiloint2double(hi, lo)));
    return r;
}
__device__ __forceinline__ double row_max(double v) {  // lane 15: over the first 16 lanes
    return dpp_max<0x118>(dpp_max<0x114>(dpp_max<0x112>(dpp_max<0x111>(v))));
}
template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) {
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true)));
}
__device__ __forceinline__ float row_max(float v) {
    return dpp_max<0x118>(dpp_max<0x114>(dpp_max<0x112>(dpp_max<0x111>(v))));
}
__device__ __forceinline__ float lane_of(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ float wave_max(float v) { return lane_of(dpp_max<0x143>(dpp_max<0x142>(row_max(v))), 63); }
__device__ __forceinline__ double lane_of(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ __forceinline__ double wave_max(double v) { return lane_of(dpp_max<0x143>(dpp_max<0x142>(row_max(v))), 63); }

template <int CTRL>
__device__ __forceinline__ int dpp_min(int v) {
    return min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, CTRL, 0xf, 0xf, false));
}
// The lane of `ties` (not empty) whose pos is lowest; a body's symmetry makes
// many entries of a column equal.
__device__ __forceinline__ int lowest_lane(uint64_t ties, int pos) {
    if (!(ties & (ties - 1))) return __ffsll((unsigned long long)ties) - 1;
    const bool in = (ties >> (threadIdx.x & 63)) & 1;
    int v = in ? pos : 0x7fffffff;
    v = dpp_min<0x118>(dpp_min<0x114>(dpp_min<0x112>(dpp_min<0x111>(v))));
    v = dpp_min<0x143>(dpp_min<0x142>(v));
    const int low = __builtin_amdgcn_readlane(v, 63);
    return __ffsll((unsigned long long)__ballot(in && pos == low)) - 1;
}

// A barrier that orders LDS accesses only: the factors' stores to memory,
// which only their own thread reads back, need not be waited for each step.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace vx
