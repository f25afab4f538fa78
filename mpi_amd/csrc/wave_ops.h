// wave_ops.h -- lane exchanges and reductions of one wave, without LDS.
#pragma once

#include <hip/hip_runtime.h>

namespace hz {
namespace {

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Lane exchanges without LDS: DPP moves within rows of 16 lanes, readlane
// across them.
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)dpp_i32<CTRL>((int)(unsigned)b);
    const unsigned hi = (unsigned)dpp_i32<CTRL>((int)(unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v of lane l (l uniform)
__device__ __forceinline__ double lane_f64(double v, int l)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// DPP controls: quad_perm [1,0,3,2] and [2,3,0,1] (lane xor 1, xor 2), then
// the half-row and row mirrors, which leave every lane with the reduction
// over its row of 16 lanes; the four rows are then combined by readlane.
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;

// Maximum of v over the wave (uniform result); v is not NaN.
__device__ __forceinline__ double wave_max_f64(double v)
{
    v = fmax(v, dpp_f64<kDppXor1>(v));
    v = fmax(v, dpp_f64<kDppXor2>(v));
    v = fmax(v, dpp_f64<kDppHalfMirror>(v));
    v = fmax(v, dpp_f64<kDppMirror>(v));
    return fmax(fmax(lane_f64(v, 0), lane_f64(v, 16)), fmax(lane_f64(v, 32), lane_f64(v, 48)));
}

// Minimum of v over the wave (uniform result).
__device__ __forceinline__ int wave_min_i32(int v)
{
    v = min(v, dpp_i32<kDppXor1>(v));
    v = min(v, dpp_i32<kDppXor2>(v));
    v = min(v, dpp_i32<kDppHalfMirror>(v));
    v = min(v, dpp_i32<kDppMirror>(v));
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Maximum of v over the wave (uniform result).
__device__ __forceinline__ int wave_max_i32(int v)
{
    v = max(v, dpp_i32<kDppXor1>(v));
    v = max(v, dpp_i32<kDppXor2>(v));
    v = max(v, dpp_i32<kDppHalfMirror>(v));
    v = max(v, dpp_i32<kDppMirror>(v));
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

}  // namespace
}  // namespace hz
