// Exchanges, reductions and sums over the lanes of a wave without the LDS unit: a lane move is a cycle or two, a trip through ds_bpermute
// (__shfl_xor) 60 to 100 of waiting, and these stand in the chains that most launches of a decode step are bound by.
#pragma once

#include "mesh_common.hpp"

namespace mesh {

template <int CTRL, class T> __device__ __forceinline__ T lane_dpp(T v) {
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// f(v, v of lane ^ O), in both lanes the same bits (f commutes)
template <int O, class T, class F> __device__ __forceinline__ T lane_fold(T v, F f) {
    static_assert(sizeof(T) == 4 && (O == 1 || O == 2 || O == 4 || O == 8 || O == 16 || O == 32), "a lane bit");
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (O == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
        const unsigned a = r[0], b = r[1];
        return f(__builtin_bit_cast(T, a), __builtin_bit_cast(T, b));
    } else if constexpr (O == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
        const unsigned a = r[0], b = r[1];
        return f(__builtin_bit_cast(T, a), __builtin_bit_cast(T, b));
    } else if constexpr (O == 8) return f(v, lane_dpp<0x128>(v));                       // row_ror 8
    else if constexpr (O == 4) return f(v, lane_dpp<0x1B>(lane_dpp<0x141>(v)));        // mirrored within eight lanes, then within four
    else return f(v, lane_dpp<O == 2 ? 0x4E : 0xB1>(v));                               // within four
#else
    return v;
#endif
}
// folds over the bits FROM, FROM / 2, ... 1: the bits of a butterfly over __shfl_xor in that order.  (After the step over 8 the lanes 8
// apart hold the same value, so that a rotation of the row by 4 is as good as an exchange over 4, and so on.)
template <int FROM, class T, class F> __device__ __forceinline__ T lanes_fold(T v, F f) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (FROM >= 32) v = lane_fold<32>(v, f);
    if constexpr (FROM >= 16) v = lane_fold<16>(v, f);
    if constexpr (FROM >= 8) {
        v = lane_fold<8>(v, f);
        v = f(v, lane_dpp<0x124>(v));
        v = f(v, lane_dpp<0x122>(v));
        v = f(v, lane_dpp<0x121>(v));
    } else {
        if constexpr (FROM >= 4) v = lane_fold<4>(v, f);
        v = lane_fold<2>(v, f);
        v = lane_fold<1>(v, f);
    }
#endif
    return v;
}
struct LaneAdd { template <class T> __device__ __forceinline__ T operator()(T a, T b) const { return a + b; } };
struct LaneMax { __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); } };
__device__ __forceinline__ float wave_sum(float v) { return lanes_fold<32>(v, LaneAdd{}); }
__device__ __forceinline__ float wave_max(float v) { return lanes_fold<32>(v, LaneMax{}); }
// over the 4, 8 or 16 neighbouring lanes of an aligned group, from the nearest on
template <int N, class T> __device__ __forceinline__ T group_sum(T v) {
    v = lane_fold<2>(lane_fold<1>(v, LaneAdd{}), LaneAdd{});
    if constexpr (N >= 8) v += lane_dpp<0x141>(v);          // (lanes of four hold the same: a mirror is as good as an exchange)
    if constexpr (N >= 16) v += lane_dpp<0x140>(v);
    return v;
}

// Sum of v over this lane and those before it.
__device__ __forceinline__ int wave_scan(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);      // row_shr 1, 2, 4, 8: within rows of 16
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);      // a row's last lane to the next row, then lane 31 to the upper half
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
#endif
    return v;
}

}  // namespace mesh
