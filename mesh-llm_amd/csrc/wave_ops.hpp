// Reductions and sums over the 64 lanes of a wave without the LDS unit.
#pragma once

#include "mesh_common.hpp"

namespace mesh {

// f(v, v of lane ^ 32), then ^ 16, 8, 4, 2, 1: the bits of the butterfly over __shfl_xor in that order, in every lane (f commutes).  Lanes 8 apart
// hold the same value after the step over 8, so that a rotation of the row by 4 is as good as an exchange over 4, and so on.  Six
// moves of a cycle or two each; a trip through ds_bpermute is 60 to 100 cycles.
template <class F> __device__ __forceinline__ float wave_fold(float v, F f) {
#if defined(__HIP_DEVICE_COMPILE__)
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = f(__uint_as_float(b[0]), __uint_as_float(b[1]));
    v = f(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false)));     // row_ror 8
    v = f(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, false)));
    v = f(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xF, 0xF, false)));
    v = f(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xF, 0xF, false)));
#endif
    return v;
}
__device__ __forceinline__ float wave_sum(float v) { return wave_fold(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ float wave_max(float v) { return wave_fold(v, [](float a, float b) { return fmaxf(a, b); }); }

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
