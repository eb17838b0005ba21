// Accesses to LDS that the compiler has no plain form for.
#pragma once

#include "mesh_common.hpp"

namespace mesh {

typedef uint32_t lds_u2 __attribute__((ext_vector_type(2)));

// byte address of a place in LDS
__device__ __forceinline__ unsigned lds_place(const void *p) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (unsigned)(unsigned long long)(__attribute__((address_space(3))) const char *)p;
#else
    return 0;
#endif
}

// 1 KB from memory to LDS without passing registers: the 16 bytes at base + off (bytes, a lane's own) go to place + 16 lane (uniform).
// As text: behind the builtin the compiler waits for every load in flight at the next access to LDS, cross-lane moves among them.
// Its own counts stay right, a load it does not know of only makes a wait stricter; who reads the place waits for its arrival.
__device__ __forceinline__ void load_to_lds_16(const void *base, uint32_t off, unsigned place) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"         // (m0 is reserved: named so that the compiler keeps its own uses away)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(place)), "v"(off), "s"(base) : "memory", "m0");
#pragma clang diagnostic pop
#endif
}

// Four halves of one column of a 4-row x 16-column tile: lane i of a group of 16 lanes hands in the address of row i / 4,
// columns 4 (i % 4) .. + 4, and receives column i of the four rows.
__device__ __forceinline__ lds_u2 lds_read_transposed(const _Float16 *p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef short s4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(lds_u2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4 *)p));
#else
    return lds_u2{0, 0};
#endif
}

// Workgroup barrier that orders LDS only.  __syncthreads() also waits for every outstanding global load.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The LDS unit executes a wave's accesses in order; the fences only keep the compiler from reordering them.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace mesh
