// Tiles of K-quants as fragments of v_mfma_f32_16x16x32_f16, formed in registers (gemm_skinny_f16.hip, expert_step.hip).
#pragma once

#include "gemv_device.hpp"

namespace mesh {
namespace f16sk {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ h2_t h2_of(float v) {
    const _Float16 h = (_Float16)v;
    return h2_t{h, h};
}
__device__ __forceinline__ h2_t h2_bits(uint32_t v) { return __builtin_bit_cast(h2_t, v); }
__device__ __forceinline__ uint32_t h2_bits(h2_t v) { return __builtin_bit_cast(uint32_t, v); }

// A choice between two values by lane, as arithmetic: written as `lane ? a : b`, the two formulas of a tile's scales are compiled
// into branches.
__device__ __forceinline__ uint32_t lanes_mask(bool b) {
    uint32_t m = b ? 0xFFFFFFFFu : 0u;
    asm("" : "+v"(m));          // (or the compiler turns the arithmetic back into the choice)
    return m;
}
__device__ __forceinline__ uint32_t bits_of(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | (b & ~mask); }

// Weight fragments of one tile, MFMA by MFMA.  frag(t) returns the fragment of MFMA t (0..7), integers exact in f16 (see below for
// q6_K): the sum of the tile's products times `d` is what the weights without their minimum contribute.  minimum(high), where a
// type has one, is the same for all MFMAs of a sub-block: its products times `ndmin` complete the sum.
template <int TYPE> struct TileFrags;

template <> struct TileFrags<MESH_Q4_K> {
    static constexpr bool MINIMUM = true;
    uint32_t w[8];
    h2_t s_lo, s_hi, o_lo, o_hi;
    uint32_t m_lo, m_hi, mask_lo, mask_hi, base_lo, base_hi;
    float d, ndmin;
    __device__ __forceinline__ void prepare(const TileRegs<MESH_Q4_K> &R, int g) {
        d = f16_bits_to_f32((uint16_t)(R.hdr.x & 0xFFFFu));
        ndmin = -f16_bits_to_f32((uint16_t)(R.hdr.x >> 16));
        // 6-bit (scale, min) of sub-blocks 2g and 2g+1 (get_scale_min_k4 of ggml-quants.c)
        const uint32_t first = lanes_mask(g < 2);
        const uint32_t scw = bits_of(first, R.hdr.y & 0x3F3F3F3Fu, (R.hdr.w & 0x0F0F0F0Fu) | ((R.hdr.y >> 2) & 0x30303030u));
        const uint32_t mnw = bits_of(first, R.hdr.z & 0x3F3F3F3Fu, ((R.hdr.w >> 4) & 0x0F0F0F0Fu) | ((R.hdr.z >> 2) & 0x30303030u));
        const int sh = (g & 1) * 16;
        s_lo = h2_of((float)((scw >> sh) & 0xFFu));                  // integers below 64: exact
        s_hi = h2_of((float)((scw >> (sh + 8)) & 0xFFu));
        o_lo = s_lo * h2_of(-1024.f);                                // (powers of two times them: exact too)
        o_hi = s_hi * h2_of(-64.f);
        m_lo = h2_bits(h2_of((float)((mnw >> sh) & 0xFFu)));
        m_hi = h2_bits(h2_of((float)((mnw >> (sh + 8)) & 0xFFu)));
        // (values the compiler cannot see make mask and base one and-or; with literals it forms an and, then an or)
        mask_lo = 0x000F000Fu; mask_hi = 0x00F000F0u; base_lo = 0x64006400u; base_hi = 0x54005400u;
        asm("" : "+s"(mask_lo), "+s"(mask_hi), "+v"(base_lo), "+v"(base_hi));
        const uint32_t q[8] = {R.qa.x, R.qa.y, R.qa.z, R.qa.w, R.qb.x, R.qb.y, R.qb.z, R.qb.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = __builtin_amdgcn_perm(0u, q[i], 0x03010200u);      // bytes 0 2 1 3: neighbours 16 bits apart
    }
    // MFMA t: t < 4 low nibbles (sub-block 2g), bytes 8t..8t+7; t >= 4 high nibbles (sub-block 2g+1).  0x6400 | q is 1024 + q, and
    // 0x5400 | q << 4 is 64 + q; one fma takes the offset off and multiplies by the sub-block's integer scale: q * sc <= 945.
    __device__ __forceinline__ h8_t frag(int t) const {
        const int tt = t & 3;
        u4_t a;                                                      // built as four dwords: no half-register moves
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t v = i & 1 ? w[2 * tt + (i >> 1)] >> 8 : w[2 * tt + (i >> 1)];
            a[i] = t < 4 ? h2_bits(__builtin_elementwise_fma(h2_bits((v & mask_lo) | base_lo), s_lo, o_lo))
                         : h2_bits(__builtin_elementwise_fma(h2_bits((v & mask_hi) | base_hi), s_hi, o_hi));
        }
        return __builtin_bit_cast(h8_t, a);
    }
    __device__ __forceinline__ h8_t minimum(int t) const {
        const uint32_t v = t < 4 ? m_lo : m_hi;
        return __builtin_bit_cast(h8_t, u4_t{v, v, v, v});
    }
};

template <> struct TileFrags<MESH_Q6_K> {
    static constexpr bool MINIMUM = false;
    uint32_t v[4][4];      // [t4][dword]: six-bit quants in bytes, elements 128n + 32 t4 + 16u + 4 dword + byte
    h2_t s[4];
    float d;
    __device__ __forceinline__ void prepare(const TileRegs<MESH_Q6_K> &R, int g) {
        const int n = g >> 1, u = g & 1;
        d = f16_bits_to_f32((uint16_t)R.d);
        const uint32_t la[4] = {R.qla.x, R.qla.y, R.qla.z, R.qla.w}, lb[4] = {R.qlb.x, R.qlb.y, R.qlb.z, R.qlb.w};
        const uint32_t qh[4] = {R.qh.x, R.qh.y, R.qh.z, R.qh.w};
        const uint32_t upper = lanes_mask(n != 0), scw0 = bits_of(upper, R.sc.z, R.sc.x), scw1 = bits_of(upper, R.sc.w, R.sc.y);
        s[0] = h2_of((float)(int8_t)((scw0 >> (8 * u)) & 0xFFu));     // int8: exact
        s[1] = h2_of((float)(int8_t)((scw0 >> (16 + 8 * u)) & 0xFFu));
        s[2] = h2_of((float)(int8_t)((scw1 >> (8 * u)) & 0xFFu));
        s[3] = h2_of((float)(int8_t)((scw1 >> (16 + 8 * u)) & 0xFFu));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[0][j] = (la[j] & 0x0F0F0F0Fu) | ((qh[j] << 4) & 0x30303030u);
            v[1][j] = (lb[j] & 0x0F0F0F0Fu) | ((qh[j] << 2) & 0x30303030u);
            v[2][j] = ((la[j] >> 4) & 0x0F0F0F0Fu) | (qh[j] & 0x30303030u);
            v[3][j] = ((lb[j] >> 4) & 0x0F0F0F0Fu) | ((qh[j] >> 2) & 0x30303030u);
        }
    }
    // MFMA t = 2 t4 + h: elements 8h..8h+7 of the 16-element scale group t4.  (q - 32) * sc reaches 32 * 128 = 4096, one bit more
    // than f16 holds exactly: products above 2048 with an odd value round by 2^-12 of themselves.
    __device__ __forceinline__ h8_t frag(int t) const {
        const int t4 = t >> 1, h = t & 1;
        const h2_t off = {(_Float16)1056.f, (_Float16)1056.f};       // 1024 + 32: quants are stored with a bias of 32
        u4_t a;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a[i] = h2_bits((h2_bits(__builtin_amdgcn_perm(0x64646464u, v[t4][2 * h + (i >> 1)], i & 1 ? 0x04030402u : 0x04010400u)) - off) * s[t4]);
        return __builtin_bit_cast(h8_t, a);
    }
    // ... and what that rounding took off, exactly: 0 or 1 up or down.
    __device__ __forceinline__ h8_t frag(int t, h8_t &rest) const {
        const int t4 = t >> 1, h = t & 1;
        const h2_t off = {(_Float16)1056.f, (_Float16)1056.f};
        u4_t a, b;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const h2_t q = h2_bits(__builtin_amdgcn_perm(0x64646464u, v[t4][2 * h + (i >> 1)], i & 1 ? 0x04030402u : 0x04010400u)) - off, p = q * s[t4];
            a[i] = h2_bits(p);
            b[i] = h2_bits(__builtin_elementwise_fma(q, s[t4], -p));
        }
        rest = __builtin_bit_cast(h8_t, b);
        return __builtin_bit_cast(h8_t, a);
    }
};

// Element offset of MFMA t's fragment from the lane's quarter, and of quarter g in its super-block.
template <int TYPE> __device__ __forceinline__ constexpr int frag_k(int t) { return TYPE == MESH_Q4_K ? 32 * (t >> 2) + 8 * (t & 3) : 32 * (t >> 1) + 8 * (t & 1); }
template <int TYPE> __device__ __forceinline__ constexpr int quarter_k(int g) { return TYPE == MESH_Q4_K ? 64 * g : 128 * (g >> 1) + 16 * (g & 1); }

// Moves a tile loaded with the dense mapping (lane 4r + c holds row r, quarter c) to the MFMA mapping
// (lane m + 16 g holds row m, quarter g).
__device__ __forceinline__ uint32_t lane_gather(uint32_t v, int src_lane4) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(src_lane4, (int)v);
}
__device__ __forceinline__ uint4 lane_gather(const uint4 &v, int src_lane4) {
    return make_uint4(lane_gather(v.x, src_lane4), lane_gather(v.y, src_lane4), lane_gather(v.z, src_lane4), lane_gather(v.w, src_lane4));
}
__device__ __forceinline__ void to_mfma_lanes(TileRegs<MESH_Q4_K> &R, int src_lane4) {
    R.hdr = lane_gather(R.hdr, src_lane4);
    R.qa = lane_gather(R.qa, src_lane4);
    R.qb = lane_gather(R.qb, src_lane4);
}
__device__ __forceinline__ void to_mfma_lanes(TileRegs<MESH_Q6_K> &R, int src_lane4) {
    R.qla = lane_gather(R.qla, src_lane4);
    R.qlb = lane_gather(R.qlb, src_lane4);
    R.qh = lane_gather(R.qh, src_lane4);
    R.sc = lane_gather(R.sc, src_lane4);
    R.d = lane_gather(R.d, src_lane4);
}

}  // namespace f16sk
}  // namespace mesh
