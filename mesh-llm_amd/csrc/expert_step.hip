// Expert products of a batch of decode steps: up to 8 (token, slot) pairs of an expert per pass over its tiled q4_K / q6_K weights, on
// v_mfma_f32_16x16x32_f16.
//
// The mat-vec kernel (gemv_grouped_kernel) pays a dot product per column and takes 4 pairs a pass; the f16 skinny GEMM (gemm_skinny_f16.hip)
// pays for a tile once, but rounds activations to 11 bits, and an expert layer keeps 16.  Here the sixteen columns of the instruction
// are eight pairs twice: an activation is a sum of two f16 (22 bits and a scale, expert_step.hpp), its halves are two columns and their products
// are added at the end.  Weights are the integers of quants and scales, exact: q4_K as in the skinny GEMM, q6_K with the one bit its
// products may have too many as a second fragment; the super-block's d and dmin multiply the sums in f32.
//
// A workgroup is an item and two or four tile-rows, its waves split K, all items of a batch of 16 are on the chip at once (four workgroups a
// CU).  Before (mat-vec kernel) / now, us, 64 experts of 2 x 768 x 2048 (q4_K) and 2048 x 768 behind a Zipf router, top 8: 16 tokens (28
// experts, 34 items) gate / up 30.5 / 20.8, down q6_K 30.4 / 16.5, q4_K 23.8 / 12.6 (with one fixed scale for all outputs 16.0 and 12.6); 4 tokens 15.4 / 12.4, 16.9 / 11.4, 13.5 / 8.9;
// 1 token 8.4 / 9.2, 7.8 / 7.0, 7.2 / 5.9; distance of the layers from 64 bits 5.2e-5 / 4.9e-5 (16 tokens).  What bounds it: an item costs 0.45 us whatever
// is left out of its tiles (lane moves, half of the MFMAs, most of the activation loads: 1-2 us each at 16 tokens), 3.8 TB/s of weights
// beside as many bytes of activations; a launch starts at 6 us.  Two segments a wave instead of four: 25.0, 19.0, 14.8; four tiles in flight instead of
// two at three workgroups a CU: 22.4, 19.1, 14.4.
#include "expert_step.hpp"

#include <algorithm>

#include "gemm.hpp"
#include "lds_ops.hpp"
#include "skinny_frags.hpp"
#include "wave_ops.hpp"

namespace mesh {
namespace f16sk {

constexpr int EX_WAVES = 4, EX_THREADS = 64 * EX_WAVES;
constexpr int EX_SEGS = 4;                // (tile-row, matrix) segments of a wave: 9-13 KB of weights to 8 KB of activations
constexpr int EX_DEPTH = 2;               // weight tiles a wave keeps in flight
constexpr int EX_ROW = 20;                // floats between rows of sums in LDS
constexpr int EX_ITEM_INTS = (2 + EXPERT_STEP_PAIRS + 3) / 4 * 4;

struct ExpertOut {
    _Float16 *ffn;
    float *ffn_scale, *y;                 // (ffn_scale: written by gate / up, read by down)
    const float *x_scale;
    int M, x_div;
};

template <int TYPE, int NU>
__global__ __launch_bounds__(EX_THREADS, 4) void expert_step_kernel(const int32_t *__restrict__ items, const int32_t *__restrict__ n_items,
                                                                                             const uint8_t *w0, const uint8_t *w1, const _Float16 *x, int K, int tile_rows,
                                                                                             size_t expert_stride, const ExpertOut o) {
    constexpr int TB = TileRegs<TYPE>::BYTES, ROWS = EX_SEGS / NU;
    constexpr bool BY_ITEM = NU == 1;
    constexpr int K8 = BY_ITEM ? 128 : 256;                  // halfs between groups of eight elements
    __shared__ float red[EX_WAVES * EX_SEGS * 16 * EX_ROW];
    __shared__ float s_scale[EXPERT_STEP_PAIRS];             // of a slot's row
    extern __shared__ __align__(16) uint32_t s_ratio[];      // down: [slot][K / 32], a block's scale over its row's, as two f16
    const int by = blockIdx.y;
    const int32_t *it = items + (size_t)by * EX_ITEM_INTS;
    const int expert = it[0], n = it[1];
    if (by >= *n_items) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), KS = blockDim.x >> 6;
    const int m = lane & 15, g = lane >> 4, src_lane4 = 4 * (4 * m + g);
    const int nsb = K / QK_K, n_i = (nsb - wave + KS - 1) / KS;         // (KS <= nsb)
    const int tr0 = blockIdx.x * ROWS;
    const size_t row_stride = (size_t)nsb * TB;
    const uint8_t *const e0 = w0 + (size_t)expert * expert_stride, *const e1 = NU == 2 ? w1 + (size_t)expert * expert_stride : e0;
    // (a segment past the last tile-row reads the first again and is dropped; no branch in the walk, see gemm_skinny_f16.hip)
    auto tile_ptr = [&](int ii, int seg) {
        const int j = tr0 + seg / NU < tile_rows ? seg / NU : 0;
        return (seg % NU ? e1 : e0) + (size_t)(tr0 + j) * row_stride + (size_t)(wave + KS * (ii < n_i ? ii : n_i - 1)) * TB;
    };
    // this lane's column: slot m % 8, plane m / 8 (slots past the item's repeat its first, or hold anything: computed, never stored)
    const int slot = m & 7, plane = m >> 3;
    // Down: blocks of 32 elements have scales of their own (their workgroup of the gate / up launch had no others).  Fragments come to the
    // row's largest scale by a power of two in f16, which takes bits of what is below 2^-28 of the row's largest alone; the row's scale
    // multiplies the sums.  (The first scales are requested ahead of the weights and needed behind them: waiting for them is no wait for those.)
    const int nb = K / 32, share = 4 * (g + 4 * plane);      // (eight lanes a slot)
    [[maybe_unused]] const float *const scales = o.ffn_scale + ((size_t)by * EXPERT_STEP_PAIRS + slot) * nb;
    [[maybe_unused]] float4 first;
    if constexpr (BY_ITEM) first = *reinterpret_cast<const float4 *>(scales + (share < nb ? share : 0));
    TileRegs<TYPE> ring[EX_DEPTH];
#pragma unroll
    for (int f = 0; f < EX_DEPTH; ++f) ring[f].load(tile_ptr(f / EX_SEGS, f % EX_SEGS), lane);
    const _Float16 *xl;
    [[maybe_unused]] float token_scale;
    if (BY_ITEM) xl = x + (size_t)by * 16 * K + m * 8;
    else {
        const int tok = it[2 + (slot < n ? slot : 0)] / o.x_div;
        xl = x + (size_t)(tok >> 4) * 32 * K + plane * 128 + (tok & 15) * 8;
        token_scale = o.x_scale[tok];
    }
    xl += quarter_k<TYPE>(g) / 8 * K8;
    uint4 xb[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) xb[t] = ldg<uint4>(xl + (size_t)wave * 32 * K8 + frag_k<TYPE>(t) / 8 * K8);
    if constexpr (BY_ITEM) {
        __builtin_amdgcn_sched_barrier(0);
        if (wave == 0) {
            auto each = [&](auto &&f) {
                if (share < nb) f(share, first);
                for (int b = 32 + share; b < nb; b += 32) f(b, *reinterpret_cast<const float4 *>(scales + b));
            };
            float most = 0.f;
            each([&](int, const float4 &v) { most = fmaxf(most, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w))); });
            most = lane_fold<32>(lane_fold<16>(lane_fold<8>(most, LaneMax{}), LaneMax{}), LaneMax{});
            const float to_row = __uint_as_float(0x7F000000u - __float_as_uint(most));      // 1 / most, a power of two
            each([&](int b, const float4 &v) {
                *reinterpret_cast<uint4 *>(s_ratio + slot * nb + b) =
                    make_uint4(h2_bits(h2_of(v.x * to_row)), h2_bits(h2_of(v.y * to_row)), h2_bits(h2_of(v.z * to_row)), h2_bits(h2_of(v.w * to_row)));
            });
            if (lane < EXPERT_STEP_PAIRS) s_scale[lane] = most;
        }
        lds_barrier();
    }
    f4_t acc[EX_SEGS];
#pragma unroll
    for (int s = 0; s < EX_SEGS; ++s) acc[s] = f4_t{0.f, 0.f, 0.f, 0.f};
    auto step = [&](const TileRegs<TYPE> &loaded, f4_t &sum_to, bool refill, int next_ii) {
        const _Float16 *nx = xl + (size_t)(wave + KS * (next_ii < n_i ? next_ii : n_i - 1)) * 32 * K8;
        TileRegs<TYPE> tile = loaded;
        to_mfma_lanes(tile, src_lane4);
        TileFrags<TYPE> F;
        F.prepare(tile, g);
        f4_t sum = {0.f, 0.f, 0.f, 0.f}, low = sum;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const h8_t b = __builtin_bit_cast(h8_t, xb[t]);
            if constexpr (TileFrags<TYPE>::MINIMUM) {
                sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, F.frag(t), sum, 0, 0, 0);
                low = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, F.minimum(t), low, 0, 0, 0);
            } else {
                h8_t rest;
                const h8_t w = F.frag(t, rest);
                sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, w, sum, 0, 0, 0);
                low = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, rest, low, 0, 0, 0);
            }
            if (refill) xb[t] = ldg<uint4>(nx + frag_k<TYPE>(t) / 8 * K8);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (TileFrags<TYPE>::MINIMUM) sum_to[i] = fmaf(F.ndmin, low[i], fmaf(F.d, sum[i], sum_to[i]));
            else sum_to[i] = fmaf(F.d, sum[i] + low[i], sum_to[i]);
        }
    };
    for (int ii = 0; ii < n_i; ++ii) {
        if constexpr (BY_ITEM) {
            // of the blocks this lane's fragments lie in
            constexpr int NS = TYPE == MESH_Q4_K ? 2 : 4;
            const uint32_t *const at = s_ratio + slot * nb + (wave + KS * ii) * 8 + quarter_k<TYPE>(g) / 32;
            uint32_t ratio[NS];
#pragma unroll
            for (int j = 0; j < NS; ++j) ratio[j] = at[j];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const h2_t f = h2_bits(ratio[frag_k<TYPE>(t) / 32]);
                xb[t] = make_uint4(h2_bits(h2_bits(xb[t].x) * f), h2_bits(h2_bits(xb[t].y) * f), h2_bits(h2_bits(xb[t].z) * f), h2_bits(h2_bits(xb[t].w) * f));
            }
        }
#pragma unroll
        for (int q = 0; q < EX_SEGS; ++q) {
            step(ring[q % EX_DEPTH], acc[q], q == EX_SEGS - 1, ii + 1);
            __builtin_amdgcn_sched_barrier(0);
            ring[q % EX_DEPTH].load(tile_ptr(ii + (q + EX_DEPTH) / EX_SEGS, (q + EX_DEPTH) % EX_SEGS), lane);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if constexpr (!BY_ITEM)
        if (wave == 0 && lane < EXPERT_STEP_PAIRS) s_scale[lane] = token_scale;
    // acc[seg]: weight row m, columns 4 g .. 4 g + 3
#pragma unroll
    for (int s = 0; s < EX_SEGS; ++s) *reinterpret_cast<f4_t *>(red + ((wave * EX_SEGS + s) * 16 + m) * EX_ROW + 4 * g) = acc[s];
    __syncthreads();
    auto total = [&](int seg, int r, int sl) {
        float hi = 0.f, lo = 0.f;
        for (int k = 0; k < KS; ++k) {
            const float *p = red + ((k * EX_SEGS + seg) * 16 + r) * EX_ROW + sl;
            hi += p[0];
            lo += p[8];
        }
        return fmaf(lo, 1.0f / EXPERT_LO, hi) * s_scale[sl];
    };
    for (int i = threadIdx.x; i < ROWS * 128; i += blockDim.x) {
        if constexpr (NU == 2) {
            // the workgroup's 32 rows of a slot side by side: a block with a scale of its own
            const int r = i & 31, sl = i >> 5, row = tr0 * 16 + r;
            if (sl >= n) break;
            const float gate = total(2 * (r >> 4), r & 15, sl), up = total(2 * (r >> 4) + 1, r & 15, sl);
            const float v = gate / (1.0f + expf(-gate)) * up;
            const PairScale ps = pair_scale(lanes_fold<16>(fabsf(v), LaneMax{}));
            _Float16 *to = o.ffn + (size_t)by * 16 * o.M + ((size_t)(row >> 3) * 16 + sl) * 8 + (row & 7);
            pair_of(v * ps.inverse, to[0], to[64]);
            if (r == 0) o.ffn_scale[((size_t)by * EXPERT_STEP_PAIRS + sl) * (o.M / 32) + row / 32] = ps.scale;
        } else {
            const int j = i >> 7, r = i & 15, sl = (i >> 4) & 7, row = (tr0 + j) * 16 + r;
            if (sl >= n || row >= o.M) continue;
            o.y[(size_t)it[2 + sl] * o.M + row] = total(j, r, sl);
        }
    }
}

}  // namespace f16sk

bool expert_step_supported(int gate_type, int down_type, int embd, int ff) {
    return type_is_tiled(gate_type) && type_is_tiled(down_type) && embd > 0 && ff > 0 && embd % QK_K == 0 && ff % QK_K == 0 && ff <= EXPERT_STEP_FF_MAX;
}

template <int TYPE, int NU> static int launch_expert_step(const ExpertStepArgs &a, hipStream_t stream) {
    using namespace f16sk;
    const int tile_rows = (a.M + TILE_ROWS - 1) / TILE_ROWS, rows = EX_SEGS / NU;
    const dim3 grid((unsigned)((tile_rows + rows - 1) / rows), (unsigned)a.max_items), block(64u * (unsigned)std::min(EX_WAVES, a.K / QK_K));
    const ExpertOut o{reinterpret_cast<_Float16 *>(a.ffn), a.ffn_scale, a.y, a.x_scale, a.M, a.x_div};
    MESH_LAUNCH((expert_step_kernel<TYPE, NU>), grid, block, NU == 1 ? (size_t)a.K : 0, stream, a.items, a.n_items, static_cast<const uint8_t *>(a.W[0]), static_cast<const uint8_t *>(a.W[1]),
                reinterpret_cast<const _Float16 *>(NU == 2 ? a.x : a.ffn), a.K, tile_rows, (size_t)tiled_bytes(a.type, a.M, a.K), o);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

int expert_step(const ExpertStepArgs &a, hipStream_t stream) {
    const bool pair = a.W[1] != nullptr;
    if (!a.W[0] || !a.items || !a.n_items || a.max_items < 1 || a.max_items > 65535 || a.x_div < 1 || !a.ffn || !a.ffn_scale || (pair ? !a.x || !a.x_scale : !a.y) ||
        !(pair ? expert_step_supported(a.type, a.type, a.K, a.M) : expert_step_supported(a.type, a.type, a.M, a.K)))
        return fail(MESH_ERR_INVALID, "expert_step: bad arguments (%d x %d, type %d, %d items)", a.M, a.K, a.type, a.max_items);
    if (a.type == MESH_Q4_K) return pair ? launch_expert_step<MESH_Q4_K, 2>(a, stream) : launch_expert_step<MESH_Q4_K, 1>(a, stream);
    return pair ? launch_expert_step<MESH_Q6_K, 2>(a, stream) : launch_expert_step<MESH_Q6_K, 1>(a, stream);
}

}  // namespace mesh
