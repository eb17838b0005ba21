// Expert products of a batch of decode steps on the f16 matrix cores (expert_step.hip).
#pragma once

#include "mesh_common.hpp"

namespace mesh {

// Activations as pairs of f16: x = (hi + lo / 2048) * scale, scale a power of two that brings the largest of a group to 2^14 .. 2^15
// (pair_scale): 22 significant bits down to 2^-27 of it, an absolute step of 2^-49 of it below, no limit of range.
// By token, a scale per token: blocks of 16 tokens, element (t, k) of plane p (0 hi, 1 lo) at ((k / 8 * 2 + p) * 16 + t % 16) * 8 + k % 8 of
// the block's 32 K halfs; scales at t.  By item, a scale per slot and 32 elements: a block per work item, element (slot, k) at (k / 8 * 16 +
// 8 p + slot) * 8 + k % 8 of its 16 K halfs, scale of elements 32 b.. at (item * 8 + slot) * (K / 32) + b.
constexpr int EXPERT_STEP_PAIRS = 8;              // pairs a work item holds at most: two planes each fill the instruction's 16 columns
constexpr float EXPERT_LO = 2048.f;
constexpr int EXPERT_STEP_TOKENS_MAX = 32;
constexpr int EXPERT_STEP_FF_MAX = 32768;         // the down launch keeps K bytes of scales in LDS
inline size_t expert_x_bytes(int K) { return (size_t)EXPERT_STEP_TOKENS_MAX * K * 4; }
inline size_t expert_ffn_bytes(int max_items, int K) { return (size_t)max_items * 16 * K * 2; }
inline size_t expert_ffn_scales(int max_items, int K) { return (size_t)max_items * EXPERT_STEP_PAIRS * (K / 32); }

// Work items as moe_group writes them, EXPERT_STEP_PAIRS pairs each; matrices tiled K-quants of one type and shape, expert 0 of each.
//   gate and up (W[1] set): x by token (pair / x_div), silu(gate) up as pairs of f16 by item to ffn
//   down (W[1] null):       ffn read, f32 rows by pair to y
struct ExpertStepArgs {
    const void *W[2] = {nullptr, nullptr};
    int type = -1, M = 0, K = 0;
    const int32_t *items = nullptr, *n_items = nullptr;
    int max_items = 0, x_div = 1;
    const uint16_t *x = nullptr;
    const float *x_scale = nullptr;
    uint16_t *ffn = nullptr;
    float *ffn_scale = nullptr;
    float *y = nullptr;
};
// gate and up of ff x embd, down of embd x ff
bool expert_step_supported(int gate_type, int down_type, int embd, int ff);
int expert_step(const ExpertStepArgs &a, hipStream_t stream);

#ifdef __HIPCC__
struct PairScale { float scale, inverse; };
// of a group whose largest magnitude is given; both powers of two.  (Below 2^-112 the smallest normal number; infinity gives a value that
// keeps it one.)
__device__ __forceinline__ PairScale pair_scale(float amax) {
    const int e = (int)(__float_as_uint(amax) >> 23) & 0xFF, s = e < 15 ? 1 : e - 14;
    return PairScale{__uint_as_float((uint32_t)s << 23), __uint_as_float((uint32_t)(254 - s) << 23)};
}
__device__ __forceinline__ void pair_of(float scaled, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)scaled;
    lo = (_Float16)((scaled - (float)hi) * EXPERT_LO);
}
#endif

}  // namespace mesh
