// Expert products of a batch of decode steps on the f16 matrix cores (expert_step.hip).
#pragma once

#include "mesh_common.hpp"

namespace mesh {

// Activations as pairs of f16: x = (hi + lo / 2048) / scale with scale a power of two, 22 significant bits (hi clamped to the f16 range).
// By token: blocks of 16 tokens, element (t, k) of plane p (0 hi, 1 lo) at ((k / 8 * 2 + p) * 16 + t % 16) * 8 + k % 8 of the block's 32 K
// halfs.  By item: a block per work item, element (slot, k) at (k / 8 * 16 + 8 p + slot) * 8 + k % 8 of its 16 K halfs.
constexpr int EXPERT_STEP_PAIRS = 8;              // pairs a work item holds at most: two planes each fill the instruction's 16 columns
constexpr float EXPERT_LO = 2048.f;
constexpr float EXPERT_FFN_SCALE = 1.0f / 64;     // of the SwiGLU outputs: up to 2^22 before they clamp, 2^-30 the smallest step
constexpr int EXPERT_STEP_TOKENS_MAX = 32;
inline size_t expert_x_bytes(int K) { return (size_t)EXPERT_STEP_TOKENS_MAX * K * 4; }
inline size_t expert_ffn_bytes(int max_items, int K) { return (size_t)max_items * 16 * K * 2; }

// Work items as moe_group writes them, EXPERT_STEP_PAIRS pairs each; matrices tiled K-quants of one type and shape, expert 0 of each.
//   gate and up (W[1] set): x by token (pair / x_div), silu(gate) up as pairs of f16 by item to ffn
//   down (W[1] null):       ffn read, f32 rows by pair to y
struct ExpertStepArgs {
    const void *W[2] = {nullptr, nullptr};
    int type = -1, M = 0, K = 0;
    const int32_t *items = nullptr, *n_items = nullptr;
    int max_items = 0, x_div = 1;
    const uint16_t *x = nullptr;
    uint16_t *ffn = nullptr;
    float *y = nullptr;
    unsigned *sat = nullptr;        // counts SwiGLU outputs that clamped
};
bool expert_step_supported(int type, int M, int K);
int expert_step(const ExpertStepArgs &a, hipStream_t stream);

}  // namespace mesh
