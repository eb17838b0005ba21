// Prefill GEMM over tiled K-quant weights with f16 activations (gemm.hip), and its elementwise companions.
#pragma once

#include "gemv.hpp"

namespace mesh {

constexpr int SKINNY_ITEM_PAIRS = 16;      // pairs per work item of an expert launch of the skinny GEMM: one MFMA's columns

struct GemmArgs {
    const void *W = nullptr;         // tiled q4_K / q6_K matrix [M][K]
    const void *Wp = nullptr;        // optional: the same matrix in the GEMM layout (gemm_pack); used instead of W when set
    const void *Wt = nullptr;        // optional: the same weights as f16 in the large tile's layout (gemm_tile_copy); used for calls of tile_min_tokens
    int tile_min_tokens = 1 << 30;   // tokens with k8-major activations.  n_seg matrices: one copy of them back to back, of any types.
    int type = -1;
    int M = 0, K = 0, T = 0;
    int M_pad = 0;                   // filled in by gemm_kquant
    const _Float16 *X = nullptr;     // [T][ldx] f16 activations; or, with x_k8, the k8-major layout of the skinny GEMM (below)
    int ldx = 0;
    bool x_k8 = false;               // X is k8-major: the matrix-core waves fetch their operand fragments from it directly
    float *Y = nullptr;              // [T][ldy] f32
    int ldy = 0;
    const float *bias = nullptr;     // [M] or null
    const float *residual = nullptr; // [T][ldres] or null; may alias Y
    int ldres = 0;
    // Several matrices sharing X in one launch (GEMM layout only: Wp holds their row blocks back to back, every matrix
    // but the last a whole number of 128-row blocks): matrix i starts at row block seg_begin[i] and has its own output,
    // bias and row count; M is the total.  n_seg == 1: the fields above describe the one matrix.
    int n_seg = 1;
    int seg_begin[3] = {0, 0, 0}, seg_M[3] = {0, 0, 0}, seg_ldy[3] = {0, 0, 0};
    float *seg_Y[3] = {nullptr, nullptr, nullptr};
    const float *seg_bias[3] = {nullptr, nullptr, nullptr};
    // Where gemm_types_ride() says so: the last of the n_seg matrices is of type_last, at Wp_last.
    const void *Wp_last = nullptr;
    int type_last = -1;
    // SwiGLU pair: Wp is a gate/up pair packed by gemm_pack_pair (every row block 64 gate rows, then the same 64 up
    // rows), M their common row count; the launch writes f16(silu(gate) * up) in the k8-major layout to y16_k8 (Y unused).
    _Float16 *y16_k8 = nullptr;
    unsigned *sat = nullptr;         // optional device counter of SwiGLU outputs clamped to the f16 range (mesh_common.hpp: note_f16_clamp)
    bool big_tile = true;            // wide projections of long calls may take the 256-row tile
    bool narrow_tile = true;         // calls of at most 64 tokens that the 256-row tile leaves may take the register-formed tile of 32 or 64 columns
    // Optional scratch for launches too narrow to fill the chip (few row blocks x token blocks): K is then split over
    // blockIdx.z, every slice writes its f32 partial tile to `part` ([slice][token][row of the launch]) and a second
    // kernel adds the slices in slice order and applies the epilogue.  Null: never split.  ksplit / k_per_split are
    // filled in by gemm_kquant.
    float *part = nullptr;
    size_t part_bytes = 0;
    int ksplit = 1, k_per_split = 0;
    // Optional, split launches only (ask gemm_split_count first): matrix i is the q / k / v projection of a layer
    // (kind[i], GEMV_KIND_*); the second kernel rotates q and k rows (neighbouring-pair RoPE) and appends k and v to
    // the f16 KV cache instead of storing them to their outputs, like the projection epilogues of the decode kernels.
    GemvRope rope;
    int kind[3] = {GEMV_KIND_PLAIN, GEMV_KIND_PLAIN, GEMV_KIND_PLAIN};
    // Optional, where gemm_norm_rides() says so: the second kernel of a split launch also writes f16(rms_norm(Y) * next_w), k8-major with
    // T padded to 16 by zeros, to next_x16 (which may be X).
    const float *next_w = nullptr;
    float next_eps = 0.f;
    _Float16 *next_x16 = nullptr;
    // Expert launch (mixture of experts; GEMM layout and k8-major activations only, plain store or SwiGLU): X holds the
    // (token, slot) pairs sorted by expert (moe.hpp: moe_sort), T is its capacity in pair slots, and tile i of `tiles` =
    // {expert, first slot, slots, 0} multiplies slots [first, first + slots) (at most 128; first a multiple of 16) by the
    // matrix at Wp + expert * expert_stride.  *n_tiles (device) tiles are live, max_tiles bounds them for the grid.
    // Outputs are indexed by slot.
    const int32_t *tiles = nullptr, *n_tiles = nullptr;
    // x_slot set: X holds plain rows of K, not sorted, and slot s's is row x_slot[s] / x_div (a slot without a pair, < 0, may take any).
    const int32_t *x_slot = nullptr;
    int x_div = 0;
    size_t expert_stride = 0;
    int max_tiles = 0;
    // SwiGLU pair of a call of at most 32 tokens, x_k8: the consumer side of SkinnyF16Args' norm hand-over (X not yet divided by the
    // token's rms, its sums of squares by [workgroup][16], from 17 tokens on [workgroup][32]).  Not split along K.
    const float *norm_part = nullptr;
    int norm_parts = 0;
    float norm_eps = 0.f;
};
// workgroups of the launch of such a pair
inline int gemm_pair_row_blocks(int64_t M) { return (int)((M + 63) / 64); }
int gemm_kquant(const GemmArgs &a, hipStream_t stream);
// Number of K slices gemm_kquant will use for this launch (1: not split).
int gemm_split_count(const GemmArgs &a);
// Whether the launch adds slices in a second kernel that can take the next norm along (one matrix and a residual).
bool gemm_norm_rides(const GemmArgs &a);

// Whether one launch takes matrices of both types (Wp_last).
bool gemm_types_ride(const GemmArgs &a);

// GEMM layout of a K-quant matrix: a second copy for the prefill GEMM, arranged by the workgroup tile that consumes it.
// One chunk per (128-row block, 64-element k-step), chunks of a row block consecutive in k.  A chunk holds, for each of
// the 256 slots s = 2 * row + h (elements 16 j + 8 h .. + 7, j = 0..3, of the row's 64), what a thread that forms them
// needs, at s * stride of each section, and per row the scales; a load of a wave covers whole lines:
//   q4_K (5120 B): [256 x 16 B quants: dword j, element e of its eight at nibble e / 2 + 4 (e % 2)]
//                  [128 x 8 B: byte sc (the integer block scale) of the first 32 elements, of the others, f16 d, f16 c = 8 d sc - dmin m
//                  of the first 32, of the others]
//   q6_K (7168 B): [256 x 16 B low nibbles, same order][256 x 8 B upper two bits: those of element e of dword j in dword j / 2
//                  at bit 2 P + 16 (e % 2), P = 4 (j % 2) + e / 2]
//                  [128 x 8 B: byte 128 + sc of each 16 elements, f16 d, twice]
// The kernel forms a weight as ((q - offset) * sc) * d + c: an exact small integer times the super-block's own f16
// scale, rounded once.  The fields are the ones the kernel would otherwise derive from the block headers, so both
// layouts give the same bits; the integer scales are bytes, 1024 + byte being an f16 that one permutation makes (five bits a weight
// of q4_K, seven of q6_K; as f16 they made it six and eight: batches of 32 decode steps of four layers 5120 wide 1.0% slower, the
// copies a sixth and an eighth larger).  Rows beyond M are zero.
size_t gemm_packed_bytes(int type, int64_t M, int64_t K);
int gemm_pack(int type, const void *tiled, void *packed, int64_t M, int64_t K, hipStream_t stream);
// gate / up pair for the SwiGLU launch: row block b = gate rows [64b, 64b + 64) followed by up rows [64b, 64b + 64)
size_t gemm_packed_pair_bytes(int type, int64_t M, int64_t K);
int gemm_pack_pair(int type, const void *gate_tiled, const void *up_tiled, void *packed, int64_t M, int64_t K, hipStream_t stream);

// f16 copy of a GEMM-layout matrix for the large tile (gemm_tile.hpp: GT_BLOCKS), rows padded to 128: the very weights the GEMM
// forms from its layout, 2 bytes each.  A pair: per 128-row block 32 gate rows, their 32 up rows, the next 32 and 32, so that a wave
// holds a gate row and its up row in the same lane.
size_t gemm_tile_bytes(int64_t M, int64_t K);
size_t gemm_tile_pair_bytes(int64_t M, int64_t K);
int gemm_tile_copy(int type, const void *packed, void *tile, int64_t M, int64_t K, bool pair, hipStream_t stream);
// The launch itself (gemm_kquant calls it): whether `a` takes it, its slices along K, and the product.
bool gemm_tile_takes(const GemmArgs &a);
int gemm_tile_slices(const GemmArgs &a);
int gemm_tile(const GemmArgs &a, hipStream_t stream);
int gemm_add_slices(const GemmArgs &a, int row_blocks, hipStream_t stream);
constexpr int GEMM_NORM_ROW_MAX = 8192;         // longest row whose next norm it writes

// Skinny GEMM for a batch of decode steps (gemm_skinny.hip): up to three tiled K-quant matrices sharing the
// activations, any T (processed 16 columns at a time), epilogues as in the mat-vec kernel, integer dot products on
// the matrix cores.  Activations come in the "q16" layout quant16_k8 produces: per block of 16 tokens
// q16_block_bytes(K) bytes holding 16-bit fixed-point values per 32-element block as two int8 planes, the f32 block
// scales and the f32 block sums (gemm_skinny.hip describes the arrangement); columns beyond T hold zeros.
struct SkinnyArgs {
    GemvMat mat[3];
    int n_mat = 1;                   // for EPI_SWIGLU exactly 2 (gate, up), written through mat[0].y
    const uint8_t *xq = nullptr;     // q16 layout, ceil(T / 16) blocks of q16_block_bytes(K), 16-byte aligned
    int K = 0, T = 0;
    int epi = EPI_STORE;
    const float *residual = nullptr; // EPI_RESIDUAL: [T][ldres]; may alias y
    int ldres = 0;
    // RoPE + KV append in the epilogue of a q/k/v launch, as in the mat-vec kernel (gemv.hpp); EPI_STORE only
    GemvRope rope;
    int kind[3] = {GEMV_KIND_PLAIN, GEMV_KIND_PLAIN, GEMV_KIND_PLAIN};
    bool pair_launch = true;         // q4_K matrices followed by one q6_K matrix (q, k and a q6_K v): one launch for both types
    // Expert launch (mixture of experts): mat[] describe expert 0 of stacked, equally shaped tiled matrices; work
    // item i (blockIdx.y) = {expert, n, pair[0..n)} in the grouping kernel's format with SKINNY_ITEM_PAIRS pairs per item
    // (moe.hpp); slot j of an item reads activation column pair[j] / x_div of xq (any block of 16) and writes output row
    // pair[j].  One matrix or a gate / up pair (EPI_SWIGLU); T is not used.
    const int32_t *items = nullptr, *n_items = nullptr;
    int max_items = 0;
    int x_div = 1;
};
int gemm_skinny(const SkinnyArgs &a, hipStream_t stream);
// Bytes of one 16-token block of the q16 layout for rows of K elements.
size_t q16_block_bytes(int K);
// y (q16 layout) = quantise(rms_norm(x) * w) for T rows of n floats (w == null: quantise(x)); n a multiple of 32
int quant16_k8(const float *x, const float *w, float eps, int T, int n, uint8_t *y, hipStream_t stream);
// Mixture of experts: x[t] += sum_s w[t][s] * y[t * top_k + s] (moe.hpp: moe_combine) and, from the new x, the q16 activations
// quant16_k8(x, norm_w, eps) would produce, in one launch: the same bits as the two launches.  Rows of n <= 8192.
bool moe_combine_quant16_supported(int n);
int moe_combine_quant16(float *x, const float *y, const float *w, int T, int n, int top_k, const float *norm_w, float eps, uint8_t *yq, hipStream_t stream);
// The "k8-major" f16 layout the large-tile GEMM reads: blocks of 16 tokens, element (t, k) of block t / 16 at
// ((k / 8) * 16 + t % 16) * 8 + k % 8 within the block of 16 * K halfs; columns beyond T hold zeros.
// The same launches on the f16 matrix cores (gemm_skinny_f16.hip): activations in the k8-major f16 layout above, weights as the
// integers of their quants and scales in f16, the super-blocks' factors on the f32 sums.  Faster than the integer kernel, less
// precise (f16 activations).
struct SkinnyF16Args {
    GemvMat mat[3];
    int n_mat = 1;                   // for EPI_SWIGLU exactly 2 (gate, up), written through mat[0].y and/or y16
    const _Float16 *x = nullptr;     // k8-major, ceil(T / 16) blocks of 16 * K halfs, 16-byte aligned
    int K = 0, T = 0;
    int epi = EPI_STORE;
    const float *residual = nullptr; // EPI_RESIDUAL: [T][ldres]; may alias y
    int ldres = 0;
    _Float16 *y16 = nullptr;         // optional f16 copy of matrix 0's output in the k8-major layout (feeds the next GEMM)
    unsigned *sat = nullptr;         // optional device counter of y16 values clamped to the f16 range
    // RoPE + KV append in the epilogue of a q/k/v launch, as in the mat-vec kernel (gemv.hpp); EPI_STORE only
    GemvRope rope;
    int kind[3] = {GEMV_KIND_PLAIN, GEMV_KIND_PLAIN, GEMV_KIND_PLAIN};
    // q4_K matrices followed by one q6_K matrix (q, k and a q6_K v): one launch for both types instead of two
    bool pair_launch = true;
    // RMS-norm hand-over between two launches (T <= 32: one launch each), in place of a norm kernel of its own between them.  The producer
    // (EPI_RESIDUAL, one matrix) also writes f16(y * norm_w) -- scaled by the next norm's weight but not yet by the
    // token's 1 / rms -- in the k8-major layout to norm_out.x16, and per workgroup the sum of y^2 of its rows for every
    // token to norm_out.part ([workgroups][16], or [workgroups][32] for a call of more than 16 tokens); gemm_skinny_f16_workgroups gives the workgroup count.  The consumer reads
    // those activations as its x, adds the partial sums in workgroup order and multiplies every accumulated product by
    // 1 / sqrt(sum / K + eps) before bias and epilogue: W . (y w / rms) = (W . (y w)) / rms.
    struct NormOut { const float *norm_w = nullptr; _Float16 *x16 = nullptr; float *part = nullptr; } norm_out;
    struct NormIn { const float *part = nullptr; int n_parts = 0; float eps = 0.f; } norm_in;
};
int gemm_skinny_f16(const SkinnyF16Args &a, hipStream_t stream);
// The same product cut along K, where gemm_skinny_f16_slices (with the scratch there is) says more than 1; no norm hand-over.  The slices meet
// in sum.part and are added by gemm_add_slices, which also writes the next norm's rows (sum.next_w, next_eps, next_x16, sat).
int gemm_skinny_f16_slices(const SkinnyF16Args &a, size_t part_bytes);
int gemm_skinny_f16_sliced(const SkinnyF16Args &a, const GemmArgs &sum, hipStream_t stream);
// workgroups a producer launch of `a` will have (= partial sums per token it writes); 0 when the launch is not valid
int gemm_skinny_f16_workgroups(const SkinnyF16Args &a);
constexpr int SKINNY_F16_NORM_PARTS_MAX = 256;
constexpr int SKINNY_F16_NORM_TOKENS_MAX = 32;

// y (k8-major) = f16(rms_norm(x) * w) for T rows of n floats; pack_f16_k8: plain conversion
// (sat: optional device counter of values clamped to the f16 range, in all of these)
int rmsnorm_f16_k8(const float *x, const float *w, float eps, int T, int n, _Float16 *y, hipStream_t stream, unsigned *sat = nullptr);
int pack_f16_k8(const float *x, int T, int n, _Float16 *y, hipStream_t stream, unsigned *sat = nullptr);
// the same as rmsnorm_f16_k8 for n_slots (a multiple of 16) gathered rows: slot i holds row row_of_slot[i] / row_div of x, zeros when negative
// (scale: optional 1 / rms of the rows of x)
int rmsnorm_f16_k8_gather(const float *x, const float *w, float eps, const int32_t *row_of_slot, int row_div, int n_slots, int n, _Float16 *y, hipStream_t stream,
                          unsigned *sat = nullptr, const float *scale = nullptr);
int swiglu_f16_k8(const float *gate, const float *up, int T, int n, _Float16 *y, hipStream_t stream, unsigned *sat = nullptr);

int rmsnorm_f16(const float *x, const float *w, float eps, int T, int n, _Float16 *y, int ldy, hipStream_t stream, unsigned *sat = nullptr);
int swiglu_f16(const float *gate, const float *up, _Float16 *out, int64_t n, hipStream_t stream, unsigned *sat = nullptr);

}  // namespace mesh
