// Prefill products of K-quant models over f16 copies of their weights: the tiles of gemm_tile.hpp with the epilogues of gemm.hip.
//
// The dequantising GEMM (gemm_big_kernel) is bound by the weight slab's way through LDS: its staging waves write it with 16-byte
// stores after ~70 vector instructions per 32 weights, and it ran at 900 TFLOP/s with the products themselves switched off at 943.  The
// copy holds the weights that GEMM forms, bit for bit, so the products and their sums are the same; it costs 2 bytes
// per weight of memory and, for calls of few tokens, their reading, which is why those stay with the quantised layouts
// (tile_min_tokens).  A chunk through eight 8B-shaped layers, us, quantised layouts / copies: 64 tokens 1122 / 1241, 128 1326 / 1328,
// 192 1770 / 1635, 333 2577 / 2030, 512 2965 / 2600, 1024 5061 / 4245, 2048 9002 / 7654; four 32B-shaped layers: 128 1128 / 1194,
// 192 1715 / 1381, 1024 5452 / 4545.  gate/up of the 8B shape at 2048 tokens: 531 -> 410 us (1170 TFLOP/s) on one box, 410 to 434 over several.
#include <algorithm>

#include "gemm.hpp"
#include "gemm_tile.hpp"

namespace mesh {

// TILE_ROWS_OUT: f32 rows with bias and residual, per matrix of the launch; TILE_SWIGLU: f16(silu(gate) up) in the k8-major layout;
// TILE_PARTIAL: this slice's sums as they are.  SwiGLU holds tokens in the lanes (four weight rows of a lane are 8 bytes of the
// output), the others weight rows (a store covers whole lines).
enum TileOut { TILE_ROWS_OUT = 0, TILE_SWIGLU = 1, TILE_PARTIAL = 2 };

template <TileOut OUT, int WM, int WT>
__global__ __launch_bounds__(64 * WM * WT, gt_waves_per_simd(WM, WT)) void gemm_f16_kernel(GemmArgs a, int row_blocks, int n_ttiles, int n_tiles) {
    __shared__ __align__(1024) char smem[gt_lds_bytes(WM, WT)];
    int mt, tt;
    gt_place(blockIdx.x, n_tiles, n_ttiles, mt, tt);
    const int n_all = a.K / GT_K, k0 = OUT == TILE_PARTIAL ? (int)blockIdx.y * a.k_per_split : 0;
    const int n_steps = OUT == TILE_PARTIAL && n_all - k0 > a.k_per_split ? a.k_per_split : n_all - k0;
    gt_f16v acc[2][2];
    gt_clear(acc);
    gt_multiply<gt_h8, GT_BLOCKS, GT_BLOCKS, WM, WT, OUT != TILE_SWIGLU>(smem, acc, a.Wt, a.K, a.X, a.K, k0, n_steps, mt * WM * 4, row_blocks * 8, tt * WT * 4, a.T);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = (mt * WM + wave % WM) * 64, t0 = (tt * WT + wave / WM) * 64;      // this wave's rows of the launch and its tokens
    const int block = m0 >> 7;
    if (block >= row_blocks) return;
    if constexpr (OUT == TILE_SWIGLU) {
        // acc[0]: gate rows, acc[1]: the up rows of the same outputs; register i of a lane: row 8 * (i / 4) + 4 * (lane / 32) + i % 4, token lane % 32
        const int t_pad = (a.T + 15) & ~15;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = t0 + 32 * j + (lane & 31);
            if (t >= t_pad) continue;
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const int m = (m0 >> 1) + 8 * e4 + 4 * (lane >> 5);
                if (m >= a.M) continue;
                float o[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float g = acc[0][j][4 * e4 + c], u = acc[1][j][4 * e4 + c];
                    o[c] = t < a.T ? g / (1.0f + expf(-g)) * u : 0.f;        // padding columns of the last token block hold zeros
                }
                note_f16_clamp(a.sat, o[0], o[1], o[2], o[3]);
                *reinterpret_cast<uint2 *>(a.y16_k8 + (size_t)(t >> 4) * 16 * a.M + ((size_t)(m >> 3) * 16 + (t & 15)) * 8 + (m & 7)) =
                    make_uint2(pack_h2(o[0], o[1]), pack_h2(o[2], o[3]));
            }
        }
        return;
    }
    // register i of a lane: token 8 * (i / 4) + 4 * (lane / 32) + i % 4, row lane % 32
    if constexpr (OUT == TILE_PARTIAL) {
        const size_t ld = (size_t)row_blocks * 128;
        float *P = a.part + (size_t)blockIdx.y * a.T * ld;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            // (a pair's partials in the order the adding kernel takes: 64 gate rows, 64 up rows)
            const int row = (a.y16_k8 ? block * 128 + b * 64 + ((m0 >> 6) & 1) * 32 : m0 + 32 * b) + (lane & 31);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int t = t0 + 32 * h + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                    if (t < a.T) P[(size_t)t * ld + row] = acc[h][b][i];
                }
        }
        return;
    }
    float *Y = a.Y;
    const float *bias = a.bias;
    int M = a.M, ldy = a.ldy, first = 0;
    if (a.n_seg > 1) {
        // (selected, not indexed: a dynamically indexed kernel-argument array would be spilled to scratch)
        const int sg = (block >= a.seg_begin[1] ? 1 : 0) + (a.n_seg > 2 && block >= a.seg_begin[2] ? 1 : 0);
        Y = sg == 0 ? a.seg_Y[0] : sg == 1 ? a.seg_Y[1] : a.seg_Y[2];
        bias = sg == 0 ? a.seg_bias[0] : sg == 1 ? a.seg_bias[1] : a.seg_bias[2];
        M = sg == 0 ? a.seg_M[0] : sg == 1 ? a.seg_M[1] : a.seg_M[2];
        ldy = sg == 0 ? a.seg_ldy[0] : sg == 1 ? a.seg_ldy[1] : a.seg_ldy[2];
        first = (sg == 0 ? 0 : sg == 1 ? a.seg_begin[1] : a.seg_begin[2]) * 128;
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int m = m0 - first + 32 * b + (lane & 31);
        if (m >= M) continue;
        const float add = bias ? bias[m] : 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int tb = t0 + 32 * h + 4 * (lane >> 5);
            float r[16];
            // the residual may be Y itself: all sixteen are read before the first is written
            if (a.residual) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int t = tb + 8 * (i >> 2) + (i & 3);
                    r[i] = a.residual[(size_t)(t < a.T ? t : a.T - 1) * a.ldres + m];
                }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int t = tb + 8 * (i >> 2) + (i & 3);
                float v = acc[h][b][i];
                if (bias) v += add;
                if (a.residual) v += r[i];
                if (t < a.T) Y[(size_t)t * ldy + m] = v;
            }
        }
    }
}

static int tile_row_blocks(const GemmArgs &a) { return a.y16_k8 ? (a.M + 63) / 64 : (a.M + 127) / 128; }

// a launch of its own adds the slices: about 5 us
static GtPlan tile_plan(const GemmArgs &a) {
    const int rows = tile_row_blocks(a) * 128;
    return gt_plan(rows, a.T, a.K, a.part ? 8 : 1, a.part_bytes / ((size_t)a.T * rows * sizeof(float)), 5000.0);
}

bool gemm_tile_takes(const GemmArgs &a) { return a.Wt && a.x_k8 && !a.tiles && a.T >= a.tile_min_tokens; }

int gemm_tile_slices(const GemmArgs &a) { return tile_plan(a).slices; }

template <TileOut OUT>
static int launch_f16(const GemmArgs &a, const GtPlan &p, int row_blocks, hipStream_t stream) {
    const int mtiles = (row_blocks * 2 + p.wm - 1) / p.wm, ttiles = (a.T + 64 * p.wt - 1) / (64 * p.wt);
    const dim3 grid((unsigned)(mtiles * ttiles), (unsigned)p.slices), block((unsigned)(64 * p.wm * p.wt));
    if (p.wt == 4) MESH_LAUNCH((gemm_f16_kernel<OUT, 4, 4>), grid, block, 0, stream, a, row_blocks, ttiles, mtiles * ttiles);
    else if (p.wt == 3) MESH_LAUNCH((gemm_f16_kernel<OUT, 4, 3>), grid, block, 0, stream, a, row_blocks, ttiles, mtiles * ttiles);
    else if (p.wm == 4) MESH_LAUNCH((gemm_f16_kernel<OUT, 4, 2>), grid, block, 0, stream, a, row_blocks, ttiles, mtiles * ttiles);
    else MESH_LAUNCH((gemm_f16_kernel<OUT, 2, 2>), grid, block, 0, stream, a, row_blocks, ttiles, mtiles * ttiles);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// (shapes and pointers checked by gemm_kquant)
int gemm_tile(const GemmArgs &a, hipStream_t stream) {
    const int row_blocks = tile_row_blocks(a);
    const GtPlan p = tile_plan(a);
    if (a.rope.pos && (p.slices <= 1 || a.y16_k8 || a.residual || a.rope.head_dim % 4 || a.rope.n_rot % 2))
        return fail(MESH_ERR_INVALID, "gemm: RoPE / KV append on a launch it does not fit");
    if (p.slices <= 1) return a.y16_k8 ? launch_f16<TILE_SWIGLU>(a, p, row_blocks, stream) : launch_f16<TILE_ROWS_OUT>(a, p, row_blocks, stream);
    GemmArgs k = a;
    k.ksplit = p.slices;
    k.k_per_split = p.k_slice;
    const int rc = launch_f16<TILE_PARTIAL>(k, p, row_blocks, stream);
    return rc != MESH_OK ? rc : gemm_add_slices(k, row_blocks, stream);
}

}  // namespace mesh
