// Main loop of the large-tile products: 16-bit operands (f16 or bf16) straight from memory into LDS, f32 sums on the matrix cores.
//
// A workgroup of WM x WT waves owns a tile of 64 WM weight rows x 64 WT tokens, a wave 64 x 64 of it (2 x 2 blocks of
// v_mfma_f32_32x32x16).  K goes by in steps of 32: a step's operands are (WM + WT) * 4 chunks of 1 KB, one per 16 rows, and
// a chunk is one global_load_lds_dwordx4 of a wave.  LDS holds STAGES steps: while step k is multiplied the ones behind it have
// been requested, so a wave waits with the loads of STAGES - 2 steps still in flight (vmcnt, exact because every wave
// issues the same number of loads per step) and one barrier per step serves both ways: behind it the step has landed for
// everybody, and everybody is done with the stage that the next loads overwrite.
//
// What bounds it: with every CU at work the clock (M 4096, K 14336, 2048 tokens: 1100-1250 TFLOP/s; half the CUs alone reach
// 82% of the matrix cores' nominal rate, all of them 50%), with few workgroups the latency of weights that come from
// memory.  Measured, weights cold, us (M, K, tokens): 64 x 64 per wave 436 against 502 with 128 x 64 (28672, 4096, 2048, weights
// warm); steps of 64 in two stages 604; s_setprio around the products 432 against 436-496.  Stages of the 128 x 128 tile, 3 / 5 / 8:
// 48 / 39 / 40 (6144, 4096, 512), 154 / 121 / 121 (4096, 14336, 512); of 256 x 128, 3 / 4 / 6: 224 / 206 / 203 (4096, 14336, 2048),
// 35 / 37 / 41 (8192, 2048, 900).
//
// The loads are issued by inline asm because the compiler counts LDS writes of the builtin as conflicting with the
// fragment reads of the other stages across the loop's back edge and waits for all of them.  The asm has no outputs; its
// operands are read when it issues.
#pragma once

#include <type_traits>

#include "lds_ops.hpp"
#include "mesh_common.hpp"

namespace mesh {

typedef float gt_f16v __attribute__((ext_vector_type(16)));
typedef uint32_t gt_u4 __attribute__((ext_vector_type(4)));
typedef _Float16 gt_h8 __attribute__((ext_vector_type(8)));
typedef __bf16 gt_b8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ gt_f16v gt_mma(gt_h8 a, gt_h8 b, gt_f16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ gt_f16v gt_mma(gt_b8 a, gt_b8 b, gt_f16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// How the operands lie in memory.
//   GT_BLOCKS: blocks of 16 rows, element (r, k) at ((k / 8) * 16 + r % 16) * 8 + k % 8 of the block's 16 * K: a chunk is
//              contiguous, and in LDS (the same order) a fragment read covers 256 contiguous bytes per 16 lanes.
//   GT_ROWS:   plain rows of K elements.  A chunk is 64 bytes of each of 16 rows, kept in LDS as 16-byte piece p of row r at
//              position p ^ ((r / 4) % 4), so that 16 rows' same piece falls on all 64 banks; the swizzle is
//              applied to the source address, because the destination of such a load is linear in the lane.
// Half lines of 16 rows cost the address path four times a contiguous chunk's lines: M 28672, K 4096, 2048 tokens take (on one box) 410 us with
// both operands in blocks, 465 with only the weights, 530 with plain rows (M 4096, K 14336: 187, 192, 233).
enum GtLayout { GT_BLOCKS = 0, GT_ROWS = 1 };

constexpr int GT_K = 32;                       // elements of K per step
constexpr int gt_stages(int WM, int WT) { return WM == 2 ? 5 : WT == 2 ? 4 : 3; }
constexpr int gt_lds_bytes(int WM, int WT, int STAGES) { return STAGES * (WM + WT) * 4096; }
constexpr int gt_lds_bytes(int WM, int WT) { return gt_lds_bytes(WM, WT, gt_stages(WM, WT)); }
// waves per SIMD of the workgroups that a CU's 160 KB of LDS hold
constexpr int gt_waves_per_simd(int WM, int WT) { return 160 * 1024 / gt_lds_bytes(WM, WT) * WM * WT / 4; }

// Tile and split of a product.  Four tiles are built; a launch's time goes as the rounds its workgroups make over the CUs times a
// round's time per element of K, which grows with the share of the chip at work (the clock).  A slice costs writing and
// reading its result, and split_ns once where the reader is a launch of its own.  Measured with cold weights, us (M, K, tokens):
//   28672, 4096, 2048: 256x256 419, 256x192 431, 256x128 451, 128x128 479     28672, 4096, 512: 111, 154, 121, 139
//   28672, 4096, 256:  88, 85, 74, 79        6144, 4096, 2048: 100, 140, 110, 108        6144, 4096, 512: 72, 62, 55, 39
//   4096, 4096, 2048:  84, 71, 68, 76        4096, 4096, 512: 71, 61, 54, 38             2048, 8192, 900: 129, 119, 88, 53
// Slices in any number where each keeps 1280 of K (us without the adding): 4096, 14336, 333 on 256x128 in 4 / 5 / 6 slices 54.3 / 49.9 / 53 (192,
// 240 and 288 workgroups), 6144, 4096, 333 on 256x128 in 2 / 3 slices 27 / 23.9, on 256x192 in 4 25.5; shorter ones gain less than the model's
// error (4096, 4096, 333 on 256x128 in 4 / 5 slices 19.5 / 19.1, their adding 1.3 more) and stay at powers of two.
// The cost is of whole tiles, as all of these were measured: halves of 32 tokens that gt_multiply leaves out since (1 to 7% of a call) are not in it.
struct GtPlan {
    int wm = 2, wt = 2, slices = 1, k_slice = 0;       // waves (of 64 rows) by waves (of 64 tokens), one of the tiles below; steps of a slice
};
inline int gt_n_cu() {
    static const int n = [] {
        int dev = 0, cu = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0) cu = 256;
        return cu;
    }();
    return n;
}
// slices_max, slices_room: the most slices the caller takes, and has room for
inline GtPlan gt_plan(int M, int T, int K, int slices_max, size_t slices_room, double split_ns, int n_cu = gt_n_cu()) {
    // one round's time per element of K: a few workgroups, and what a full chip adds
    static constexpr struct { int wm, wt; double few, full; } tiles[4] = {{2, 2, 9.2, 0.3}, {4, 2, 13.0, 3.5}, {4, 3, 14.0, 7.0}, {4, 4, 15.5, 10.5}};
    GtPlan best;
    double least = 0;
    const int steps = K / GT_K;
    for (const auto &t : tiles)
        for (int s = 1; s <= slices_max && (s == 1 || ((size_t)s <= slices_room && K / s >= 256)); ++s) {
            if ((s & (s - 1)) != 0 && K / s < 1280) continue;
            const long n = (long)((M + 64 * t.wm - 1) / (64 * t.wm)) * ((T + 64 * t.wt - 1) / (64 * t.wt)) * s;
            const int k_slice = (steps + s - 1) / s;
            const double ns = t.few + t.full * (n < n_cu ? (double)n / n_cu : 1.0);
            const double cost = (double)((n + n_cu - 1) / n_cu) * ns * k_slice * GT_K + (s > 1 ? s * (double)T * M * 0.00145 + split_ns : 0.0);
            if (least != 0 && cost >= least) continue;
            least = cost;
            best.wm = t.wm; best.wt = t.wt; best.k_slice = k_slice;
            best.slices = (steps + k_slice - 1) / k_slice;      // no empty slice
        }
    return best;
}

// acc += W x over steps [k0, k0 + n_steps), n_steps >= 1.  w, x: 16-bit elements, rows of ldw and ldx (GT_BLOCKS: both K); w_block, x_block: first 16-row block of the
// tile; w_blocks: blocks the matrix holds; x_rows: rows x holds (GT_BLOCKS: up to a whole block).  Blocks and rows past the end
// repeat the last one; what they multiply is never stored.  A wave's half of 32 tokens past the last one is brought into LDS with the tile, but neither read from there nor
// multiplied: a clock that falls with the products at work gains on whole launches what those would have cost.  Chunks, us, multiplied / left out: four
// 32B-shaped layers 270 tokens 1731 / 1620, 600 3014 / 2877, 800 3688 / 3518; eight 8B-shaped ones 333 2046 / 2023, 700 3405 / 3366,
// 1600 6247 / 6124, whole tiles (1536) as before.  SWAP: result rows = tokens, columns (lanes) = weight rows.
template <class V, GtLayout LW, GtLayout LX, int WM, int WT, bool SWAP, int STAGES = gt_stages(WM, WT)>
__device__ __forceinline__ void gt_multiply(char *smem, gt_f16v (&acc)[2][2], const void *w, int ldw, const void *x, int ldx, int k0, int n_steps, int w_block, int w_blocks,
                                            int x_block, int x_rows) {
    constexpr int WAVES = WM * WT, CHUNKS = (WM + WT) * 4, PER = (CHUNKS + WAVES - 1) / WAVES, STAGE = CHUNKS * 1024;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    // this wave's chunks: uniform base, byte offset of the lane, place in the stage.  (A wave with fewer chunks than PER brings the last
    // one again: the same bytes to the same place, and every wave has PER loads per step in flight.)
    const char *src[PER];
    uint32_t off[PER], place[PER], step_bytes[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int c = wave * PER + j < CHUNKS ? wave * PER + j : CHUNKS - 1;
        const bool is_w = c < WM * 4;
        int b = is_w ? w_block + c : x_block + c - WM * 4;
        const int last = is_w ? w_blocks - 1 : (x_rows - 1) / 16;
        b = b < last ? b : last;
        const int ld = is_w ? ldw : ldx;
        src[j] = static_cast<const char *>(is_w ? w : x) + (size_t)b * 32 * (size_t)ld;
        place[j] = lds0 + c * 1024;
        const bool blocks = (is_w ? LW : LX) == GT_BLOCKS;
        step_bytes[j] = blocks ? 1024 : 64;             // from one step's chunk to the next one's
        if (blocks) {
            off[j] = (uint32_t)k0 * 1024u + lane * 16;
        } else {
            int r = lane >> 2;
            const int piece = (lane & 3) ^ ((r >> 2) & 3);
            if (!is_w && r > x_rows - 1 - 16 * b) r = x_rows - 1 - 16 * b;
            off[j] = (uint32_t)r * (uint32_t)ld * 2u + piece * 16 + (uint32_t)k0 * 64u;
        }
    }
    auto load = [&](int stage, int k) {
        const uint32_t at = (uint32_t)(k < n_steps ? k : n_steps - 1);        // (past the end: the last step again, read by nobody)
#pragma unroll
        for (int j = 0; j < PER; ++j) load_to_lds_16(src[j], off[j] + at * step_bytes[j], place[j] + stage * STAGE);
    };
    // fragments of this wave's 64 rows: lane -> row lane % 32 of a 32-row half, 8 elements from 8 * (lane / 32) of a k16 step
    const int r16 = lane & 15, half = lane >> 5;
    const int in_blocks = ((lane & 31) >> 4) * 1024 + half * 256 + r16 * 16, in_rows = ((lane & 31) >> 4) * 1024 + r16 * 64 + (half ^ (r16 >> 2)) * 16;
    const int wf_at = (wave % WM) * 4096 + (LW == GT_BLOCKS ? in_blocks : in_rows), xf_at = (WM + wave / WM) * 4096 + (LX == GT_BLOCKS ? in_blocks : in_rows);
    V wf[2][2], xf[2][2];
    // LIVE: 32-token halves of this wave that hold tokens
    auto read = [&](auto live, const char *st, int ks) {
        constexpr int LIVE = decltype(live)::value;
        auto place_of = [&](GtLayout l, int at) { return l == GT_BLOCKS ? at + 512 * ks : at ^ (32 * ks); };
#pragma unroll
        for (int j = 0; j < LIVE; ++j) xf[ks][j] = *reinterpret_cast<const V *>(st + place_of(LX, xf_at) + 2048 * j);
#pragma unroll
        for (int i = 0; i < (LIVE ? 2 : 0); ++i) wf[ks][i] = *reinterpret_cast<const V *>(st + place_of(LW, wf_at) + 2048 * i);
    };
    auto step = [&](auto live, int stage, auto more, int next_stage, int next_k) {
        constexpr int LIVE = decltype(live)::value;
        const char *st = smem + stage * STAGE;
        read(live, st, 0);
        if constexpr (decltype(more)::value) load(next_stage, next_k);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            if (ks == 0) read(live, st, 1);
#pragma unroll
            for (int i = 0; i < (SWAP ? LIVE : 2); ++i)
#pragma unroll
                for (int j = 0; j < (SWAP ? 2 : LIVE); ++j) acc[i][j] = SWAP ? gt_mma(xf[ks][i], wf[ks][j], acc[i][j]) : gt_mma(wf[ks][i], xf[ks][j], acc[i][j]);
            if (ks == 0 && LIVE == 2) {
                // the second half's fragments are requested between the first half's products
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
    };
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i) load(i, i);
    // (every wave passes the same barriers, whichever of the loops it runs)
    auto steps = [&](auto live) {
        int k = 0;
        for (; k + STAGES <= n_steps; k += STAGES) {
#pragma unroll
            for (int i = 0; i < STAGES; ++i) {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PER * (STAGES - 2)) : "memory");
                step(live, i, std::true_type{}, (i + STAGES - 1) % STAGES, k + i + STAGES - 1);
            }
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int i = 0; i < STAGES - 1; ++i)
            if (k + i < n_steps) step(live, i, std::false_type{}, 0, 0);
    };
    const int tokens = x_rows - x_block * 16 - (wave / WM) * 64;        // from this wave's first on
    if (tokens > 32) steps(std::integral_constant<int, 2>{});
    else if (tokens > 0) steps(std::integral_constant<int, 1>{});
    else steps(std::integral_constant<int, 0>{});
}

__device__ __forceinline__ void gt_clear(gt_f16v (&acc)[2][2]) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
}

// 1-D grid of row tiles x token tiles: the workgroups a die is dealt (every eighth) take a contiguous run of tiles, the token tile
// running fastest, so that a die's cache keeps the weight rows of its run
__device__ __forceinline__ void gt_place(int tile, int n_tiles, int n_ttiles, int &mt, int &tt) {
    const int per = n_tiles >> 3, whole = per << 3;
    if (tile < whole) tile = (tile & 7) * per + (tile >> 3);
    mt = tile / n_ttiles;
    tt = tile % n_ttiles;
}

}  // namespace mesh
