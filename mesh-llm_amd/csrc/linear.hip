// Products of bf16 weight matrices with many token rows, on the matrix cores.
//
// linear_rows_kernel streams the weights: a workgroup owns 16 weight rows and 16 * NT tokens, its four waves split K and
// meet in LDS.  The A operand is the weight row as it lies in memory (lane = row, 8 consecutive k), the B operand the
// activation row (lane = token).  With f32 activations the same fragments feed eight v_mfma_f32_16x16x4_f32 instead of one
// v_mfma_f32_16x16x32_bf16: step j multiplies element j of every lane's 8, and the sum over lanes groups and steps covers
// the same 32 products.
//
// linear_tile_kernel is the large-tile product of gemm_tile.hpp: plain bf16 activation rows, weights in blocks of 16 rows where the
// stage keeps such a copy, else plain rows.
#include "linear.hpp"

#include "gemm_tile.hpp"

namespace mesh {

typedef __bf16 ln_b8 __attribute__((ext_vector_type(8)));
typedef float ln_f4 __attribute__((ext_vector_type(4)));

constexpr int ROWS_WAVES = 4;

template <ActType ACT> struct RowsFrag;
template <> struct RowsFrag<ACT_BF16> {
    uint4 v;
    __device__ __forceinline__ void load(const void *x, size_t at) { v = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(x) + at); }
};
template <> struct RowsFrag<ACT_F32> {
    float4 a, b;
    __device__ __forceinline__ void load(const void *x, size_t at) {
        const float *p = static_cast<const float *>(x) + at;
        a = *reinterpret_cast<const float4 *>(p);
        b = *reinterpret_cast<const float4 *>(p + 4);
    }
};

__device__ __forceinline__ ln_f4 rows_mma(const uint4 &w, const RowsFrag<ACT_BF16> &x, ln_f4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ln_b8, w), __builtin_bit_cast(ln_b8, x.v), acc, 0, 0, 0);
}
__device__ __forceinline__ ln_f4 rows_mma(const uint4 &w, const RowsFrag<ACT_F32> &x, ln_f4 acc) {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
    const float xf[8] = {x.a.x, x.a.y, x.a.z, x.a.w, x.b.x, x.b.y, x.b.z, x.b.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float wf = __uint_as_float((j & 1) ? (u[j >> 1] & 0xFFFF0000u) : (u[j >> 1] << 16));
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf, xf[j], acc, 0, 0, 0);
    }
    return acc;
}

// what becomes of a result: stored as it is, or as an activation of the product that follows
enum LinearOut { LINEAR_OUT_F32 = 0, LINEAR_OUT_RELU2 = 1 };
template <ActType ACT, LinearOut OUT> __device__ __forceinline__ void linear_store(void *y, size_t at, float v) {
    if constexpr (OUT == LINEAR_OUT_RELU2) {
        v = fmaxf(v, 0.f);
        v *= v;
    }
    if constexpr (OUT == LINEAR_OUT_F32 || ACT == ACT_F32) static_cast<float *>(y)[at] = v;
    else static_cast<uint16_t *>(y)[at] = f32_to_bf16_bits(v);
}

// grid (row blocks of 16, token blocks of 16 * NT)
template <ActType ACT, int NT, LinearOut OUT>
__global__ __launch_bounds__(64 * ROWS_WAVES) void linear_rows_kernel(const uint16_t *w, const void *x, void *y, int K, int M, int T, int ldy) {
    __shared__ float red[ROWS_WAVES][NT][16][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.x * 16, t0 = blockIdx.y * 16 * NT;
    const uint16_t *wp = w + (size_t)(m0 + c) * K + 8 * g;
    size_t xo[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int t = t0 + 16 * n + c;
        xo[n] = (size_t)(t < T ? t : T - 1) * K + 8 * g;       // columns past the call repeat its last token and are not stored
    }
    ln_f4 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = ln_f4{0.f, 0.f, 0.f, 0.f};
    // several steps' loads go out together; a step past the end multiplies zero weights
    constexpr int UN = NT == 4 ? 2 : 4;
    for (int kb = wave * 32; kb < K; kb += UN * 32 * ROWS_WAVES) {
        uint4 wf[UN];
        RowsFrag<ACT> xf[UN][NT];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int k = kb + u * 32 * ROWS_WAVES;
            const int at = k < K ? k : 0;
            wf[u] = *reinterpret_cast<const uint4 *>(wp + at);
            if (k >= K) wf[u] = make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int n = 0; n < NT; ++n) xf[u][n].load(x, xo[n] + at);
        }
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[n] = rows_mma(wf[u], xf[u][n], acc[n]);
    }
    // register i of a lane: weight row 4 * g + i, token c
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][n][c][4 * g + i] = acc[n][i];
    __syncthreads();
    for (int idx = tid; idx < NT * 256; idx += 64 * ROWS_WAVES) {
        const int r = idx & 15, tk = (idx >> 4) & 15, n = idx >> 8;
        float s = red[0][n][tk][r];
#pragma unroll
        for (int v = 1; v < ROWS_WAVES; ++v) s += red[v][n][tk][r];
        const int m = m0 + r, t = t0 + 16 * n + tk;
        if (m < M && t < T) linear_store<ACT, OUT>(y, (size_t)t * ldy + m, s);
    }
}

// ---- large tile -----------------------------------------------------------------------------------------------
// blockIdx.y: slice of K (k_slice steps) and the partial result it writes, y_slice floats apart
template <LinearOut OUT, GtLayout LW, int WM, int WT>
__global__ __launch_bounds__(64 * WM * WT, gt_waves_per_simd(WM, WT)) void linear_tile_kernel(const uint16_t *w, const uint16_t *x, void *y, int K, int M, int T, int ldy, int row_blocks,
                                                                                           int n_ttiles, int n_tiles, int k_slice, size_t y_slice) {
    __shared__ __align__(1024) char smem[gt_lds_bytes(WM, WT)];
    int mt, tt;
    gt_place(blockIdx.x, n_tiles, n_ttiles, mt, tt);
    const int n_all = K / GT_K, k0 = blockIdx.y * k_slice, n_steps = n_all - k0 < k_slice ? n_all - k0 : k_slice;
    gt_f16v acc[2][2];
    gt_clear(acc);
    gt_multiply<gt_b8, LW, GT_ROWS, WM, WT, true>(smem, acc, w, K, x, K, k0, n_steps, mt * WM * 4, row_blocks * 8, tt * WT * 4, T);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = (mt * WM + wave % WM) * 64, t0 = (tt * WT + wave / WM) * 64;
    y = static_cast<float *>(y) + blockIdx.y * y_slice;          // (slices are f32 results)
    // register i of a lane: token 8 * (i / 4) + 4 * (lane / 32) + i % 4, weight row lane % 32: a store covers whole lines of y
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int m = m0 + 32 * b + (lane & 31);
        if (m >= M) continue;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int t = t0 + 32 * a + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                if (t < T) linear_store<ACT_BF16, OUT>(y, (size_t)t * ldy + m, acc[a][b][i]);
            }
    }
}

// M: columns of y to write, at least W.M (the rows of W behind it are zeros)
template <ActType ACT, LinearOut OUT>
static int launch_rows(const LinearWeight &W, const void *x, int T, void *y, int ldy, int M, hipStream_t stream) {
    const unsigned mb = (unsigned)((M + 15) / 16);
    const dim3 block(64 * ROWS_WAVES);
    if (T <= 16) MESH_LAUNCH((linear_rows_kernel<ACT, 1, OUT>), dim3(mb, 1), block, 0, stream, W.w, x, y, W.Kp, M, T, ldy);
    else if (T <= 32) MESH_LAUNCH((linear_rows_kernel<ACT, 2, OUT>), dim3(mb, 1), block, 0, stream, W.w, x, y, W.Kp, M, T, ldy);
    else MESH_LAUNCH((linear_rows_kernel<ACT, 4, OUT>), dim3(mb, (unsigned)((T + 63) / 64)), block, 0, stream, W.w, x, y, W.Kp, M, T, ldy);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

__global__ __launch_bounds__(256) void linear_blocks_kernel(const uint16_t *w, uint16_t *dst, int K, size_t pieces) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;        // 16-byte piece of dst: row i % 16 of its block, k from 8 * (i / 16 % (K / 8))
    if (i >= pieces) return;
    const size_t k8 = i / 16 % (K / 8), row = i / (2 * (size_t)K) * 16 + i % 16;
    reinterpret_cast<uint4 *>(dst)[i] = *reinterpret_cast<const uint4 *>(w + row * K + k8 * 8);
}

int linear_make_blocks(const LinearWeight &W, uint16_t *dst, hipStream_t stream) {
    if (!W.w || !dst || W.Mp % 16 || W.Kp % 8) return fail(MESH_ERR_INVALID, "linear_make_blocks: bad operands (%d x %d)", W.M, W.K);
    const size_t pieces = (size_t)W.Mp * W.Kp / 8;
    MESH_LAUNCH(linear_blocks_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, W.w, dst, W.Kp, pieces);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

template <LinearOut OUT, GtLayout LW>
static int launch_tile_layout(const uint16_t *w, const LinearWeight &W, const void *x, int T, void *y, int ldy, int M, const GtPlan &p, size_t stride, hipStream_t stream) {
    const int row_blocks = W.Mp / 128, mtiles = (M + 64 * p.wm - 1) / (64 * p.wm), ttiles = (T + 64 * p.wt - 1) / (64 * p.wt);
    const dim3 grid((unsigned)(mtiles * ttiles), (unsigned)p.slices), block((unsigned)(64 * p.wm * p.wt));
    const uint16_t *xb = static_cast<const uint16_t *>(x);
    if (p.wt == 4) MESH_LAUNCH((linear_tile_kernel<OUT, LW, 4, 4>), grid, block, 0, stream, w, xb, y, W.Kp, M, T, ldy, row_blocks, ttiles, mtiles * ttiles, p.k_slice, stride);
    else if (p.wt == 3) MESH_LAUNCH((linear_tile_kernel<OUT, LW, 4, 3>), grid, block, 0, stream, w, xb, y, W.Kp, M, T, ldy, row_blocks, ttiles, mtiles * ttiles, p.k_slice, stride);
    else if (p.wm == 4) MESH_LAUNCH((linear_tile_kernel<OUT, LW, 4, 2>), grid, block, 0, stream, w, xb, y, W.Kp, M, T, ldy, row_blocks, ttiles, mtiles * ttiles, p.k_slice, stride);
    else MESH_LAUNCH((linear_tile_kernel<OUT, LW, 2, 2>), grid, block, 0, stream, w, xb, y, W.Kp, M, T, ldy, row_blocks, ttiles, mtiles * ttiles, p.k_slice, stride);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}
template <LinearOut OUT>
static int launch_tile(const LinearWeight &W, const void *x, int T, void *y, int ldy, int M, const GtPlan &p, size_t stride, hipStream_t stream) {
    return W.blocks ? launch_tile_layout<OUT, GT_BLOCKS>(static_cast<const uint16_t *>(W.blocks), W, x, T, y, ldy, M, p, stride, stream) : launch_tile_layout<OUT, GT_ROWS>(W.w, W, x, T, y, ldy, M, p, stride, stream);
}

static bool linear_ok(const LinearWeight &W, const void *x, int T, const void *y, int ldy) {
    return W.w && x && y && W.M >= 1 && W.Kp % LINEAR_K_PAD == 0 && W.Mp % LINEAR_ROW_PAD == 0 && W.Mp >= W.M && W.Kp >= W.K && ldy >= W.M && (T + 63) / 64 <= 65535;
}

int linear_sliced(const LinearWeight &W, const void *x, ActType act, int T, float *y, size_t stride, size_t y_floats, int big_from, hipStream_t stream) {
    if (T <= 0) return 1;
    if (!linear_ok(W, x, T, y, W.M) || stride < (size_t)T * W.M || y_floats < stride) return fail(MESH_ERR_INVALID, "linear_sliced: bad operands (%d x %d, %d tokens)", W.M, W.K, T);
    GtPlan p;
    if (act == ACT_BF16 && T >= big_from) p = gt_plan(W.M, T, W.Kp, LINEAR_SLICES_MAX, y_floats / stride, 0.0);
    if (p.slices <= 1) {
        const int rc = linear(W, x, act, T, y, W.M, big_from, stream);
        return rc == MESH_OK ? 1 : rc;
    }
    const int rc = launch_tile<LINEAR_OUT_F32>(W, x, T, y, W.M, W.M, p, stride, stream);
    return rc == MESH_OK ? p.slices : rc;
}

int linear(const LinearWeight &W, const void *x, ActType act, int T, float *y, int ldy, int big_from, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    if (!linear_ok(W, x, T, y, ldy)) return fail(MESH_ERR_INVALID, "linear: bad operands (%d x %d, %d tokens)", W.M, W.K, T);
    if (act == ACT_F32) return launch_rows<ACT_F32, LINEAR_OUT_F32>(W, x, T, y, ldy, W.M, stream);
    if (T < big_from || W.M < 128) return launch_rows<ACT_BF16, LINEAR_OUT_F32>(W, x, T, y, ldy, W.M, stream);
    return launch_tile<LINEAR_OUT_F32>(W, x, T, y, ldy, W.M, gt_plan(W.M, T, W.Kp, 1, 1, 0.0), 0, stream);
}

int linear_relu2(const LinearWeight &W, const void *x, ActType act, int T, void *out, int ld, int big_from, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    if (!linear_ok(W, x, T, out, ld) || ld > W.Mp) return fail(MESH_ERR_INVALID, "linear_relu2: bad operands (%d x %d, %d tokens)", W.M, W.K, T);
    if (act == ACT_F32) return launch_rows<ACT_F32, LINEAR_OUT_RELU2>(W, x, T, out, ld, ld, stream);
    if (T < big_from || W.M < 128) return launch_rows<ACT_BF16, LINEAR_OUT_RELU2>(W, x, T, out, ld, ld, stream);
    return launch_tile<LINEAR_OUT_RELU2>(W, x, T, out, ld, ld, gt_plan(ld, T, W.Kp, 1, 1, 0.0), 0, stream);
}

}  // namespace mesh
