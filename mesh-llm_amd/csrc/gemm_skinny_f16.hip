// Skinny GEMM for batched decode on the f16 matrix cores: Y[T][M] = W[M][K] . X[T][K] with up to 16 or up to 32 tokens per
// pass, W a tiled q4_K / q6_K matrix, X in f16 (the k8-major layout of gemm.hpp).
//
// The alternative to the integer kernel of gemm_skinny.hip for the same launches: the weight stream is organised as in
// the mat-vec kernel -- a workgroup owns a few tile-rows (16 rows each), its waves split K and each keeps two
// weight tiles in flight -- and a tile is formed in registers as f16 and multiplied with 16 activation columns at
// once (v_mfma_f32_16x16x32_f16).  Activations are f16 (11 significant bits against the integer kernel's 16-bit fixed point).
// A fragment holds the integers q * sc of q4_K (at most 945, exact) or (q - 32) * sc of q6_K (exact up to 2048; odd ones above, up
// to 4096, are rounded by 2^-12 of themselves), the sub-block minimum's integers go through MFMAs of their own, and the super-block's
// d and dmin multiply the tile's sums in f32.  (Before, every weight was rounded to f16 once; a first version multiplied by d * sc
// rounded to f16, which does not average out over K.)
//
// What bounds it.  By time stamps (gate / up of 28672 x 4096, 66 MB, 5 tokens): first loads requested at 2.3 us, a workgroup's weight
// stream done at 11.2, its slowest wave at 14.9, its end 16.1; the last workgroup ends at 20.3, so the launch as a whole streams at
// 3.2 TB/s of the 5.9 - 6.1 that reads reach.  Before, every round waited for all it had requested (a branch around
// a tile makes the compiler assume the worst), the norm's partial sums were fetched behind it (2.9 us) and the epilogue's operands
// behind the barrier (1.5 - 2).
// Before / now, us: 5 tokens gate / up 22.6 / 20.5, q/k/v 11.8 - 12.0 / 10.1 - 10.7, output 7.4 / 7.6, q4_K down 16.4 / 14.4, q6_K down
// 19.4 / 17.2; 16 tokens 23.3 / 21.0, 12.6 - 12.9 / 10.8 - 11.6, 7.9 / 7.6, 16.7 / 14.8, 19.7 / 17.7; 32 tokens of the 32B shape (160
// workgroups of two tile-rows) q6_K down 59.0 / 52.4, q4_K down 57.4 / 44.8, output 17.0 / 14.5, q/k/v 16.7 - 18.4 / 15.8 - 16.2.
//
// Register dequantisation: lane (m = l % 16, g = l / 16) loads what lane 4m + g of the mat-vec kernel loads, i.e.
// quarter g of row m of the super-block (gemv.hpp).  An MFMA's k-slots of lane group g are then 8 consecutive
// elements of that quarter; the B operand (activations) is read with the same element indices, so the k-order of
// the instruction never has to match the order in memory.  Nibbles become f16 through the exponent trick
// (0x6400 | q is 1024 + q exactly).  Weight tiles are loaded with the mat-vec kernel's dense lane mapping and moved to
// the MFMA lanes with ds_bpermute, so that a wave's load touches whole cache lines.
//
// Same place in the worker's graph as the mat-vec kernel: mul_mat for K-quant weights, reached from
// rpc_server::graph_compute (third_party/llama.cpp/patches/0002-rpc-add-direct-peer-tensor-transfers.patch:443-451).

#include "gemm.hpp"
#include "lds_ops.hpp"
#include "skinny_frags.hpp"
#include "wave_ops.hpp"

namespace mesh {
namespace f16sk {

constexpr int SK_THREADS = 512;
constexpr int SK_WAVES = SK_THREADS / 64;
constexpr int SK_DEPTH = 2;               // weight tiles a wave keeps in flight (three or four: 1-5% of a step slower)
constexpr int SK_NT = 16;                 // activation columns of one MFMA (a launch takes one or two such blocks)
constexpr int SK_SEGS_MAX = 4;            // (tile-row, matrix) segments one wave may own (8 spills registers)
constexpr size_t SK_LDS_LIMIT = 160 * 1024;

struct SkinnyKernelArgs {
    const uint8_t *wbase[3];      // matrix base minus its first tile-row, so a global tile-row index addresses it
    int tile_begin[4];            // first global tile-row of each matrix; unused slots hold the total
    float *y[3];
    const float *bias[3];
    int M[3];
    int ldy[3];
    const _Float16 *x;            // k8-major block of 16 columns
    int K, T;
    const float *residual;
    int ldres;
    int epi;
    _Float16 *y16;                // optional f16 copy of the output (matrix 0): k8-major block with M16 rows as its k
    unsigned *sat;                // optional counter of y16 values clamped to the f16 range
    int M16;
    int ks;                       // waves along K
    GemvRope rope;                // rope.pos / rope.seq point at the launch's first column
    int kind[3];
    // RMS-norm hand-over (gemm.hpp: SkinnyF16Args::NormOut / NormIn)
    const float *no_w;            // producer: weight of the norm that follows
    _Float16 *no_x16;
    float *no_part;
    const float *ni_part;         // consumer: [ni_parts][16] partial sums of squares
    int ni_parts;
    float ni_eps;
};

// B fragments of one super-block for this lane: 8 MFMAs x 8 f16
template <int TYPE>
struct BFrags {
    uint4 b[8];
    // base: the super-block's k8-major activations (uniform), lane_off: this lane's column and quarter offset in halfs
    __device__ __forceinline__ void load(const _Float16 *base, int lane_off) {
#pragma unroll
        for (int t = 0; t < 8; ++t) b[t] = ldg<uint4>(base + lane_off + frag_k<TYPE>(t) * 16);
    }
};

// Where a lane's share of the activation fragments lies: lane (n = m, g) supplies column n, quarter g.  A column past the call's tokens is
// its block's last one again, which takes no line of its own, and what it yields is dropped: the fragments of a super-block are 8 KB to
// 2.3 of weights, and half of their lines go (eight 8B-shaped layers, 5 tokens 612 -> 590 us; the zeros that lie there read before).
template <int TYPE, int NC>
struct SkinnyColumns {
    int at[NC];
    __device__ __forceinline__ SkinnyColumns(int m, int g, int T) {
#pragma unroll
        for (int c = 0; c < NC; ++c) at[c] = quarter_k<TYPE>(g) * 16 + min(m, max(T - 1 - SK_NT * c, 0)) * 8;
    }
};

// A wave's walk: its n_i super-blocks of SEGS (tile-row, matrix) segments each, tile_ptr(ii, seg) the tile of one, times NC blocks of 16
// activation columns.  x: the activations of its first super-block; x_step, x_block: halfs to its next one and to the next block of columns.
template <int TYPE, int SEGS, int NC>
struct SkinnyWalk {
    static constexpr int RB = SEGS % SK_DEPTH == 0 ? 1 : SK_DEPTH;      // super-blocks per round: ring slots static inside it
    static_assert(RB <= 2 && RB * SEGS % SK_DEPTH == 0, "ring slots must be static inside a round, and at most one super-block left over");
    const _Float16 *x;
    unsigned x_step, x_block;         // (32 bits: an address is one scalar product and a sum)
    int n_i, lane, g, src_lane4;
    SkinnyColumns<TYPE, NC> cols;
    TileRegs<TYPE> ring[SK_DEPTH];
    BFrags<TYPE> Bw[NC];

    // (a constructor: braces around the members would clear the registers of ring and Bw before the first load)
    __device__ __forceinline__ SkinnyWalk(const _Float16 *x_, unsigned x_step_, unsigned x_block_, int n_i_, int lane_, int g_, int src_lane4_, const SkinnyColumns<TYPE, NC> &cols_)
        : x(x_), x_step(x_step_), x_block(x_block_), n_i(n_i_), lane(lane_), g(g_), src_lane4(src_lane4_), cols(cols_) {}

    // The walk has no branch inside a round of tiles: a tile past the end is the wave's last one again (a cache hit).  The compiler
    // then knows how many loads are in flight at every point and waits for one tile without draining the others; with a branch
    // around a tile or a load it assumes the worst at the join, and every round waited for everything it had just requested.
    template <class TilePtr> __device__ __forceinline__ void load_tile(TileRegs<TYPE> &dst, int ii, int seg, const TilePtr &tile_ptr) {
        dst.load(tile_ptr(ii < n_i ? ii : n_i - 1, seg), lane);
    }
    // Activation fragments: 8 KB per super-block, column block and wave.  Only ONE super-block is held (32 registers per
    // column block) and every fragment is fetched again, for the next super-block, right behind the last MFMAs that read
    // it: one tile's time ahead of its use, enough for a hit in L2.  (Two whole super-blocks in registers, fetched a
    // super-block ahead, cost 32 more registers per column block and measured 6% slower at 16 columns.)
    __device__ __forceinline__ void step(const TileRegs<TYPE> &loaded, f4_t (&acc)[NC], bool refill, int next_ii) {
        const _Float16 *nb = x + (unsigned)(next_ii < n_i ? next_ii : n_i - 1) * x_step;
        TileRegs<TYPE> tile = loaded;
        to_mfma_lanes(tile, src_lane4);
        TileFrags<TYPE> F;
        F.prepare(tile, g);
        f4_t sum[NC];
        [[maybe_unused]] f4_t low[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) sum[c] = low[c] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const h8_t wf = F.frag(t);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                sum[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, Bw[c].b[t]), wf, sum[c], 0, 0, 0);
                if constexpr (TileFrags<TYPE>::MINIMUM)
                    low[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, Bw[c].b[t]), F.minimum(t), low[c], 0, 0, 0);
            }
            if (refill) {
#pragma unroll
                for (int c = 0; c < NC; ++c) Bw[c].b[t] = ldg<uint4>(nb + c * x_block + cols.at[c] + frag_k<TYPE>(t) * 16);
            }
        }
        // a lane's outputs are all of weight row m, whose scales it holds
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[c][i] = fmaf(F.d, sum[c][i], acc[c][i]);
                if constexpr (TileFrags<TYPE>::MINIMUM) acc[c][i] = fmaf(F.ndmin, low[c][i], acc[c][i]);
            }
    }
    // clears the sums and requests the first tiles and fragments
    template <class TilePtr> __device__ __forceinline__ void start(f4_t (&D)[SEGS][NC], bool any, const TilePtr &tile_ptr) {
#pragma unroll
        for (int s = 0; s < SEGS; ++s)
#pragma unroll
            for (int c = 0; c < NC; ++c) D[s][c] = f4_t{0.f, 0.f, 0.f, 0.f};
        if (any) {
#pragma unroll
            for (int f = 0; f < SK_DEPTH; ++f) load_tile(ring[f], f / SEGS, f % SEGS, tile_ptr);
#pragma unroll
            for (int c = 0; c < NC; ++c) Bw[c].load(x + c * x_block, cols.at[c]);
        }
    }
    template <class TilePtr> __device__ __forceinline__ void run(f4_t (&D)[SEGS][NC], const TilePtr &tile_ptr) {
        int ii = 0;
        for (; ii + RB <= n_i; ii += RB) {
#pragma unroll
            for (int q = 0; q < RB * SEGS; ++q) {
                const int seg = q % SEGS, slot = q % SK_DEPTH;
                step(ring[slot], D[seg], seg == SEGS - 1, ii + q / SEGS + 1);
                // (the tile goes out behind the fragments, which are needed first: loads return in order)
                __builtin_amdgcn_sched_barrier(0);
                load_tile(ring[slot], ii + (q + SK_DEPTH) / SEGS, (q + SK_DEPTH) % SEGS, tile_ptr);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (RB > 1 && ii < n_i) {
#pragma unroll
            for (int seg = 0; seg < SEGS; ++seg) {
                step(ring[seg % SK_DEPTH], D[seg], false, 0);
                if (seg + SK_DEPTH < SEGS) load_tile(ring[seg % SK_DEPTH], ii, seg + SK_DEPTH, tile_ptr);
            }
        }
    }
};

// element (row k, column t) of k8-major f16 activations with K rows per column: block t / 16 of 16 * K halfs
__device__ __forceinline__ size_t k8_at(int K, int k, int t) { return (size_t)(t >> 4) * 16 * K + ((size_t)(k >> 3) * 16 + (t & 15)) * 8 + (k & 7); }

// KB per wave and column block that hold a wave's share of the partial sums
constexpr int NORM_CHUNKS = SKINNY_F16_NORM_PARTS_MAX / SK_WAVES * SK_NT / 256;
static_assert(NORM_CHUNKS * 256 * SK_WAVES == SKINNY_F16_NORM_PARTS_MAX * SK_NT, "shares of whole KB");

// most tile-rows a workgroup of the launch has (p_split = tile-rows per workgroup | workgroups with one more << 16)
__device__ __forceinline__ int rows_here_max(unsigned p_split) { return (int)(p_split & 0xFFFFu) + ((p_split >> 16) ? 1 : 0); }

// NC: blocks of 16 activation columns one pass over the weights multiplies with (1: up to 16 tokens, 2: up to 32).
// bx: the workgroup's index among those of its launch part (the whole launch, or one side of a pair launch).
template <int TYPE, int NU, int SEGS, int NC>
__device__ __forceinline__ void skinny_workgroup(int bx, const _Float16 *p_x, const uint8_t *p_w0, const uint8_t *p_w1, const uint8_t *p_w2, int p_K,
                                                 int p_ks, unsigned p_begins, unsigned p_split, const SkinnyKernelArgs &a) {
    // (p_ks = waves along K | columns << 16; p_begins = first tile-row of matrix 1 | of matrix 2 << 16; p_split = tile-rows per workgroup | workgroups with one
    // more << 16, computed on the host: no division and no grid-size load stand before the first weight load)
    const int p_begin1 = (int)(p_begins & 0xFFFFu), p_begin2 = (int)(p_begins >> 16);
    // (leading scalar arguments: preloaded into SGPRs, see gemv.hip)
    extern __shared__ __align__(16) uint8_t smem[];
    float *red = reinterpret_cast<float *>(smem);         // [KS][rows_here][NU][16 rows][16 NC columns]
    constexpr int TB = TileRegs<TYPE>::BYTES;
    const int K = p_K, nsb = K / QK_K;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);       // scalar: tile addresses become SGPR base + lane offset
    const int m = lane & 15, g = lane >> 4;
    const int src_lane4 = 4 * (4 * m + g);                // byte address, for ds_bpermute, of the lane that loaded row m, quarter g
    const int KS = p_ks & 0xFFFF, T = p_ks >> 16, LK = __builtin_ctz((unsigned)KS), RS = SK_WAVES >> LK;      // KS is a power of two
    const int ks = wave & (KS - 1), rs = wave >> LK;
    const int sq = (int)(p_split & 0xFFFFu), sr = (int)(p_split >> 16);
    const int tr0 = bx * sq + (bx < sr ? bx : sr);
    const int rows_here = sq + (bx < sr ? 1 : 0);
    const int n_i = rs < RS ? (nsb - ks + KS - 1) >> LK : 0;        // super-blocks of this wave (ks < KS <= nsb)
    const size_t row_stride = (size_t)nsb * TB;
    const SkinnyColumns<TYPE, NC> cols(m, g, T);
    // flat tile index f = ii * SEGS + seg; seg -> (local tile-row j, matrix u).  A segment past the workgroup's rows reads the wave's
    // first one again and is dropped at the end: the walk has no branch (see below).
    auto seg_valid = [&](int seg) { return rs + RS * (seg / NU) < rows_here; };
    auto tile_ptr = [&](int ii, int seg) -> const uint8_t * {
        const int tr = tr0 + rs + (seg_valid(seg) ? RS * (seg / NU) : 0);
        int mi = seg % NU;
        if (NU == 1) mi = (tr >= p_begin1 ? 1 : 0) + (tr >= p_begin2 ? 1 : 0);
        // (offsets added under conditions: an indexed kernel-argument array is fetched with a load, and a three-way
        // select of preloaded pointers becomes a table in scratch memory)
        const uint8_t *wb = p_w0 + (mi >= 1 ? p_w1 - p_w0 : (ptrdiff_t)0) + (mi >= 2 ? p_w2 - p_w1 : (ptrdiff_t)0);
        return wb + (size_t)tr * row_stride + (size_t)(ks + KS * ii) * TB;
    };
    // a wave without a valid first segment has nothing at all
    const bool any = n_i > 0 && seg_valid(0);
    constexpr int NT = SK_NT * NC;                        // activation columns of this launch
    f4_t D[SEGS][NC];
    SkinnyWalk<TYPE, SEGS, NC> walk(p_x + (size_t)ks * (QK_K * 16), (unsigned)KS * (QK_K * 16), (unsigned)SK_NT * K, n_i, lane, g, src_lane4, cols);
    walk.start(D, any, tile_ptr);
    // What the tail of the workgroup reads is requested here, behind the first tiles: fetched where it is used, the norm's
    // partial sums cost 2.9 us behind the weight stream, the residual or the rotation's operands 1.5 - 2.
    // (Branch-free: a launch or thread that has no use for an operand reads the first activations instead.)
    const float *const idle = reinterpret_cast<const float *>(p_x);
    float *const nrm = red + (size_t)KS * rows_here_max(p_split) * NU * 16 * NT;        // [SK_WAVES][NT] sums of the consumer side
    float *const wsum = nrm + SK_WAVES * NT;                                            // [SK_WAVES][NT] of the producer side
    float *const my_parts = wsum + SK_WAVES * NT + wave * (NORM_CHUNKS * NC * 256);     // this wave's share of the partial sums
    const int parts_per = a.ni_part ? (a.ni_parts + SK_WAVES - 1) / SK_WAVES : 0, parts_end = a.ni_part ? a.ni_parts : 0;
    {
        const float *src = a.ni_part ? a.ni_part : idle;
        const int last = a.ni_part ? a.ni_parts * NT - 4 : 4 * 63;
#pragma unroll
        for (int i = 0; i < NORM_CHUNKS * NC; ++i) {
            const int at = wave * parts_per * NT + i * 256 + lane * 4;
            load_to_lds_16(src, 4u * (at < last ? at : last), lds_place(my_parts + i * 256));
        }
    }
    // outputs of a thread: column tid % NT and row (tid / NT) % 16 of the tile-rows out_j, out_j + OUT_STEP, ...
    constexpr int OUT_STEP = SK_THREADS / (16 * NT), OUT_PRE = 2;
    // (a wave's outputs lie in one tile-row: which matrix that is of stays a scalar)
    const int out_t = tid % NT, out_r = (tid / NT) % 16, out_j = __builtin_amdgcn_readfirstlane(tid / (16 * NT));
    const bool roped = NU == 1 && a.rope.pos;
    [[maybe_unused]] float pre_res[OUT_PRE], pre_w[OUT_PRE], pre_freq[OUT_PRE];
    [[maybe_unused]] bool pre_rot[OUT_PRE];
    [[maybe_unused]] int pre_pos = 0;
    auto matrix_of = [&](int tr) { return NU == 1 ? (tr >= a.tile_begin[1] ? 1 : 0) + (tr >= a.tile_begin[2] ? 1 : 0) : 0; };
    if constexpr (NU == 1) {
        pre_pos = *(roped && out_t < a.T ? a.rope.pos + out_t : reinterpret_cast<const int32_t *>(idle));
#pragma unroll
        for (int k = 0; k < OUT_PRE; ++k) {
            const int tr = tr0 + out_j + k * OUT_STEP, mi = matrix_of(tr), row = (tr - a.tile_begin[mi]) * TILE_ROWS + out_r;
            const bool ok = out_j + k * OUT_STEP < rows_here && row < a.M[mi] && out_t < a.T;
            pre_res[k] = *(ok && a.epi == EPI_RESIDUAL ? a.residual + (size_t)out_t * a.ldres + row : idle);
            pre_w[k] = *(ok && a.no_x16 ? a.no_w + row : idle);
            const int dd = roped ? row % a.rope.head_dim : 0;
            pre_rot[k] = ok && roped && dd < a.rope.n_rot && (a.kind[mi] == GEMV_KIND_Q || a.kind[mi] == GEMV_KIND_K);
            pre_freq[k] = *(pre_rot[k] ? a.rope.inv_freq + (dd >> 1) : idle);
        }
    }
    if (any) walk.run(D, tile_ptr);
    // partial sums of this wave: D[seg] holds row m, columns 4g..4g+3 of segment seg
#pragma unroll
    for (int seg = 0; seg < SEGS; ++seg) {
        if (any && seg_valid(seg)) {
            const int j = rs + RS * (seg / NU), u = seg % NU;
#pragma unroll
            for (int c = 0; c < NC; ++c) *reinterpret_cast<f4_t *>(red + ((((size_t)ks * rows_here + j) * NU + u) * 16 + m) * NT + c * SK_NT + 4 * g) = D[seg][c];
        }
    }
    // norm hand-over, consumer side: this wave's share of the partial sums of squares of every column, in order
    if (a.ni_part) {
        // (loads return in order: a wave that has walked a second super-block has used activations that it requested behind the
        // partial sums, and its sums with them stand before this in memory's order; any other waits for all it has requested)
        if (any && n_i >= 2) asm volatile("" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        float ss = 0.f;
        for (int p = lane / NT; p < parts_per; p += 64 / NT) ss += wave * parts_per + p < parts_end ? my_parts[p * NT + lane % NT] : 0.f;
        if (NT == 16) ss = lane_fold<16>(ss, LaneAdd{});
        ss = lane_fold<32>(ss, LaneAdd{});
        if (lane < NT) nrm[wave * NT + lane] = ss;
    }
    [[maybe_unused]] float pre_sin[OUT_PRE], pre_cos[OUT_PRE];
    if constexpr (NU == 1) {
#pragma unroll
        for (int k = 0; k < OUT_PRE; ++k) {
            pre_sin[k] = pre_cos[k] = 0.f;
            if (pre_rot[k]) sincosf((float)pre_pos * pre_freq[k], &pre_sin[k], &pre_cos[k]);
        }
    }
    __syncthreads();
    // 1 / rms of this thread's column (every output of a thread is of column tid % NT): waves added in order
    float inv_rms = 1.0f;
    if (a.ni_part) {
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < SK_WAVES; ++q) ss += nrm[q * NT + out_t];
        inv_rms = 1.0f / sqrtf(ss / (float)K + a.ni_eps);
    }
    float no_ss = 0.f;         // producer side: sum of squares of this thread's outputs (one column)
    // outputs of this workgroup: rows_here x 16 rows x T columns; column t is column t % 16 of the f16 layouts' block t / 16
    const int t = out_t, r = out_r;
    for (int j = out_j, k = 0; j < rows_here; j += OUT_STEP, ++k) {
        const int tr = tr0 + j, mi = matrix_of(tr);
        const int row = (tr - a.tile_begin[mi]) * TILE_ROWS + r;
        if (row >= a.M[mi]) continue;
        if (t >= a.T) {                                    // unused columns of the f16 output block stay finite
            if (a.y16 && mi == 0) a.y16[k8_at(a.M16, row, t)] = (_Float16)0.f;
            if (a.no_x16) a.no_x16[k8_at(a.M[0], row, t)] = (_Float16)0.f;
            continue;
        }
        float s0 = 0.f, s1 = 0.f;
        for (int k2 = 0; k2 < KS; ++k2) {
            s0 += red[((((size_t)k2 * rows_here + j) * NU + 0) * 16 + r) * NT + t];
            if (NU == 2) s1 += red[((((size_t)k2 * rows_here + j) * NU + 1) * 16 + r) * NT + t];
        }
        s0 *= inv_rms;
        if (NU == 2) s1 *= inv_rms;
        if (a.bias[mi]) s0 += a.bias[mi][row];
        if (NU == 1 && a.rope.pos && a.kind[mi] != GEMV_KIND_PLAIN) {
            // q / k / v row of a token (see gemv.hpp): rotate q and k with the neighbouring row, k and v go to the cache
            const int kind = a.kind[mi], hd = a.rope.head_dim;
            const int head = row / hd, dd = row - head * hd;
            const int pos = pre_pos;
            float val = s0;
            if (kind != GEMV_KIND_V && dd < a.rope.n_rot) {
                float sp = 0.f;
                for (int k2 = 0; k2 < KS; ++k2) sp += red[((((size_t)k2 * rows_here + j) * NU + 0) * 16 + (r ^ 1)) * NT + t];
                sp *= inv_rms;
                if (a.bias[mi]) sp += a.bias[mi][row ^ 1];
                float sn = k == 0 ? pre_sin[0] : pre_sin[1], cs = k == 0 ? pre_cos[0] : pre_cos[1];
                if (k >= OUT_PRE) sincosf((float)pos * a.rope.inv_freq[dd >> 1], &sn, &cs);
                val = (dd & 1) ? sp * sn + s0 * cs : s0 * cs - sp * sn;
            }
            if (kind == GEMV_KIND_Q) {
                a.y[mi][(size_t)t * a.ldy[mi] + row] = val;
            } else {
                uint16_t *cache = kind == GEMV_KIND_K ? a.rope.kcache : a.rope.vcache;
                cache[(((size_t)a.rope.seq[t] * a.rope.n_kv + head) * a.rope.n_ctx + pos) * hd + dd] = f32_to_f16_bits(val);
            }
            continue;
        }
        float out = s0;
        if constexpr (NU == 2) {
            if (a.bias[1]) s1 += a.bias[1][row];
            out = (s0 / (1.0f + expf(-s0))) * s1;
        } else if (a.epi == EPI_RESIDUAL) {
            out = (k == 0 ? pre_res[0] : k == 1 ? pre_res[1] : a.residual[(size_t)t * a.ldres + row]) + s0;
        }
        if (a.y[mi]) a.y[mi][(size_t)t * a.ldy[mi] + row] = out;
        // (saturating: a SwiGLU product beyond the f16 range becomes +-65504, not an infinity the next GEMM would spread)
        if (a.y16 && mi == 0) {
            note_f16_clamp(a.sat, out, 0.f);
            a.y16[k8_at(a.M16, row, t)] = (_Float16)__builtin_amdgcn_fmed3f(out, -65504.f, 65504.f);
        }
        if (a.no_x16) {
            float v = out;
            if constexpr (NU == 1) v *= k == 0 ? pre_w[0] : k == 1 ? pre_w[1] : a.no_w[row];
            note_f16_clamp(a.sat, v, 0.f);
            a.no_x16[k8_at(a.M[0], row, t)] = (_Float16)__builtin_amdgcn_fmed3f(v, -65504.f, 65504.f);
            no_ss = fmaf(out, out, no_ss);
        }
    }
    if (a.no_part) {
        // this workgroup's sum of squares per column: the lanes of a wave that share a column, then the waves in order
        if (NT == 16) no_ss = lane_fold<16>(no_ss, LaneAdd{});
        no_ss = lane_fold<32>(no_ss, LaneAdd{});
        if (lane < NT) wsum[wave * NT + lane] = no_ss;
        __syncthreads();
        if (tid < NT) {
            float ss = 0.f;
            for (int w = 0; w < SK_WAVES; ++w) ss += wsum[w * NT + tid];
            a.no_part[(size_t)bx * NT + tid] = ss;
        }
    }
}

template <int TYPE, int NU, int SEGS, int NC>
__global__ __launch_bounds__(SK_THREADS, 2) void gemm_skinny_kernel(const _Float16 *p_x, const uint8_t *p_w0, const uint8_t *p_w1, const uint8_t *p_w2, int p_K,
                                                                 int p_ks, int p_rows, unsigned p_begins, unsigned p_split,
                                                                 const SkinnyKernelArgs a) {
    (void)p_rows;
    skinny_workgroup<TYPE, NU, SEGS, NC>((int)blockIdx.x, p_x, p_w0, p_w1, p_w2, p_K, p_ks, p_begins, p_split, a);
}

// Two launches that read the same activations as one: the first grid_a workgroups run a q4_K launch, the others a q6_K launch
// (the q and k projections of a layer next to a q6_K v projection: 160 + 64 workgroups at Llama-3-8B shape, one wave of
// workgroups instead of two dependent launches).  Same arithmetic per workgroup as the separate launches.
template <int SEGS_A, int SEGS_B, int NC>
__global__ __launch_bounds__(SK_THREADS, 2) void gemm_skinny_pair_kernel(const _Float16 *p_x, const uint8_t *p_w0, const uint8_t *p_w1, int p_K, int p_ks,
                                                                      int grid_a, unsigned p_begins, unsigned p_split_a, unsigned p_split_b,
                                                                      const uint8_t *p_wb, const SkinnyKernelArgs a, const SkinnyKernelArgs b) {
    const int bx = (int)blockIdx.x;
    if (bx < grid_a) skinny_workgroup<MESH_Q4_K, 1, SEGS_A, NC>(bx, p_x, p_w0, p_w1, p_w1, p_K, p_ks, p_begins, p_split_a, a);
    else skinny_workgroup<MESH_Q6_K, 1, SEGS_B, NC>(bx - grid_a, p_x, p_wb, p_wb, p_wb, p_K, p_ks, 0xFFFFFFFFu, p_split_b, b);
}

// A launch cut along K: workgroup (slice, group) multiplies SEGS tile-rows by one slice of the super-blocks, which its eight waves share, and
// writes the sums to part[slice][column][row]; gemm_add_slices adds them.
template <int TYPE, int SEGS, int NC>
__global__ __launch_bounds__(SK_THREADS, 2) void gemm_skinny_slice_kernel(const _Float16 *p_x, const uint8_t *p_w, int p_K, int p_T, int p_rows, int p_per, int p_ld, float *p_part) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int NT = SK_NT * NC, TB = TileRegs<TYPE>::BYTES;
    float *red = reinterpret_cast<float *>(smem);         // [SK_WAVES][SEGS][NT columns][16 rows]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int nsb = p_K / QK_K, sb0 = (int)blockIdx.x * p_per, here = min(p_per, nsb - sb0), tr0 = (int)blockIdx.y * SEGS, rows_here = min(SEGS, p_rows - tr0);
    const int n_i = (here - wave + SK_WAVES - 1) / SK_WAVES;
    const size_t row_stride = (size_t)nsb * TB;
    auto tile_ptr = [&](int ii, int seg) { return p_w + (size_t)(tr0 + (seg < rows_here ? seg : 0)) * row_stride + (size_t)(sb0 + wave + SK_WAVES * ii) * TB; };
    f4_t D[SEGS][NC];
    SkinnyWalk<TYPE, SEGS, NC> walk(p_x + (size_t)(sb0 + wave) * (QK_K * 16), (unsigned)SK_WAVES * (QK_K * 16), (unsigned)SK_NT * p_K, n_i, lane, g, 4 * (4 * m + g),
                                    SkinnyColumns<TYPE, NC>(m, g, p_T));
    walk.start(D, n_i > 0, tile_ptr);
    if (n_i > 0) walk.run(D, tile_ptr);
    // D[seg] holds row m, columns 4 g .. 4 g + 3 of segment seg
#pragma unroll
    for (int seg = 0; seg < SEGS; ++seg)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[((size_t)(wave * SEGS + seg) * NT + SK_NT * c + 4 * g + i) * 16 + m] = D[seg][c][i];
    __syncthreads();
    float *part = p_part + (size_t)blockIdx.x * p_T * p_ld;
    for (int i = tid; i < SEGS * NT * 4; i += SK_THREADS) {
        const int r4 = i & 3, seg = (i >> 2) % SEGS, t = (i >> 2) / SEGS;
        if (t >= p_T || seg >= rows_here) continue;
        f4_t v = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < SK_WAVES; ++w) v += *reinterpret_cast<const f4_t *>(red + ((size_t)(w * SEGS + seg) * NT + t) * 16 + 4 * r4);
        *reinterpret_cast<f4_t *>(part + (size_t)t * p_ld + (tr0 + seg) * TILE_ROWS + 4 * r4) = v;
    }
}

template <int TYPE, int NU, int SEGS, int NC>
static int launch_skinny(const SkinnyKernelArgs &ka, int grid, size_t smem, hipStream_t stream) {
    static bool attr_set = false;
    if (!attr_set) {
        MESH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_skinny_kernel<TYPE, NU, SEGS, NC>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)SK_LDS_LIMIT));
        attr_set = true;
    }
    MESH_LAUNCH((gemm_skinny_kernel<TYPE, NU, SEGS, NC>), dim3((unsigned)grid), dim3(SK_THREADS), smem, stream, ka.x, ka.wbase[0], ka.wbase[1] ? ka.wbase[1] : ka.wbase[0],
                ka.wbase[2] ? ka.wbase[2] : ka.wbase[0], ka.K, ka.ks | ka.T << 16, ka.tile_begin[3], (unsigned)ka.tile_begin[1] | ((unsigned)ka.tile_begin[2] << 16),
                (unsigned)(ka.tile_begin[3] / grid) | ((unsigned)(ka.tile_begin[3] % grid) << 16), ka);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

template <int TYPE, int NU, int NC>
static int launch_skinny_segs(int segs, const SkinnyKernelArgs &ka, int grid, size_t smem, hipStream_t stream) {
    if (segs <= 1) return launch_skinny<TYPE, NU, NU, NC>(ka, grid, smem, stream);   // NU == 2 needs two segments at least
    if (segs <= 2) return launch_skinny<TYPE, NU, 2, NC>(ka, grid, smem, stream);
    return launch_skinny<TYPE, NU, 4, NC>(ka, grid, smem, stream);
}
template <int TYPE, int NU>
static int launch_skinny_cols(int nc, int segs, const SkinnyKernelArgs &ka, int grid, size_t smem, hipStream_t stream) {
    return nc == 2 ? launch_skinny_segs<TYPE, NU, 2>(segs, ka, grid, smem, stream) : launch_skinny_segs<TYPE, NU, 1>(segs, ka, grid, smem, stream);
}

static int skinny_n_cu() {
    static int n = 0;
    if (!n) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) n = p.multiProcessorCount;
        if (n <= 0) n = 256;
    }
    return n;
}

// waves along K: a power of two (the kernel splits its waves with shifts)
static int skinny_ks(int nsb) {
    int KS = 1;
    while (KS * 2 <= nsb && KS * 2 <= SK_WAVES) KS *= 2;
    return KS;
}
// workgroups of a launch over total_rows tile-rows: spread over the CUs, bounded by the segments a wave can hold
static int skinny_grid(int total_rows, int NU, int KS) {
    const int RS = SK_WAVES / KS;
    const int rows_cap = std::max(1, SK_SEGS_MAX / NU) * RS;
    const int ncu = skinny_n_cu();
    int rows_per_wg = std::min((total_rows + ncu - 1) / ncu, rows_cap);
    rows_per_wg = std::max(1, rows_per_wg);
    return (total_rows + rows_per_wg - 1) / rows_per_wg;
}

// What a launch over the matrices of `a` (tiled K-quants of one type) needs, before the token chunk is chosen
struct SkinnyLaunch {
    SkinnyKernelArgs ka;
    int type, NU, KS, total_rows, grid, rows_max, segs;
    size_t smem(int nt) const { return sizeof(float) * ((size_t)KS * rows_max * NU * 16 * nt + 2 * (size_t)SK_WAVES * nt + (size_t)SKINNY_F16_NORM_PARTS_MAX * nt); }
};
static int skinny_prepare(const SkinnyF16Args &a, SkinnyLaunch &L) {
    L.type = a.mat[0].type;
    const int nsb = a.K / QK_K, NU = a.epi == EPI_SWIGLU ? 2 : 1;
    L.NU = NU;
    const size_t row_stride = (size_t)nsb * (L.type == MESH_Q4_K ? Q4K_TILE_BYTES : Q6K_TILE_BYTES);
    SkinnyKernelArgs &ka = L.ka;
    ka = SkinnyKernelArgs{};
    int total_rows = 0;
    for (int i = 0; i < a.n_mat; ++i) {
        const int begin = (NU == 2 && i == 1) ? 0 : total_rows;     // gate and up share tile-row indices
        ka.tile_begin[i] = begin;
        ka.wbase[i] = static_cast<const uint8_t *>(a.mat[i].W) - (size_t)begin * row_stride;
        ka.y[i] = a.mat[i].y;
        ka.bias[i] = a.mat[i].bias;
        ka.M[i] = a.mat[i].M;
        ka.ldy[i] = a.mat[i].ldy;
        ka.kind[i] = a.kind[i];
        if (!(NU == 2 && i == 1)) total_rows += (a.mat[i].M + TILE_ROWS - 1) / TILE_ROWS;
    }
    const int n_bound = NU == 2 ? 1 : a.n_mat;          // matrix boundaries the kernel searches
    for (int i = n_bound; i < 4; ++i) ka.tile_begin[i] = total_rows;
    ka.K = a.K;
    ka.ldres = a.ldres; ka.epi = a.epi;
    ka.rope = a.rope;
    ka.M16 = a.mat[0].M;
    ka.sat = a.sat;
    ka.no_w = a.norm_out.norm_w; ka.no_x16 = a.norm_out.x16; ka.no_part = a.norm_out.part;
    ka.ni_part = a.norm_in.part; ka.ni_parts = a.norm_in.n_parts; ka.ni_eps = a.norm_in.eps;
    L.KS = skinny_ks(nsb);
    const int RS = SK_WAVES / L.KS;
    ka.ks = L.KS;
    L.total_rows = total_rows;
    if (total_rows > 0xFFFF) return fail(MESH_ERR_UNSUPPORTED, "gemm_skinny_f16: %d tile-rows in one launch", total_rows);
    L.grid = skinny_grid(total_rows, NU, L.KS);
    L.rows_max = (total_rows + L.grid - 1) / L.grid;
    L.segs = ((L.rows_max + RS - 1) / RS) * NU;         // per wave
    if (L.segs > SK_SEGS_MAX) return fail(MESH_ERR_UNSUPPORTED, "gemm_skinny_f16: %d segments per wave", L.segs);
    return MESH_OK;
}
// the kernel arguments of the launch for columns t .. t + nt - 1 of the call
static SkinnyKernelArgs skinny_chunk(const SkinnyF16Args &a, const SkinnyLaunch &L, int t, int nt) {
    SkinnyKernelArgs kb = L.ka;
    kb.T = std::min(nt, a.T - t);
    if (kb.rope.pos) { kb.rope.pos += t; kb.rope.seq += t; }
    kb.x = a.x + (size_t)t * a.K;                  // block t / 16 of the k8-major activations
    kb.residual = a.residual ? a.residual + (size_t)t * a.ldres : nullptr;
    kb.y16 = a.y16 ? a.y16 + (size_t)t * a.mat[0].M : nullptr;
    for (int i = 0; i < a.n_mat; ++i)
        if (kb.y[i]) kb.y[i] = a.mat[i].y + (size_t)t * a.mat[i].ldy;
    return kb;
}

// all matrices of `a` are tiled K-quants of one type
static int skinny_one_type(const SkinnyF16Args &a, hipStream_t stream) {
    SkinnyLaunch L;
    int rc = skinny_prepare(a, L);
    if (rc != MESH_OK) return rc;
    // a pass over the weights takes 32 columns while more than 16 remain, else 16 (a call of up to 32 tokens is one launch)
    for (int t = 0; t < a.T;) {
        const int nc = a.T - t > SK_NT ? 2 : 1, nt = nc * SK_NT;
        const size_t smem = L.smem(nt);
        if (smem > SK_LDS_LIMIT) return fail(MESH_ERR_UNSUPPORTED, "gemm_skinny_f16: reduction buffer of %zu bytes does not fit LDS", smem);
        const SkinnyKernelArgs kb = skinny_chunk(a, L, t, nt);
        if (L.type == MESH_Q4_K) rc = L.NU == 2 ? launch_skinny_cols<MESH_Q4_K, 2>(nc, L.segs, kb, L.grid, smem, stream) : launch_skinny_cols<MESH_Q4_K, 1>(nc, L.segs, kb, L.grid, smem, stream);
        else rc = L.NU == 2 ? launch_skinny_cols<MESH_Q6_K, 2>(nc, L.segs, kb, L.grid, smem, stream) : launch_skinny_cols<MESH_Q6_K, 1>(nc, L.segs, kb, L.grid, smem, stream);
        if (rc != MESH_OK) return rc;
        t += nt;
    }
    return MESH_OK;
}

template <int SEGS_A, int SEGS_B, int NC>
static int launch_pair(const SkinnyKernelArgs &ka, const SkinnyKernelArgs &kb, int grid_a, int grid_b, size_t smem, hipStream_t stream) {
    static bool attr_set = false;
    if (!attr_set) {
        MESH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_skinny_pair_kernel<SEGS_A, SEGS_B, NC>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)SK_LDS_LIMIT));
        attr_set = true;
    }
    MESH_LAUNCH((gemm_skinny_pair_kernel<SEGS_A, SEGS_B, NC>), dim3((unsigned)(grid_a + grid_b)), dim3(SK_THREADS), smem, stream, ka.x, ka.wbase[0],
                ka.wbase[1] ? ka.wbase[1] : ka.wbase[0], ka.K, ka.ks | ka.T << 16, grid_a, (unsigned)ka.tile_begin[1] | ((unsigned)ka.tile_begin[2] << 16),
                (unsigned)(ka.tile_begin[3] / grid_a) | ((unsigned)(ka.tile_begin[3] % grid_a) << 16),
                (unsigned)(kb.tile_begin[3] / grid_b) | ((unsigned)(kb.tile_begin[3] % grid_b) << 16), kb.wbase[0], ka, kb);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}
template <int NC>
static int launch_pair_segs(int segs_a, int segs_b, const SkinnyKernelArgs &ka, const SkinnyKernelArgs &kb, int grid_a, int grid_b, size_t smem, hipStream_t stream) {
    const int sa = segs_a <= 1 ? 1 : segs_a <= 2 ? 2 : 4;
    if (segs_b <= 1) {
        if (sa == 1) return launch_pair<1, 1, NC>(ka, kb, grid_a, grid_b, smem, stream);
        if (sa == 2) return launch_pair<2, 1, NC>(ka, kb, grid_a, grid_b, smem, stream);
        return launch_pair<4, 1, NC>(ka, kb, grid_a, grid_b, smem, stream);
    }
    if (sa == 1) return launch_pair<1, 2, NC>(ka, kb, grid_a, grid_b, smem, stream);
    if (sa == 2) return launch_pair<2, 2, NC>(ka, kb, grid_a, grid_b, smem, stream);
    return launch_pair<4, 2, NC>(ka, kb, grid_a, grid_b, smem, stream);
}

// `qa`: one or two q4_K matrices, `qb`: one q6_K matrix, same activations, plain-store epilogues (with or without RoPE):
// one launch whose first workgroups are qa's and whose last are qb's.  MESH_ERR_UNSUPPORTED when the shapes do not fit
// (the caller then launches them one after the other).
static int skinny_pair(const SkinnyF16Args &qa, const SkinnyF16Args &qb, hipStream_t stream) {
    SkinnyLaunch A, B;
    int rc = skinny_prepare(qa, A);
    if (rc != MESH_OK) return rc;
    if ((rc = skinny_prepare(qb, B)) != MESH_OK) return rc;
    if (B.segs > 2 || A.KS != B.KS) return MESH_ERR_UNSUPPORTED;
    for (int t = 0; t < qa.T;) {
        const int nc = qa.T - t > SK_NT ? 2 : 1, nt = nc * SK_NT;
        const size_t smem = std::max(A.smem(nt), B.smem(nt));
        if (smem > SK_LDS_LIMIT) return MESH_ERR_UNSUPPORTED;
        const SkinnyKernelArgs ka = skinny_chunk(qa, A, t, nt), kb = skinny_chunk(qb, B, t, nt);
        rc = nc == 2 ? launch_pair_segs<2>(A.segs, B.segs, ka, kb, A.grid, B.grid, smem, stream) : launch_pair_segs<1>(A.segs, B.segs, ka, kb, A.grid, B.grid, smem, stream);
        if (rc != MESH_OK) return rc;
        t += nt;
    }
    return MESH_OK;
}

// ---- cut along K
constexpr int SLICE_SEGS_MAX = 5;
struct SlicePlan { int segs, slices, per; };
template <int TYPE, int SEGS, int NC>
static int launch_slice(const SkinnyF16Args &a, const SlicePlan &p, float *part, hipStream_t stream) {
    constexpr size_t smem = sizeof(float) * SK_WAVES * SEGS * SK_NT * NC * 16;
    static_assert(smem <= SK_LDS_LIMIT, "sums of a workgroup");
    static bool attr_set = false;
    if (!attr_set) {
        MESH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_skinny_slice_kernel<TYPE, SEGS, NC>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)SK_LDS_LIMIT));
        attr_set = true;
    }
    const int rows = (a.mat[0].M + TILE_ROWS - 1) / TILE_ROWS;
    MESH_LAUNCH((gemm_skinny_slice_kernel<TYPE, SEGS, NC>), dim3((unsigned)p.slices, (unsigned)((rows + SEGS - 1) / SEGS)), dim3(SK_THREADS), smem, stream, a.x,
                static_cast<const uint8_t *>(a.mat[0].W), a.K, a.T, rows, p.per, (a.mat[0].M + 127) / 128 * 128, part);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}
template <int TYPE, int NC>
static int launch_slice_segs(const SkinnyF16Args &a, const SlicePlan &p, float *part, hipStream_t stream) {
    return p.segs == 3 ? launch_slice<TYPE, 3, NC>(a, p, part, stream) : p.segs == 4 ? launch_slice<TYPE, 4, NC>(a, p, part, stream) : launch_slice<TYPE, 5, NC>(a, p, part, stream);
}
// Whether a launch is cut, and how: groups of three to five tile-rows by two to four slices, as many workgroups as the CUs take at once.  For
// launches that leave a quarter of the CUs idle otherwise, if no wave multiplies more tiles than before.  A workgroup of several rows
// reads its slice's activations once for all of them (5120 x 27648 at 32 tokens: 0.44 MB a workgroup instead of 1.8); what is paid is the
// launch that adds the slices, 2 to 4 us, which also writes the next norm's rows.
// Cut / whole, us a layer less, 24 tokens: 5120 x 27648 (160 workgroups of two rows, 28 tiles a wave) five rows by four 15.5, four by three 10.5,
// three by two 9.4; 5120 x 13824 2.3 and 3.1 (three by two); 3072 x 8192 three by four 1.8; 2048 x 16384 three by four 3.2; 2560 x 10240 (no
// such cut) 0.1 at the best; with more workgroups to begin with 4096 x 14336 0, 3584 x 18944 2.  Up to 16 tokens there is half as much to
// read: 3072 x 8192 0.5, 2048 x 16384 -0.7; rows of 5120 by tiles a wave, 4 / 8 / 16 tokens: 14 -1.2 -1.5 -0.8, 16 -0.9 -0.6 0.0, 18 0.1 -0.2 1.4,
// 20 0.6 0.8 2.3, 22 -0.6 -0.7 1.6, 24 0.4 0.4 2.5, 26 1.9 1.8 4.4, 28 2.1 2.6 5.3: from 24 on it gains at every count (9 to 16 tokens alone would
// from 18 on).
static SlicePlan slice_plan(const SkinnyF16Args &a, size_t part_bytes) {
    const SlicePlan whole{1, 1, 0};
    const GemvMat &w = a.mat[0];
    if (a.n_mat != 1 || a.epi != EPI_RESIDUAL || a.y16 || a.rope.pos || w.bias || a.T > 2 * SK_NT || a.K % QK_K || w.M % 8 || w.ldy % 4 || a.ldres % 4) return whole;
    const int nsb = a.K / QK_K, rows = (w.M + TILE_ROWS - 1) / TILE_ROWS, ncu = skinny_n_cu(), ks = skinny_ks(nsb), grid = skinny_grid(rows, 1, ks);
    const int tiles = (rows + grid - 1) / grid * ((nsb + ks - 1) / ks);
    if (ks != SK_WAVES || 4 * grid > 3 * ncu || (a.T <= SK_NT && tiles < 24)) return whole;
    SlicePlan best = whole;
    int most = grid;
    for (int segs = 3; segs <= SLICE_SEGS_MAX; ++segs)
        for (int slices = 2; slices <= 4; ++slices) {
            const int per = (nsb + slices - 1) / slices, n = (nsb + per - 1) / per, wgs = (rows + segs - 1) / segs * n;
            if (wgs > ncu || wgs <= most || segs * ((per + SK_WAVES - 1) / SK_WAVES) > tiles) continue;
            if ((size_t)n * a.T * ((w.M + 127) / 128 * 128) * sizeof(float) > part_bytes) continue;
            most = wgs;
            best = SlicePlan{segs, n, per};
        }
    return best;
}

}  // namespace f16sk

int gemm_skinny_f16_workgroups(const SkinnyF16Args &a) {
    using namespace f16sk;
    if (a.n_mat != 1 || a.K <= 0 || a.K % QK_K || a.mat[0].M <= 0) return 0;
    return skinny_grid((a.mat[0].M + TILE_ROWS - 1) / TILE_ROWS, 1, skinny_ks(a.K / QK_K));
}

int gemm_skinny_f16_slices(const SkinnyF16Args &a, size_t part_bytes) { return f16sk::slice_plan(a, part_bytes).slices; }

int gemm_skinny_f16_sliced(const SkinnyF16Args &a, const GemmArgs &sum, hipStream_t stream) {
    using namespace f16sk;
    const SlicePlan p = sum.part ? slice_plan(a, sum.part_bytes) : SlicePlan{1, 1, 0};
    if (p.slices <= 1 || !a.x || (reinterpret_cast<uintptr_t>(a.x) & 15) || !a.mat[0].W || !a.mat[0].y || !a.residual || a.T <= 0 || !type_is_tiled(a.mat[0].type) ||
        (sum.next_x16 && a.mat[0].M > GEMM_NORM_ROW_MAX))
        return fail(MESH_ERR_INVALID, "gemm_skinny_f16_sliced: a launch it does not fit");
    GemmArgs k = sum;
    k.M = a.mat[0].M; k.K = a.K; k.T = a.T; k.Y = a.mat[0].y; k.ldy = a.mat[0].ldy; k.residual = a.residual; k.ldres = a.ldres;
    k.ksplit = p.slices;
    const bool two = a.T > SK_NT;
    const int rc = a.mat[0].type == MESH_Q4_K ? (two ? launch_slice_segs<MESH_Q4_K, 2>(a, p, sum.part, stream) : launch_slice_segs<MESH_Q4_K, 1>(a, p, sum.part, stream))
                                              : (two ? launch_slice_segs<MESH_Q6_K, 2>(a, p, sum.part, stream) : launch_slice_segs<MESH_Q6_K, 1>(a, p, sum.part, stream));
    return rc != MESH_OK ? rc : gemm_add_slices(k, (k.M + 127) / 128, stream);
}

int gemm_skinny_f16(const SkinnyF16Args &a, hipStream_t stream) {
    using namespace f16sk;
    if (a.norm_out.x16 || a.norm_out.part || a.norm_out.norm_w) {
        if (!a.norm_out.x16 || !a.norm_out.part || !a.norm_out.norm_w || a.n_mat != 1 || a.epi != EPI_RESIDUAL || a.T > SKINNY_F16_NORM_TOKENS_MAX || a.mat[0].M % 8 ||
            gemm_skinny_f16_workgroups(a) > SKINNY_F16_NORM_PARTS_MAX)
            return fail(MESH_ERR_INVALID, "gemm_skinny_f16: the norm hand-over needs one matrix with a residual epilogue, at most 32 tokens and a row count that is a multiple of 8");
    }
    if (a.norm_in.part && (a.norm_in.n_parts < 1 || a.norm_in.n_parts > SKINNY_F16_NORM_PARTS_MAX || a.T > SKINNY_F16_NORM_TOKENS_MAX))
        return fail(MESH_ERR_INVALID, "gemm_skinny_f16: bad norm hand-over input (%d partial sums, %d tokens)", a.norm_in.n_parts, a.T);
    if (a.n_mat < 1 || a.n_mat > 3 || !a.x || a.T <= 0 || a.K <= 0) return fail(MESH_ERR_INVALID, "gemm_skinny_f16: bad arguments");
    if (a.K % QK_K || (reinterpret_cast<uintptr_t>(a.x) & 15))
        return fail(MESH_ERR_INVALID, "gemm_skinny_f16: K %d must be a multiple of 256 and the activations 16-byte aligned", a.K);
    if (a.y16 && a.mat[0].M % 8) return fail(MESH_ERR_INVALID, "gemm_skinny_f16: f16 output needs a row count that is a multiple of 8");
    if (a.epi == EPI_SWIGLU && (a.n_mat != 2 || a.mat[0].M != a.mat[1].M || a.mat[0].type != a.mat[1].type))
        return fail(MESH_ERR_INVALID, "gemm_skinny_f16: SwiGLU needs a gate and an up matrix of equal shape and type");
    if (a.epi == EPI_RESIDUAL && !a.residual) return fail(MESH_ERR_INVALID, "gemm_skinny_f16: residual epilogue without residual");
    if (a.rope.pos && (a.epi != EPI_STORE || a.rope.head_dim % 2 || a.rope.n_rot % 2)) return fail(MESH_ERR_INVALID, "gemm_skinny_f16: rope epilogue needs a plain store");
    for (int i = 0; i < a.n_mat; ++i) {
        if (!a.mat[i].W || a.mat[i].M <= 0 || !type_is_tiled(a.mat[i].type)) return fail(MESH_ERR_INVALID, "gemm_skinny_f16: matrix %d is not a tiled K-quant", i);
        if (!a.mat[i].y && !(i == 1 && a.epi == EPI_SWIGLU) && !(i == 0 && a.y16)) return fail(MESH_ERR_INVALID, "gemm_skinny_f16: matrix %d has no output", i);
    }
    bool same = true;
    for (int i = 1; i < a.n_mat; ++i) same = same && a.mat[i].type == a.mat[0].type;
    if (same) return skinny_one_type(a, stream);
    // mixed types (q/k in q4_K, v in q6_K): q4_K matrices followed by one q6_K matrix share a launch ...
    if (a.pair_launch && a.epi == EPI_STORE && !a.y16 && a.mat[a.n_mat - 1].type == MESH_Q6_K) {
        bool lead_q4 = true;
        for (int k2 = 0; k2 + 1 < a.n_mat; ++k2) lead_q4 = lead_q4 && a.mat[k2].type == MESH_Q4_K;
        if (lead_q4) {
            SkinnyF16Args qa = a, qb = a;
            qa.n_mat = a.n_mat - 1;
            qb.n_mat = 1;
            qb.mat[0] = a.mat[a.n_mat - 1]; qb.kind[0] = a.kind[a.n_mat - 1];
            const int rc = skinny_pair(qa, qb, stream);
            if (rc != MESH_ERR_UNSUPPORTED) return rc;
        }
    }
    // ... anything else: one launch per run of equal type
    int i = 0;
    while (i < a.n_mat) {
        int j = i + 1;
        while (j < a.n_mat && a.mat[j].type == a.mat[i].type) ++j;
        SkinnyF16Args sub = a;
        sub.n_mat = j - i;
        for (int k2 = 0; k2 < sub.n_mat; ++k2) { sub.mat[k2] = a.mat[i + k2]; sub.kind[k2] = a.kind[i + k2]; }
        sub.y16 = i == 0 ? a.y16 : nullptr;
        int rc = skinny_one_type(sub, stream);
        if (rc != MESH_OK) return rc;
        i = j;
    }
    return MESH_OK;
}

}  // namespace mesh
