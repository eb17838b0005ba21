// Causal GQA attention for a prefill chunk on the matrix cores (head_dim 64 or 128, written below for 128; f16 or quantised KV cache rows, which
// are dequantised to f16 on their way into LDS).
//
// The chunk is T consecutive positions pos0 .. pos0 + T - 1 of one sequence whose keys and values are already in
// the cache (rope_kv appended them); token t attends to cache positions [0, pos0 + t], or to the last `window` of them
// (a workgroup then starts its walk at the first key its first query sees).  A workgroup takes 32
// queries of every head of one KV-head group (one wave per head), walks the keys in tiles of 32 and keeps the
// running softmax in registers:
//   S^T = K . Q^T        (32 keys x 32 queries, v_mfma_f32_32x32x16_f16 over the 128 dims)
//   O^T += V^T . P^T     (128 dims x 32 queries, contraction over the 32 keys)
// Both products are arranged transposed so that a lane owns ONE query column: the softmax maximum and sum of a
// query are reductions over the lane's own 16 registers plus one cross-half shuffle, and the rescale of O is a
// per-lane scalar.  K and V tiles are staged once per workgroup in LDS (all heads of the group share them), as rows; the
// contraction index (keys) has to be contiguous in an MFMA operand, so V is read back with ds_read_b64_tr_b16, which
// transposes.  f16 rows go from memory to LDS without passing registers, into the buffer the step before has left: the
// loads of a step have the whole step before it to arrive, and a step costs one barrier.
// The MFMA k-slots of the second product are the lane's own S^T registers, in the order the hardware leaves them:
// slot (half, j) of the first MFMA is key 4*half + j (j < 4) or 8 + 4*half + j - 4; the V^T operand is read from LDS
// with the same key order, so no data moves between lanes.
//
// What bounds it: a step of a wave is 32 MFMAs of 32 cycles and ~180 vector instructions with 33 exponentials (~1 200 cycles), two waves
// to a SIMD.  Llama-3-8B shape, a layer: 2048 tokens 78.7 -> 59.3 us (padded tiles with V transposed on the way in, two barriers a step,
// four waves a workgroup; of that 74 with rows by direct loads, 63 with two key groups, the rest by the order of pieces and addresses
// that are constants), 333 tokens behind 1500 36.7 -> 29.5; expert shard 600 tokens 24.2 -> 19.6.
//
// Same result as the per-token kernel of attn.hip (ggml's soft_max + mul_mat of the attention block, reached from
// rpc_server::graph_compute, third_party/llama.cpp/patches/0002-rpc-add-direct-peer-tensor-transfers.patch:443-451)
// except that Q and the probabilities are rounded to f16 for the matrix cores; sums are f32.

#include <algorithm>
#include <type_traits>

#include "act_math.hpp"
#include "attn.hpp"
#include "lds_ops.hpp"
#include "wave_ops.hpp"

namespace mesh {

constexpr int PF_TILE = 32;                 // queries per workgroup

// Rows of a tile lie in LDS without padding (a load to LDS writes 1 KB in one piece), the 16-byte pieces of row r in the order
// piece ^ pf_swizzle(r): equal pieces of the 16 rows that a read of K touches at once, and equal 64-byte runs of the 4 rows that a
// transposing read touches, lie on different banks.  (Rows of 128 halfs all start on bank 0, rows of 64 and 192 on 0 and 32 in turn.)
template <int D> __host__ __device__ constexpr int pf_swizzle(int row) { return D == 128 ? (row & 3) << 2 | (row >> 2 & 3) : (row & 2) << 1 | (row >> 2 & 3); }
constexpr int PF_TWO_GROUPS_WALK = 320;      // two groups of waves share walks of more keys than this
constexpr int PF_EXPAND_HD = 128;            // kv_expand_kernel's head_dim
constexpr int PF_EXPAND_MIN_T = 128;         // chunks from this many tokens decode a quantised cache to f16 once, ahead of the walk
constexpr float PF_RESCALE_STEP = 8.f;      // the softmax reference moves only when the running maximum exceeds it by this (log2)

typedef _Float16 pf_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 pf_h2 __attribute__((ext_vector_type(2)));
typedef float pf_f16v __attribute__((ext_vector_type(16)));
typedef uint32_t pf_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void pf_step_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#endif
}

__device__ __forceinline__ uint32_t pf_pack(float a, float b) {
    const pf_h2 h = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, h);
}

// the 8 values a (key, piece) pair contributes to a tile, as packed f16
template <int TYPE>
__device__ __forceinline__ uint4 pf_decode(const KvRaw<TYPE> &r) {
    if constexpr (TYPE == MESH_F16) {
        return r.v;
    } else {
        float u[8];
        const float d = kv_decode<TYPE>(r, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = (u[e] - KvAffine<TYPE>::off) * d;
        return make_uint4(pf_pack(u[0], u[1]), pf_pack(u[2], u[3]), pf_pack(u[4], u[5]), pf_pack(u[6], u[7]));
    }
}
template <int TYPE, int HD>
__device__ __forceinline__ uint4 pf_row_piece(const uint8_t *row, int piece) { return pf_decode<TYPE>(kv_load<TYPE, HD>(row, piece * 8)); }

// HD, VD: entries of a key and of a value row.  NP: KB of a step's keys (and at most as many of its values) that a wave brings, at least
// HD / 8 / (waves of the workgroup); for quantised rows (key, 8-dim piece) pairs of a thread, which are as many.
template <int HD, int VD, int KT, int VT, int NP, int KG>
__global__ __launch_bounds__(512) void attn_chunk_kernel(const AttnArgs a, int T, int pos0, int seq, int hpw, int qtiles, int n_ksplit) {
    constexpr int KRB = kv_row_bytes(KT, HD), VRB = kv_row_bytes(VT, VD);
    constexpr int PIECES = HD / 8, VPIECES = VD / 8;      // 8-dim pieces of a row
    constexpr int NKC = HD / 16, NDB = VD / 32;     // steps of the score product along the dims, 32-dim blocks of the output
    constexpr int NT = 2;                           // tiles of 32 keys per step: two independent score chains
    constexpr int PF_KEYS = 32 * NT;                // keys per step
    constexpr bool DIRECT = KT == MESH_F16 && VT == MESH_F16;
    static_assert(!DIRECT || (KRB == HD * 2 && VRB == VD * 2), "f16 rows without gaps");
    constexpr int PF_STAGE = PF_KEYS * KG;          // keys brought at a time
    __shared__ __align__(16) _Float16 sK[2][PF_STAGE * HD];
    __shared__ __align__(16) _Float16 sV[2][PF_STAGE * VD];
    const int tid = threadIdx.x, lane = tid & 63, nthreads = blockDim.x;
    // wave -> (head of the workgroup, one of its `qtiles` consecutive query tiles): groups of fewer than four heads fill the
    // workgroup with several query tiles of the same heads, which share the K / V tiles like heads do
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), n_waves = nthreads >> 6, own = wv % (hpw * qtiles), kg = wv / (hpw * qtiles);
    const int wave = own % hpw, qtl = own / hpw;
    const int qcol = lane & 31, half = lane >> 5;
    // the last query tile of a chunk walks the most keys: the launch hands the tiles out from the last one backwards, so
    // that the longest walks start first when the workgroups do not all fit on the chip at once
    const int lin = (int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)), across = (int)(gridDim.y * gridDim.z);
    const int qg = (int)gridDim.x - 1 - (KG > 1 ? lin / across : (int)blockIdx.x);
    const int kvh = KG > 1 ? lin % across % (int)gridDim.y : (int)blockIdx.y, bz = KG > 1 ? lin % across / (int)gridDim.y : (int)blockIdx.z;
    const int qt = qg * qtiles + qtl;           // (past the last tile of the chunk: a wave without queries, q_live false)
    // bz = (head group, key split): with n_ksplit > 1 the workgroup walks one n_ksplit-th of the keys and leaves
    // an un-normalised partial for attn_combine_kernel (short chunks on a long history, which have few query tiles)
    const int ks = bz % n_ksplit;
    const int h = kvh * a.group + (bz / n_ksplit) * hpw + wave;
    const int tq = qt * PF_TILE + qcol;
    const bool q_live = tq < T;
    const int pos_q = pos0 + tq;
    const int win_lo = a.window > 0 ? pos_q - a.window : -1;      // keys up to this one are out of the query's sight

    // Q^T fragments of this lane's query, scaled so that the scores are in log2 units
    const float qs = a.scale * 1.44269504088896341f;
    pf_h8 qf[NKC];
    {
        const float *qp = a.q + ((size_t)(q_live ? tq : 0) * a.n_head + h) * HD + 8 * half;
#pragma unroll
        for (int kc = 0; kc < NKC; ++kc) {
            const float4 v0 = *reinterpret_cast<const float4 *>(qp + kc * 16), v1 = *reinterpret_cast<const float4 *>(qp + kc * 16 + 4);
            const float z = q_live ? qs : 0.f;
            const pf_u4 p = {pf_pack(v0.x * z, v0.y * z), pf_pack(v0.z * z, v0.w * z), pf_pack(v1.x * z, v1.y * z), pf_pack(v1.z * z, v1.w * z)};
            qf[kc] = __builtin_bit_cast(pf_h8, p);
        }
    }
    pf_f16v o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    float m = -INFINITY, l = 0.f;

    const size_t base = ((size_t)seq * a.n_kv + kvh) * a.n_ctx;
    const int q_end = qt * PF_TILE + PF_TILE < T ? qt * PF_TILE + PF_TILE : T;      // queries of this tile: [qt*32, q_end)
    const int n_keys_own = qt * PF_TILE < T ? pos0 + q_end : 0;                     // keys any of them may see
    const int wg_end = (qg + 1) * qtiles * PF_TILE < T ? (qg + 1) * qtiles * PF_TILE : T;
    const int n_keys_wg = pos0 + wg_end;                                            // keys the workgroup's last tile walks
    // keys before the window of the workgroup's (and of this wave's) first query are not walked
    const int wg_first = a.window > 0 ? (pos0 + qg * qtiles * PF_TILE - a.window + 1 > 0 ? (pos0 + qg * qtiles * PF_TILE - a.window + 1) & ~(PF_KEYS - 1) : 0) : 0;
    const int own_first = a.window > 0 ? pos0 + qt * PF_TILE - a.window + 1 : 0;
    const int full_from = a.window > 0 ? pos0 + qt * PF_TILE + PF_TILE - a.window : 0;     // from this key on, inside every query's window
    const int per_split = (((n_keys_wg - wg_first + n_ksplit - 1) / n_ksplit) + 63) & ~63;
    const int k_lo = wg_first + ks * per_split;
    const int n_keys = k_lo + per_split < n_keys_wg ? k_lo + per_split : n_keys_wg;   // end of this workgroup's walk
    const int n_keys_mine = n_keys_own < n_keys ? n_keys_own : n_keys;              // and of this wave's
    // Staging.  Rows past the context end are clamped (masked below).
    const uint8_t *const k_rows = a.kcache + base * KRB, *const v_rows = a.vcache + base * VRB;
    auto row_of = [&](int key) { return (uint32_t)(key < a.n_ctx ? key : a.n_ctx - 1); };
    // f16: a wave brings every n_waves-th KB of the tiles
    auto bring = [&](int k0, int buf) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int kb = wv + i * n_waves, at = kb * 64 + lane, row = at / PIECES, piece = (at % PIECES) ^ pf_swizzle<HD>(row);
            if (kb < PF_STAGE * HD / 512) load_to_lds_16(k_rows, row_of(k0 + row) * KRB + piece * 16, lds_place(sK[buf] + kb * 512));
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int kb = wv + i * n_waves, at = kb * 64 + lane, row = at / VPIECES, piece = (at % VPIECES) ^ pf_swizzle<VD>(row);
            if (kb < PF_STAGE * VD / 512) load_to_lds_16(v_rows, row_of(k0 + row) * VRB + piece * 16, lds_place(sV[buf] + kb * 512));
        }
    };
    // quantised rows travel through registers: requested ahead of a step's products, decoded and written behind them
    KvRaw<KT> rk[DIRECT ? 1 : NP];
    KvRaw<VT> rv[DIRECT ? 1 : NP];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = tid + i * nthreads;
            if (p < PF_STAGE * PIECES) rk[i] = kv_load<KT, HD>(k_rows + (size_t)row_of(k0 + p / PIECES) * KRB, p % PIECES * 8);
            if (p < PF_STAGE * VPIECES) rv[i] = kv_load<VT, VD>(v_rows + (size_t)row_of(k0 + p / VPIECES) * VRB, p % VPIECES * 8);
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int p = tid + i * nthreads;
            if (p < PF_STAGE * PIECES) *reinterpret_cast<uint4 *>(sK[buf] + (p / PIECES) * HD + ((p % PIECES) ^ pf_swizzle<HD>(p / PIECES)) * 8) = pf_decode<KT>(rk[i]);
            if (p < PF_STAGE * VPIECES) *reinterpret_cast<uint4 *>(sV[buf] + (p / VPIECES) * VD + ((p % VPIECES) ^ pf_swizzle<VD>(p / VPIECES)) * 8) = pf_decode<VT>(rv[i]);
        }
    };
    // V^T operand: dim 32 db + lane % 32, keys of a 32-key tile 8 quad + 4 half .. + 4 (lds_read_transposed: this lane hands in row
    // (lane % 16) / 4 of the four, 4 dims)
    const int tr_row = 4 * half + ((lane & 15) >> 2), tr_piece = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), tr_at = 4 * (lane & 1);
    if (k_lo < n_keys) {
        if constexpr (DIRECT) bring(k_lo, 0);
        else { fetch(k_lo); put(0); }
    }
    // (which buffer is known when compiling: with a switch in a register every LDS address of a step is an addition)
    auto stage = [&](int ks0, auto which) {
        constexpr int buf = decltype(which)::value;
        pf_step_barrier();          // the step's tiles are there, and every wave is done with the other buffer
        if (ks0 + PF_STAGE < n_keys) {
            if constexpr (DIRECT) bring(ks0 + PF_STAGE, buf ^ 1);
            else fetch(ks0 + PF_STAGE);
        }
        const int k0 = ks0 + kg * PF_KEYS;          // this wave's keys of the step
        const _Float16 *const tK = sK[buf] + kg * (PF_KEYS * HD), *const tV = sV[buf] + kg * (PF_KEYS * VD);
        // (an earlier query tile of the workgroup is done before the last one, and with a window starts before it)
        if (k0 < n_keys_mine && k0 + PF_KEYS > own_first) {
        // the second 32 keys of the step lie past every query of the tile at the end of the walk
        const bool two = NT == 2 && k0 + 32 < n_keys_mine;

        // S^T = K . Q^T, two tiles of 32 keys x 32 queries: lane (key row = lane % 32 of the A operand, query column =
        // lane % 32 of the result); two independent accumulation chains
        pf_f16v s[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) s[t][i] = t == 0 ? 0.f : (two ? 0.f : -INFINITY);
        if (two) {
#pragma unroll
            for (int kc = 0; kc < NKC; ++kc)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const pf_h8 kf = *reinterpret_cast<const pf_h8 *>(tK + (32 * t + qcol) * HD + ((2 * kc + half) ^ pf_swizzle<HD>(qcol)) * 8);
                    s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[kc], s[t], 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int kc = 0; kc < NKC; ++kc) {
                const pf_h8 kf = *reinterpret_cast<const pf_h8 *>(tK + qcol * HD + ((2 * kc + half) ^ pf_swizzle<HD>(qcol)) * 8);
                s[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[kc], s[0], 0, 0, 0);
            }
        }
        // register i of tile t is key k0 + 32 * t + 8 * (i / 4) + 4 * half + i % 4 for query qcol.  Only a step that
        // reaches past the first query's position, or starts before the last query's window, has anything to mask (a dead query column has q = 0 and is never stored).
        if (k0 + PF_KEYS - 1 > pos0 + qt * PF_TILE || k0 < full_from) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int key = k0 + 32 * t + 8 * (i >> 2) + 4 * half + (i & 3);
                    s[t][i] = key <= pos_q && key > win_lo ? s[t][i] : -INFINITY;
                }
        }
        float mxt[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) mxt[t] = s[t][0];
#pragma unroll
        for (int i = 1; i < 16; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) mxt[t] = fmaxf(mxt[t], s[t][i]);
        float mx = NT == 2 ? fmaxf(mxt[0], mxt[NT - 1]) : mxt[0];
        mx = lane_fold<32>(mx, LaneMax{});
        // m is the reference the exponentials are taken against.  It follows the running maximum only when that has
        // moved by more than PF_RESCALE_STEP (log2 units), so that most steps skip the rescale of the 64 accumulator
        // registers; in between p <= 2^PF_RESCALE_STEP, which f16 holds comfortably.  (Without a window key 0
        // is visible to every query, so after the first step m is finite for every live column.)
        if (__builtin_amdgcn_ballot_w64(mx > m + PF_RESCALE_STEP) != 0ull) {
            const float m_new = mx > m + PF_RESCALE_STEP ? mx : m;
            // 1 for lanes that stay, exp2(-inf) = 0 while nothing is accumulated.  A query that has seen no key yet and
            // sees none in this step either (a key split that begins inside the tile's position range) has m = m_new =
            // -inf: its l and o are still zero, and -inf - -inf must not reach them as NaN.
            const float corr = m_new == -INFINITY ? 1.f : exp2f(m - m_new);
            l *= corr;
            m = m_new;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[db][i] *= corr;
        }
        // (In a later split, or in the first steps of a windowed walk, a query may see no key at all: all its scores are -inf and so is m; the reference 0 then gives p = 0, not NaN.)
        const float mref = m == -INFINITY ? 0.f : m;
        // P^T as the B operand: the lane's own registers, 8 per MFMA
        pf_h8 pf[NT][2];
        float ps0 = 0.f, ps1 = 0.f;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float p[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) p[i] = __builtin_amdgcn_exp2f(s[t][i] - mref);  // s - m <= PF_RESCALE_STEP; far below, 0
#pragma unroll
            for (int i = 0; i < 16; i += 2) { ps0 += p[i]; ps1 += p[i + 1]; }
            const pf_u4 pu1 = {pf_pack(p[0], p[1]), pf_pack(p[2], p[3]), pf_pack(p[4], p[5]), pf_pack(p[6], p[7])};
            const pf_u4 pu2 = {pf_pack(p[8], p[9]), pf_pack(p[10], p[11]), pf_pack(p[12], p[13]), pf_pack(p[14], p[15])};
            pf[t][0] = __builtin_bit_cast(pf_h8, pu1);
            pf[t][1] = __builtin_bit_cast(pf_h8, pu2);
        }
        float ps = ps0 + ps1;
        ps = lane_fold<32>(ps, LaneAdd{});
        l += ps;
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
            // keys 8 quad + 4 half .. + 4 of tile t, quad = 0 .. 3: the order of P^T's registers
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (t == 1 && !two) break;
                lds_u2 v[4];
#pragma unroll
                for (int quad = 0; quad < 4; ++quad) {
                    const int row = 32 * t + 8 * quad + tr_row;
                    v[quad] = lds_read_transposed(tV + row * VD + ((4 * db + tr_piece) ^ pf_swizzle<VD>(row)) * 8 + tr_at);
                }
                const pf_u4 v1 = {v[0][0], v[0][1], v[1][0], v[1][1]}, v2 = {v[2][0], v[2][1], v[3][0], v[3][1]};
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pf_h8, v1), pf[t][0], o[db], 0, 0, 0);
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pf_h8, v2), pf[t][1], o[db], 0, 0, 0);
            }
        }
        }
        if constexpr (!DIRECT) {
            if (ks0 + PF_STAGE < n_keys) put(buf ^ 1);
        }
    };
    for (int ks0 = k_lo; ks0 < n_keys; ks0 += 2 * PF_STAGE) {
        stage(ks0, std::integral_constant<int, 0>{});
        if (ks0 + PF_STAGE < n_keys) stage(ks0 + PF_STAGE, std::integral_constant<int, 1>{});
    }
    if constexpr (KG > 1) {
        // the second key group's result joins the first's, through the tiles' memory
        static_assert(KG == 2 && sizeof(sK) >= 4 * 64 * (VD / 2) * sizeof(float) && sizeof(sV) >= 2 * 4 * 64 * sizeof(float), "four waves' results");
        float *const s_m = reinterpret_cast<float *>(&sV[0][0]) + own * 64 + lane, *const s_l = s_m + 4 * 64;
        float *const s_o = reinterpret_cast<float *>(&sK[0][0]) + (size_t)own * 64 * (VD / 2) + lane;
        __syncthreads();
        if (kg == 1) {
            *s_m = m;
            *s_l = l;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) s_o[(db * 16 + i) * 64] = o[db][i];
        }
        __syncthreads();
        if (kg == 1) return;
        // (a group that has seen no key has m = -inf, l = 0 and o = 0)
        const float m1 = *s_m, mm = fmaxf(m, m1), w0 = m == -INFINITY ? 0.f : exp2f(m - mm), w1 = m1 == -INFINITY ? 0.f : exp2f(m1 - mm);
        l = l * w0 + *s_l * w1;
        m = mm;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[db][i] = o[db][i] * w0 + s_o[(db * 16 + i) * 64] * w1;
    }
    if (n_ksplit > 1) {
        // un-normalised partial and (maximum, sum) of this key split, in the layout of the split-KV decode kernels
        if (q_live) {
            const size_t prow = ((size_t)tq * a.n_head + h) * n_ksplit + ks;
            float *pp = a.part + prow * VD;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4)
                    *reinterpret_cast<float4 *>(pp + db * 32 + 8 * i4 + 4 * half) =
                        make_float4(o[db][4 * i4], o[db][4 * i4 + 1], o[db][4 * i4 + 2], o[db][4 * i4 + 3]);
            if (half == 0) { a.ml[prow * 2] = m; a.ml[prow * 2 + 1] = l; }
        }
        return;
    }
    if (a.out16_k8) {
        // f16, in the k8-major layout the output projection's GEMM reads (gemm.hpp); the padding columns of the last
        // block of 16 tokens are written as zeros
        const int t_pad = (T + 15) & ~15;
        if (tq < t_pad) {
            const float inv = q_live ? 1.0f / l : 0.f;
            const size_t KK = (size_t)a.n_head * VD;
            _Float16 *ob = a.out16_k8 + (size_t)(tq >> 4) * 16 * KK + (size_t)(tq & 15) * 8;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const size_t kk = (size_t)h * VD + db * 32 + 8 * i4 + 4 * half;
                    *reinterpret_cast<uint2 *>(ob + (kk >> 3) * 128 + (kk & 7)) =
                        make_uint2(pf_pack(o[db][4 * i4] * inv, o[db][4 * i4 + 1] * inv), pf_pack(o[db][4 * i4 + 2] * inv, o[db][4 * i4 + 3] * inv));
                }
        }
    } else if (a.out_bf16) {
        if (q_live) {
            const float inv = (a.head_gate ? act_sigmoid(a.head_gate[(size_t)tq * a.gate_ld + h]) : 1.0f) / l;
            uint16_t *op = a.out_bf16 + ((size_t)tq * a.n_head + h) * VD;
            auto two16 = [&](float lo, float hi) { return (uint32_t)f32_to_bf16_bits(lo * inv) | ((uint32_t)f32_to_bf16_bits(hi * inv) << 16); };
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4)
                    *reinterpret_cast<uint2 *>(op + db * 32 + 8 * i4 + 4 * half) =
                        make_uint2(two16(o[db][4 * i4], o[db][4 * i4 + 1]), two16(o[db][4 * i4 + 2], o[db][4 * i4 + 3]));
        }
    } else if (q_live) {
        const float inv = 1.0f / l;
        float *op = a.out + ((size_t)tq * a.n_head + h) * VD;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4)
                *reinterpret_cast<float4 *>(op + db * 32 + 8 * i4 + 4 * half) =
                    make_float4(o[db][4 * i4] * inv, o[db][4 * i4 + 1] * inv, o[db][4 * i4 + 2] * inv, o[db][4 * i4 + 3] * inv);
    }
}

// Rows [0, n_keys) of one sequence's K and V, every KV head, as f16 rows [n_kv][n_ctx][128] (the values the staging
// of attn_chunk_kernel would decode): one thread per (row, 8-dim piece).
template <int KT, int VT>
__global__ __launch_bounds__(256) void kv_expand_kernel(const uint8_t *kcache, const uint8_t *vcache, uint4 *k16, uint4 *v16, int n_keys, int n_ctx,
                                                        int n_kv, int seq) {
    constexpr int KRB = kv_row_bytes(KT, PF_EXPAND_HD), VRB = kv_row_bytes(VT, PF_EXPAND_HD);
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int piece = (int)(idx & 15);
    const size_t row = idx >> 4;
    if (row >= (size_t)n_kv * n_keys) return;
    const int kvh = (int)(row / n_keys), key = (int)(row % n_keys);
    const size_t src = ((size_t)seq * n_kv + kvh) * n_ctx + key, dst = (size_t)kvh * n_ctx + key;
    k16[dst * 16 + piece] = pf_row_piece<KT, PF_EXPAND_HD>(kcache + src * KRB, piece);
    v16[dst * 16 + piece] = pf_row_piece<VT, PF_EXPAND_HD>(vcache + src * VRB, piece);
}

static int pf_n_cu() {
    static int n = 0;
    if (!n) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) n = p.multiProcessorCount;
        if (n <= 0) n = 256;
    }
    return n;
}

int attention_chunk(const AttnArgs &a_in, int T, int pos0, int seq, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    AttnArgs a = a_in;
    const int v_dim = a.v_dim ? a.v_dim : a.head_dim;
    const bool apart = v_dim != a.head_dim;         // keys and values of different lengths
    if (apart ? a.group != 1 || a.k_type != MESH_F16 || a.v_type != MESH_F16 || !((a.head_dim == 128 && v_dim == 64) || (a.head_dim == 192 && v_dim == 128))
              : a.head_dim != 128 && (a.head_dim != 64 || a.k_type != MESH_F16))
        return fail(MESH_ERR_UNSUPPORTED, "attention_chunk: head_dim %d, values of %d, cache type %d (128, and 64 with f16 rows; 128 with 64 and 192 with 128)", a.head_dim, v_dim, a.k_type);
    if (a.head_gate && !a.out_bf16) return fail(MESH_ERR_INVALID, "attention_chunk: gated output is bf16");
    if (a.group < 1 || a.n_head != a.group * a.n_kv || pos0 < 0 || pos0 + T > a.n_ctx || seq < 0)
        return fail(MESH_ERR_INVALID, "attention_chunk: bad head layout or chunk [%d, %d) outside the context of %d", pos0, pos0 + T, a.n_ctx);
    if (a.k_type != MESH_F16 && a.chunk_kv16 && T >= PF_EXPAND_MIN_T) {
        // Every query tile's workgroup would decode the quantised rows it walks.  Decode them once instead, into the
        // caller's f16 scratch, and run the f16 kernel on that: the same values reach the matrix cores.
        const int n_keys = pos0 + T;
        uint4 *k16 = reinterpret_cast<uint4 *>(a.chunk_kv16), *v16 = k16 + (size_t)a.n_kv * a.n_ctx * 16;
        const unsigned blocks = (unsigned)(((size_t)a.n_kv * n_keys * 16 + 255) / 256);
        if (a.k_type == MESH_Q8_0 && a.v_type == MESH_Q4_0)
            MESH_LAUNCH((kv_expand_kernel<MESH_Q8_0, MESH_Q4_0>), dim3(blocks), dim3(256), 0, stream, a.kcache, a.vcache, k16, v16, n_keys, a.n_ctx, a.n_kv, seq);
        else if (a.k_type == MESH_Q4_0 && a.v_type == MESH_Q4_0)
            MESH_LAUNCH((kv_expand_kernel<MESH_Q4_0, MESH_Q4_0>), dim3(blocks), dim3(256), 0, stream, a.kcache, a.vcache, k16, v16, n_keys, a.n_ctx, a.n_kv, seq);
        else return fail(MESH_ERR_UNSUPPORTED, "attention_chunk: KV cache types %d/%d", a.k_type, a.v_type);
        MESH_LAUNCH_CHECK();
        a.kcache = reinterpret_cast<const uint8_t *>(k16);
        a.vcache = reinterpret_cast<const uint8_t *>(v16);
        a.k_type = a.v_type = MESH_F16;
        seq = 0;
    }
    int hpw = a.group;                       // heads (waves) per workgroup: the largest divisor of the group up to 8
    while (hpw > 8 || a.group % hpw) --hpw;
    // eight heads per KV head: two workgroups of four waves when one of eight per (query tile, KV head) would leave CUs idle
    if (hpw == 8 && ((T + PF_TILE - 1) / PF_TILE) * a.n_kv < pf_n_cu()) hpw = 4;
    // groups of fewer than four heads: several consecutive query tiles per workgroup (they share the K / V tiles like heads do)
    const int qtiles = hpw >= 4 ? 1 : hpw == 1 ? 4 : 2;
    const int waves = hpw * qtiles, n_tiles = (T + PF_TILE - 1) / PF_TILE;
    dim3 grid((unsigned)((n_tiles + qtiles - 1) / qtiles), (unsigned)a.n_kv, (unsigned)(a.group / hpw));
    // A short chunk on a long history has few query tiles, each with a long walk: split the keys of every walk over
    // several workgroups (partials in the caller's split buffers, merged by attn_combine_kernel) until the launch has a
    // workgroup per CU, at most 8 ways, at least 256 keys each, within the buffers' rows of (token, split).
    int n_ksplit = 1;
    const int n_keys = a.window > 0 ? std::min(pos0 + T, a.window + PF_TILE) : pos0 + T;
    {
        const int wgs = (int)(grid.x * grid.y * grid.z);
        if (a.part && a.ml && a.part_rows > 0 && wgs < pf_n_cu())
            n_ksplit = std::max(1, std::min(std::min(pf_n_cu() / wgs, 8), std::min(n_keys / 256, (int)(a.part_rows / (size_t)T))));
        if (n_ksplit > ATTN_SPLITS_CAP) n_ksplit = ATTN_SPLITS_CAP;
    }
    grid.z *= (unsigned)n_ksplit;
    // Workgroups of four waves leave a SIMD one wave, whose products wait for its softmax and the other way round (two workgroups fit
    // a CU, but the longest walks end alone): a second group of four waves takes every other step of 64 keys of the same walks.  Short
    // walks have few steps to share and pay for the larger workgroup and the merge.  One group / two, us, 8B shape: 17 tokens alone 6.7 /
    // 10.5, 200 12.6 / 13.8, 128 behind 500 (walks of 314) 15.3 / 16.7, 333 16.1 / 16.1, 17 behind 1000 (339) 15.0 / 14.7, 1024 32.4 / 27.3,
    // 2048 75.7 / 57.8; quantised rows 17 behind 1000 18.9 / 17.2; 16 heads of 192 with values of 128 320 tokens 18.7 / 19.3, 400 21.2 / 20.6.
    const int key_groups = waves == 4 && (n_keys + n_ksplit - 1) / n_ksplit > PF_TWO_GROUPS_WALK ? 2 : 1;
    const dim3 block((unsigned)(64 * waves * key_groups));
    // (Two tiles per step everywhere.  With 5 heads per KV head one tile per step keeps the kernel under 170 registers, so
    // that two 5-wave workgroups share a CU instead of one: measured slower, 16.5 against 14.8 ms over 32 layers of 4096 tokens.)
    // NP by the threads of the workgroup: 1024 / threads pairs each, rounded up
#define MESH_CHUNK_LAUNCH(HD, KT, VT)                                                                                     \
    do {                                                                                                                  \
        if (waves == 8) MESH_LAUNCH((attn_chunk_kernel<HD, HD, KT, VT, 2, 1>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit);      \
        else if (waves == 6) MESH_LAUNCH((attn_chunk_kernel<HD, HD, KT, VT, 3, 1>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit); \
        else if (key_groups == 2) MESH_LAUNCH((attn_chunk_kernel<HD, HD, KT, VT, 4, 2>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit); \
        else MESH_LAUNCH((attn_chunk_kernel<HD, HD, KT, VT, 4, 1>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit);                  \
    } while (0)
    // (a group of one: four waves)
    if (apart && a.head_dim == 192) {
        if (key_groups == 2) MESH_LAUNCH((attn_chunk_kernel<192, 128, MESH_F16, MESH_F16, 6, 2>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit);
        else MESH_LAUNCH((attn_chunk_kernel<192, 128, MESH_F16, MESH_F16, 6, 1>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit);
    } else if (apart) {
        if (key_groups == 2) MESH_LAUNCH((attn_chunk_kernel<128, 64, MESH_F16, MESH_F16, 4, 2>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit);
        else MESH_LAUNCH((attn_chunk_kernel<128, 64, MESH_F16, MESH_F16, 4, 1>), grid, block, 0, stream, a, T, pos0, seq, hpw, qtiles, n_ksplit);
    }
    else if (a.head_dim == 64) MESH_CHUNK_LAUNCH(64, MESH_F16, MESH_F16);
    else if (a.k_type == MESH_F16 && a.v_type == MESH_F16) MESH_CHUNK_LAUNCH(128, MESH_F16, MESH_F16);
    else if (a.k_type == MESH_Q8_0 && a.v_type == MESH_Q4_0) MESH_CHUNK_LAUNCH(128, MESH_Q8_0, MESH_Q4_0);
    else if (a.k_type == MESH_Q4_0 && a.v_type == MESH_Q4_0) MESH_CHUNK_LAUNCH(128, MESH_Q4_0, MESH_Q4_0);
    else return fail(MESH_ERR_UNSUPPORTED, "attention_chunk: KV cache types %d/%d", a.k_type, a.v_type);
#undef MESH_CHUNK_LAUNCH
    MESH_LAUNCH_CHECK();
    if (n_ksplit > 1) {
        a.n_splits = n_ksplit;
        return attention_combine(a, T, stream);
    }
    return MESH_OK;
}

}  // namespace mesh
