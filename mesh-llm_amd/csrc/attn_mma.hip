// GQA decode attention on the matrix cores, for batches of decode tokens over long KV ranges.
//
// Same contract as attn_kernel of attn.hip (token t attends to cache positions [0, pos[t]] of sequence seq[t], or the last `window` of them; split-KV
// partials merged by attn_combine_kernel), same place in the worker's graph (flash_attn_ext under -fa on,
// mesh-llm/src/inference/launch.rs:1350-1353).  The per-key work of that kernel is vector ALU work that grows with the
// number of query heads per KV head; here the query heads of a KV head are the 16 columns of an MFMA tile, so the
// cost per key does not depend on the group size (up to 16), and the cache rows cross the vector ALUs only to be
// converted (quantised rows) and transposed (V).
//
// A workgroup takes one (split, kv head, token); each of its 4 waves walks its own 32-key blocks of the range and
// keeps its own running softmax, merged at the end:
//   S^T (2 x 16 keys x 16 heads) = K . Q^T   v_mfma_f32_16x16x32_f16 per 32 dims; the K operand is the cache row as it
//                                             lies in memory (lane = key, 8 consecutive dims), loaded straight from HBM
//   O^T (16 dims x 16 heads) += V^T . P^T     v_mfma_f32_16x16x32_f16 per 16 dims and 32 keys; the result registers of
//                                             S^T (4 keys of one head per lane and half) are the P^T operand as they are;
//                                             V^T needs the keys along a lane: V rows pass a wave-private LDS tile as
//                                             they are (long walks of f16: K rows too), and ds_read_b64_tr_b16 hands them back transposed
// A lane owns one head column throughout: the softmax maximum is a reduction over its 8 registers and the 4 lane
// groups, the rescale of O is a per-lane scalar, and its share of the sum meets the others' once, at the end.
// Q and the probabilities are rounded to f16 for the matrix cores; sums are f32.
//
// What bounds it: the walk of a workgroup is a chain of row loads (29 GB/s per workgroup), beside it the conversion of
// quantised rows (~300 vector instructions per 32 keys; ~490 with the results in
// accumulation registers and nibbles masked and biased apart, which took 206 registers for 166 and was two waves a SIMD for three:
// 60.7 -> 54.6 us, 32 sequences of 2000 to 6000 keys, 8 heads, q8_0 / q4_0).  Against blocks of 16 keys with V scattered into the transposed
// tile by 32 two-byte stores a lane: 64.4 -> 55.9 us (32 sequences of 2000 to 6000 keys, 8 heads, q8_0 / q4_0: 213 MB),
// 17.4 -> 15.4 (16 sequences, 4 heads), f16 rows 41.4 -> 39.5 (16 sequences, 179 MB: 4.5 TB/s), 7.3 -> 6.8 (one); f16 rows and whole
// lines of V (RowBlock) against those blocks of 16 keys, 8 heads of 128, 4000 keys, with the merge: 64 sequences 177 -> 177, 33 140 -> 129,
// 20 69 -> 59, 5 23.6 -> 22.6, one 11.5 -> 10.9; of 64: 128 sequences 180 -> 172, 33 62 -> 62, 40 66 -> 69, 20 49 -> 33.

#include "attn.hpp"
#include "lds_ops.hpp"
#include "q16.hpp"
#include "wave_ops.hpp"

#include <type_traits>

namespace mesh {

constexpr int MMA_THREADS = 256, MMA_WAVES = 4, MMA_KEYS = 32;
constexpr float MMA_RESCALE_STEP = 8.f;  // log2 units
// Blocks in flight per wave.  A block of f16 rows is 16 KB, of quantised rows 4.6 - 6.7 KB: a second one of those covers the
// latency of the walk (61.6 -> 55.9 us at 32 tokens), a third one and a second one of f16 rows cost more waves than they
// bring (step of eight 8B-shaped layers at 16 tokens 910 -> 920 us).
constexpr int MMA_DEPTH_F16 = 1, MMA_DEPTH_Q = 2;
// halfs added to a key row of the V tile: rows of 272 (144) bytes put the 16 rows of a wave's stores on different banks
constexpr int MMA_VPAD = 8;

typedef _Float16 mm_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 mm_h2 __attribute__((ext_vector_type(2)));
typedef float mm_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t mm_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t mm_u4a8 __attribute__((ext_vector_type(4), aligned(8)));

__device__ __forceinline__ uint32_t mm_pack(float a, float b) {
    const mm_h2 h = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, h);
}

// Bytes / nibbles -> f16 without conversions: 0x6400 | u is the half 1024 + u (0x5400 | u << 4 the half 64 + u), so one
// packed subtraction of that and the offset leaves the signed quant exactly, and one packed multiply by the block scale
// (an f16 in the cache) gives d * q rounded to f16 -- the same value as the f32 product rounded once.
__device__ __forceinline__ uint32_t mm_scale_pair(uint32_t biased, float bias, mm_h2 d2) {
    const mm_h2 v = (__builtin_bit_cast(mm_h2, biased) - mm_h2{(_Float16)bias, (_Float16)bias}) * d2;
    return __builtin_bit_cast(uint32_t, v);
}

// What a lane (key row c, lane group g) holds of a cache row: HD / 4 values as HD / 32 pieces of 8.
//   f16         piece cc is dims 32 cc + 8 g .. + 8: the four groups of a row read 64 consecutive bytes per load
//   quantised   piece cc is dims (HD / 4) g + 8 cc .. + 8: whole 16-byte loads, and one block scale per lane
// q4_0 pieces come out with their dims in the order 0 4 1 5 2 6 3 7 (mm_dim_slot), which takes one shift per eight
// nibbles; Q is packed in the same order for K, and the merge undoes it for V.
template <int TYPE, int HD>
struct RowShare {
    static constexpr int NC = HD / 32;
    static constexpr int BYTES = TYPE == MESH_F16 ? HD / 2 : TYPE == MESH_Q8_0 ? HD / 4 : HD / 8;
    uint32_t w[BYTES / 4];
    uint16_t d;
    __device__ __forceinline__ void load(const uint8_t *row, int g) {
        if constexpr (TYPE == MESH_F16) {
#pragma unroll
            for (int cc = 0; cc < NC; ++cc) {
                const uint4 v = *reinterpret_cast<const uint4 *>(row + 64 * cc + 16 * g);
                w[4 * cc] = v.x; w[4 * cc + 1] = v.y; w[4 * cc + 2] = v.z; w[4 * cc + 3] = v.w;
            }
        } else {
            // (rows are multiples of 8 bytes, not of 16)
            const uint8_t *p = row + BYTES * g;
            if constexpr (BYTES >= 16) {
#pragma unroll
                for (int i = 0; i < BYTES / 16; ++i) {
                    const mm_u4a8 v = *reinterpret_cast<const mm_u4a8 *>(p + 16 * i);
                    w[4 * i] = v[0]; w[4 * i + 1] = v[1]; w[4 * i + 2] = v[2]; w[4 * i + 3] = v[3];
                }
            } else {
                const uint2 v = *reinterpret_cast<const uint2 *>(p);
                w[0] = v.x; w[1] = v.y;
            }
            d = *reinterpret_cast<const uint16_t *>(row + kv_quant_bytes(TYPE, HD) + (HD / 4 * g >> 5) * 2);
        }
    }
    __device__ __forceinline__ mm_u4 piece(int cc) const {
        if constexpr (TYPE == MESH_F16) {
            return mm_u4{w[4 * cc], w[4 * cc + 1], w[4 * cc + 2], w[4 * cc + 3]};
        } else {
            const _Float16 dh = __builtin_bit_cast(_Float16, d);
            const mm_h2 d2 = {dh, dh};
            if constexpr (TYPE == MESH_Q8_0) {
                const uint32_t a = w[2 * cc] ^ 0x80808080u, b = w[2 * cc + 1] ^ 0x80808080u;       // int8 -> biased uint8
                return mm_u4{mm_scale_pair(__builtin_amdgcn_perm(0x64646464u, a, 0x04010400u), 1024.f + 128.f, d2),
                             mm_scale_pair(__builtin_amdgcn_perm(0x64646464u, a, 0x04030402u), 1024.f + 128.f, d2),
                             mm_scale_pair(__builtin_amdgcn_perm(0x64646464u, b, 0x04010400u), 1024.f + 128.f, d2),
                             mm_scale_pair(__builtin_amdgcn_perm(0x64646464u, b, 0x04030402u), 1024.f + 128.f, d2)};
            } else {
                // (masks in scalar registers and biases in vector ones: the form one v_and_or_b32 takes, which reads one scalar)
                uint32_t lo = 0x000F000Fu, hi = 0x00F000F0u, lo_bias = 0x64006400u, hi_bias = 0x54005400u;
                asm("" : "+s"(lo), "+s"(hi), "+v"(lo_bias), "+v"(hi_bias));
                const uint32_t x = w[cc], y = x >> 8;
                return mm_u4{mm_scale_pair((x & lo) | lo_bias, 1024.f + 8.f, d2), mm_scale_pair((x & hi) | hi_bias, 64.f + 8.f, d2),
                             mm_scale_pair((y & lo) | lo_bias, 1024.f + 8.f, d2), mm_scale_pair((y & hi) | hi_bias, 64.f + 8.f, d2)};
            }
        }
    }
    // first dim of piece cc
    static __device__ __forceinline__ int dim0(int cc, int g) { return TYPE == MESH_F16 ? 32 * cc + 8 * g : HD / 4 * g + 8 * cc; }
};
// What a lane holds of the rows of a 32-key block; rows past the range are clamped to its last key (the scores are masked, the
// probabilities zero).
// A lane's shares of rows c and 16 + c, as above:
template <int TYPE, int HD, int PITCH>
struct ShareBlock {
    RowShare<TYPE, HD> r[2];
    __device__ __forceinline__ void load(const uint8_t *rows, int kb, int j1, int lane) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int key = kb + 16 * h + (lane & 15);
            key = key < j1 ? key : j1 - 1;
            r[h].load(rows + (size_t)key * kv_row_bytes(TYPE, HD), lane >> 4);
        }
    }
    __device__ __forceinline__ void put(_Float16 *tile, int lane) const {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int cc = 0; cc < RowShare<TYPE, HD>::NC; ++cc)
                *reinterpret_cast<mm_u4 *>(tile + (16 * h + (lane & 15)) * PITCH + RowShare<TYPE, HD>::dim0(cc, lane >> 4)) = r[h].piece(cc);
    }
};
// Whole rows on their way to the wave's LDS tile [key][dim], for f16 rows, which pass as they are: the 16 lanes that the memory pipe
// works on at a time lie in two cache lines instead of 16.  Lines that one load takes whole and nothing reads again need no place in
// the caches, and memory gives more without them (a plain walk of 140 MB: 5.7 TB/s, and 6.2 with the hint; of lines taken in halves
// the hint makes it less).  V / K rows read so, us, 8 KV heads, rows of 128: 32 sequences of 4090 keys 92.1 as shares of rows, 81.5
// with V, 81.9 with V and K whole; 32 of 1400 to 4090 69.1, 63.6, 60.2; 16 of 4090 49.2, 44.7, 43.5; 16 of 1400 to 4090 40.0, 37.5,
// 34.7; 5 of 1000 to 3000 12.8, 12.1, 12.0.
template <int HD, int PITCH>
struct RowBlock {
    static constexpr int PIECES = HD / 8, ROWS = 64 / PIECES;       // 16-byte pieces of a row, rows of a load
    mm_u4 v[MMA_KEYS / ROWS];
    __device__ __forceinline__ void load(const uint8_t *rows, int kb, int j1, int lane) {
#pragma unroll
        for (int i = 0; i < MMA_KEYS / ROWS; ++i) {
            int key = kb + i * ROWS + lane / PIECES;
            key = key < j1 ? key : j1 - 1;
            v[i] = __builtin_nontemporal_load(reinterpret_cast<const mm_u4 *>(rows + (size_t)key * (HD * 2) + lane % PIECES * 16));
        }
    }
    __device__ __forceinline__ void put(_Float16 *tile, int lane) const {
#pragma unroll
        for (int i = 0; i < MMA_KEYS / ROWS; ++i) *reinterpret_cast<mm_u4 *>(tile + (i * ROWS + lane / PIECES) * PITCH + lane % PIECES * 8) = v[i];
    }
};
// place, within its eight, of dim dd of a q4_0 piece
__device__ __forceinline__ int mm_dim_slot(int dd) { return (dd & ~7) | ((dd & 3) << 1) | ((dd >> 2) & 1); }

__device__ __forceinline__ void mm_wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// grid (n_splits, n_kv, T), 256 threads.  group <= 16.
// KROWS: K rows of f16 come whole, through the tile that V takes afterwards (RowBlock), else as shares, which a walk of one block a
// wave has sooner (one token, 4090 keys over 32 splits: 6.4 us, and 6.6 with whole rows).
// (the arguments on the way to the first K / V loads come first, as scalars, so that they are preloaded into SGPRs:
// see gemv.hip)
template <int HD, int KT, int VT, bool KROWS>
__global__ __launch_bounds__(MMA_THREADS) void attn_mma_kernel(const float *p_q, const int32_t *p_pos, const int32_t *p_seq,
                                                               const uint8_t *p_kcache, const uint8_t *p_vcache, int p_n_splits,
                                                               int p_n_ctx, int p_n_kv, int p_group, int p_n_head, float p_scale, int p_window,
                                                               const AttnArgs a) {
    constexpr int NC = HD / 32;             // steps of the score product
    constexpr int NDB = HD / 16;            // 16-dim blocks of the output
    constexpr int KRB = kv_row_bytes(KT, HD), VRB = kv_row_bytes(VT, HD);
    constexpr int VPITCH = HD + MMA_VPAD;   // halfs per key row of the V tile
    constexpr int OPITCH = HD + 4;          // floats per head row of the merge buffer
    // the V tiles (one per wave) and, after the key loop, the per-wave results share this memory
    constexpr int STAGE_BYTES = MMA_WAVES * MMA_KEYS * VPITCH * 2, MERGE_BYTES = MMA_WAVES * 16 * OPITCH * 4;
    constexpr int SH_BYTES = STAGE_BYTES > MERGE_BYTES ? STAGE_BYTES : MERGE_BYTES;
    __shared__ __align__(16) uint8_t s_raw[SH_BYTES];
    __shared__ float s_m[MMA_WAVES][16], s_l[MMA_WAVES][16];

    const int split = blockIdx.x, kvh = blockIdx.y, t = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, g = lane >> 4;         // head column / key row of a tile, lane group
    const int G = p_group;
    const int seq = p_seq[t];
    const int n_keys = p_pos[t] + 1;
    const int first = p_window > 0 && n_keys > p_window ? n_keys - p_window : 0;
    const int per = (n_keys - first + p_n_splits - 1) / p_n_splits;
    const int j0 = first + split * per;
    const int j1 = j0 + per < n_keys ? j0 + per : n_keys;

    // Q^T operand: head column c, the dims a lane of the K operand has, in log2 units
    mm_h8 qf[NC];
    {
        const float qs = c < G ? p_scale * 1.44269504088896341f : 0.f;
        const float *qp = p_q + ((size_t)t * p_n_head + (size_t)kvh * G + (c < G ? c : 0)) * HD;
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) {
            const float *qd = qp + RowShare<KT, HD>::dim0(cc, g);
            const float4 v0 = *reinterpret_cast<const float4 *>(qd), v1 = *reinterpret_cast<const float4 *>(qd + 4);
            const mm_u4 p = KT == MESH_Q4_0
                                ? mm_u4{mm_pack(v0.x * qs, v1.x * qs), mm_pack(v0.y * qs, v1.y * qs), mm_pack(v0.z * qs, v1.z * qs), mm_pack(v0.w * qs, v1.w * qs)}
                                : mm_u4{mm_pack(v0.x * qs, v0.y * qs), mm_pack(v0.z * qs, v0.w * qs), mm_pack(v1.x * qs, v1.y * qs), mm_pack(v1.z * qs, v1.w * qs)};
            qf[cc] = __builtin_bit_cast(mm_h8, p);
        }
    }
    mm_f4 o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) o[db] = mm_f4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;           // l: of this lane's keys only

    _Float16 *const sV = reinterpret_cast<_Float16 *>(s_raw) + wave * MMA_KEYS * VPITCH;
    const _Float16 *const v_get = sV + (4 * g + (c >> 2)) * VPITCH + 4 * (c & 3);         // (lds_read_transposed: rows 4 g .. + 4)
    const size_t base = ((size_t)seq * p_n_kv + kvh) * p_n_ctx;
    // what a lane fetches of a 32-key block: its shares of key rows c and 16 + c (rows past the range are clamped to its
    // last key, and masked below), and of the value rows
    constexpr int STEP = MMA_WAVES * MMA_KEYS;
    constexpr int DEPTH = KT == MESH_F16 && VT == MESH_F16 ? MMA_DEPTH_F16 : MMA_DEPTH_Q;
    typedef typename std::conditional<KROWS, RowBlock<HD, VPITCH>, ShareBlock<KT, HD, VPITCH>>::type KBlock;
    typedef typename std::conditional<VT == MESH_F16, RowBlock<HD, VPITCH>, ShareBlock<VT, HD, VPITCH>>::type VBlock;
    KBlock krs[DEPTH];
    VBlock vrs[DEPTH];
    auto fetch = [&](KBlock &kr, VBlock &vr, int kb) {
        kr.load(p_kcache + base * KRB, kb, j1, lane);
        vr.load(p_vcache + base * VRB, kb, j1, lane);
    };
    const int kb0 = j0 + __builtin_amdgcn_readfirstlane(wave) * MMA_KEYS;
    if (kb0 < j1) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) fetch(krs[d], vrs[d], kb0 + d * STEP);
    }
    for (int kbb = kb0; kbb < j1; kbb += DEPTH * STEP) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        const int kb = kbb + d * STEP;
        if (kb >= j1) break;
        KBlock &kr = krs[d];
        VBlock &vr = vrs[d];
        // S^T = K . Q^T : register i of half h is key kb + 16 h + 4 g + i for head c
        mm_f4 s[2];
        if constexpr (KROWS) { kr.put(sV, lane); mm_wave_lds_sync(); }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            s[h] = mm_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int cc = 0; cc < NC; ++cc) {
                mm_u4 kp;
                if constexpr (KROWS) kp = *reinterpret_cast<const mm_u4 *>(sV + (16 * h + c) * VPITCH + RowShare<KT, HD>::dim0(cc, g));
                else kp = kr.r[h].piece(cc);
                s[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mm_h8, kp), qf[cc], s[h], 0, 0, 0);
            }
        }
        if constexpr (KROWS) mm_wave_lds_sync();
        // V rows as they are: sV[key][dim]
        vr.put(sV, lane);
        // rows of a later block travel while this one is worked on (two blocks deep without a branch: the compiler then
        // counts the loads in flight exactly, 56 against 60 us; one block deep waits for all of them anyway, and the walks
        // of one block save the fetch)
        if (DEPTH > 1 || kb + DEPTH * STEP < j1) fetch(kr, vr, kb + DEPTH * STEP);

        if (kb + MMA_KEYS > j1) {       // the range's last, shorter block
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) s[h][i] = kb + 16 * h + 4 * g + i < j1 ? s[h][i] : -INFINITY;
        }
        float mx = s[0][0];
#pragma unroll
        for (int i = 1; i < 8; ++i) mx = fmaxf(mx, s[i >> 2][i & 3]);
        mx = lane_fold<32>(lane_fold<16>(mx, LaneMax{}), LaneMax{});
        // The reference point m of the exponentials only moves when a score exceeds it by more than 2^RESCALE_STEP
        // (probabilities then stay below that factor, harmless in f16 / f32), and then for the whole wave at once:
        // the rescale of the 32 accumulator registers becomes rare instead of once per block.
        if (__builtin_amdgcn_ballot_w64(mx > m + MMA_RESCALE_STEP) != 0) {      // first block: m = -inf
            const float m_new = fmaxf(m, mx);
            const float corr = __builtin_amdgcn_exp2f(m - m_new);               // exp2(-inf) = 0 on the first block
            l *= corr;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[db][i] *= corr;
            m = m_new;
        }
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f(s[i >> 2][i & 3] - m);
        l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        // P^T operand: head column c, keys 4 g + j, then 16 + 4 g + j
        const mm_u4 pu = {mm_pack(p[0], p[1]), mm_pack(p[2], p[3]), mm_pack(p[4], p[5]), mm_pack(p[6], p[7])};
        const mm_h8 pf = __builtin_bit_cast(mm_h8, pu);

        mm_wave_lds_sync();
        // O^T += V^T . P^T : the V^T operand is place 16 db + c of the rows, keys in the order of P^T
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
            const lds_u2 v0 = lds_read_transposed(v_get + 16 * db), v1 = lds_read_transposed(v_get + 16 * VPITCH + 16 * db);
            const mm_u4 vv = {v0[0], v0[1], v1[0], v1[1]};
            o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mm_h8, vv), pf, o[db], 0, 0, 0);
        }
        mm_wave_lds_sync();        // the tile is rewritten by the next block
      }
    }

    // merge the waves: o[db][i] is place 16 db + 4 g + i of head c
    l = lane_fold<32>(lane_fold<16>(l, LaneAdd{}), LaneAdd{});
    __syncthreads();               // every wave is done with its V tile: the memory becomes the merge buffer
    float *s_o = reinterpret_cast<float *>(s_raw);          // [wave][16 heads][place]
    if (g == 0) { s_m[wave][c] = m; s_l[wave][c] = l; }
    if (c < G) {
#pragma unroll
        for (int db = 0; db < NDB; ++db) *reinterpret_cast<mm_f4 *>(s_o + (wave * 16 + c) * OPITCH + 16 * db + 4 * g) = o[db];
    }
    __syncthreads();
    const bool single = p_n_splits == 1;
    for (int idx = tid; idx < G * HD; idx += MMA_THREADS) {
        const int h = idx / HD, dd = idx % HD, slot = VT == MESH_Q4_0 ? mm_dim_slot(dd) : dd;
        float mh = -INFINITY;
#pragma unroll
        for (int w = 0; w < MMA_WAVES; ++w) mh = fmaxf(mh, s_m[w][h]);
        float sum = 0.f, ll = 0.f;
#pragma unroll
        for (int w = 0; w < MMA_WAVES; ++w) {
            const float mw = s_m[w][h];
            const float wgt = mw == -INFINITY ? 0.f : exp2f(mw - mh);
            sum = fmaf(s_o[(w * 16 + h) * OPITCH + slot], wgt, sum);
            ll = fmaf(s_l[w][h], wgt, ll);
        }
        const size_t row = (size_t)t * p_n_head + (size_t)kvh * G + h;
        if (single) {
            if (a.out_q16) {
                q16_store_block32(a.out_q16, p_n_head * HD, t, (kvh * G + h) * HD + dd, sum / ll);
            } else if (a.out16_k8) {
                const size_t kk = ((size_t)kvh * G + h) * HD + dd, KK = (size_t)p_n_head * HD;
                a.out16_k8[(size_t)(t / 16) * 16 * KK + ((kk >> 3) * 16 + (t % 16)) * 8 + (kk & 7)] = (_Float16)(sum / ll);
            } else if (a.out_bf16) {
                a.out_bf16[row * HD + dd] = f32_to_bf16_bits(sum / ll);
            } else {
                a.out[row * HD + dd] = sum / ll;
            }
        } else {
            a.part[(row * p_n_splits + split) * HD + dd] = sum;
            if (dd == 0) {
                a.ml[(row * p_n_splits + split) * 2 + 0] = mh;
                a.ml[(row * p_n_splits + split) * 2 + 1] = ll;
            }
        }
    }
}

template <int HD, int KT, int VT, bool KROWS>
static void launch_mma_as(const AttnArgs &a, int T, hipStream_t stream) {
    MESH_LAUNCH((attn_mma_kernel<HD, KT, VT, KROWS>), dim3((unsigned)a.n_splits, (unsigned)a.n_kv, (unsigned)T), dim3(MMA_THREADS), 0, stream, a.q, a.pos, a.seq, a.kcache, a.vcache, a.n_splits,
                a.n_ctx, a.n_kv, a.group, a.n_head, a.scale, a.window, a);
}

// f16 rows, at most one block of keys a wave (attn_mma_kernel, KROWS)
bool attention_mma_one_block(const AttnArgs &a) {
    return a.k_type == MESH_F16 && a.v_type == MESH_F16 && a.max_keys > 0 && a.max_keys <= a.n_splits * MMA_WAVES * MMA_KEYS;
}

template <int HD>
static int launch_mma(const AttnArgs &a, int T, hipStream_t stream) {
    if (a.k_type == MESH_F16 && a.v_type == MESH_F16) {
        if (attention_mma_one_block(a)) launch_mma_as<HD, MESH_F16, MESH_F16, false>(a, T, stream);
        else launch_mma_as<HD, MESH_F16, MESH_F16, true>(a, T, stream);
    } else if (a.k_type == MESH_Q8_0 && a.v_type == MESH_Q4_0) launch_mma_as<HD, MESH_Q8_0, MESH_Q4_0, false>(a, T, stream);
    else if (a.k_type == MESH_Q4_0 && a.v_type == MESH_Q4_0) launch_mma_as<HD, MESH_Q4_0, MESH_Q4_0, false>(a, T, stream);
    else return fail(MESH_ERR_UNSUPPORTED, "attention_mma: KV cache types %d/%d", a.k_type, a.v_type);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

bool attention_mma_supported(const AttnArgs &a) {
    return (a.head_dim == 64 || a.head_dim == 128) && a.group >= 1 && a.group <= 16 && kv_pair_supported(a.k_type, a.v_type);
}

int attention_mma(const AttnArgs &a, int T, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    if (a.n_splits < 1 || a.n_splits > ATTN_SPLITS_CAP || a.group < 1 || a.n_head != a.group * a.n_kv)
        return fail(MESH_ERR_INVALID, "attention_mma: bad head layout or split count");
    if (a.n_splits > 1 && (!a.part || !a.ml)) return fail(MESH_ERR_INVALID, "attention_mma: split buffers missing");
    if (!attention_mma_supported(a)) return fail(MESH_ERR_UNSUPPORTED, "attention_mma: head_dim %d / group %d", a.head_dim, a.group);
    int rc = a.head_dim == 128 ? launch_mma<128>(a, T, stream) : launch_mma<64>(a, T, stream);
    if (rc != MESH_OK || a.n_splits == 1) return rc;
    return attention_combine(a, T, stream);
}

}  // namespace mesh
