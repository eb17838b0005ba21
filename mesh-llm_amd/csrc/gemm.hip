// Prefill GEMM: Y[T][M] = X[T][K] . W^T with W in tiled q4_K / q6_K blocks (gemv.hpp) and X in f16.
// The many-token counterpart of the decode GEMV -- what ggml_backend_graph_compute runs for mul_mat when a prompt is
// ingested (third_party/llama.cpp/patches/0002-rpc-add-direct-peer-tensor-transfers.patch:443-451).
//
// Design (gfx950): a 256-thread workgroup owns a 128 (weight rows) x 128 (tokens) output tile and walks K in
// steps of 64.  Per step the 128 x 64 weight slab is dequantised from its K-quant blocks straight into LDS as
// f16 (each thread: one row, one 32-element sub-block), the 128 x 64 activation slab is copied next to it, and
// the four waves (2 x 2, 64 x 64 each) issue v_mfma_f32_32x32x16_f16 on 16-byte LDS fragments with f32
// accumulation.  Weights cross HBM once per 128 tokens; dequantisation is amortised over 128 columns.  The two
// LDS stages alternate: the raw bytes of step k+1 are fetched into registers before the MFMAs of step k and
// dequantised after them, so global-memory latency and the dequant VALU work overlap the matrix cores (two
// workgroups fit a CU).  Calls of at most 64 tokens and the experts of a chunk form their fragments in registers instead
// (reg_tile below); wide projections of long calls take a 256-row tile (gemm_big_kernel), or f16 copies (gemm_f16.hip).
//
// MFMA operand layout used below (checked on hardware): A lane l = row l%32, k = 8*(l/32)+j; B lane l = column
// l%32, same k; accumulator register i of lane l = D[8*(i/4) + 4*(l/32) + i%4][l%32].

#include "gemm.hpp"
#include "gemm_tile.hpp"
#include "lds_ops.hpp"
#include "wave_ops.hpp"

#include <algorithm>
#include <type_traits>

namespace mesh {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int GM = 128, GN = 128, GK = 64;     // workgroup tile: weight rows x tokens x k-step
constexpr int LDS_LD = GK + 8;                 // f16 elements per LDS row (16-byte pad against bank conflicts)
constexpr int GEMM_THREADS = 512;              // 4 matrix-core waves + 4 staging waves

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// four bytes (values < 64) -> four f16 holding ((value - off) * sc) * d + c, as two packed dwords.  0x6400 | q is the f16
// 1024 + q exactly and the offset comes off exactly; sc is the block's integer scale, so (q - off) * sc is an exact
// small integer (|.| <= 504 for q4_K with off = 1024 + 8; q6_K's reaches 4064, where integers above 2048 round to even);
// d is the super-block's f16 scale as stored in the file.  One packed fma then makes the weight with a single
// rounding: products of ROUNDED per-block scales (f16(d * sc), f16(dmin * m)) carry their rounding error into every
// weight of the block, three times the error of this form on q4_K.
__device__ __forceinline__ void dequant4(uint32_t q, half2v off, half2v sc, half2v d, half2v c, uint32_t &lo, uint32_t &hi) {
    const half2v a = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, q, 0x04010400u)) - off) * sc;
    const half2v b = (__builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, q, 0x04030402u)) - off) * sc;
    lo = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(a, d, c));
    hi = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(b, d, c));
}
// q4_K: w = d sc (q - 8) + c with c = 8 d sc - dmin m (f32, rounded to f16 once).  {sc, c} of a sub-block:
__device__ __forceinline__ half2v q4k_sc_c(float d, float dmin, uint32_t scb, uint32_t mnb) {
    const float sc = (float)scb;
    return half2v{(_Float16)sc, (_Float16)(8.0f * d * sc - dmin * (float)mnb)};
}
__device__ __forceinline__ half2v h2_splat(float v) {
    const _Float16 h = (_Float16)v;
    return half2v{h, h};
}

// eight nibbles (elements 0..3 in the bytes of lo, 4..7 in those of hi) in the GEMM layout's order: element e at nibble e / 2 + 4 (e % 2)
__device__ __forceinline__ uint32_t pair_nibbles(uint32_t lo, uint32_t hi) {
    uint32_t r = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) r |= (((e < 4 ? lo : hi) >> (8 * (e & 3))) & 0xFu) << (4 * (e >> 1) + 16 * (e & 1));
    return r;
}

// Raw bytes of one (row, 32-element sub-block) of a tile: what a staging thread prefetches one k-step ahead.
template <int TYPE> struct RawSub;

// q4_K: row r of the tile, k-chunk c (64 elements) of the super-block, half h (sub-block 2c + h)
template <> struct RawSub<MESH_Q4_K> {
    uint4 hdr, qa, qb;
    __device__ __forceinline__ void load(const uint8_t *__restrict__ tile, int r, int c, int) {
        hdr = *reinterpret_cast<const uint4 *>(tile + r * 16);
        qa = *reinterpret_cast<const uint4 *>(tile + 256 + r * 128 + c * 32);
        qb = *reinterpret_cast<const uint4 *>(tile + 256 + r * 128 + c * 32 + 16);
    }
    __device__ __forceinline__ void store(int c, int h, _Float16 *dst) const {
        const float d = f16_bits_to_f32((uint16_t)(hdr.x & 0xFFFFu)), dmin = f16_bits_to_f32((uint16_t)(hdr.x >> 16));
        const uint32_t scw = c < 2 ? (hdr.y & 0x3F3F3F3Fu) : ((hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u));
        const uint32_t mnw = c < 2 ? (hdr.z & 0x3F3F3F3Fu) : (((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u));
        const int sh = (c & 1) * 16 + h * 8;
        const half2v sc_c = q4k_sc_c(d, dmin, (scw >> sh) & 0xFFu, (mnw >> sh) & 0xFFu);
        const half2v sc = {sc_c[0], sc_c[0]}, cc = {sc_c[1], sc_c[1]}, dd = h2_splat(d);
        const half2v off = {(_Float16)1032.f, (_Float16)1032.f};
        const uint32_t w[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
        uint4 *d4 = reinterpret_cast<uint4 *>(dst);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint4 o;
            dequant4((w[2 * i] >> (4 * h)) & 0x0F0F0F0Fu, off, sc, dd, cc, o.x, o.y);
            dequant4((w[2 * i + 1] >> (4 * h)) & 0x0F0F0F0Fu, off, sc, dd, cc, o.z, o.w);
            d4[i] = o;
        }
    }
    // this thread's part of a GEMM-layout chunk (gemm.hpp); s = 2 * row + h
    __device__ __forceinline__ void pack(int c, int h, uint8_t *chunk, int s) const {
        const float d = f16_bits_to_f32((uint16_t)(hdr.x & 0xFFFFu)), dmin = f16_bits_to_f32((uint16_t)(hdr.x >> 16));
        const uint32_t scw = c < 2 ? (hdr.y & 0x3F3F3F3Fu) : ((hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u));
        const uint32_t mnw = c < 2 ? (hdr.z & 0x3F3F3F3Fu) : (((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u));
        const int sh = (c & 1) * 16 + h * 8;
        const half2v sc_c = q4k_sc_c(d, dmin, (scw >> sh) & 0xFFu, (mnw >> sh) & 0xFFu);
        const uint32_t w[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<uint32_t *>(chunk + (s - h + (j & 1)) * 16 + (2 * h + (j >> 1)) * 4) = pair_nibbles((w[2 * j] >> (4 * h)) & 0x0F0F0F0Fu, (w[2 * j + 1] >> (4 * h)) & 0x0F0F0F0Fu);
        uint8_t *row = chunk + 4096 + (s >> 1) * 8;
        row[h] = (uint8_t)(scw >> sh);
        *reinterpret_cast<uint16_t *>(row + 4 + 2 * h) = (uint16_t)(__builtin_bit_cast(uint32_t, sc_c) >> 16);
        if (h == 0) *reinterpret_cast<uint16_t *>(row + 2) = (uint16_t)hdr.x;
    }
};

// q6_K: row r, k-chunk c: half n = c/2, elements 128n + 32*t4 + l with t4 = 2*(c%2) + h, l = 0..31
template <> struct RawSub<MESH_Q6_K> {
    uint4 la, lb, ha, hb;
    uint32_t sc, d;
    __device__ __forceinline__ void load(const uint8_t *__restrict__ tile, int r, int c, int h) {
        const int n = c >> 1, t4 = 2 * (c & 1) + h;
        const uint8_t *ql = tile + r * 128 + 64 * n + 32 * (t4 & 1);
        const uint8_t *qh = tile + 2048 + r * 64 + 32 * n;
        la = *reinterpret_cast<const uint4 *>(ql); lb = *reinterpret_cast<const uint4 *>(ql + 16);
        ha = *reinterpret_cast<const uint4 *>(qh); hb = *reinterpret_cast<const uint4 *>(qh + 16);
        sc = *reinterpret_cast<const uint16_t *>(tile + 3072 + r * 16 + 8 * n + 2 * t4);
        d = *reinterpret_cast<const uint16_t *>(tile + 3328 + r * 2);
    }
    __device__ __forceinline__ void store(int c, int h, _Float16 *dst) const {
        const int t4 = 2 * (c & 1) + h;
        const half2v dd = h2_splat(f16_bits_to_f32((uint16_t)d));
        const half2v s0 = h2_splat((float)(int8_t)(sc & 0xFFu)), s1 = h2_splat((float)(int8_t)(sc >> 8));
        const half2v off = {(_Float16)1056.f, (_Float16)1056.f}, zero = {(_Float16)0.f, (_Float16)0.f};
        const uint32_t lw[8] = {la.x, la.y, la.z, la.w, lb.x, lb.y, lb.z, lb.w};
        const uint32_t hw[8] = {ha.x, ha.y, ha.z, ha.w, hb.x, hb.y, hb.z, hb.w};
        uint4 *d4 = reinterpret_cast<uint4 *>(dst);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t q[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int j = 2 * i + e;
                const uint32_t nib = (t4 & 2) ? (lw[j] >> 4) & 0x0F0F0F0Fu : lw[j] & 0x0F0F0F0Fu;
                q[e] = nib | (((hw[j] >> (2 * t4)) & 0x03030303u) << 4);
            }
            const half2v s = i < 2 ? s0 : s1;       // one scale per 16 elements
            uint4 o;
            dequant4(q[0], off, s, dd, zero, o.x, o.y);
            dequant4(q[1], off, s, dd, zero, o.z, o.w);
            d4[i] = o;
        }
    }
    __device__ __forceinline__ void pack(int c, int h, uint8_t *chunk, int s) const {
        const int t4 = 2 * (c & 1) + h;
        const uint32_t lw[8] = {la.x, la.y, la.z, la.w, lb.x, lb.y, lb.z, lb.w};
        const uint32_t hw[8] = {ha.x, ha.y, ha.z, ha.w, hb.x, hb.y, hb.z, hb.w};
        uint32_t q[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t nib = (t4 & 2) ? (lw[j] >> 4) & 0x0F0F0F0Fu : lw[j] & 0x0F0F0F0Fu;
            q[j] = nib | (((hw[j] >> (2 * t4)) & 0x03030303u) << 4);
        }
        uint32_t hb2[2] = {0u, 0u};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            *reinterpret_cast<uint32_t *>(chunk + (s - h + (j & 1)) * 16 + (2 * h + (j >> 1)) * 4) = pair_nibbles(q[2 * j] & 0x0F0F0F0Fu, q[2 * j + 1] & 0x0F0F0F0Fu);
            // element e of the eight: bits 2 P and up of the word's lower half (e even) or upper half, P = 4 (j / 2) + e / 2
#pragma unroll
            for (int e = 0; e < 8; ++e)
                hb2[j & 1] |= ((q[2 * j + (e >> 2)] >> (8 * (e & 3) + 4)) & 3u) << (2 * (4 * (j >> 1) + (e >> 1)) + 16 * (e & 1));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) *reinterpret_cast<uint32_t *>(chunk + 4096 + (s - h + j) * 8 + h * 4) = hb2[j];
        uint8_t *row = chunk + 6144 + (s >> 1) * 8;
        *reinterpret_cast<uint16_t *>(row + 2 * h) = (uint16_t)(sc ^ 0x8080u);
        *reinterpret_cast<uint16_t *>(row + 4 + 2 * h) = (uint16_t)d;
    }
};

// Half a row of a chunk out of the GEMM layout (gemm.hpp): slot s = 2 row + h holds elements 16 j + 8 h .. + 7, j = 0..3, of the
// row's 64: what one lane of a v_mfma_f32_32x32x16_f16 fragment holds in each of four steps.
// Eight weights of it are a dword of nibbles, element e at nibble e / 2 + 4 (e % 2): one shift puts a pair into bits 4..7 and
// 20..23, where or-ing 0x5400 makes two f16 of exactly 64 + q (64 to 127: sixteenths in the lowest bits), and one packed fma with
// the scale then takes the offset off: (64 + q) sc - (64 + off) sc is (q - off) sc, exactly or rounded once, as (q - off)
// times sc is; 72 sc (off 8, sc <= 63) and 96 sc (off 32, |sc| <= 128) are f16.  15 instructions for 8 weights of q4_K, 23 of q6_K,
// and up to two a scale to make it an f16.
template <int TYPE> struct PackedSub;
// Loads of a staging wave's loop (load_staged), from a uniform base plus a 32-bit offset of the lane that stays in its register.  Left to
// itself the compiler adds 64-bit addresses in the loop, into registers of loads under way, and waits for those.  Down projection of
// 4096 x 14336, q6_K: 25.6 -> 23.5 us at 100 tokens, 76.4 -> 70.8 at 512, on the 256-row tile at 2048 tokens 258 -> 248 (with the stores of
// staged_slot); gate / up, q4_K: 48.3 -> 46.6 at 100 tokens, 478 -> 466 at 2048.
struct StagedSlot { unsigned quants, bits, scales; };
__device__ __forceinline__ StagedSlot staged_offsets(unsigned s) { return StagedSlot{s * 16, s * 8, (s >> 1) * 8}; }
template <class V> __device__ __forceinline__ V load_section(const uint8_t *chunk, int at, unsigned &off) {
    uint64_t base = reinterpret_cast<uint64_t>(chunk) + at;
    asm volatile("" : "+s"(base), "+v"(off));
    typedef uint32_t W __attribute__((ext_vector_type(sizeof(V) / 4)));
    typedef const __attribute__((address_space(1))) uint8_t *Bytes;
    typedef const __attribute__((address_space(1))) W *Words;
    return __builtin_bit_cast(V, *(Words)((Bytes)base + off));
}
__device__ __forceinline__ half2v fma2(uint32_t x, half2v b, half2v c) { return __builtin_elementwise_fma(__builtin_bit_cast(half2v, x), b, c); }
// (x & mask) | y in one instruction: it takes one constant from scalar registers, so the other has to be held in a vector register
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t y) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(mask), "v"(y));
    return r;
}
__device__ __forceinline__ uint32_t nibble_pair(uint32_t w, int p) {
    uint32_t mask = 0x00F000F0u, base = 0x54005400u;
    asm("" : "+s"(mask), "+v"(base));
    return ((p == 0 ? w << 4 : w >> (4 * (p - 1))) & mask) | base;
}
// 1024 + byte i of w, twice, exactly
__device__ __forceinline__ half2v byte_pair(uint32_t w, int i) { return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u + 0x00010001u * i)); }
template <> struct PackedSub<MESH_Q4_K> {
    static constexpr int CHUNK = 5120;
    uint4 q;
    uint2 sm;          // {byte sc of elements 0..31, of 32..63, f16 d}, {f16 c of elements 0..31, of 32..63}
    __device__ __forceinline__ void load(const uint8_t *__restrict__ chunk, unsigned s) {
        q = *reinterpret_cast<const uint4 *>(chunk + s * 16);
        sm = *reinterpret_cast<const uint2 *>(chunk + 4096 + (s >> 1) * 8);
    }
    __device__ __forceinline__ void load_staged(const uint8_t *chunk, StagedSlot &s) {
        q = load_section<uint4>(chunk, 0, s.quants);
        sm = load_section<uint2>(chunk, 4096, s.scales);
    }
    // the eight weights of step j (known at compile time)
    __device__ __forceinline__ uint4 form(int j) const {
        const half2v sc = byte_pair(sm.x, j >> 1) - half2v{(_Float16)1024.f, (_Float16)1024.f}, off = sc * half2v{(_Float16)-72.f, (_Float16)-72.f};
        const half2v dd = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sm.x, sm.x, 0x03020302u));
        const half2v cc = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sm.y, sm.y, j < 2 ? 0x01000100u : 0x03020302u));
        const uint32_t w = j == 0 ? q.x : j == 1 ? q.y : j == 2 ? q.z : q.w;
        uint32_t o[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) o[p] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(fma2(nibble_pair(w, p), sc, off), dd, cc));
        return make_uint4(o[0], o[1], o[2], o[3]);
    }
};
template <> struct PackedSub<MESH_Q6_K> {
    static constexpr int CHUNK = 7168;
    uint4 q;
    uint2 hb;
    uint2 sc;          // bytes 128 + sc of elements 0..15, 16..31, 32..47, 48..63; f16 d, twice
    __device__ __forceinline__ void load(const uint8_t *__restrict__ chunk, unsigned s) {
        q = *reinterpret_cast<const uint4 *>(chunk + s * 16);
        hb = *reinterpret_cast<const uint2 *>(chunk + 4096 + s * 8);
        sc = *reinterpret_cast<const uint2 *>(chunk + 6144 + (s >> 1) * 8);
    }
    __device__ __forceinline__ void load_staged(const uint8_t *chunk, StagedSlot &s) {
        q = load_section<uint4>(chunk, 0, s.quants);
        hb = load_section<uint2>(chunk, 4096, s.bits);
        sc = load_section<uint2>(chunk, 6144, s.scales);
    }
    __device__ __forceinline__ uint4 form(int j) const {
        const half2v s = byte_pair(sc.x, j) - half2v{(_Float16)1152.f, (_Float16)1152.f};
        const half2v off = s * half2v{(_Float16)-96.f, (_Float16)-96.f};
        const half2v dd = __builtin_bit_cast(half2v, sc.y), zero = {(_Float16)0.f, (_Float16)0.f};
        const uint32_t w = j == 0 ? q.x : j == 1 ? q.y : j == 2 ? q.z : q.w, hw = j < 2 ? hb.x : hb.y;
        uint32_t o[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int at = 2 * (4 * (j & 1) + p);
            const uint32_t x = and_or(at < 8 ? hw << (8 - at) : hw >> (at - 8), 0x03000300u, nibble_pair(w, p));
            o[p] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(fma2(x, s, off), dd, zero));
        }
        return make_uint4(o[0], o[1], o[2], o[3]);
    }
};
// ... to its places in a row of the weight slab, dst being the row's element 8 h
template <int TYPE>
__device__ __forceinline__ void store_sub(const PackedSub<TYPE> &w, _Float16 *dst) {
    uint4 *d4 = reinterpret_cast<uint4 *>(dst);
#pragma unroll
    for (int j = 0; j < 4; ++j) d4[2 * j] = w.form(j);
}

// The slot that staging thread s (0..255) brings: within its wave's 64 slots, eight lanes side by side take eight rows and the same
// h, so that their 16-byte stores (rows of 36 banks) fall on different banks; slot = s would put h = 1 of one row on h = 0 of the next
// (down projection of 4096 x 14336, q6_K, 2048 tokens on the 256-row tile: 270 -> 266 us).
__device__ __forceinline__ int staged_slot(int s) { return (s & ~63) + 2 * ((s & 7) + ((s >> 4) & 3) * 8) + ((s >> 3) & 1); }

// (Barriers here are lds_barrier: __syncthreads() also waits for every outstanding global load, i.e. at the end of each k-step for the
// activation fragments requested a moment ago for the NEXT step -- with one matrix-core wave per SIMD nothing else would run
// during that wait.)

// Role split: waves 0-3 only multiply (each a 64 x 64 corner of the tile out of LDS stage kc & 1), waves 4-7 only
// stage (fetch the raw weight bytes and activations of step kc + 2, dequantise step kc + 1 into the other LDS
// stage).  A SIMD then holds one wave of each kind per workgroup, and the dequantisation (vector ALU) of one runs
// while the MFMAs (matrix core) of the other execute -- in one wave doing both, the ~110 dequant instructions of
// a step only start once its 16 MFMAs have been issued, and the four waves move in lockstep between barriers.
// PACKED: the weights come from the GEMM layout (a.Wp) instead of the mat-vec tiles (a.W).
// XDIRECT: the activations are k8-major (gemm.hpp) and never enter LDS: a matrix-core wave's B fragment of 32 tokens x
// 16 k is four contiguous 256-byte pieces of that layout, so each lane fetches its 16 bytes straight from memory (L2),
// four k16 steps ahead, into a ring of registers.  That halves the LDS reads per MFMA and leaves the staging waves only
// the weights.
// Wp, w_block: a GEMM layout, and the workgroup's row block in it.
template <int TYPE, bool PACKED, bool XDIRECT, bool SPLIT>
__device__ __forceinline__ void kq_tile(const GemmArgs &a, const uint8_t *Wp, int w_block) {
    extern __shared__ __align__(16) _Float16 gemm_smem[];
    _Float16 *Ws = gemm_smem;                                  // [2][GM][LDS_LD]
    _Float16 *Xs = gemm_smem + 2 * GM * LDS_LD;                // [2][GN][LDS_LD]
    constexpr int TB = TYPE == MESH_Q4_K ? Q4K_TILE_BYTES : Q6K_TILE_BYTES;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = blockIdx.y * GN, t_end = a.T;
    const int m0 = blockIdx.x * GM;
    const int nsb = a.K / QK_K, n_all = a.K / GK;
    // k-steps [k0, k0 + n_steps) of this workgroup: all of them, or slice blockIdx.z of a split launch
    // (a template parameter: the unsplit kernel must not carry the offsets, they cost it 6%)
    const int k0 = SPLIT ? (int)blockIdx.z * a.k_per_split : 0;
    const int n_steps = SPLIT ? (n_all - k0 < a.k_per_split ? n_all - k0 : a.k_per_split) : n_all;

    if (wave >= 4) {
        // ---- staging waves: thread s (0..255): weights -- row s/2, sub-block half s%2 (PACKED: a slot of the chunk); activations --
        // token s/2, 32 elements s%2
        const int st = tid - 256;
        const int srow = st >> 1, sh = st & 1, slot = staged_slot(st);
        const int wrow = m0 + srow;                                  // rows beyond M are zero tiles (M padded to 16)
        const bool wlive = PACKED || wrow < a.M_pad;                 // (the GEMM layout holds its zero rows)
        const uint8_t *wtile_row = PACKED ? Wp + ((size_t)w_block * n_all + k0) * PackedSub<TYPE>::CHUNK
                                          : static_cast<const uint8_t *>(a.W) + (size_t)((wlive ? wrow : 0) >> 4) * nsb * TB;
        using Sub = typename std::conditional<PACKED, PackedSub<TYPE>, RawSub<TYPE>>::type;
        const int tok = t0 + srow;
        const bool xlive = tok < a.T;
        const _Float16 *xrow = XDIRECT ? a.X : a.X + (size_t)(xlive ? tok : 0) * a.ldx + 32 * sh;
        StagedSlot offsets = staged_offsets(slot);
        Sub rw[2];
        uint4 rx[2][4];
        auto fetch = [&](int kc, Sub &w, uint4 (&x)[4]) {
            if constexpr (PACKED) w.load_staged(wtile_row + (size_t)kc * PackedSub<TYPE>::CHUNK, offsets);
            else w.load(wtile_row + (size_t)((k0 + kc) >> 2) * TB, wrow & 15, (k0 + kc) & 3, sh);
            if constexpr (!XDIRECT) {
                const uint4 *s4 = reinterpret_cast<const uint4 *>(xrow + (size_t)(k0 + kc) * GK);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = s4[i];
            }
        };
        auto stage = [&](int kc, int buf, const Sub &w, const uint4 (&x)[4]) {
            _Float16 *wdst = PACKED ? Ws + (buf * GM + (slot >> 1)) * LDS_LD + 8 * (slot & 1) : Ws + (buf * GM + srow) * LDS_LD + 32 * sh;
            if constexpr (PACKED) {
                store_sub(w, wdst);
            } else if (wlive) {
                w.store((k0 + kc) & 3, sh, wdst);
            } else {
                uint4 *d4 = reinterpret_cast<uint4 *>(wdst);
#pragma unroll
                for (int i = 0; i < 4; ++i) d4[i] = make_uint4(0, 0, 0, 0);
            }
            if constexpr (!XDIRECT) {
                uint4 *x4 = reinterpret_cast<uint4 *>(Xs + (buf * GN + srow) * LDS_LD + 32 * sh);
#pragma unroll
                for (int i = 0; i < 4; ++i) x4[i] = xlive ? x[i] : make_uint4(0, 0, 0, 0);
            }
        };
        fetch(0, rw[0], rx[0]);
        fetch(n_steps > 1 ? 1 : 0, rw[1], rx[1]);
        stage(0, 0, rw[0], rx[0]);
        __syncthreads();
        // step kc (its slot parity = kc & 1): the slot of step kc was staged already -> refill it with step kc + 2;
        // then dequantise step kc + 1 (the other slot) into the LDS stage the multiplying waves are not reading
        for (int kc0 = 0; kc0 < n_steps; kc0 += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int kc = kc0 + u;
                if (kc >= n_steps) break;
                fetch(kc + 2 < n_steps ? kc + 2 : n_steps - 1, rw[u], rx[u]);
                if (kc + 1 < n_steps) stage(kc + 1, u ^ 1, rw[u ^ 1], rx[u ^ 1]);
                __syncthreads();
            }
        }
        return;
    }

    // ---- multiplying waves
    // wave's corner of the tile: 64 rows x 64 tokens
    constexpr int MI = 2;
    const int wm = (wave & 1) * 64, wn = (wave >> 1) * 64;
    float16v acc[MI][2];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    if constexpr (XDIRECT) {
        // lane's slot in the fragments of its two 32-token groups: token (lane & 31), k8 group (lane >> 5) of a k16 step;
        // consecutive k16 steps are 256 halfs apart.  Token blocks past the batch re-read the last one (never stored).
        const int n_blk = (a.T + 15) >> 4, n_g = n_all * (GK / 16), g0 = k0 * (GK / 16);
        const _Float16 *bp[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int tok = t0 + wn + 32 * i + (lane & 31);
            const int blk = (tok >> 4) < n_blk ? (tok >> 4) : n_blk - 1;
            bp[i] = a.X + (size_t)blk * 16 * a.K + ((lane >> 5) * 16 + (tok & 15)) * 8;
        }
        half8 ring[GK / 16][2];
#pragma unroll
        for (int ks = 0; ks < GK / 16; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i) ring[ks][i] = *reinterpret_cast<const half8 *>(bp[i] + (size_t)(g0 + ks < n_g ? g0 + ks : n_g - 1) * 256);
        __syncthreads();
        for (int kc = 0; kc < n_steps; ++kc) {
            const _Float16 *Wb = Ws + (kc & 1) * GM * LDS_LD;
#pragma unroll
            for (int ks = 0; ks < GK / 16; ++ks) {
                half8 af[MI];
#pragma unroll
                for (int i = 0; i < MI; ++i)
                    af[i] = *reinterpret_cast<const half8 *>(Wb + (wm + 32 * i + (lane & 31)) * LDS_LD + 16 * ks + 8 * (lane >> 5));
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], ring[ks][j], acc[i][j], 0, 0, 0);
                int gn = g0 + (kc + 1) * (GK / 16) + ks;
                gn = gn < n_g ? gn : n_g - 1;
#pragma unroll
                for (int i = 0; i < 2; ++i) ring[ks][i] = *reinterpret_cast<const half8 *>(bp[i] + (size_t)gn * 256);
                // keep each refill where it is written: left to itself the scheduler sinks all eight loads to the end
                // of the step, where the next step's first MFMA waits for them at full memory latency
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
        }
    } else {
    __syncthreads();
    for (int kc = 0; kc < n_steps; ++kc) {
        const int buf = kc & 1;
        const _Float16 *Wb = Ws + buf * GM * LDS_LD, *Xb = Xs + buf * GN * LDS_LD;
#pragma unroll
        for (int ks = 0; ks < GK / 16; ++ks) {
            half8 af[2], bf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                af[i] = *reinterpret_cast<const half8 *>(Wb + (wm + 32 * i + (lane & 31)) * LDS_LD + 16 * ks + 8 * (lane >> 5));
                bf[i] = *reinterpret_cast<const half8 *>(Xb + (wn + 32 * i + (lane & 31)) * LDS_LD + 16 * ks + 8 * (lane >> 5));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    }

    // D[m][t]: lane holds column t = lane%32 and rows 8*(e/4) + 4*(lane/32) + e%4 -> four consecutive m per store
    if constexpr (SPLIT) {
        // slice of a split launch: the raw sums go to part[slice][token][row of the launch]
        const size_t ld = (size_t)gridDim.x * GM;
        float *P = a.part + (size_t)blockIdx.z * a.T * ld + m0;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int t = t0 + wn + 32 * j + (lane & 31);
                if (t >= a.T) continue;
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4)
                    *reinterpret_cast<float4 *>(P + (size_t)t * ld + wm + 32 * i + 8 * e4 + 4 * (lane >> 5)) =
                        make_float4(acc[i][j][4 * e4], acc[i][j][4 * e4 + 1], acc[i][j][4 * e4 + 2], acc[i][j][4 * e4 + 3]);
            }
        return;
    }
    if (a.y16_k8) {
        // SwiGLU pair: the waves of the upper half of the tile hold the up rows of the gate rows in the lower half, at
        // the same (register, lane).  They hand them over through LDS (free by now: the staging waves have left, and
        // the barrier makes sure every matrix-core wave has read its last fragments).
        float *xch = reinterpret_cast<float *>(gemm_smem);         // [pair of waves][64 registers][64 lanes]
        const bool is_up = wm != 0;
        const int pair = (wn >> 6) * 4;  // first 16-register group of this pair of waves
        __syncthreads();
        if (is_up) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) xch[((pair + i * 2 + j) * 16 + e) * 64 + lane] = acc[i][j][e];
        }
        __syncthreads();
        if (is_up) return;
        const int t_pad = (t_end + 15) & ~15;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int t = t0 + wn + 32 * j + (lane & 31);
                if (t >= t_pad) continue;
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const int m = (int)blockIdx.x * (GM / 2) + 32 * i + 8 * e4 + 4 * (lane >> 5);
                    if (m >= a.M) continue;
                    float o[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const float g = acc[i][j][4 * e4 + c], u = xch[((pair + i * 2 + j) * 16 + 4 * e4 + c) * 64 + lane];
                        o[c] = t < t_end ? g / (1.0f + expf(-g)) * u : 0.f;       // padding columns of the last token block hold zeros
                    }
                    note_f16_clamp(a.sat, o[0], o[1], o[2], o[3]);
                    *reinterpret_cast<uint2 *>(a.y16_k8 + (size_t)(t >> 4) * 16 * a.M + ((size_t)(m >> 3) * 16 + (t & 15)) * 8 + (m & 7)) =
                        make_uint2(pack_h2(o[0], o[1]), pack_h2(o[2], o[3]));
                }
            }
        return;
    }
    float *Y = a.Y;
    const float *bias = a.bias;
    int M = a.M, ldy = a.ldy, mb0 = m0;
    if (a.n_seg > 1) {
        // (selected, not indexed: a dynamically indexed kernel-argument array would be spilled to scratch)
        const int bx = blockIdx.x;
        const int sg = (bx >= a.seg_begin[1] ? 1 : 0) + (a.n_seg > 2 && bx >= a.seg_begin[2] ? 1 : 0);
        Y = sg == 0 ? a.seg_Y[0] : sg == 1 ? a.seg_Y[1] : a.seg_Y[2];
        bias = sg == 0 ? a.seg_bias[0] : sg == 1 ? a.seg_bias[1] : a.seg_bias[2];
        M = sg == 0 ? a.seg_M[0] : sg == 1 ? a.seg_M[1] : a.seg_M[2];
        ldy = sg == 0 ? a.seg_ldy[0] : sg == 1 ? a.seg_ldy[1] : a.seg_ldy[2];
        mb0 = (bx - (sg == 0 ? 0 : sg == 1 ? a.seg_begin[1] : a.seg_begin[2])) * GM;
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = t0 + wn + 32 * j + (lane & 31);
            if (t >= t_end) continue;
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const int m = mb0 + wm + 32 * i + 8 * e4 + 4 * (lane >> 5);
                if (m >= M) continue;      // M is a multiple of 4 for every projection
                float4 o = make_float4(acc[i][j][4 * e4], acc[i][j][4 * e4 + 1], acc[i][j][4 * e4 + 2], acc[i][j][4 * e4 + 3]);
                if (bias) {
                    const float4 b = *reinterpret_cast<const float4 *>(bias + m);
                    o.x += b.x; o.y += b.y; o.z += b.z; o.w += b.w;
                }
                if (a.residual) {
                    const float4 r = *reinterpret_cast<const float4 *>(a.residual + (size_t)t * a.ldres + m);
                    o.x += r.x; o.y += r.y; o.z += r.z; o.w += r.w;
                }
                *reinterpret_cast<float4 *>(Y + (size_t)t * ldy + m) = o;
            }
        }
}

template <int TYPE, bool PACKED, bool XDIRECT, bool SPLIT>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_kq_kernel(GemmArgs a) {
    kq_tile<TYPE, PACKED, XDIRECT, SPLIT>(a, static_cast<const uint8_t *>(a.Wp), (int)blockIdx.x);
}

// Several matrices of which the last is of another type: its few row blocks beside the others' instead of in a launch of their own, which
// must split K to fill the chip and add the slices in one more.
template <int TYPE, int LAST, bool SPLIT>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_kq_types_kernel(GemmArgs a) {
    const int bx = (int)blockIdx.x, begin = a.n_seg > 2 ? a.seg_begin[2] : a.seg_begin[1];
    if (bx < begin) kq_tile<TYPE, true, true, SPLIT>(a, static_cast<const uint8_t *>(a.Wp), bx);
    else kq_tile<LAST, true, true, SPLIT>(a, static_cast<const uint8_t *>(a.Wp_last), bx - begin);
}

// ---- expert launches ------------------------------------------------------------------------------------------------------
// 128 weight rows x the pairs of one tile of the list (1 to 128 of one expert) per workgroup of four waves.  A wave owns 32 rows
// and all pairs: a lane of the multiplied fragment holds one row, and the GEMM layout's slot (row, half of a chunk) is
// that lane's, so it forms the fragments of four MFMA steps from its own 32 or 40 bytes, in registers.  The activations go through LDS, k8-major as they lie in memory: 16-byte pieces at consecutive
// addresses both ways.  NT groups of 32 pairs: an expert's remainder costs the groups it fills.
// Bound by forming the weights (77 vector instructions per 2048 of them and wave, 112 of q6_K; of 77 about 300 cycles of a SIMD: a packed f16 instruction takes
// five, and_or and perm 4.5, a shift 2.4) next to multiplying them (33 cycles a product), at the 1.4 to 1.6 GHz that the chip holds with all
// of it busy, and by how evenly the tiles fill the chip.  Gate / up of 64 experts of 2 x 768 rows x 2048 (q4_K), 4800 pairs of a Zipf router
// (86 tiles, 44 of at most 32 pairs): 98 us with the staging waves of gemm_kq_kernel on tiles of 128 columns, 80 with fragments formed in
// registers, 70 with the larger tiles first (moe_sort) and and_or, 62 with a step's fragments formed between the products of the step
// before, three workgroups a CU kept (two: 67) and small tiles' activations in groups of up to four chunks; down projection of 2048 x 768:
// 53 -> 40 (q4_K), 56 -> 46 -> 43 (q6_K).  In turn on one card, fragments formed before the products / between them: gate / up 66.8 / 60.7 (rows by
// their slots), down q6_K 46.0 / 43.0, q4_K 39.1 / 39.4, which gains nothing.  113 MB of weights at the rate of a large copy: 22 us.
// Rows of a SwiGLU pair are dealt out so that a wave holds 16 gate rows and the 16 up rows of the same outputs, in one lane's
// registers e and e + 8.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// KG groups of four waves, each over its own part of the k-steps; the partial products meet in LDS.
// The k order of the sums is the 128-column tile's, within a group.
// MODE: REG_DENSE, REG_SPLIT (raw sums of slice blockIdx.z to a.part), REG_EXPERT (one group), REG_NORM (a pair with a.norm_part), REG_EXPERT_ROWS (a.x_slot).
enum { REG_DENSE, REG_SPLIT, REG_EXPERT, REG_NORM, REG_EXPERT_ROWS };
constexpr int reg_lds_bytes(int NT, int KG) { return KG * NT * 8192; }        // two buffers of activations per group; half the groups' sums
template <int TYPE, int NT, int MODE, int KG>
__device__ __forceinline__ void reg_tile(const GemmArgs &a, const uint8_t *wp, int bx, int t0, int t_end, int k0, int n_steps, u32x4 *lds) {
    constexpr bool EXPERT = MODE == REG_EXPERT || MODE == REG_EXPERT_ROWS, ROWS = MODE == REG_EXPERT_ROWS;
    // Activations of a chunk in LDS: [32 columns][16 of them][group of 8 of k][column], in 16-byte pieces.  A thread of ROWS brings a piece of a row, whose
    // eight would lie 256 bytes apart, all on the same banks: there a group takes 17 places.
    constexpr int K8 = ROWS ? 17 : 16, COLS = 16 * K8;
    constexpr int AHEAD = 4, STEP = NT * COLS;                 // chunks of weights on their way; pieces of a chunk's activations
    const int tid = threadIdx.x & 255, lane = tid & 63, hh = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    const int n_all = a.K / GK;
    // this group's k-steps [k0, k0 + n) and the rounds that every group walks (the barriers are the workgroup's)
    const int per = (n_steps + KG - 1) / KG;
    k0 += group * per;
    const int n = KG == 1 ? n_steps : n_steps - group * per < per ? n_steps - group * per : per;
    const bool pair = MODE != REG_SPLIT && a.y16_k8 != nullptr;
    const unsigned slot = 2 * (pair ? 16 * wave + (r & 15) + (r >> 4) * 64 : 32 * wave + r) + hh;
    wp += ((size_t)bx * n_all + k0) * PackedSub<TYPE>::CHUNK;
    const int n_blk = (a.T + 15) >> 4;
    const u32x4 *const xbase = ROWS ? reinterpret_cast<const u32x4 *>(a.X) : reinterpret_cast<const u32x4 *>(a.X + (size_t)(t0 >> 4) * 16 * a.K) + (size_t)k0 * 128;
    constexpr int X_CHUNK = ROWS ? 8 : 128;                    // pieces from a chunk's activations to the next one's
    unsigned xo[NT];                                           // 16-byte pieces from the tile's first block
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        if constexpr (ROWS) {
            const int s = t0 + 32 * i + (tid >> 3), of = a.x_slot[s < a.T ? s : a.T - 1];       // (slots past the tile's: any row, never stored)
            xo[i] = (of > 0 ? (unsigned)of / (unsigned)a.x_div : 0u) * (unsigned)(a.K / 8) + (unsigned)(tid & 7);
        } else {
            const int b = 2 * i + (tid >> 7), last = n_blk - 1 - (t0 >> 4);        // (blocks past the list re-read the last one, never stored)
            xo[i] = (unsigned)(b < last ? b : last) * (unsigned)(2 * a.K) + (unsigned)(tid & 127);
        }
    }
    const int put = ROWS ? (tid >> 7) * 8 * K8 + (tid & 7) * K8 + ((tid >> 3) & 15) : tid;
    u32x4 *xs = lds + group * 2 * STEP;
    float16v acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
    const int last = n > 0 ? n - 1 : 0;                        // (a group without steps of its own reads the first and multiplies none)
    if (n <= 0) { wp -= (size_t)k0 * PackedSub<TYPE>::CHUNK; }
    const u32x4 *const xb = n > 0 ? xbase : xbase - (size_t)k0 * 128;
    // (fewer on their way where more would cost a workgroup of a CU its registers)
    constexpr int RING = EXPERT && TYPE == MESH_Q6_K && NT > 2 ? 2 : AHEAD;
    PackedSub<TYPE> rw[RING];
    // Loads return in order: activations stored a step after they were asked for would have the weights asked for before them arrive
    // by then too, two chunks ahead instead of AHEAD.  Activations asked for XA steps before, against one: a batch of 32 decode steps of
    // four layers 5120 wide 821 -> 809 us, eight layers of a 40-token chunk 4096 wide 971 -> 953.  Two columns of tiles in a dense call with AHEAD spill (40 tokens: 995).
    constexpr int XA = NT == 1 ? AHEAD : NT > 2 ? 1 : 2;       // (the registers that are left at the occupancy)
    // Expert tiles: activations in groups of G chunks, 16 KB at most; a group is asked for while the one before it is multiplied.
    constexpr int G = EXPERT ? (NT > 2 ? 1 : 4 / NT) : 1, GROUP = 4 * COLS;
    u32x4 rx[EXPERT ? G * NT : XA * NT];
    auto fetch = [&](int kc) {
#pragma unroll
        for (int i = 0; i < G * NT; ++i) rx[i] = (xb + (size_t)(kc + i / NT < last ? kc + i / NT : last) * X_CHUNK)[xo[i % NT]];
    };
    if constexpr (EXPERT) {
        fetch(0);
#pragma unroll
        for (int i = 0; i < G * NT; ++i) xs[i * COLS + put] = rx[i];
        fetch(G);
    } else {
#pragma unroll
        for (int i = 0; i < NT; ++i) xs[i * 256 + tid] = xb[xo[i]];
#pragma unroll
        for (int v = 1; v <= XA; ++v)
#pragma unroll
            for (int i = 0; i < NT; ++i) rx[v % XA * NT + i] = (xb + (size_t)(v < last ? v : last) * 128)[xo[i]];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < RING; ++u) rw[u].load(wp + (size_t)(EXPERT || u < last ? u : last) * PackedSub<TYPE>::CHUNK, slot);
    lds_barrier();
    const int at = (lane & 15) + ((lane >> 4) & 1) * 8 * K8 + hh * K8;
    if constexpr (EXPERT) {
        // A step's fragments are formed between the products of the step before, whose issue leaves the vector ALU idle, and its activations
        // read ahead of those.  The barrier of a group of chunks stands before its last step: behind it the next group's activations
        // have landed, whose first fragments that step reads, and the buffer they lie in has been read by everybody a group ago.
        u32x4 f[NT];
        half8 w[2];
        w[0] = __builtin_bit_cast(half8, rw[0].form(0));
        const u32x4 *x = xs + at;
        int to_next = GROUP;
#pragma unroll
        for (int j = 0; j < NT; ++j) f[j] = x[j * COLS];
        for (int kc0 = 0; kc0 < per; kc0 += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const int kc = kc0 + u, c = u % G;
#pragma unroll
                for (int st = 0; st < 4; ++st) {
                    const bool turn = c == G - 1 && st == 3;
                    if (turn) {
                        lds_barrier();
                        x += to_next;
                        to_next = -to_next;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    w[(st + 1) & 1] = __builtin_bit_cast(half8, st < 3 ? rw[u % RING].form(st + 1) : rw[(u + 1) % RING].form(0));
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[st & 1], __builtin_bit_cast(half8, f[j]), acc[j], 0, 0, 0);
                        f[j] = x[(turn ? 0 : st < 3 ? c * STEP + (st + 1) * 2 * K8 : (c + 1) * STEP) + j * COLS];
                    }
#pragma unroll
                    for (int j = 0; j < NT; ++j) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, (24 + NT - 1) / NT, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (c == 0 && st == 0) {
                        // (the other buffer's last readers stand before the barrier of the group before)
                        u32x4 *const nx = const_cast<u32x4 *>(x) - at + put + to_next;
#pragma unroll
                        for (int i = 0; i < G * NT; ++i) nx[i * COLS] = rx[i];
                        fetch(kc + 2 * G);
                    }
                    if (st == 2) rw[u % RING].load(wp + (size_t)(kc + RING < last ? kc + RING : last) * PackedSub<TYPE>::CHUNK, slot);
                }
            }
        }
    } else
    for (int kc0 = 0; kc0 < per; kc0 += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int kc = kc0 + u;
            // (the other buffer was read a step ago; the step's barrier hands it over)
#pragma unroll
            for (int i = 0; i < NT; ++i) xs[((u + 1) & 1) * STEP + i * 256 + tid] = rx[(u + 1) % XA * NT + i];
#pragma unroll
            for (int i = 0; i < NT; ++i) rx[(u + 1) % XA * NT + i] = (xb + (size_t)(kc + 1 + XA < last ? kc + 1 + XA : last) * 128)[xo[i]];
            const u32x4 *x = xs + (u & 1) * STEP + at;
            if (kc < n) {
                u32x4 f[2][NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) f[0][j] = x[j * 256];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int st = 0; st < 4; ++st) {
                    if (st < 3)
#pragma unroll
                        for (int j = 0; j < NT; ++j) f[(st + 1) & 1][j] = x[j * 256 + (st + 1) * 32];
                    const half8 w = __builtin_bit_cast(half8, rw[u].form(st));
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, __builtin_bit_cast(half8, f[st & 1][j]), acc[j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            rw[u].load(wp + (size_t)(kc + AHEAD < last ? kc + AHEAD : last) * PackedSub<TYPE>::CHUNK, slot);
            lds_barrier();
        }
    }
    float inv_rms = 1.0f;
    float *const nrm = reinterpret_cast<float *>(lds) + reg_lds_bytes(NT, KG) / 4;     // [8 KG][32 columns]
    if (MODE == REG_NORM && a.norm_part) {
        // (after the weight stream: before it, the wave would wait for them ahead of its first tile loads)
        const int cols = a.T > 16 ? 32 : 16;
        float ss = 0.f;
        if (r < cols)
            for (int p = threadIdx.x >> 5; p < a.norm_parts; p += 8 * KG) ss += a.norm_part[(size_t)p * cols + r];
        nrm[threadIdx.x] = ss;
    }
    // the groups' sums, the upper half of them added to the lower until one is left
#pragma unroll
    for (int half = KG / 2; half > 0; half /= 2) {
        float *part = reinterpret_cast<float *>(lds) + ((group % half) * 4 + wave) * NT * 1024 + lane;
        if (group >= half && group < 2 * half) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) part[(j * 16 + e) * 64] = acc[j][e];
        }
        __syncthreads();
        if (group < half) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[j][e] += part[(j * 16 + e) * 64];
        }
        if (half > 1) __syncthreads();
    }
    if (group > 0) return;
    if (MODE == REG_NORM && a.norm_part) {
        float ss = 0.f;
        for (int q = 0; q < 8 * KG; ++q) ss += nrm[q * 32 + r];
        inv_rms = 1.0f / sqrtf(ss / (float)a.K + a.norm_eps);
    }
    if constexpr (MODE == REG_SPLIT) {
        // slice of a split launch: the raw sums go to part[slice][token][row of the launch]
        const size_t ld = (size_t)gridDim.x * GM;
        float *P = a.part + (size_t)blockIdx.z * a.T * ld + (size_t)bx * GM + 32 * wave + 4 * hh;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int t = t0 + 32 * j + r;
            if (t >= t_end) continue;
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4)
                *reinterpret_cast<float4 *>(P + (size_t)t * ld + 8 * e4) = make_float4(acc[j][4 * e4], acc[j][4 * e4 + 1], acc[j][4 * e4 + 2], acc[j][4 * e4 + 3]);
        }
        return;
    }
    if (pair) {
        const int t_pad = (t_end + 15) & ~15;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int t = t0 + 32 * j + r;
            if (t >= t_pad) continue;
#pragma unroll
            for (int e4 = 0; e4 < 2; ++e4) {
                const int m = bx * (GM / 2) + 16 * wave + 8 * e4 + 4 * hh;
                if (m >= a.M) continue;
                float o[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float g = acc[j][4 * e4 + c] * inv_rms, up = acc[j][8 + 4 * e4 + c] * inv_rms;
                    o[c] = t < t_end ? g / (1.0f + expf(-g)) * up : 0.f;       // padding columns of the last token block hold zeros
                }
                note_f16_clamp(a.sat, o[0], o[1], o[2], o[3]);
                *reinterpret_cast<uint2 *>(a.y16_k8 + (size_t)(t >> 4) * 16 * a.M + ((size_t)(m >> 3) * 16 + (t & 15)) * 8 + (m & 7)) =
                    make_uint2(pack_h2(o[0], o[1]), pack_h2(o[2], o[3]));
            }
        }
        return;
    }
    float *Y = a.Y;
    const float *bias = MODE == REG_DENSE ? a.bias : nullptr, *res = MODE == REG_DENSE ? a.residual : nullptr;
    int M = a.M, ldy = a.ldy, mb0 = bx * GM;
    if (MODE == REG_DENSE && a.n_seg > 1) {
        // (selected, not indexed: a dynamically indexed kernel-argument array would be spilled to scratch)
        const int sg = (bx >= a.seg_begin[1] ? 1 : 0) + (a.n_seg > 2 && bx >= a.seg_begin[2] ? 1 : 0);
        Y = sg == 0 ? a.seg_Y[0] : sg == 1 ? a.seg_Y[1] : a.seg_Y[2];
        bias = sg == 0 ? a.seg_bias[0] : sg == 1 ? a.seg_bias[1] : a.seg_bias[2];
        M = sg == 0 ? a.seg_M[0] : sg == 1 ? a.seg_M[1] : a.seg_M[2];
        ldy = sg == 0 ? a.seg_ldy[0] : sg == 1 ? a.seg_ldy[1] : a.seg_ldy[2];
        mb0 = (bx - (sg == 0 ? 0 : sg == 1 ? a.seg_begin[1] : a.seg_begin[2])) * GM;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int t = t0 + 32 * j + r;
        if (t >= t_end) continue;
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            const int m = mb0 + 32 * wave + 8 * e4 + 4 * hh;
            if (m >= M) continue;              // M is a multiple of 4 for every projection
            float4 o = make_float4(acc[j][4 * e4], acc[j][4 * e4 + 1], acc[j][4 * e4 + 2], acc[j][4 * e4 + 3]);
            if (bias) {
                const float4 b = *reinterpret_cast<const float4 *>(bias + m);
                o.x += b.x; o.y += b.y; o.z += b.z; o.w += b.w;
            }
            if (res) {
                const float4 q = *reinterpret_cast<const float4 *>(res + (size_t)t * a.ldres + m);
                o.x += q.x; o.y += q.y; o.z += q.z; o.w += q.w;
            }
            *reinterpret_cast<float4 *>(Y + (size_t)t * ldy + m) = o;
        }
    }
}
// REG_EXPERT_ROWS: a tile's activations straight from the rows the router has left, a token's 128 bytes of a chunk by eight lanes, where a launch before had to
// sort copies of them: 600 tokens of 64 experts, top 8, gather 11.8 + gate / up 57 us before, 61 now (and the router 13 -> 14.4); eight expert
// layers 40 tokens 972 -> 920 us, 200 1249 -> 1193, 600 1865 -> 1777, 2000 4375 -> 4112.
template <int TYPE, int MODE>
__global__ __launch_bounds__(256, 2) void gemm_expert_kernel(GemmArgs a) {
    __shared__ u32x4 xs[2 * 4 * (MODE == REG_EXPERT_ROWS ? 272 : 256)];
    // workgroups go to the eight XCDs in turn: every row block of a tile on one of them, whose L2 fetches the tile's activations once
    // (gate / up as above: 66 us then, 82 with the row blocks dealt over the XCDs)
    const int g = (int)(blockIdx.y * gridDim.x + blockIdx.x), bx = (g >> 3) % (int)gridDim.x, nt = *a.n_tiles;
    int eight = (g >> 3) / (int)gridDim.x;                     // of the list, eight tiles at a time
    // Down: the list's halves in turn, so that a CU has large tiles, bound by their products, beside small ones, bound by forming weights
    // (2048 x 768 as above, largest first / in halves: q6_K 43.5 / 43.0 us, q4_K 39.0 / 39.4: next to nothing).  Gate / up walk longer rows and would
    // end behind their largest tiles (65 -> 71).
    if (!a.y16_k8) {
        const int n8 = (nt + 7) >> 3;
        if (eight >= n8) return;
        eight = (eight & 1) ? ((n8 + 1) >> 1) + (eight >> 1) : eight >> 1;
    }
    const int by = eight * 8 + (g & 7);
    if (by >= nt) return;
    const int4 tl = reinterpret_cast<const int4 *>(a.tiles)[by];
    const uint8_t *wp = static_cast<const uint8_t *>(a.Wp) + (size_t)tl.x * a.expert_stride;
    const int n = a.K / GK;
    switch ((tl.z + 31) >> 5) {
        case 1: return reg_tile<TYPE, 1, MODE, 1>(a, wp, bx, tl.y, tl.y + tl.z, 0, n, xs);
        case 2: return reg_tile<TYPE, 2, MODE, 1>(a, wp, bx, tl.y, tl.y + tl.z, 0, n, xs);
        case 3: return reg_tile<TYPE, 3, MODE, 1>(a, wp, bx, tl.y, tl.y + tl.z, 0, n, xs);
        default: return reg_tile<TYPE, 4, MODE, 1>(a, wp, bx, tl.y, tl.y + tl.z, 0, n, xs);
    }
}
// Dense calls of at most 64 tokens, at most 32 or 64 columns.  A launch of few workgroups per CU needs its waves from K: four groups
// (16 waves), two in a slice of a split launch, whose k range is short already.  Gate / up of 2 x 14336 rows x 4096 (q4_K, 66 MB):
// 41 us at 40 tokens with the staging waves of gemm_kq_kernel, 31 with two groups, 28 with four; 22 at 20 tokens; down projection of
// 4096 x 14336 (q6_K): 23 -> 18 us.  From 65 tokens on every wave reads every activation fragment, LDS gives out and the
// 128-column tile is the better one (128 tokens: 45 us against 48 for gate / up, but 29 against 27 and 16 against 13 for the others).
template <int TYPE, int NT, int MODE, int KG>
__global__ __launch_bounds__(256 * KG, 4) void gemm_reg_kernel(GemmArgs a) {
    __shared__ u32x4 lds[reg_lds_bytes(NT, KG) / 16 + (MODE == REG_NORM ? 64 * KG : 0)];
    const int n_all = a.K / GK, k0 = MODE == REG_SPLIT ? (int)blockIdx.z * a.k_per_split : 0;
    const int n = MODE == REG_SPLIT && n_all - k0 > a.k_per_split ? a.k_per_split : n_all - k0;
    reg_tile<TYPE, NT, MODE, KG>(a, static_cast<const uint8_t *>(a.Wp), (int)blockIdx.x, 0, a.T, k0, n, lds);
}

// ---- the same product on a 256 x 128 workgroup tile ----------------------------------------------------------
// What bounds the 128 x 128 kernel above is operand traffic, not the matrix cores: a wave that owns 64 x 64 of the tile
// needs 1 KB of fragments per v_mfma_f32_32x32x16_f16 (2 x 2 register blocking: two weight fragments from LDS and two
// activation fragments from memory per four MFMAs), and four SIMDs at one MFMA per 32 cycles then ask the vector memory
// path for its whole 64 B per cycle and LDS for three quarters of its 128.  Here a matrix-core wave owns 128 weight rows x
// 64 tokens (4 x 2 blocking, 128 accumulator registers): 0.5 KB of weight fragments and 0.25 KB of activation fragments
// per MFMA, half of either path.  The price is one workgroup per CU and one matrix-core wave per SIMD, which therefore
// fetches the weight fragments of the next k16 step before it multiplies the current one; a staging wave shares the
// SIMD and dequantises while the MFMAs execute.
// Production layout only (GEMM-layout weights, k8-major activations), K not split, an even number of 128-row blocks:
// a workgroup takes row blocks 2 * blockIdx.x and + 1, one per pair of matrix-core waves, so everything that depends on
// the row block (matrix of a multi-matrix launch, SwiGLU pairing) is per wave.
constexpr int BGM = 256;
template <int TYPE>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_big_kernel(GemmArgs a) {
    extern __shared__ __align__(16) _Float16 gemm_smem[];
    _Float16 *Ws = gemm_smem;                                  // [2][BGM][LDS_LD]
    using Sub = PackedSub<TYPE>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = blockIdx.y * GN;
    const int n_steps = a.K / GK;

    if (wave >= 4) {
        // ---- staging waves: a slot of both row blocks
        const int st = staged_slot(tid - 256);
        const uint8_t *chunk0 = static_cast<const uint8_t *>(a.Wp) + (size_t)(2 * blockIdx.x) * n_steps * Sub::CHUNK;
        const uint8_t *chunk1 = chunk0 + (size_t)n_steps * Sub::CHUNK;
        _Float16 *dst = Ws + (st >> 1) * LDS_LD + 8 * (st & 1);
        StagedSlot offsets = staged_offsets(st);
        Sub rw[2][2];
        auto fetch = [&](int kc, Sub (&w)[2]) {
            w[0].load_staged(chunk0 + (size_t)kc * Sub::CHUNK, offsets);
            w[1].load_staged(chunk1 + (size_t)kc * Sub::CHUNK, offsets);
        };
        auto stage = [&](int buf, const Sub (&w)[2]) {
            store_sub(w[0], dst + buf * BGM * LDS_LD);
            store_sub(w[1], dst + (buf * BGM + GM) * LDS_LD);
        };
        fetch(0, rw[0]);
        fetch(n_steps > 1 ? 1 : 0, rw[1]);
        stage(0, rw[0]);
        lds_barrier();
        for (int kc0 = 0; kc0 < n_steps; kc0 += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int kc = kc0 + u;
                if (kc >= n_steps) break;
                fetch(kc + 2 < n_steps ? kc + 2 : n_steps - 1, rw[u]);
                if (kc + 1 < n_steps) stage(u ^ 1, rw[u ^ 1]);
                lds_barrier();
            }
        }
        return;
    }

    // ---- multiplying waves: row block (wave & 1), token half (wave >> 1)
    const int vb = 2 * (int)blockIdx.x + (wave & 1);           // this wave's 128-row block of the launch
    const int wm = (wave & 1) * GM, wn = (wave >> 1) * 64;
    float16v acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    const int n_blk = (a.T + 15) >> 4, n_g = n_steps * (GK / 16);
    const _Float16 *bp[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int tok = t0 + wn + 32 * i + (lane & 31);
        const int blk = (tok >> 4) < n_blk ? (tok >> 4) : n_blk - 1;
        bp[i] = a.X + (size_t)blk * 16 * a.K + ((lane >> 5) * 16 + (tok & 15)) * 8;
    }
    half8 ring[GK / 16][2];
#pragma unroll
    for (int ks = 0; ks < GK / 16; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i) ring[ks][i] = *reinterpret_cast<const half8 *>(bp[i] + (size_t)(ks < n_g ? ks : n_g - 1) * 256);
    const int a_off = (wm + (lane & 31)) * LDS_LD + 8 * (lane >> 5);
    lds_barrier();
    for (int kc = 0; kc < n_steps; ++kc) {
        const _Float16 *Wb = Ws + (kc & 1) * BGM * LDS_LD + a_off;
        half8 af[2][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) af[0][i] = *reinterpret_cast<const half8 *>(Wb + 32 * i * LDS_LD);
#pragma unroll
        for (int ks = 0; ks < GK / 16; ++ks) {
            if (ks + 1 < GK / 16) {
#pragma unroll
                for (int i = 0; i < 4; ++i) af[(ks + 1) & 1][i] = *reinterpret_cast<const half8 *>(Wb + 32 * i * LDS_LD + 16 * (ks + 1));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[ks & 1][i], ring[ks][j], acc[i][j], 0, 0, 0);
            int gn = (kc + 1) * (GK / 16) + ks;
            gn = gn < n_g ? gn : n_g - 1;
#pragma unroll
            for (int i = 0; i < 2; ++i) ring[ks][i] = *reinterpret_cast<const half8 *>(bp[i] + (size_t)gn * 256);
            // Issue order inside the step: the next step's four fragment reads go out between the first MFMAs (an MFMA
            // holds the matrix pipe for 32 cycles, the wave is free to issue meanwhile), the two activation refills after
            // the last.  Left to itself the scheduler puts the reads behind all eight MFMAs, and the next step then
            // starts by waiting out the LDS latency.
            if (ks + 1 < GK / 16) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);      // one LDS read
                }
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
            } else {
                __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);              // the two global loads
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_barrier();
    }

    // D[m][t]: lane holds column t = lane % 32 and rows 8 * (e / 4) + 4 * (lane / 32) + e % 4 of each 32 x 32 block
    if (a.y16_k8) {
        // SwiGLU pair: the row block's rows 0..63 are gate rows, 64..127 the up rows of the same outputs: blocks
        // acc[0..1] and acc[2..3] of this very lane
        const int t_pad = (a.T + 15) & ~15;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int t = t0 + wn + 32 * j + (lane & 31);
                if (t >= t_pad) continue;
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const int m = vb * (GM / 2) + 32 * i + 8 * e4 + 4 * (lane >> 5);
                    if (m >= a.M) continue;
                    float o[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const float g = acc[i][j][4 * e4 + c], u = acc[i + 2][j][4 * e4 + c];
                        o[c] = t < a.T ? g / (1.0f + expf(-g)) * u : 0.f;
                    }
                    note_f16_clamp(a.sat, o[0], o[1], o[2], o[3]);
                    *reinterpret_cast<uint2 *>(a.y16_k8 + (size_t)(t >> 4) * 16 * a.M + ((size_t)(m >> 3) * 16 + (t & 15)) * 8 + (m & 7)) =
                        make_uint2(pack_h2(o[0], o[1]), pack_h2(o[2], o[3]));
                }
            }
        return;
    }
    float *Y = a.Y;
    const float *bias = a.bias;
    int M = a.M, ldy = a.ldy, mb0 = vb * GM;
    if (a.n_seg > 1) {
        const int sg = (vb >= a.seg_begin[1] ? 1 : 0) + (a.n_seg > 2 && vb >= a.seg_begin[2] ? 1 : 0);
        Y = sg == 0 ? a.seg_Y[0] : sg == 1 ? a.seg_Y[1] : a.seg_Y[2];
        bias = sg == 0 ? a.seg_bias[0] : sg == 1 ? a.seg_bias[1] : a.seg_bias[2];
        M = sg == 0 ? a.seg_M[0] : sg == 1 ? a.seg_M[1] : a.seg_M[2];
        ldy = sg == 0 ? a.seg_ldy[0] : sg == 1 ? a.seg_ldy[1] : a.seg_ldy[2];
        mb0 = (vb - (sg == 0 ? 0 : sg == 1 ? a.seg_begin[1] : a.seg_begin[2])) * GM;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = t0 + wn + 32 * j + (lane & 31);
            if (t >= a.T) continue;
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const int m = mb0 + 32 * i + 8 * e4 + 4 * (lane >> 5);
                if (m >= M) continue;
                float4 o = make_float4(acc[i][j][4 * e4], acc[i][j][4 * e4 + 1], acc[i][j][4 * e4 + 2], acc[i][j][4 * e4 + 3]);
                if (bias) {
                    const float4 b = *reinterpret_cast<const float4 *>(bias + m);
                    o.x += b.x; o.y += b.y; o.z += b.z; o.w += b.w;
                }
                if (a.residual) {
                    const float4 r = *reinterpret_cast<const float4 *>(a.residual + (size_t)t * a.ldres + m);
                    o.x += r.x; o.y += r.y; o.z += r.z; o.w += r.w;
                }
                *reinterpret_cast<float4 *>(Y + (size_t)t * ldy + m) = o;
            }
        }
}

template <int TYPE>
static int launch_gemm_big(const GemmArgs &k, int row_blocks, int t_blocks, hipStream_t stream) {
    constexpr size_t smem = sizeof(_Float16) * 2 * BGM * LDS_LD;
    static bool attr_set = false;
    if (!attr_set) {
        MESH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_big_kernel<TYPE>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_set = true;
    }
    MESH_LAUNCH((gemm_big_kernel<TYPE>), dim3((unsigned)(row_blocks / 2), (unsigned)t_blocks), dim3(GEMM_THREADS), smem, stream, k);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// Second kernel of a split launch: adds the slices of part[slice][token][row] in slice order and applies the epilogue
// of the unsplit kernel.  One thread per (token, four consecutive rows); rows run fastest, so partial reads and output
// writes are contiguous.
__global__ __launch_bounds__(256) void gemm_splitk_epilogue_kernel(GemmArgs a, int row_blocks) {
    const size_t ld = (size_t)row_blocks * GM;
    const int t_pad = a.y16_k8 ? (a.T + 15) & ~15 : a.T;
    const int per_block = a.y16_k8 ? GM / 8 : GM / 4;          // threads per row block: 64 gate rows or 128 rows, four each
    const size_t n = (size_t)t_pad * row_blocks * per_block;
    for (size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x; idx < n; idx += (size_t)gridDim.x * 256) {
        const int q = (int)(idx % per_block), bx = (int)((idx / per_block) % row_blocks), t = (int)(idx / ((size_t)per_block * row_blocks));
        auto sum4 = [&](size_t row) {
            // four slices in flight at a time (indices past the end re-read the last slice and are not added)
            float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
            for (int z0 = 0; z0 < a.ksplit; z0 += 4) {
                float4 p[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int z = z0 + u < a.ksplit ? z0 + u : a.ksplit - 1;
                    p[u] = *reinterpret_cast<const float4 *>(a.part + ((size_t)z * a.T + t) * ld + row);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (z0 + u < a.ksplit) { o.x += p[u].x; o.y += p[u].y; o.z += p[u].z; o.w += p[u].w; }
            }
            return o;
        };
        if (a.y16_k8) {
            const int m = bx * (GM / 2) + 4 * q;
            if (m >= a.M) continue;
            float o[4] = {0.f, 0.f, 0.f, 0.f};                 // padding columns of the last token block hold zeros
            if (t < a.T) {
                const float4 g = sum4((size_t)bx * GM + 4 * q), u = sum4((size_t)bx * GM + GM / 2 + 4 * q);
                o[0] = g.x / (1.0f + expf(-g.x)) * u.x; o[1] = g.y / (1.0f + expf(-g.y)) * u.y;
                o[2] = g.z / (1.0f + expf(-g.z)) * u.z; o[3] = g.w / (1.0f + expf(-g.w)) * u.w;
            }
            note_f16_clamp(a.sat, o[0], o[1], o[2], o[3]);
            *reinterpret_cast<uint2 *>(a.y16_k8 + (size_t)(t >> 4) * 16 * a.M + ((size_t)(m >> 3) * 16 + (t & 15)) * 8 + (m & 7)) =
                make_uint2(pack_h2(o[0], o[1]), pack_h2(o[2], o[3]));
            continue;
        }
        float *Y = a.Y;
        const float *bias = a.bias;
        int M = a.M, ldy = a.ldy, mb0 = bx * GM, kind = a.kind[0];
        if (a.n_seg > 1) {
            const int sg = (bx >= a.seg_begin[1] ? 1 : 0) + (a.n_seg > 2 && bx >= a.seg_begin[2] ? 1 : 0);
            kind = sg == 0 ? a.kind[0] : sg == 1 ? a.kind[1] : a.kind[2];
            Y = sg == 0 ? a.seg_Y[0] : sg == 1 ? a.seg_Y[1] : a.seg_Y[2];
            bias = sg == 0 ? a.seg_bias[0] : sg == 1 ? a.seg_bias[1] : a.seg_bias[2];
            M = sg == 0 ? a.seg_M[0] : sg == 1 ? a.seg_M[1] : a.seg_M[2];
            ldy = sg == 0 ? a.seg_ldy[0] : sg == 1 ? a.seg_ldy[1] : a.seg_ldy[2];
            mb0 = (bx - (sg == 0 ? 0 : sg == 1 ? a.seg_begin[1] : a.seg_begin[2])) * GM;
        }
        const int m = mb0 + 4 * q;
        if (m >= M) continue;
        float4 o = sum4((size_t)bx * GM + 4 * q);
        if (bias) {
            const float4 b = *reinterpret_cast<const float4 *>(bias + m);
            o.x += b.x; o.y += b.y; o.z += b.z; o.w += b.w;
        }
        if (a.rope.pos && kind != GEMV_KIND_PLAIN) {
            // rows m..m+3 of a q / k / v projection: two neighbouring pairs of one head (head_dim % 4 == 0)
            const int hd = a.rope.head_dim, head = m / hd, dd = m - head * hd, pos = a.rope.pos[t];
            if (kind != GEMV_KIND_V) {
                if (dd < a.rope.n_rot) {
                    float sn, cs;
                    sincosf((float)pos * a.rope.inv_freq[dd >> 1], &sn, &cs);
                    const float x0 = o.x, x1 = o.y;
                    o.x = x0 * cs - x1 * sn; o.y = x0 * sn + x1 * cs;
                }
                if (dd + 2 < a.rope.n_rot) {
                    float sn, cs;
                    sincosf((float)pos * a.rope.inv_freq[(dd >> 1) + 1], &sn, &cs);
                    const float x0 = o.z, x1 = o.w;
                    o.z = x0 * cs - x1 * sn; o.w = x0 * sn + x1 * cs;
                }
            }
            if (kind == GEMV_KIND_Q) {
                *reinterpret_cast<float4 *>(Y + (size_t)t * ldy + m) = o;
            } else {
                uint16_t *cache = kind == GEMV_KIND_K ? a.rope.kcache : a.rope.vcache;
                *reinterpret_cast<uint2 *>(cache + (((size_t)a.rope.seq[t] * a.rope.n_kv + head) * a.rope.n_ctx + pos) * hd + dd) =
                    make_uint2(pack_h2(o.x, o.y), pack_h2(o.z, o.w));
            }
            continue;
        }
        if (a.residual) {
            const float4 r = *reinterpret_cast<const float4 *>(a.residual + (size_t)t * a.ldres + m);
            o.x += r.x; o.y += r.y; o.z += r.z; o.w += r.w;
        }
        *reinterpret_cast<float4 *>(Y + (size_t)t * ldy + m) = o;
    }
}

// The same for one matrix whose result is the hidden state, with the RMS norm of the next launch's input: a workgroup per token holds
// the row, so the norm costs a reduction over the workgroup instead of a launch that reads the row again.  The sums are those of
// the kernel above, in its order.  Bound by the latency of its loads, all of a row's in flight at once; two launches of 5 to 8 us
// become one of about that.  Chunks through eight 8B-shaped layers, us with it / without: 20 tokens 795 / 841, 40 921 / 970, 64 963 / 1082,
// 100 1157 / 1273, 200 1596 / 1704, 333 behind 1500 2137 / 2210, 512 2500 / 2625, 800 3849 / 3876; four 32B-shaped layers 40 tokens
// 734 / 754, 150 1296 / 1338, 400 2217 / 2274: at every count that splits.
constexpr int SN_THREADS = 512;
static_assert(GEMM_NORM_ROW_MAX == 2 * 8 * SN_THREADS, "two groups of eight a thread");
template <int NG>              // groups of 8 elements a thread has: rows of up to NG * 4096
__global__ __launch_bounds__(SN_THREADS) void gemm_splitk_epilogue_norm_kernel(GemmArgs a, int row_blocks) {
    __shared__ float s_ss[SN_THREADS / 64];
    const size_t ld = (size_t)row_blocks * GM;
    const int t = blockIdx.x, tid = threadIdx.x;
    const bool live = t < a.T;
    float4 v[NG][2], w[NG][2], res[NG][2];
    float ss = 0.f;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int i = 8 * (tid + SN_THREADS * g);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v[g][h] = w[g][h] = res[g][h] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!live || i >= a.M) continue;
            w[g][h] = *reinterpret_cast<const float4 *>(a.next_w + i + 4 * h);
            res[g][h] = *reinterpret_cast<const float4 *>(a.residual + (size_t)t * a.ldres + i + 4 * h);
        }
    }
    for (int z0 = 0; z0 < a.ksplit; z0 += 4) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int i = 8 * (tid + SN_THREADS * g);
            if (!live || i >= a.M) continue;
            float4 p[4][2];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int z = z0 + u < a.ksplit ? z0 + u : a.ksplit - 1;
                const float *src = a.part + ((size_t)z * a.T + t) * ld + i;
                p[u][0] = *reinterpret_cast<const float4 *>(src);
                p[u][1] = *reinterpret_cast<const float4 *>(src + 4);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (z0 + u < a.ksplit)
#pragma unroll
                    for (int h = 0; h < 2; ++h) { v[g][h].x += p[u][h].x; v[g][h].y += p[u][h].y; v[g][h].z += p[u][h].z; v[g][h].w += p[u][h].w; }
        }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int i = 8 * (tid + SN_THREADS * g);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float4 &o = v[g][h];
            o.x += res[g][h].x; o.y += res[g][h].y; o.z += res[g][h].z; o.w += res[g][h].w;
            if (live && i < a.M) *reinterpret_cast<float4 *>(a.Y + (size_t)t * a.ldy + i + 4 * h) = o;
            ss += (o.x * o.x + o.y * o.y) + (o.z * o.z + o.w * o.w);
        }
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) s_ss[tid >> 6] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int k = 0; k < SN_THREADS / 64; ++k) tot += s_ss[k];
    const float sc = 1.0f / sqrtf(tot / (float)a.M + a.next_eps);
    _Float16 *yb = a.next_x16 + (size_t)(t >> 4) * 16 * a.M + (size_t)(t & 15) * 8;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int i = 8 * (tid + SN_THREADS * g);
        if (i >= a.M) continue;
        float o[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            o[4 * h] = v[g][h].x * sc * w[g][h].x; o[4 * h + 1] = v[g][h].y * sc * w[g][h].y;
            o[4 * h + 2] = v[g][h].z * sc * w[g][h].z; o[4 * h + 3] = v[g][h].w * sc * w[g][h].w;
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) note_f16_clamp(a.sat, o[2 * h], o[2 * h + 1]);
        *reinterpret_cast<uint4 *>(yb + (size_t)(i >> 3) * 128) = make_uint4(pack_h2(o[0], o[1]), pack_h2(o[2], o[3]), pack_h2(o[4], o[5]), pack_h2(o[6], o[7]));
    }
}

bool gemm_norm_rides(const GemmArgs &a) {
    return a.n_seg <= 1 && !a.y16_k8 && !a.bias && a.residual && !a.tiles && a.M % 8 == 0 && a.M <= GEMM_NORM_ROW_MAX &&
           a.ldy % 4 == 0 && a.ldres % 4 == 0 && gemm_split_count(a) > 1;
}

int gemm_add_slices(const GemmArgs &k, int row_blocks, hipStream_t stream) {
    if (k.next_x16) {
        const dim3 grid((unsigned)((k.T + 15) & ~15)), block(SN_THREADS);
        if (k.M <= 8 * SN_THREADS) MESH_LAUNCH(gemm_splitk_epilogue_norm_kernel<1>, grid, block, 0, stream, k, row_blocks);
        else MESH_LAUNCH(gemm_splitk_epilogue_norm_kernel<2>, grid, block, 0, stream, k, row_blocks);
        MESH_LAUNCH_CHECK();
        return MESH_OK;
    }
    const int t_pad = k.y16_k8 ? (k.T + 15) & ~15 : k.T;
    const size_t n = (size_t)t_pad * row_blocks * (k.y16_k8 ? GM / 8 : GM / 4);
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
    MESH_LAUNCH(gemm_splitk_epilogue_kernel, dim3(blocks), dim3(256), 0, stream, k, row_blocks);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

template <int TYPE, bool PACKED, bool XDIRECT, bool SPLIT>
static int launch_gemm_kernel(const GemmArgs &k, dim3 grid, hipStream_t stream) {
    // two stages of the weight slab, and of the activation slab unless the activations bypass LDS: 73 728 / 36 864 B
    constexpr size_t smem = sizeof(_Float16) * 2 * (GM + (XDIRECT ? 0 : GN)) * LDS_LD;
    static bool attr_set = false;
    if (!attr_set) {
        MESH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_kq_kernel<TYPE, PACKED, XDIRECT, SPLIT>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_set = true;
    }
    MESH_LAUNCH((gemm_kq_kernel<TYPE, PACKED, XDIRECT, SPLIT>), grid, dim3(GEMM_THREADS), smem, stream, k);
    MESH_LAUNCH_CHECK();
    return SPLIT ? gemm_add_slices(k, (int)grid.x, stream) : MESH_OK;
}

template <int TYPE, int LAST, bool SPLIT>
static int launch_gemm_types(const GemmArgs &k, dim3 grid, hipStream_t stream) {
    constexpr size_t smem = sizeof(_Float16) * 2 * GM * LDS_LD;
    MESH_LAUNCH((gemm_kq_types_kernel<TYPE, LAST, SPLIT>), grid, dim3(GEMM_THREADS), smem, stream, k);
    MESH_LAUNCH_CHECK();
    return SPLIT ? gemm_add_slices(k, (int)grid.x, stream) : MESH_OK;
}

// groups of waves along K: four where a CU gets one workgroup (16 waves), two where it gets several or K is split already
template <int TYPE, int NT, int MODE>
static int launch_gemm_reg(const GemmArgs &k, dim3 grid, hipStream_t stream) {
    if (k.ksplit > 1) MESH_LAUNCH((gemm_reg_kernel<TYPE, NT, REG_SPLIT, 2>), grid, dim3(512), 0, stream, k);
    else if ((int)grid.x > gt_n_cu()) MESH_LAUNCH((gemm_reg_kernel<TYPE, NT, MODE, 2>), grid, dim3(512), 0, stream, k);
    else MESH_LAUNCH((gemm_reg_kernel<TYPE, NT, MODE, 4>), grid, dim3(1024), 0, stream, k);
    MESH_LAUNCH_CHECK();
    return k.ksplit > 1 ? gemm_add_slices(k, (int)grid.x, stream) : MESH_OK;
}

template <int TYPE, bool PACKED, bool XDIRECT>
static int launch_gemm(const GemmArgs &k, dim3 grid, hipStream_t stream) {
    // calls of at most 64 tokens on the production layout (GEMM-layout weights, k8-major activations)
    if constexpr (PACKED && XDIRECT) {
        if (k.T <= GN / 2 && k.narrow_tile) return k.T <= GN / 4 ? launch_gemm_reg<TYPE, 1, REG_DENSE>(k, grid, stream) : launch_gemm_reg<TYPE, 2, REG_DENSE>(k, grid, stream);
    }
    return k.ksplit > 1 ? launch_gemm_kernel<TYPE, PACKED, XDIRECT, true>(k, grid, stream) : launch_gemm_kernel<TYPE, PACKED, XDIRECT, false>(k, grid, stream);
}

// slices of K for a launch of row_blocks x t_blocks workgroups (1: not split); *k_per_split = k-steps per slice
static int split_plan(const GemmArgs &a, int row_blocks, int t_blocks, int *k_per_split) {
    const int n_all = a.K / GK;
    *k_per_split = n_all;
    if (!a.part) return 1;
    const int wgs = row_blocks * t_blocks, ncu = gt_n_cu();
    int ks = 1;
    while (ks < 16 && wgs * ks * 2 <= ncu && n_all / (ks * 2) >= 8 &&
           (size_t)(ks * 2) * a.T * row_blocks * GM * sizeof(float) <= a.part_bytes) ks *= 2;
    // Any number where each keeps 1280 of K, as in gt_plan, us: two / three slices of 2048 x 4096 at 600 tokens (160 / 240 workgroups of 256 CUs) eight layers of
    // the expert shard 1897 / 1876; four / six of 5120 rows, four 32B-shaped layers of 40 tokens 683 / 650, without f16 copies 100 940 / 880, 250 1580 / 1446.
    for (int more = ks + 1, most = std::min({16, ncu / wgs, n_all / 20}); more <= most && (size_t)more * a.T * row_blocks * GM * sizeof(float) <= a.part_bytes; ++more) ks = more;
    if (ks <= 1) return 1;
    *k_per_split = (n_all + ks - 1) / ks;
    return (n_all + *k_per_split - 1) / *k_per_split;      // no empty slice
}

int gemm_split_count(const GemmArgs &a) {
    if (a.M <= 0 || a.K <= 0 || a.T <= 0) return 1;
    if (gemm_tile_takes(a)) return gemm_tile_slices(a);
    const int row_blocks = a.y16_k8 ? (a.M + GM / 2 - 1) / (GM / 2) : (a.M + GM - 1) / GM;
    int kps;
    return split_plan(a, row_blocks, (a.T + GN - 1) / GN, &kps);
}

// the 256 x 128 tile, where its workgroups give every CU one
static bool takes_big(const GemmArgs &a, int row_blocks, int slices) {
    return a.x_k8 && a.Wp && slices <= 1 && !a.rope.pos && row_blocks % 2 == 0 && a.big_tile && (row_blocks / 2) * ((a.T + GN - 1) / GN) >= gt_n_cu();
}

// Where the others are not cut along K, or v gets no fewer slices than alone; not where q and k would get fewer by it, take the 256-row tile or make
// more than two rounds over the CUs, beside which v is little.  Calls whose v alone is cut finer, 130 to 384 tokens of the expert shard, keep three
// launches though two are faster there: 130 tokens 1193 / 1146, 200 1265 / 1217, 384 1541 / 1493.  Their sums in fewer slices are no less
// exact; they move rows whose router has a near tie, and no test tells such rows from wrong ones.
// q and k of q4_K, v of q6_K, apart / together, us: 4096 + 512 and 512 x 2048, 600 tokens 22.4 + 9.4 + 5.0 (the slices of v) / 26.0; eight layers of
// the expert shard 70 tokens 1095 / 1043, 600 1950 / 1902, 1300 3151 / 3099, 1700 3864 / 3865; eight 8B-shaped layers
// without f16 copies 70 tokens 1041 / 999, 900 4635 / 4564.
bool gemm_types_ride(const GemmArgs &a) {
    if (!a.Wp || !a.Wp_last || !a.x_k8 || a.n_seg < 2 || a.y16_k8 || a.tiles || gemm_tile_takes(a)) return false;
    if (!((a.type == MESH_Q4_K && a.type_last == MESH_Q6_K) || (a.type == MESH_Q6_K && a.type_last == MESH_Q4_K))) return false;
    if (a.T <= GN / 2 && a.narrow_tile) return false;
    const int first = a.seg_begin[a.n_seg - 1], t_blocks = (a.T + GN - 1) / GN;
    int kps;
    const int slices = split_plan(a, first, t_blocks, &kps), all = (a.M + GM - 1) / GM;
    if (first * t_blocks > 2 * gt_n_cu() || takes_big(a, first, slices)) return false;
    return slices <= 1 || (split_plan(a, all, t_blocks, &kps) == slices && split_plan(a, all - first, t_blocks, &kps) <= slices);
}

int gemm_kquant(const GemmArgs &a, hipStream_t stream) {
    if (a.next_x16 && !gemm_norm_rides(a)) return fail(MESH_ERR_INVALID, "gemm: the next norm on a launch it does not fit");
    if (!a.X || a.M <= 0 || a.K <= 0 || a.T <= 0) return fail(MESH_ERR_INVALID, "gemm: null pointer or empty shape");
    if (a.y16_k8 || a.n_seg > 1) {
        if ((!a.Wp && !gemm_tile_takes(a)) || (a.y16_k8 && (a.n_seg > 1 || a.bias || a.residual)) || a.n_seg > 3)
            return fail(MESH_ERR_INVALID, "gemm: multi-matrix and SwiGLU launches need the GEMM layout (and no bias / residual for SwiGLU)");
        for (int i = 0; i < a.n_seg && !a.y16_k8; ++i)
            if (!a.seg_Y[i] || a.seg_M[i] <= 0 || a.seg_M[i] % 4 || a.seg_ldy[i] % 4 || (i + 1 < a.n_seg && a.seg_M[i] % GM) || (a.residual))
                return fail(MESH_ERR_INVALID, "gemm: bad matrix %d of a multi-matrix launch", i);
    } else if ((!a.W && !gemm_tile_takes(a)) || !a.Y) return fail(MESH_ERR_INVALID, "gemm: null pointer");
    if (a.K % QK_K || a.M % 4 || a.ldx % 8 || a.ldy % 4 || (a.residual && a.ldres % 4))
        return fail(MESH_ERR_INVALID, "gemm: shape M=%d K=%d not supported (K %% 256, M %% 4)", a.M, a.K);
    if ((reinterpret_cast<uintptr_t>(a.X) | reinterpret_cast<uintptr_t>(a.Y)) & 15) return fail(MESH_ERR_INVALID, "gemm: X and Y must be 16-byte aligned");
    if (!a.norm_part && gemm_tile_takes(a)) return gemm_tile(a, stream);
    GemmArgs k = a;
    k.M_pad = (a.M + TILE_ROWS - 1) / TILE_ROWS * TILE_ROWS;
    const int row_blocks = a.y16_k8 ? (a.M + GM / 2 - 1) / (GM / 2) : (a.M + GM - 1) / GM;
    if (a.norm_part) {
        if (!a.y16_k8 || !a.Wp || !a.x_k8 || a.T > GN / 4 || a.tiles || a.norm_parts < 1) return fail(MESH_ERR_INVALID, "gemm: a norm hand-over needs a SwiGLU pair, the GEMM layout and at most 32 tokens");
        if (a.type != MESH_Q4_K && a.type != MESH_Q6_K) return fail(MESH_ERR_UNSUPPORTED, "gemm: no MFMA kernel for ggml type %d", a.type);
        k.ksplit = 1;
        const dim3 g((unsigned)row_blocks);
        return a.type == MESH_Q4_K ? launch_gemm_reg<MESH_Q4_K, 1, REG_NORM>(k, g, stream) : launch_gemm_reg<MESH_Q6_K, 1, REG_NORM>(k, g, stream);
    }
    if (a.tiles) {
        // expert launch: one workgroup row per tile of the list (those past *n_tiles leave at once)
        if (!a.Wp || !a.x_k8 || !a.n_tiles || a.max_tiles <= 0 || a.n_seg > 1 || a.bias || a.residual || a.rope.pos || a.expert_stride % 16)
            return fail(MESH_ERR_INVALID, "gemm: an expert launch needs the GEMM layout, k8-major activations and a plain or SwiGLU epilogue");
        if (a.type != MESH_Q4_K && a.type != MESH_Q6_K) return fail(MESH_ERR_UNSUPPORTED, "gemm: no MFMA kernel for ggml type %d", a.type);
        const dim3 g((unsigned)row_blocks, (unsigned)((a.max_tiles + 7) / 8 * 8));       // (the kernel deals them to the XCDs in eights)
        if (a.x_slot && a.x_div < 1) return fail(MESH_ERR_INVALID, "gemm: rows of an expert launch without their divisor");
        if (a.x_slot && a.type == MESH_Q4_K) MESH_LAUNCH((gemm_expert_kernel<MESH_Q4_K, REG_EXPERT_ROWS>), g, dim3(256), 0, stream, k);
        else if (a.x_slot) MESH_LAUNCH((gemm_expert_kernel<MESH_Q6_K, REG_EXPERT_ROWS>), g, dim3(256), 0, stream, k);
        else if (a.type == MESH_Q4_K) MESH_LAUNCH((gemm_expert_kernel<MESH_Q4_K, REG_EXPERT>), g, dim3(256), 0, stream, k);
        else MESH_LAUNCH((gemm_expert_kernel<MESH_Q6_K, REG_EXPERT>), g, dim3(256), 0, stream, k);
        MESH_LAUNCH_CHECK();
        return MESH_OK;
    }
    dim3 grid((unsigned)row_blocks, (unsigned)((a.T + GN - 1) / GN));
    // A launch of fewer workgroups than CUs walks all of K in each of them while the rest of the chip idles: split K
    // over blockIdx.z (slices of at least 8 k-steps, at most one workgroup per CU in total, partial tiles within the
    // scratch the caller gave).
    k.k_per_split = a.K / GK;
    k.ksplit = split_plan(a, row_blocks, (int)grid.y, &k.k_per_split);
    grid.z = (unsigned)k.ksplit;
    if (a.rope.pos && k.ksplit <= 1) return fail(MESH_ERR_INVALID, "gemm: RoPE / KV append needs a split launch");
    if (a.rope.pos && (a.y16_k8 || a.residual || a.rope.head_dim % 4 || a.rope.n_rot % 2))
        return fail(MESH_ERR_INVALID, "gemm: RoPE / KV append on a launch it does not fit");
    if (a.type != MESH_Q4_K && a.type != MESH_Q6_K) return fail(MESH_ERR_UNSUPPORTED, "gemm: no MFMA kernel for ggml type %d", a.type);
    const bool q4 = a.type == MESH_Q4_K, packed = a.Wp != nullptr;
    if (a.Wp_last) {
        if (!gemm_types_ride(a)) return fail(MESH_ERR_INVALID, "gemm: matrices of two types in a launch they do not fit");
        if (k.ksplit > 1) return q4 ? launch_gemm_types<MESH_Q4_K, MESH_Q6_K, true>(k, grid, stream) : launch_gemm_types<MESH_Q6_K, MESH_Q4_K, true>(k, grid, stream);
        return q4 ? launch_gemm_types<MESH_Q4_K, MESH_Q6_K, false>(k, grid, stream) : launch_gemm_types<MESH_Q6_K, MESH_Q4_K, false>(k, grid, stream);
    }
    // enough workgroups of the 256 x 128 tile to give every CU one: the big tile (gemm_big_kernel).  A pair of 512 row blocks and more
    // does at any token count: calls of 17 to 64 tokens over such a pair take it too, though the register-formed tile is the faster one
    // there (two layers 4096 wide with 33024 feed-forward rows: 388 against 286 us at 17 tokens, 473 against 377 at 64).
    if (takes_big(a, row_blocks, k.ksplit))
        return q4 ? launch_gemm_big<MESH_Q4_K>(k, row_blocks, (int)grid.y, stream) : launch_gemm_big<MESH_Q6_K>(k, row_blocks, (int)grid.y, stream);
    if (a.x_k8) {
        if (packed) return q4 ? launch_gemm<MESH_Q4_K, true, true>(k, grid, stream) : launch_gemm<MESH_Q6_K, true, true>(k, grid, stream);
        return q4 ? launch_gemm<MESH_Q4_K, false, true>(k, grid, stream) : launch_gemm<MESH_Q6_K, false, true>(k, grid, stream);
    }
    if (packed) return q4 ? launch_gemm<MESH_Q4_K, true, false>(k, grid, stream) : launch_gemm<MESH_Q6_K, true, false>(k, grid, stream);
    return q4 ? launch_gemm<MESH_Q4_K, false, false>(k, grid, stream) : launch_gemm<MESH_Q6_K, false, false>(k, grid, stream);
}

// ---- GEMM layout ----------------------------------------------------------------------------------------------
// One workgroup writes one chunk: thread s re-reads its (row, sub-block) from the mat-vec tiles the way the staging
// thread of the unpacked kernel does, and writes it in the packed form.
// tiled2 set: a gate / up pair -- the chunk's rows 0..63 are rows [64 mb, 64 mb + 64) of `tiled`, rows 64..127 those of tiled2.
template <int TYPE>
__global__ __launch_bounds__(256) void gemm_pack_kernel(const uint8_t *__restrict__ tiled, const uint8_t *__restrict__ tiled2,
                                                        uint8_t *__restrict__ packed, int M_pad, int nsb) {
    constexpr int TB = TYPE == MESH_Q4_K ? Q4K_TILE_BYTES : Q6K_TILE_BYTES;
    constexpr int CH = PackedSub<TYPE>::CHUNK;
    const int kc = blockIdx.x, mb = blockIdx.y, n_steps = gridDim.x, s = threadIdx.x;
    const int h = s & 1;
    int wrow = mb * GM + (s >> 1);
    if (tiled2) {
        wrow = mb * (GM / 2) + ((s >> 1) & (GM / 2 - 1));
        if ((s >> 1) >= GM / 2) tiled = tiled2;
    }
    uint8_t *chunk = packed + ((size_t)mb * n_steps + kc) * CH;
    if (wrow >= M_pad) {
        *reinterpret_cast<uint4 *>(chunk + s * 16) = make_uint4(0, 0, 0, 0);
        if (TYPE == MESH_Q6_K) *reinterpret_cast<uint2 *>(chunk + 4096 + s * 8) = make_uint2(0, 0);
        *reinterpret_cast<uint32_t *>(chunk + (TYPE == MESH_Q6_K ? 6144 : 4096) + s * 4) = 0u;
        return;
    }
    RawSub<TYPE> r;
    r.load(tiled + ((size_t)(wrow >> 4) * nsb + (kc >> 2)) * TB, wrow & 15, kc & 3, h);
    r.pack(kc & 3, h, chunk, s);
}

size_t gemm_packed_bytes(int type, int64_t M, int64_t K) {
    if ((type != MESH_Q4_K && type != MESH_Q6_K) || M <= 0 || K <= 0 || K % QK_K) return 0;
    const size_t chunk = type == MESH_Q4_K ? PackedSub<MESH_Q4_K>::CHUNK : PackedSub<MESH_Q6_K>::CHUNK;
    return (size_t)((M + GM - 1) / GM) * (size_t)(K / GK) * chunk;
}

int gemm_pack(int type, const void *tiled, void *packed, int64_t M, int64_t K, hipStream_t stream) {
    if (!tiled || !packed || gemm_packed_bytes(type, M, K) == 0) return fail(MESH_ERR_INVALID, "gemm_pack: bad arguments (type %d, M %lld, K %lld)", type, (long long)M, (long long)K);
    const dim3 grid((unsigned)(K / GK), (unsigned)((M + GM - 1) / GM));
    const int M_pad = (int)((M + TILE_ROWS - 1) / TILE_ROWS * TILE_ROWS), nsb = (int)(K / QK_K);
    if (grid.y > 65535u) return fail(MESH_ERR_UNSUPPORTED, "gemm_pack: %lld rows are too many", (long long)M);
    if (type == MESH_Q4_K) MESH_LAUNCH(gemm_pack_kernel<MESH_Q4_K>, grid, dim3(256), 0, stream, static_cast<const uint8_t *>(tiled), nullptr, static_cast<uint8_t *>(packed), M_pad, nsb);
    else MESH_LAUNCH(gemm_pack_kernel<MESH_Q6_K>, grid, dim3(256), 0, stream, static_cast<const uint8_t *>(tiled), nullptr, static_cast<uint8_t *>(packed), M_pad, nsb);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// one workgroup per chunk: thread s forms its (row, sub-block) as the staging thread of the GEMM does
template <int TYPE>
__global__ __launch_bounds__(256) void gemm_tile_copy_kernel(const uint8_t *__restrict__ packed, _Float16 *__restrict__ tile, int pair) {
    const int kc = blockIdx.x, mb = blockIdx.y, n_steps = gridDim.x, s = threadIdx.x, h = s & 1;
    int r = s >> 1;
    PackedSub<TYPE> sub;
    sub.load(packed + ((size_t)mb * n_steps + kc) * PackedSub<TYPE>::CHUNK, s);
    if (pair) r = (r & 32) * 2 + (r >> 6) * 32 + (r & 31);
    _Float16 *dst = tile + (size_t)(mb * 8 + (r >> 4)) * 16 * n_steps * GK + ((size_t)(kc * 8 + h) * 16 + (r & 15)) * 8;
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<uint4 *>(dst + j * 256) = sub.form(j);
}

size_t gemm_tile_bytes(int64_t M, int64_t K) { return (size_t)((M + GM - 1) / GM) * GM * (size_t)K * 2; }
size_t gemm_tile_pair_bytes(int64_t M, int64_t K) { return (size_t)((M + GM / 2 - 1) / (GM / 2)) * GM * (size_t)K * 2; }

int gemm_tile_copy(int type, const void *packed, void *tile, int64_t M, int64_t K, bool pair, hipStream_t stream) {
    if (!packed || !tile || gemm_packed_bytes(type, M, K) == 0) return fail(MESH_ERR_INVALID, "gemm_tile_copy: bad arguments (type %d, M %lld, K %lld)", type, (long long)M, (long long)K);
    const int rows = pair ? GM / 2 : GM;
    const dim3 grid((unsigned)(K / GK), (unsigned)((M + rows - 1) / rows));
    if (type == MESH_Q4_K) MESH_LAUNCH(gemm_tile_copy_kernel<MESH_Q4_K>, grid, dim3(256), 0, stream, static_cast<const uint8_t *>(packed), static_cast<_Float16 *>(tile), pair ? 1 : 0);
    else MESH_LAUNCH(gemm_tile_copy_kernel<MESH_Q6_K>, grid, dim3(256), 0, stream, static_cast<const uint8_t *>(packed), static_cast<_Float16 *>(tile), pair ? 1 : 0);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

size_t gemm_packed_pair_bytes(int type, int64_t M, int64_t K) {
    if ((type != MESH_Q4_K && type != MESH_Q6_K) || M <= 0 || K <= 0 || K % QK_K) return 0;
    const size_t chunk = type == MESH_Q4_K ? PackedSub<MESH_Q4_K>::CHUNK : PackedSub<MESH_Q6_K>::CHUNK;
    return (size_t)((M + GM / 2 - 1) / (GM / 2)) * (size_t)(K / GK) * chunk;
}

int gemm_pack_pair(int type, const void *gate_tiled, const void *up_tiled, void *packed, int64_t M, int64_t K, hipStream_t stream) {
    if (!gate_tiled || !up_tiled || !packed || gemm_packed_pair_bytes(type, M, K) == 0)
        return fail(MESH_ERR_INVALID, "gemm_pack_pair: bad arguments (type %d, M %lld, K %lld)", type, (long long)M, (long long)K);
    const dim3 grid((unsigned)(K / GK), (unsigned)((M + GM / 2 - 1) / (GM / 2)));
    const int M_pad = (int)((M + TILE_ROWS - 1) / TILE_ROWS * TILE_ROWS), nsb = (int)(K / QK_K);
    if (grid.y > 65535u) return fail(MESH_ERR_UNSUPPORTED, "gemm_pack_pair: %lld rows are too many", (long long)M);
    const uint8_t *g = static_cast<const uint8_t *>(gate_tiled), *u = static_cast<const uint8_t *>(up_tiled);
    if (type == MESH_Q4_K) MESH_LAUNCH(gemm_pack_kernel<MESH_Q4_K>, grid, dim3(256), 0, stream, g, u, static_cast<uint8_t *>(packed), M_pad, nsb);
    else MESH_LAUNCH(gemm_pack_kernel<MESH_Q6_K>, grid, dim3(256), 0, stream, g, u, static_cast<uint8_t *>(packed), M_pad, nsb);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// ---- small elementwise companions of the prefill path ---------------------------------------------------------
// y16[t] = f16( x[t] * rsqrt(mean(x[t]^2) + eps) * w ), one workgroup per token
__global__ __launch_bounds__(256) void rmsnorm_f16_kernel(const float *__restrict__ x, const float *__restrict__ w, float eps,
                                                          int n, _Float16 *__restrict__ y, int ldy, unsigned *sat) {
    __shared__ float red[4];
    const int t = blockIdx.x, tid = threadIdx.x;
    const float *xt = x + (size_t)t * n;
    float ss = 0.f;
    for (int i = tid * 4; i < n; i += 1024) {
        const float4 v = *reinterpret_cast<const float4 *>(xt + i);
        ss += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    const float scale = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)n + eps);
    for (int i = tid * 4; i < n; i += 1024) {
        const float4 v = *reinterpret_cast<const float4 *>(xt + i);
        const float4 g = *reinterpret_cast<const float4 *>(w + i);
        note_f16_clamp(sat, v.x * scale * g.x, v.y * scale * g.y, v.z * scale * g.z, v.w * scale * g.w);
        *reinterpret_cast<uint2 *>(y + (size_t)t * ldy + i) =
            make_uint2(pack_h2(v.x * scale * g.x, v.y * scale * g.y), pack_h2(v.z * scale * g.z, v.w * scale * g.w));
    }
}

int rmsnorm_f16(const float *x, const float *w, float eps, int T, int n, _Float16 *y, int ldy, hipStream_t stream, unsigned *sat) {
    if (T <= 0) return MESH_OK;
    if (n % 4 || ldy % 4) return fail(MESH_ERR_INVALID, "rmsnorm: row length %d not a multiple of 4", n);
    MESH_LAUNCH(rmsnorm_f16_kernel, dim3((unsigned)T), dim3(256), 0, stream, x, w, eps, n, y, ldy, sat);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// out16 = f16( silu(gate) * up )
__global__ __launch_bounds__(256) void swiglu_f16_kernel(const float *__restrict__ g, const float *__restrict__ u,
                                                         _Float16 *__restrict__ o, int64_t n4, unsigned *sat) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const float4 a = reinterpret_cast<const float4 *>(g)[i], b = reinterpret_cast<const float4 *>(u)[i];
    const float r0 = a.x / (1.0f + expf(-a.x)) * b.x, r1 = a.y / (1.0f + expf(-a.y)) * b.y;
    const float r2 = a.z / (1.0f + expf(-a.z)) * b.z, r3 = a.w / (1.0f + expf(-a.w)) * b.w;
    note_f16_clamp(sat, r0, r1, r2, r3);
    reinterpret_cast<uint2 *>(o)[i] = make_uint2(pack_h2(r0, r1), pack_h2(r2, r3));
}

int swiglu_f16(const float *gate, const float *up, _Float16 *out, int64_t n, hipStream_t stream, unsigned *sat) {
    if (n <= 0) return MESH_OK;
    if (n % 4) return fail(MESH_ERR_INVALID, "swiglu: count not a multiple of 4");
    MESH_LAUNCH(swiglu_f16_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, stream, gate, up, out, n / 4, sat);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

}  // namespace mesh
