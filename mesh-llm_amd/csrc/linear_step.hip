// The single-token product: y = W x for a bf16 matrix and one f32 vector, bound by the weight stream.
//
// A wave takes R rows at a time; its 64 lanes cover 512 consecutive k per 16-byte load and R * U loads are in flight while
// the R * U before them are multiplied.  The input vector sits in LDS as f32.  Every workgroup derives it itself from what
// the launch before left (residual update with its output norm, polynomial activation: linear.hpp), which saves a launch
// between two products.  Loads return in order, so the vectors it is derived from are requested first, the first weights
// right behind them, and no branch lies around a weight load (the compiler would wait for all of them at its join): the
// weights travel while norms are worked out.  What an epilogue reads (state, biases, side embedding) is requested with the
// weights of its rows.
// In models that cycle through their weights, against products whose weights were requested first, us: 8192 x 2048 behind two layer
// norms 12.4 -> 11.5 (as long where the weights wait for the vectors to arrive: the norms' four sums and the start of the stream are
// what is left), behind an RMS norm 10.2 -> 8.8, three of 2048 x 2048 with the recurrence's update 9.4 -> 7.5, 2048 x 8192 of squares
// 10.2 -> 7.8, of the polynomial 10.8 -> 8.8, 2048 x 2048 4.1 -> 3.7.
// Sums of squares a later norm needs are left per workgroup and added in workgroup order by the consumer, so the result does
// not depend on timing.
#include "act_math.hpp"
#include "linear.hpp"
#include "wave_ops.hpp"

#include <algorithm>

namespace mesh {

constexpr int STEP_THREADS = 512, STEP_WAVES = STEP_THREADS / 64;
constexpr size_t STEP_LDS_MAX = 160 * 1024 - 1024;

// over the wave, in every lane, from the nearest lanes on
__device__ __forceinline__ float step_wave_sum(float v) { return lane_fold<32>(lane_fold<16>(group_sum<16>(v), LaneAdd{}), LaneAdd{}); }
// N sums over the workgroup in a fixed order, the same in every thread.  Two sums in a row use different slots: the barrier of the
// second is what keeps a third from overwriting what the first's readers still need.
typedef float StepScratch[2][STEP_WAVES][4];
template <int SLOT, int N>
__device__ __forceinline__ void step_block_sums(float (&v)[N], StepScratch &scratch, int lane, int wave) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = step_wave_sum(v[i]);
    if (lane == 0)
#pragma unroll
        for (int i = 0; i < N; ++i) scratch[SLOT][wave][i] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        v[i] = 0.f;
#pragma unroll
        for (int w = 0; w < STEP_WAVES; ++w) v[i] += scratch[SLOT][w][i];
    }
}
template <int SLOT>
__device__ __forceinline__ float step_block_sum(float v, StepScratch &scratch, int lane, int wave) {
    float s[1] = {v};
    step_block_sums<SLOT>(s, scratch, lane, wave);
    return s[0];
}

// four elements of a vector of K, zeros behind its end
__device__ __forceinline__ float4 ln_load4(const float *p, int k, int K) {
    if (k + 4 <= K) return *reinterpret_cast<const float4 *>(p + k);
    return make_float4(k < K ? p[k] : 0.f, k + 1 < K ? p[k + 1] : 0.f, k + 2 < K ? p[k + 2] : 0.f, 0.f);
}
// The same requested ahead, in two parts: loads that no branch lies around, of 16 bytes where K is a multiple of four (WHOLE) and of 4
// each otherwise, and, once they are needed, their zeros.  (With a branch for a row's last elements the weights wait for the vectors:
// products of rows of 1031 0.6 us later each; both kinds in one kernel cost rows of 4096 as much.)
template <bool WHOLE> __device__ __forceinline__ float4 ln_request4(const float *p, int k, int K) {
    if constexpr (WHOLE) return *reinterpret_cast<const float4 *>(p + (k < K ? k : K - 4));
    auto at = [&](int i) { return p[i < K ? i : K - 1]; };
    return make_float4(at(k), at(k + 1), at(k + 2), at(k + 3));
}
template <bool WHOLE> __device__ __forceinline__ void ln_settle4(float4 &v, int k, int K) {
    if constexpr (!WHOLE) v = make_float4(k < K ? v.x : 0.f, k + 1 < K ? v.y : 0.f, k + 2 < K ? v.z : 0.f, k + 3 < K ? v.w : 0.f);
    else if (k >= K) v = make_float4(0.f, 0.f, 0.f, 0.f);
}

// A thread's first N groups of four elements of a vector, requested ahead; xs[k .. k + 3] = map(k, them) over [0, Kp), the groups
// behind them loaded on the way.
template <int N, bool WHOLE> struct StepVec {
    static constexpr int STRIDE = STEP_THREADS * 4;
    float4 v[N];
    __device__ __forceinline__ void load(const float *p, int tid, int K) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = ln_request4<WHOLE>(p, tid * 4 + i * STRIDE, K);
    }
    template <typename Map> __device__ __forceinline__ void put(const float *p, int tid, int K, int Kp, Map map, float *xs) {
        for (int k0 = tid * 4; k0 < Kp; k0 += N * STRIDE) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                if (k0 == tid * 4) ln_settle4<WHOLE>(v[i], k0 + i * STRIDE, K);
                else v[i] = ln_load4(p, k0 + i * STRIDE, K);
            }
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int k = k0 + i * STRIDE;
                if (k < Kp) *reinterpret_cast<float4 *>(xs + k) = map(k, v[i]);
            }
        }
    }
};

template <int R, int U, StepIn IN, StepOut OUT, bool WHOLE>
__global__ __launch_bounds__(STEP_THREADS, 4) void linear_step_kernel(const uint16_t *p_w, int p_Kp, int p_groups, int p_width, int p_K, const StepArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ StepScratch scratch;
    float *xs = reinterpret_cast<float *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = p_K, Kp = p_Kp;
    const int batches = (Kp + 512 * U - 1) / (512 * U);
    const int g_step = gridDim.x * STEP_WAVES;
    auto row_of = [&](int gr, int r) { return OUT == STEP_OUT_MIN_GRU ? r * p_width + gr : gr * R + r; };
    // a batch of weights and what the epilogue of their rows reads
    struct Batch {
        uint4 w[R][U];
        float e[3];
    };
    static_assert(R <= 3, "e holds one number a row");
    int seq0 = 0, pos0 = 0, tok0 = 0;
    if constexpr (OUT == STEP_OUT_MIN_GRU) { seq0 = a.seq[0]; pos0 = a.pos[0]; }
    if constexpr (OUT == STEP_OUT_SIDE) tok0 = a.tok[0];
    auto fetch = [&](Batch &b, int gr, int bt) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint16_t *wr = p_w + (size_t)row_of(gr, r) * Kp;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = (bt * U + u) * 512 + lane * 8;
                b.w[r][u] = *reinterpret_cast<const uint4 *>(wr + (k < Kp ? k : Kp - 8));       // (past the row's end: not used)
            }
        }
        if constexpr (OUT == STEP_OUT_MIN_GRU) { b.e[0] = a.bias_z[gr]; b.e[1] = a.bias_x[gr]; b.e[2] = a.state[(size_t)seq0 * p_width + gr]; }
        if constexpr (OUT == STEP_OUT_SIDE) {
#pragma unroll
            for (int r = 0; r < R; ++r) b.e[r] = bf16_bits_to_f32(a.side[(size_t)tok0 * a.side_stride + a.side_offset + (gr * R + r < a.W.M ? gr * R + r : a.W.M - 1)]);
        }
    };
    Batch b0, b1;
    const int first = blockIdx.x * STEP_WAVES + wave;
    const int turns = first < p_groups ? (p_groups - first + g_step - 1) / g_step : 0;
    auto fetch_first = [&]() {
        asm volatile("" ::: "memory");          // (or the compiler moves the vectors' loads to where they are used, behind these)
        fetch(b0, turns ? first : p_groups - 1, 0);
    };

    // ---- the input vector
    static_assert(STEP_PARTS_MAX <= STEP_THREADS, "a partial sum per thread");
    if constexpr (IN == STEP_IN_VEC || IN == STEP_IN_RELU2) {
        StepVec<4, WHOLE> in;
        in.load(a.in, tid, K);
        fetch_first();
        auto sq = [](float v) { const float p = fmaxf(v, 0.f); return p * p; };
        in.put(a.in, tid, K, Kp, [&](int, const float4 &v) { return IN == STEP_IN_VEC ? v : make_float4(sq(v.x), sq(v.y), sq(v.z), sq(v.w)); }, xs);
    } else if constexpr (IN == STEP_IN_POLY) {
        float p[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) p[i] = tid < a.n_part ? a.part[i * a.n_part + tid] : 0.f;
        const float f1 = a.coef[0], f2 = a.coef[1], f3 = a.coef[2], c0 = a.coef[3];
        StepVec<4, WHOLE> in;
        in.load(a.in, tid, K);
        fetch_first();
        step_block_sums<0>(p, scratch, lane, wave);
        const float c1 = f1 / sqrtf(p[0] / (float)K + a.eps), c2 = f2 / sqrtf(p[1] / (float)K + a.eps), c3 = f3 / sqrtf(p[2] / (float)K + a.eps);
        auto poly = [&](float u) { return ((c3 * u + c2) * u + c1) * u + c0; };
        in.put(a.in, tid, K, Kp,
               [&](int k, const float4 &u) {
                   return make_float4(k < K ? poly(u.x) : 0.f, k + 1 < K ? poly(u.y) : 0.f, k + 2 < K ? poly(u.z) : 0.f, k + 3 < K ? poly(u.w) : 0.f);
               }, xs);
    } else if constexpr (IN == STEP_IN_UNIT_RMS) {
        StepVec<1, WHOLE> in, gain;
        in.load(a.in, tid, K);
        gain.load(a.gain, tid, K);
        fetch_first();
        float ss = 0.f;
        in.put(a.in, tid, K, Kp, [&](int, const float4 &v) { ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w; return v; }, xs);
        const float rinv = 1.0f / sqrtf(step_block_sum<0>(ss, scratch, lane, wave) / (float)K + a.eps);
        gain.put(a.gain, tid, K, Kp,
                 [&](int k, const float4 &g) {
                     const float4 v = *reinterpret_cast<const float4 *>(xs + k);
                     return make_float4(v.x * (rinv * g.x), v.y * (rinv * g.y), v.z * (rinv * g.z), v.w * (rinv * g.w));
                 }, xs);
    } else if constexpr (IN == STEP_IN_HEADS) {
        // a head's four-element groups lie in neighbouring lanes of a wave
        constexpr int AHEAD = 2, STRIDE = STEP_THREADS * 4;
        const int width = a.head_width, k0 = tid * 4;
        float4 o4[AHEAD], g4[AHEAD], n4[AHEAD];
        auto request = [&](int k, float4 &o, float4 &g, float4 &n) {
            const int at = k < K ? k : K - 4;
            o = *reinterpret_cast<const float4 *>(a.in + at);
            g = *reinterpret_cast<const float4 *>(a.head_gate + at);
            n = *reinterpret_cast<const float4 *>(a.gain + (at & (width - 1)));
        };
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) request(k0 + i * STRIDE, o4[i], g4[i], n4[i]);
        fetch_first();
        auto put = [&](int k, const float4 &o, const float4 &g, const float4 &n) {
            float ss = fmaf(o.x, o.x, fmaf(o.y, o.y, fmaf(o.z, o.z, o.w * o.w)));
            if (width > 4) ss = lane_fold<1>(ss, LaneAdd{});
            if (width > 8) ss = lane_fold<2>(ss, LaneAdd{});
            if (width > 16) ss = lane_fold<4>(ss, LaneAdd{});
            if (width > 32) ss = lane_fold<8>(ss, LaneAdd{});
            if (width > 64) ss = lane_fold<16>(ss, LaneAdd{});
            if (width > 128) ss = lane_fold<32>(ss, LaneAdd{});
            const float r = 1.0f / sqrtf(ss / (float)width + a.eps);
            if (k < Kp)
                *reinterpret_cast<float4 *>(xs + k) = k < K ? make_float4(o.x * r * n.x * act_silu(g.x), o.y * r * n.y * act_silu(g.y), o.z * r * n.z * act_silu(g.z), o.w * r * n.w * act_silu(g.w))
                                                            : make_float4(0.f, 0.f, 0.f, 0.f);
        };
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) put(k0 + i * STRIDE, o4[i], g4[i], n4[i]);
        for (int first_k = (tid & ~63) * 4 + AHEAD * STRIDE; first_k < Kp; first_k += STRIDE) {       // (whole waves)
            const int k = first_k + lane * 4;
            request(k, o4[0], g4[0], n4[0]);
            put(k, o4[0], g4[0], n4[0]);
        }
    } else if constexpr (IN == STEP_IN_LAYER) {
        // a thread's first AHEAD groups of four, of every vector, are requested before the first sum; means first, then squared
        // deviations
        constexpr int AHEAD = 2, STRIDE = STEP_THREADS * 4;
        const int k0 = tid * 4;
        const float inv_n = 1.0f / (float)K;
        float4 x4[AHEAD], y4[AHEAD], g4[AHEAD], b4[AHEAD], ng4[AHEAD], nb4[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int k = k0 + i * STRIDE;
            auto get = [&](const float *p) { return ln_request4<WHOLE>(p, k, K); };
            x4[i] = get(a.in);
            if (a.y) { y4[i] = get(a.y); g4[i] = get(a.gain); b4[i] = get(a.bias); }
            ng4[i] = get(a.norm_gain); nb4[i] = get(a.norm_bias);
        }
        fetch_first();
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int k = k0 + i * STRIDE;
            ln_settle4<WHOLE>(x4[i], k, K);
            if (a.y) { ln_settle4<WHOLE>(y4[i], k, K); ln_settle4<WHOLE>(g4[i], k, K); ln_settle4<WHOLE>(b4[i], k, K); }
            ln_settle4<WHOLE>(ng4[i], k, K); ln_settle4<WHOLE>(nb4[i], k, K);
        }
        auto sum4 = [](const float4 &v) { return (v.x + v.y) + (v.z + v.w); };
        auto dev4 = [&](int k, const float4 &v, float mean) {
            const float d[4] = {v.x - mean, v.y - mean, v.z - mean, v.w - mean};
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) s = fmaf(k + j < K ? d[j] : 0.f, d[j], s);
            return s;
        };
        if (a.y) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) s += sum4(y4[i]);
            for (int k = k0 + AHEAD * STRIDE; k < K; k += STRIDE) s += sum4(ln_load4(a.y, k, K));
            const float mean = step_block_sum<0>(s, scratch, lane, wave) * inv_n;
            s = 0.f;
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) s += dev4(k0 + i * STRIDE, y4[i], mean);
            for (int k = k0 + AHEAD * STRIDE; k < K; k += STRIDE) s += dev4(k, ln_load4(a.y, k, K), mean);
            const float rs = 1.0f / sqrtf(step_block_sum<1>(s, scratch, lane, wave) * inv_n + a.eps);
            auto update = [&](int k, const float4 &x, const float4 &y, const float4 &g, const float4 &b) {
                const float4 v = make_float4(x.x + ((y.x - mean) * rs * g.x + b.x), x.y + ((y.y - mean) * rs * g.y + b.y), x.z + ((y.z - mean) * rs * g.z + b.z),
                                             x.w + ((y.w - mean) * rs * g.w + b.w));
                if (blockIdx.x == 0) {
                    const float o[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (k + j < K) a.x_out[k + j] = o[j];
                }
                return v;
            };
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) x4[i] = update(k0 + i * STRIDE, x4[i], y4[i], g4[i], b4[i]);
            for (int k = k0 + AHEAD * STRIDE; k < Kp; k += STRIDE)
                *reinterpret_cast<float4 *>(xs + k) = update(k, ln_load4(a.in, k, K), ln_load4(a.y, k, K), ln_load4(a.gain, k, K), ln_load4(a.bias, k, K));
        } else {
            for (int k = k0 + AHEAD * STRIDE; k < Kp; k += STRIDE) *reinterpret_cast<float4 *>(xs + k) = ln_load4(a.in, k, K);
        }
        // (groups behind the first AHEAD wait in LDS, every thread's its own)
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) s += sum4(x4[i]);
        for (int k = k0 + AHEAD * STRIDE; k < Kp; k += STRIDE) s += sum4(*reinterpret_cast<const float4 *>(xs + k));
        const float mean = step_block_sum<0>(s, scratch, lane, wave) * inv_n;
        s = 0.f;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) s += dev4(k0 + i * STRIDE, x4[i], mean);
        for (int k = k0 + AHEAD * STRIDE; k < Kp; k += STRIDE) s += dev4(k, *reinterpret_cast<const float4 *>(xs + k), mean);
        const float rs = 1.0f / sqrtf(step_block_sum<1>(s, scratch, lane, wave) * inv_n + a.eps);
        auto put = [&](int k, const float4 &v, const float4 &g, const float4 &b) {
            if (k < Kp) *reinterpret_cast<float4 *>(xs + k) = make_float4((v.x - mean) * rs * g.x + b.x, (v.y - mean) * rs * g.y + b.y, (v.z - mean) * rs * g.z + b.z, (v.w - mean) * rs * g.w + b.w);
        };
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) put(k0 + i * STRIDE, x4[i], ng4[i], nb4[i]);
        for (int k = k0 + AHEAD * STRIDE; k < Kp; k += STRIDE) put(k, *reinterpret_cast<const float4 *>(xs + k), ln_load4(a.norm_gain, k, K), ln_load4(a.norm_bias, k, K));
    } else {
        float ss = tid < a.n_part ? a.part[tid] : 0.f;
        constexpr int AHEAD = 2;
        float4 x4[AHEAD], y4[AHEAD], g4[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int k = (tid + i * STEP_THREADS) * 4;
            auto get = [&](const float *p) { return ln_request4<WHOLE>(p, k, K); };
            x4[i] = get(a.in); y4[i] = get(a.y); g4[i] = get(a.gain);
        }
        fetch_first();
        ss = step_block_sum<0>(ss, scratch, lane, wave);
        const float rinv = 1.0f / sqrtf(ss / (float)K + a.eps);
        float sx = 0.f;
        auto update = [&](int k, const float4 &x, const float4 &y, const float4 &g) {
            if (k >= Kp) return;
            const float4 v = make_float4(x.x + y.x * rinv * g.x, x.y + y.y * rinv * g.y, x.z + y.z * rinv * g.z, x.w + y.w * rinv * g.w);
            *reinterpret_cast<float4 *>(xs + k) = v;
            sx += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
            if (blockIdx.x == 0) {
                const float o[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (k + j < K) a.x_out[k + j] = o[j];
            }
        };
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int k = (tid + i * STEP_THREADS) * 4;
            ln_settle4<WHOLE>(x4[i], k, K); ln_settle4<WHOLE>(y4[i], k, K); ln_settle4<WHOLE>(g4[i], k, K);
            update(k, x4[i], y4[i], g4[i]);
        }
        for (int k = (tid + AHEAD * STEP_THREADS) * 4; k < Kp; k += STEP_THREADS * 4) update(k, ln_load4(a.in, k, K), ln_load4(a.y, k, K), ln_load4(a.gain, k, K));
        if constexpr (IN == STEP_IN_RESIDUAL_NORM) {
            sx = step_block_sum<1>(sx, scratch, lane, wave);
            const float z = a.norm_gain[0] / sqrtf(sx / (float)K + a.eps);
            for (int k = tid; k < Kp; k += STEP_THREADS) xs[k] *= z;
        }
    }
    __syncthreads();

    // ---- rows
    float acc[R], s2 = 0.f, s4 = 0.f, s6 = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    auto finish = [&](int gr, const float (&e)[3]) {
        float v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) { v[r] = step_wave_sum(acc[r]); acc[r] = 0.f; }
        if constexpr (OUT == STEP_OUT_MIN_GRU) {
            if (lane == 0) {
                const MinGruGate g = min_gru_gate(v[0] + e[0], v[1] + e[1]);
                const float s = pos0 == 0 ? g.in : fmaf(g.keep, e[2], g.in);
                a.state[(size_t)seq0 * p_width + gr] = s;
                a.out[gr] = s * act_silu(v[2]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int m = gr * R + r;
                if (m >= a.W.M) continue;
                float o = v[r];
                if constexpr (OUT == STEP_OUT_SIDE) o = act_gelu_tanh(o) * e[r];
                if (lane == 0) a.out[m] = o;
                const float q = o * o;
                if constexpr (OUT == STEP_OUT_SUMSQ || OUT == STEP_OUT_POWERS) s2 += q;
                if constexpr (OUT == STEP_OUT_POWERS) { s4 += q * q; s6 += q * q * q; }
            }
        }
    };
    auto use = [&](const Batch &b, int gr, int bt) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = (bt * U + u) * 512 + lane * 8;
            if (k < Kp) {
                const float4 xa = *reinterpret_cast<const float4 *>(xs + k), xb = *reinterpret_cast<const float4 *>(xs + k + 4);
                const float xf[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t w[4] = {b.w[r][u].x, b.w[r][u].y, b.w[r][u].z, b.w[r][u].w};
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[r] = fmaf(__uint_as_float((j & 1) ? (w[j >> 1] & 0xFFFF0000u) : (w[j >> 1] << 16)), xf[j], acc[r]);
                }
            }
        }
        if (bt == batches - 1) finish(gr, b.e);
    };
    // (group, batch) pairs in order; each is fetched while the one before it is used
    int gr0 = first, bt0 = 0, gr1, bt1;
    auto after = [&](int gr, int bt, int &gr_next, int &bt_next) {
        const bool turn = bt + 1 == batches;
        bt_next = turn ? 0 : bt + 1;
        gr_next = turn ? gr + g_step : gr;
    };
    int left = turns * batches;
    for (; left > 2; left -= 2) {
        after(gr0, bt0, gr1, bt1);
        fetch(b1, gr1, bt1);
        use(b0, gr0, bt0);
        after(gr1, bt1, gr0, bt0);
        fetch(b0, gr0, bt0);
        use(b1, gr1, bt1);
    }
    if (left == 2) {
        after(gr0, bt0, gr1, bt1);
        fetch(b1, gr1, bt1);
        use(b0, gr0, bt0);
        use(b1, gr1, bt1);
    } else if (left == 1) {
        use(b0, gr0, bt0);
    }
    if constexpr (OUT == STEP_OUT_SUMSQ || OUT == STEP_OUT_POWERS) {
        // (every lane of a wave holds the wave's sums)
        __syncthreads();
        if (lane == 0) { scratch[0][wave][0] = s2; scratch[0][wave][1] = s4; scratch[0][wave][2] = s6; }
        __syncthreads();
        if (tid < (OUT == STEP_OUT_POWERS ? 3 : 1)) {
            float s = 0.f;
            for (int w = 0; w < STEP_WAVES; ++w) s += scratch[0][w][tid];
            a.out_part[(size_t)tid * gridDim.x + blockIdx.x] = s;
        }
    }
}

bool linear_step_supported(const LinearWeight &W) { return (size_t)W.Kp * sizeof(float) <= STEP_LDS_MAX; }

static int rows_per_group(const StepArgs &a) { return a.out_kind == STEP_OUT_MIN_GRU ? 3 : a.W.M < 4096 ? 1 : 2; }
static int step_groups(const StepArgs &a) { return a.out_kind == STEP_OUT_MIN_GRU ? a.width : (a.W.M + rows_per_group(a) - 1) / rows_per_group(a); }

int linear_step_grid(const StepArgs &a) {
    // as many workgroups as the chip holds at once, two per CU; more rows mean more turns per wave, equally many for all
    const int wgs = (step_groups(a) + STEP_WAVES - 1) / STEP_WAVES;
    const int turns = (wgs + STEP_PARTS_MAX - 1) / STEP_PARTS_MAX;
    return (wgs + turns - 1) / turns;
}

template <int R, int U, StepIn IN, StepOut OUT, bool WHOLE>
static int launch_step_of(const StepArgs &a, hipStream_t stream) {
    const size_t lds = (size_t)a.W.Kp * sizeof(float);
    static bool ready = false;        // (hosts are single-threaded per session; a second thread sets the same attribute)
    if (!ready) {
        MESH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(linear_step_kernel<R, U, IN, OUT, WHOLE>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)STEP_LDS_MAX));
        ready = true;
    }
    MESH_LAUNCH((linear_step_kernel<R, U, IN, OUT, WHOLE>), dim3((unsigned)linear_step_grid(a)), dim3(STEP_THREADS), lds, stream, a.W.w, a.W.Kp, step_groups(a), a.width, a.W.K, a);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}
template <int R, int U, StepIn IN, StepOut OUT>
static int launch_step(const StepArgs &a, hipStream_t stream) {
    return a.W.K % 4 ? launch_step_of<R, U, IN, OUT, false>(a, stream) : launch_step_of<R, U, IN, OUT, true>(a, stream);
}
template <StepIn IN, StepOut OUT>
static int launch_step_rows(const StepArgs &a, hipStream_t stream) {
    return rows_per_group(a) == 1 ? launch_step<1, 4, IN, OUT>(a, stream) : launch_step<2, 4, IN, OUT>(a, stream);
}

int linear_step(const StepArgs &a, hipStream_t stream) {
    const LinearWeight &W = a.W;
    if (!W.w || !a.in || !a.out || W.M < 1 || W.Kp % LINEAR_K_PAD || W.Kp < W.K || W.Mp < W.M || !linear_step_supported(W))
        return fail(MESH_ERR_INVALID, "linear_step: bad operands (%d x %d)", W.M, W.K);
    const bool resid = a.in_kind == STEP_IN_RESIDUAL || a.in_kind == STEP_IN_RESIDUAL_NORM;
    if ((resid && (!a.y || !a.gain || !a.part || !a.x_out || a.x_out == a.in || a.n_part < 1 || a.n_part > STEP_PARTS_MAX)) ||
        (a.in_kind == STEP_IN_RESIDUAL_NORM && !a.norm_gain) || (a.in_kind == STEP_IN_POLY && (!a.part || !a.coef || a.n_part < 1 || a.n_part > STEP_PARTS_MAX)))
        return fail(MESH_ERR_INVALID, "linear_step: input description incomplete");
    if ((a.in_kind == STEP_IN_LAYER && (!a.norm_gain || !a.norm_bias || (a.y && (!a.gain || !a.bias || !a.x_out || a.x_out == a.in)))) || (a.in_kind == STEP_IN_UNIT_RMS && !a.gain))
        return fail(MESH_ERR_INVALID, "linear_step: input description incomplete");
    if (a.in_kind == STEP_IN_HEADS && (!a.gain || !a.head_gate || a.head_width < 4 || a.head_width > 256 || (a.head_width & (a.head_width - 1)) || W.K % a.head_width ||
                                       ((reinterpret_cast<uintptr_t>(a.in) | reinterpret_cast<uintptr_t>(a.head_gate) | reinterpret_cast<uintptr_t>(a.gain)) & 15)))
        return fail(MESH_ERR_INVALID, "linear_step: input description incomplete");
    if (((a.out_kind == STEP_OUT_SUMSQ || a.out_kind == STEP_OUT_POWERS) && !a.out_part) ||
        (a.out_kind == STEP_OUT_MIN_GRU && (!a.state || !a.pos || !a.seq || !a.bias_z || !a.bias_x || a.width < 1 || W.M != 3 * a.width)) ||
        (a.out_kind == STEP_OUT_SIDE && (!a.side || !a.tok)))
        return fail(MESH_ERR_INVALID, "linear_step: output description incomplete");
#define MESH_STEP_CASE(IN, OUT) \
    if (a.in_kind == IN && a.out_kind == OUT) return launch_step_rows<IN, OUT>(a, stream);
    MESH_STEP_CASE(STEP_IN_VEC, STEP_OUT_PLAIN)
    MESH_STEP_CASE(STEP_IN_RESIDUAL, STEP_OUT_PLAIN)
    MESH_STEP_CASE(STEP_IN_RESIDUAL_NORM, STEP_OUT_PLAIN)
    MESH_STEP_CASE(STEP_IN_LAYER, STEP_OUT_PLAIN)
    MESH_STEP_CASE(STEP_IN_UNIT_RMS, STEP_OUT_PLAIN)
    MESH_STEP_CASE(STEP_IN_RELU2, STEP_OUT_PLAIN)
    MESH_STEP_CASE(STEP_IN_HEADS, STEP_OUT_PLAIN)
    MESH_STEP_CASE(STEP_IN_HEADS, STEP_OUT_SUMSQ)
    MESH_STEP_CASE(STEP_IN_VEC, STEP_OUT_SUMSQ)
    MESH_STEP_CASE(STEP_IN_POLY, STEP_OUT_SUMSQ)
    MESH_STEP_CASE(STEP_IN_RESIDUAL, STEP_OUT_POWERS)
    MESH_STEP_CASE(STEP_IN_RESIDUAL, STEP_OUT_SIDE)
#undef MESH_STEP_CASE
    if (a.in_kind == STEP_IN_VEC && a.out_kind == STEP_OUT_MIN_GRU) return launch_step<3, 2, STEP_IN_VEC, STEP_OUT_MIN_GRU>(a, stream);
    if (a.in_kind == STEP_IN_RESIDUAL && a.out_kind == STEP_OUT_MIN_GRU) return launch_step<3, 2, STEP_IN_RESIDUAL, STEP_OUT_MIN_GRU>(a, stream);
    return fail(MESH_ERR_UNSUPPORTED, "linear_step: no kernel for input %d with output %d", (int)a.in_kind, (int)a.out_kind);
}

}  // namespace mesh
