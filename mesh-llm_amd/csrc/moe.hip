// Mixture-of-experts routing for decode: softmax gate, expert mask, top-k, and the weighted sum of expert outputs.
// Follows llama.cpp's build_moe_ffn as patched by mesh-llm
// (third_party/llama.cpp/patches/0003-moe-add-expert-analysis-and-split-tools.patch:86-104): probabilities are the
// softmax of the router logits over every expert in the file; a 0 / -inf mask is ADDED to the probabilities used
// for selection only; the weights are the unmasked probabilities of the selected experts, renormalised to sum 1.

#include <algorithm>

#include "moe.hpp"
#include "expert_step.hpp"
#include "gemv.hpp"
#include "lds_ops.hpp"
#include "wave_ops.hpp"

namespace mesh {

constexpr int ROUTE_MAX_PER_LANE = MOE_EXPERTS_MAX / 64;

// softmax -> (+mask) -> top-k of one token's logits by one wave; NPL = experts per lane (n_expert <= 64 * NPL)
// (ids_copy: optional second destination of the expert ids, e.g. the workgroup's LDS)
template <int NPL>
__device__ __forceinline__ void route_wave(const float *lg, const float *mask, int n_expert, int top_k, int norm_w,
                                           int32_t *ids, float *weights, int lane, int32_t *ids_copy = nullptr) {
    float p[NPL], sel[NPL];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
        const int e = lane + 64 * i;
        p[i] = e < n_expert ? lg[e] : -INFINITY;
        mx = fmaxf(mx, p[i]);
    }
    mx = wave_max(mx);
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
        p[i] = lane + 64 * i < n_expert ? expf(p[i] - mx) : 0.f;
        den += p[i];
    }
    den = wave_sum(den);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
        const int e = lane + 64 * i;
        p[i] = p[i] / den;
        sel[i] = e < n_expert ? p[i] + (mask ? mask[e] : 0.f) : -INFINITY;
    }
    float wsum = 0.f, my_w = 0.f;
    int my_id = 0;
    // The best value left, then the first expert (ascending) that holds it and is not taken: a masked expert can still win once every allowed
    // one is, as in the reference's top-k over probabilities plus mask.  (An earlier form had every candidate count those before it,
    // one broadcast per expert: 64 of them cost more than top_k rounds whose maximum does not pass the LDS unit.)
    unsigned taken = 0;        // bit i: expert lane + 64 i has been selected
    for (int k = 0; k < top_k; ++k) {
        float best = -INFINITY;
#pragma unroll
        for (int i = 0; i < NPL; ++i) best = (taken >> i) & 1u ? best : fmaxf(best, sel[i]);
        best = wave_max(best);
        int bi = 0;
        float bp = p[0];        // (no candidate: values that are no numbers)
        bool found = false;
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
            const unsigned long long m = __builtin_amdgcn_ballot_w64(!((taken >> i) & 1u) && lane + 64 * i < n_expert && sel[i] == best);
            if (!found && m != 0ull) {
                found = true;
                const int src = __builtin_ctzll(m);
                bi = src + 64 * i;
                bp = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p[i]), src));
                if (lane == src) taken |= 1u << i;
            }
        }
        if (lane == k) { my_id = bi; my_w = bp; }
        wsum += bp;
    }
    if (lane < top_k) {
        ids[lane] = my_id;
        if (ids_copy) ids_copy[lane] = my_id;
        weights[lane] = norm_w && wsum > 0.f ? my_w / wsum : my_w;
    }
}

__device__ __forceinline__ void route_wave_any(const float *lg, const MoeRouteArgs &a, int t, int lane, int32_t *ids_copy = nullptr) {
    int32_t *ids = a.ids + (size_t)t * a.top_k;
    float *w = a.weights + (size_t)t * a.top_k;
    if (ids_copy) ids_copy += (size_t)t * a.top_k;
    if (a.n_expert <= 64) route_wave<1>(lg, a.mask, a.n_expert, a.top_k, a.norm_w, ids, w, lane, ids_copy);
    else if (a.n_expert <= 128) route_wave<2>(lg, a.mask, a.n_expert, a.top_k, a.norm_w, ids, w, lane, ids_copy);
    else route_wave<ROUTE_MAX_PER_LANE>(lg, a.mask, a.n_expert, a.top_k, a.norm_w, ids, w, lane, ids_copy);
}

// one wave per token
__global__ __launch_bounds__(64) void moe_route_kernel(MoeRouteArgs a) {
    const int t = blockIdx.x, lane = threadIdx.x;
    route_wave_any(a.logits + (size_t)t * a.n_expert, a, t, lane);
}

// Router logits and routing in one launch, one workgroup per token: every wave holds the token's normalised hidden
// state in registers (E / 64 values per lane) and takes every fourth expert row of the f32 router matrix; the
// logits meet in LDS and the first wave routes.  logits[t] = W . (x[t] * rsqrt(mean(x^2) + eps) * norm_w).
constexpr int ROUTER_THREADS = 1024, ROUTER_WAVES = ROUTER_THREADS / 64;
// (RT: threads of the workgroup.  A decode batch has few tokens and wants every wave it can get on a token's expert rows;
// a prefill chunk has a workgroup per token anyway, and small workgroups, eight to a CU, hide each other's row loads.)
constexpr int ROUTER_THREADS_WIDE = 256, ROUTER_WIDE_MIN_TOKENS = 512;
// four neighbouring elements of a token's row as pairs of f16 (expert_step.hpp, by token)
__device__ __forceinline__ void store_planes(_Float16 *planes, int E, int t, int k, const float4 &v, float inverse) {
    const float x[4] = {v.x, v.y, v.z, v.w};
    _Float16 hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) pair_of(x[i] * inverse, hi[i], lo[i]);
    _Float16 *to = planes + (size_t)(t >> 4) * 32 * E + ((size_t)(k >> 3) * 32 + (t & 15)) * 8 + (k & 7);
    *reinterpret_cast<uint2 *>(to) = __builtin_bit_cast(uint2, hi);
    *reinterpret_cast<uint2 *>(to + 128) = __builtin_bit_cast(uint2, lo);
}
// the logits of this workgroup's token, into s_logits and logits_out
template <int NV, int RT>      // float4 groups per lane = E / 256
__device__ __forceinline__ void router_logits(const float *__restrict__ x, const float *__restrict__ norm_w, const float *__restrict__ W,
                                              float *__restrict__ logits_out, int ldx, float eps, int p_n_expert, float *s_logits,
                                              float *__restrict__ scale_out = nullptr) {
    constexpr int E = NV * 256, ROUTER_WAVES = RT / 64;
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // element index of a lane's values: 4 * (lane + 64 * i) + c
    const float *xt = x + (size_t)t * ldx;
    float4 xr[NV];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        xr[i] = *reinterpret_cast<const float4 *>(xt + 4 * (lane + 64 * i));
        ss += xr[i].x * xr[i].x + xr[i].y * xr[i].y + xr[i].z * xr[i].z + xr[i].w * xr[i].w;
    }
    const float scale = 1.0f / sqrtf(wave_sum(ss) / (float)E + eps);
    if (scale_out && threadIdx.x == 0) scale_out[t] = scale;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const float4 w = *reinterpret_cast<const float4 *>(norm_w + 4 * (lane + 64 * i));
        xr[i].x = xr[i].x * scale * w.x; xr[i].y = xr[i].y * scale * w.y;
        xr[i].z = xr[i].z * scale * w.z; xr[i].w = xr[i].w * scale * w.w;
    }
    // two expert rows per step, all of their loads in flight together
    for (int e0 = wave; e0 < p_n_expert; e0 += 2 * ROUTER_WAVES) {
        const int e1 = e0 + ROUTER_WAVES;
        const bool has1 = e1 < p_n_expert;
        const float *w0 = W + (size_t)e0 * E, *w1 = W + (size_t)(has1 ? e1 : e0) * E;
        float4 r0[NV], r1[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            r0[i] = *reinterpret_cast<const float4 *>(w0 + 4 * (lane + 64 * i));
            r1[i] = *reinterpret_cast<const float4 *>(w1 + 4 * (lane + 64 * i));
        }
        float a0 = 0.f, a1 = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            a0 = fmaf(xr[i].x, r0[i].x, a0); a0 = fmaf(xr[i].y, r0[i].y, a0); a0 = fmaf(xr[i].z, r0[i].z, a0); a0 = fmaf(xr[i].w, r0[i].w, a0);
            a1 = fmaf(xr[i].x, r1[i].x, a1); a1 = fmaf(xr[i].y, r1[i].y, a1); a1 = fmaf(xr[i].z, r1[i].z, a1); a1 = fmaf(xr[i].w, r1[i].w, a1);
        }
        a0 = wave_sum(a0);
        a1 = wave_sum(a1);
        if (lane == 0) {
            s_logits[e0] = a0;
            if (logits_out) logits_out[(size_t)t * p_n_expert + e0] = a0;
            if (has1) {
                s_logits[e1] = a1;
                if (logits_out) logits_out[(size_t)t * p_n_expert + e1] = a1;
            }
        }
    }
}

template <int NV, int RT>
// (scalar arguments first: preloaded into SGPRs, see gemv.hip)
__global__ __launch_bounds__(RT) void moe_router_fused_kernel(const float *__restrict__ x, const float *__restrict__ norm_w,
                                                                          const float *__restrict__ W, float *__restrict__ logits_out,
                                                                          int ldx, float eps, int p_n_expert, const MoeRouteArgs a, float *__restrict__ scale_out) {
    __shared__ float s_logits[64 * ROUTE_MAX_PER_LANE];
    router_logits<NV, RT>(x, norm_w, W, logits_out, ldx, eps, p_n_expert, s_logits, scale_out);
    __syncthreads();
    if ((threadIdx.x >> 6) == 0) route_wave_any(s_logits, a, blockIdx.x, threadIdx.x & 63);
}

// The same for hidden sizes up to 2048, TOKENS of a call per workgroup: every wave keeps their normalised hidden states in registers and
// walks every eighth expert row, the next one on its way, the first while the states are normalised.  Every (token, expert) logit is the
// sum the kernel above forms, in its order; the first waves then route one token each.
// Bound by the CU's fetch of the whole router matrix from L2 (512 KB at about 95 GB/s: 5.4 us), before it the rows' and the norm's chain,
// behind it the picks.  So a workgroup takes as many tokens as leave one for every CU.  64 experts x 2048, us, a token a workgroup of sixteen
// waves / four tokens a workgroup, both with no row ahead (before) and two, three or four tokens: 40 tokens 19.2 / - / 12.6, 333 25.1
// / - / 12.0, 512 - / 15.9 / 12.6, 600 - / 16.4 / 14.2, 1024 - / 16.9 / 16.7, 2048 - / 29.1 / 29.2.  16 experts x 2048: one token 6.5 / - / 5.0, 16 7.8 / - / 6.2.
constexpr int CHUNK_WAVES = 8;
template <int NV, int TOKENS>
__global__ __launch_bounds__(64 * CHUNK_WAVES) void moe_router_chunk_kernel(const float *__restrict__ x, const float *__restrict__ norm_w,
                                                                      const float *__restrict__ W, float *__restrict__ logits_out,
                                                                      int ldx, float eps, int T, const MoeRouteArgs a, float *__restrict__ scale_out,
                                                                      _Float16 *__restrict__ rows_out, unsigned *sat) {
    constexpr int E = NV * 256;
    __shared__ float s_logits[TOKENS][64 * ROUTE_MAX_PER_LANE];
    const int t0 = blockIdx.x * TOKENS, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float4 xr[TOKENS][NV], nw[NV], r[2][NV];
    float sc[TOKENS];
    auto fetch = [&](float4 (&to)[NV], int e) {
        const float *wr = W + (size_t)(e < a.n_expert ? e : a.n_expert - 1) * E;       // (past the last row: not used)
#pragma unroll
        for (int i = 0; i < NV; ++i) to[i] = *reinterpret_cast<const float4 *>(wr + 4 * (lane + 64 * i));
    };
#pragma unroll
    for (int k = 0; k < TOKENS; ++k) {
        const float *xt = x + (size_t)(t0 + k < T ? t0 + k : T - 1) * ldx;
#pragma unroll
        for (int i = 0; i < NV; ++i) xr[k][i] = *reinterpret_cast<const float4 *>(xt + 4 * (lane + 64 * i));
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) nw[i] = *reinterpret_cast<const float4 *>(norm_w + 4 * (lane + 64 * i));
    fetch(r[0], wave);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < TOKENS; ++k) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) ss += xr[k][i].x * xr[k][i].x + xr[k][i].y * xr[k][i].y + xr[k][i].z * xr[k][i].z + xr[k][i].w * xr[k][i].w;
        const float scale = 1.0f / sqrtf(wave_sum(ss) / (float)E + eps);
        sc[k] = scale;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            xr[k][i].x = xr[k][i].x * scale * nw[i].x; xr[k][i].y = xr[k][i].y * scale * nw[i].y;
            xr[k][i].z = xr[k][i].z * scale * nw[i].z; xr[k][i].w = xr[k][i].w * scale * nw[i].w;
        }
    }
    // (a wave a token; the stores are on their way while the experts' rows go by)
    if (rows_out)
#pragma unroll
        for (int k = 0; k < TOKENS; ++k)
            if (wave == k && t0 + k < T)
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    const float4 v = xr[k][i];
                    if (sat) {
                        const unsigned clamped = (fmaxf(fabsf(v.x), fabsf(v.y)) > 65504.f ? 1u : 0u) + (fmaxf(fabsf(v.z), fabsf(v.w)) > 65504.f ? 1u : 0u);
                        if (clamped) atomicAdd(sat, clamped * (unsigned)a.top_k);
                    }
                    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                    const h4 h = {(_Float16)__builtin_amdgcn_fmed3f(v.x, -65504.f, 65504.f), (_Float16)__builtin_amdgcn_fmed3f(v.y, -65504.f, 65504.f),
                                  (_Float16)__builtin_amdgcn_fmed3f(v.z, -65504.f, 65504.f), (_Float16)__builtin_amdgcn_fmed3f(v.w, -65504.f, 65504.f)};
                    *reinterpret_cast<h4 *>(rows_out + (size_t)(t0 + k) * E + 4 * (lane + 64 * i)) = h;
                }
    for (int e0 = wave; e0 < a.n_expert; e0 += 2 * CHUNK_WAVES) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = e0 + u * CHUNK_WAVES;
            if (e >= a.n_expert) break;
            fetch(r[u ^ 1], e + CHUNK_WAVES);
            float acc[TOKENS];
#pragma unroll
            for (int k = 0; k < TOKENS; ++k) {
                float v = 0.f;
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    v = fmaf(xr[k][i].x, r[u][i].x, v); v = fmaf(xr[k][i].y, r[u][i].y, v); v = fmaf(xr[k][i].z, r[u][i].z, v); v = fmaf(xr[k][i].w, r[u][i].w, v);
                }
                acc[k] = v;
            }
#pragma unroll
            for (int k = 0; k < TOKENS; ++k) acc[k] = wave_sum(acc[k]);
            if (lane == 0) {
#pragma unroll
                for (int k = 0; k < TOKENS; ++k) {
                    s_logits[k][e] = acc[k];
                    if (logits_out && t0 + k < T) logits_out[(size_t)(t0 + k) * a.n_expert + e] = acc[k];
                }
            }
        }
    }
    if (scale_out && wave == 0 && lane == 0)
#pragma unroll
        for (int k = 0; k < TOKENS; ++k)
            if (t0 + k < T) scale_out[t0 + k] = sc[k];
    __syncthreads();
    if (wave < TOKENS && t0 + wave < T) route_wave_any(s_logits[wave], a, t0 + wave, lane);
}
template <int TOKENS>
static void launch_router_chunk(const MoeRouteArgs &a, const float *x, int ldx, const float *norm_w, float eps, const float *W, int E, float *logits_out, int T, hipStream_t stream,
                                float *scale_out, _Float16 *rows_out, unsigned *sat) {
    const dim3 grid((unsigned)((T + TOKENS - 1) / TOKENS)), block(64 * CHUNK_WAVES);
    switch (E / 256) {
        case 2: MESH_LAUNCH((moe_router_chunk_kernel<2, TOKENS>), grid, block, 0, stream, x, norm_w, W, logits_out, ldx, eps, T, a, scale_out, rows_out, sat); break;
        case 4: MESH_LAUNCH((moe_router_chunk_kernel<4, TOKENS>), grid, block, 0, stream, x, norm_w, W, logits_out, ldx, eps, T, a, scale_out, rows_out, sat); break;
        default: MESH_LAUNCH((moe_router_chunk_kernel<8, TOKENS>), grid, block, 0, stream, x, norm_w, W, logits_out, ldx, eps, T, a, scale_out, rows_out, sat); break;
    }
}

// Router logits of a batch of decode steps, a workgroup per token and four experts, one row of the matrix per wave.  The bits of router_logits:
// the sums of a lane's elements and of the lanes go the same way.  planes (optional): the normalised row as pairs of f16.
// Bound by its chain (row, sum of squares, dot product).  16 tokens, 64 experts x 2048: 3.6 us (3.5-4.0 in traces of whole steps); 9.4 with sixteen rows a workgroup, each wave of which
// loaded and normalised the token's row for itself and added lanes up through the LDS unit.  (Before, the last of those workgroups to
// arrive routed and grouped behind a hand-over between workgroups: 19.4 us in one launch, against 3.6 + 5.6 now.)
constexpr int SLICE_THREADS = 256, SLICE_WAVES = SLICE_THREADS / 64;
static_assert(SLICE_WAVES == 4, "the maxima of a row's four shares");
template <int NV>
__global__ __launch_bounds__(SLICE_THREADS) void moe_router_slice_kernel(const float *__restrict__ x, const float *__restrict__ norm_w, const float *__restrict__ W,
                                                                         float *__restrict__ logits, int ldx, float eps, int n_expert, _Float16 *__restrict__ planes, float *__restrict__ plane_scale) {
    constexpr int E = NV * 256, PER = E / 4 / SLICE_THREADS > 0 ? E / 4 / SLICE_THREADS : 1;       // float4 groups of the row a thread brings
    __shared__ __align__(16) float s_x[E];
    __shared__ float s_sq[E / 4], s_max[SLICE_WAVES];
    const int t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int e = blockIdx.x * SLICE_WAVES + wave, row = e < n_expert ? e : n_expert - 1;
    const float *xt = x + (size_t)t * ldx;
    float4 xv[PER], nw[PER], r[NV];
#pragma unroll
    for (int i = 0; i < PER; ++i) xv[i] = *reinterpret_cast<const float4 *>(xt + 4 * ((tid + SLICE_THREADS * i) % (E / 4)));
#pragma unroll
    for (int i = 0; i < PER; ++i) nw[i] = *reinterpret_cast<const float4 *>(norm_w + 4 * ((tid + SLICE_THREADS * i) % (E / 4)));
    // the row of the matrix is on its way while the token's is normalised
#pragma unroll
    for (int i = 0; i < NV; ++i) r[i] = *reinterpret_cast<const float4 *>(W + (size_t)row * E + 4 * (lane + 64 * i));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < PER; ++i)
        if (tid + SLICE_THREADS * i < E / 4) s_sq[tid + SLICE_THREADS * i] = xv[i].x * xv[i].x + xv[i].y * xv[i].y + xv[i].z * xv[i].z + xv[i].w * xv[i].w;
    lds_barrier();
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) ss += s_sq[lane + 64 * i];
    const float scale = 1.0f / sqrtf(wave_sum(ss) / (float)E + eps);
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int g = tid + SLICE_THREADS * i;
        xv[i] = make_float4(xv[i].x * scale * nw[i].x, xv[i].y * scale * nw[i].y, xv[i].z * scale * nw[i].z, xv[i].w * scale * nw[i].w);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(xv[i].x), fabsf(xv[i].y)), fmaxf(fabsf(xv[i].z), fabsf(xv[i].w))));
        if (g < E / 4) *reinterpret_cast<float4 *>(s_x + 4 * g) = xv[i];
    }
    const bool writes_planes = planes && blockIdx.x == 0;
    if (writes_planes) {
        mx = wave_max(mx);
        if (lane == 0) s_max[wave] = mx;
    }
    lds_barrier();
    if (writes_planes) {
        const PairScale ps = pair_scale(fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3])));
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (tid + SLICE_THREADS * i < E / 4) store_planes(planes, E, t, 4 * (tid + SLICE_THREADS * i), xv[i], ps.inverse);
        if (tid == 0) plane_scale[t] = ps.scale;
    }
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const float4 v = *reinterpret_cast<const float4 *>(s_x + 4 * (lane + 64 * i));
        acc = fmaf(v.x, r[i].x, acc); acc = fmaf(v.y, r[i].y, acc); acc = fmaf(v.z, r[i].z, acc); acc = fmaf(v.w, r[i].w, acc);
    }
    acc = wave_sum(acc);
    if (lane == 0 && e < n_expert) logits[(size_t)t * n_expert + e] = acc;
}

bool moe_router_writes_rows(int E, int n_expert, int T) {
    return E <= 2048 && !(T <= 256 && E <= 1024 && n_expert >= 96);
}

int moe_router_fused(const MoeRouteArgs &a, const float *x, int ldx, const float *norm_w, float eps, const float *W, int E,
                     float *logits_out, int T, hipStream_t stream, float *scale_out, uint16_t *rows_out, unsigned *sat) {
    if (T <= 0) return MESH_OK;
    if (!moe_router_fused_supported(E, a.n_expert, a.top_k)) return fail(MESH_ERR_UNSUPPORTED, "moe: fused router for hidden size %d / %d experts", E, a.n_expert);
    const dim3 grid((unsigned)T);
    // Up to 256 tokens every token has a CU of its own either way, and of many short rows sixteen waves walk half as many each: us, two tokens a
    // workgroup of eight waves / one a workgroup of sixteen, 200 tokens: E 512 with 96 experts 9.1 / 7.4, 128 10.0 / 8.4, 256 18.6 / 15.0,
    // 512 29.9 / 21.0; E 1024 with 96 10.0 / 9.0, 128 11.8 / 10.3, 256 20.8 / 18.3, 512 34.5 / 28.6; E 2048 with 64 9.9 / 17.9, 512 53 / 112
    // (those two with sums through the LDS unit).  300 tokens, E 512, 512 experts: 29.4 / 33.
    const bool chunk = moe_router_writes_rows(E, a.n_expert, T);
    if (rows_out && !chunk) return fail(MESH_ERR_UNSUPPORTED, "moe: rows of a router that writes none");
    if (chunk) {
        _Float16 *const rows = reinterpret_cast<_Float16 *>(rows_out);
        if (T <= 2 * 256) launch_router_chunk<2>(a, x, ldx, norm_w, eps, W, E, logits_out, T, stream, scale_out, rows, sat);
        else if (T <= 3 * 256) launch_router_chunk<3>(a, x, ldx, norm_w, eps, W, E, logits_out, T, stream, scale_out, rows, sat);
        else launch_router_chunk<4>(a, x, ldx, norm_w, eps, W, E, logits_out, T, stream, scale_out, rows, sat);
        MESH_LAUNCH_CHECK();
        return MESH_OK;
    }
    if (T >= ROUTER_WIDE_MIN_TOKENS) MESH_LAUNCH((moe_router_fused_kernel<16, ROUTER_THREADS_WIDE>), grid, dim3(ROUTER_THREADS_WIDE), 0, stream, x, norm_w, W, logits_out, ldx, eps, a.n_expert, a, scale_out);
    else if (E == 512) MESH_LAUNCH((moe_router_fused_kernel<2, ROUTER_THREADS>), grid, dim3(ROUTER_THREADS), 0, stream, x, norm_w, W, logits_out, ldx, eps, a.n_expert, a, scale_out);
    else if (E == 1024) MESH_LAUNCH((moe_router_fused_kernel<4, ROUTER_THREADS>), grid, dim3(ROUTER_THREADS), 0, stream, x, norm_w, W, logits_out, ldx, eps, a.n_expert, a, scale_out);
    else MESH_LAUNCH((moe_router_fused_kernel<16, ROUTER_THREADS>), grid, dim3(ROUTER_THREADS), 0, stream, x, norm_w, W, logits_out, ldx, eps, a.n_expert, a, scale_out);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}
bool moe_router_fused_supported(int E, int n_expert, int top_k) {
    return (E == 512 || E == 1024 || E == 2048 || E == 4096) && n_expert >= 1 && n_expert <= 64 * ROUTE_MAX_PER_LANE && top_k >= 1 && top_k <= 64 && top_k <= n_expert;
}

int moe_route(const MoeRouteArgs &a, int T, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    if (a.n_expert < 1 || a.n_expert > 64 * ROUTE_MAX_PER_LANE || a.top_k < 1 || a.top_k > 64 || a.top_k > a.n_expert)
        return fail(MESH_ERR_UNSUPPORTED, "moe: %d experts / top-%d outside what the router kernel handles", a.n_expert, a.top_k);
    MESH_LAUNCH(moe_route_kernel, dim3((unsigned)T), dim3(64), 0, stream, a);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// Pairs -> per-expert work items, one workgroup.  The pair list sits in LDS; a wave takes every 16th expert and finds
// its pairs with ballots over the list (64 pairs per step), first to count, then -- after a prefix sum over the
// experts' item counts -- to write each pair into its item.
constexpr int GROUP_THREADS = 1024, GROUP_WAVES = GROUP_THREADS / 64;
// (whole workgroup; lds: n_pairs + 2 * n_expert ints)
// ipairs: most pairs per item; an item takes iints = moe_item_ints(ipairs) int32
// ids == nullptr: the pair list is in lds[0 .. n_pairs) already and a barrier has been passed since it was written
__device__ __forceinline__ void group_pairs(const int32_t *__restrict__ ids, int n_pairs, int n_expert, int32_t *__restrict__ items,
                                            int32_t *__restrict__ n_items, int32_t *lds, int ipairs) {
    const int iints = moe_item_ints(ipairs), shift = __builtin_ctz((unsigned)ipairs);       // (a power of two)
    int32_t *s_ids = lds, *s_cnt = lds + n_pairs, *s_base = s_cnt + n_expert;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (ids) {
        for (int p = tid; p < n_pairs; p += GROUP_THREADS) s_ids[p] = ids[p];
        __syncthreads();
    }
    // the first pairs of the list stay in a lane's registers: a wave's experts find theirs among them without a trip to LDS
    constexpr int HELD = 4;
    int held[HELD];
#pragma unroll
    for (int j = 0; j < HELD; ++j) held[j] = lane + 64 * j < n_pairs ? s_ids[lane + 64 * j] : -1;
    for (int e = wave; e < n_expert; e += GROUP_WAVES) {
        int c = 0;
#pragma unroll
        for (int j = 0; j < HELD; ++j) c += __popcll(__ballot(held[j] == e));
        for (int p0 = 64 * HELD; p0 < n_pairs; p0 += 64) {
            const int p = p0 + lane;
            c += __popcll(__ballot(p < n_pairs && s_ids[p] == e));
        }
        if (lane == 0) s_cnt[e] = c;
    }
    lds_barrier();
    if (wave == 0) {
        // exclusive prefix of items per expert: each lane sums a run of experts, the runs are scanned across the wave
        const int per = (n_expert + 63) / 64, e0 = lane * per;
        int mine = 0;
        for (int e = e0; e < e0 + per && e < n_expert; ++e) mine += (s_cnt[e] + ipairs - 1) >> shift;
        const int incl = wave_scan(mine);
        int run = incl - mine;
        for (int e = e0; e < e0 + per && e < n_expert; ++e) {
            s_base[e] = run;
            run += (s_cnt[e] + ipairs - 1) >> shift;
        }
        if (lane == 63) n_items[0] = incl;
    }
    lds_barrier();
    for (int e = wave; e < n_expert; e += GROUP_WAVES) {
        const int cnt = s_cnt[e], base = s_base[e];
        int seen = 0;
        auto place = [&](int p, bool hit) {
            const unsigned long long m = __ballot(hit);
            if (hit) {
                const int r = seen + __popcll(m & ((1ull << lane) - 1ull));
                items[(size_t)(base + (r >> shift)) * iints + 2 + (r & (ipairs - 1))] = p;
            }
            seen += __popcll(m);
        };
#pragma unroll
        for (int j = 0; j < HELD; ++j) place(lane + 64 * j, held[j] == e);
        for (int p0 = 64 * HELD; p0 < n_pairs && seen < cnt; p0 += 64) place(p0 + lane, p0 + lane < n_pairs && s_ids[p0 + lane] == e);
        const int n_it = (cnt + ipairs - 1) >> shift;
        for (int i = lane; i < n_it; i += 64) {
            items[(size_t)(base + i) * iints + 0] = e;
            items[(size_t)(base + i) * iints + 1] = i + 1 < n_it ? ipairs : cnt - i * ipairs;
        }
    }
}

__global__ __launch_bounds__(GROUP_THREADS) void moe_group_kernel(const int32_t *__restrict__ ids, int n_pairs, int n_expert,
                                                                  int32_t *__restrict__ items, int32_t *__restrict__ n_items, int ipairs) {
    extern __shared__ int32_t g_lds[];
    group_pairs(ids, n_pairs, n_expert, items, n_items, g_lds, ipairs);
}

// Routing of a small batch and the grouping of its pairs in one single-workgroup launch: wave w routes tokens w,
// w + 16, ... from their logits, then the workgroup groups the pairs it has just written (the barrier in between
// also makes those writes visible to the whole workgroup).  A chain: 9.1 us with reductions through the LDS unit and a rank counted
// over all candidates, 5.6 now (16 tokens, 64 experts, top 8, timed apart; 4.5 of it without the grouping; 6.8-7.2 in traces of whole steps).
// (the routing arguments as leading scalars: preloaded into SGPRs, see gemv.hip)
__global__ __launch_bounds__(GROUP_THREADS) void moe_route_group_kernel(const float *p_logits, const float *p_mask, int32_t *p_ids, float *p_weights,
                                                                        int T, int p_n_expert, int p_top_k, int p_norm_w,
                                                                        int32_t *__restrict__ items, int32_t *__restrict__ n_items, int ipairs) {
    extern __shared__ int32_t g_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    MoeRouteArgs a;
    a.logits = p_logits; a.mask = p_mask; a.ids = p_ids; a.weights = p_weights; a.n_expert = p_n_expert; a.top_k = p_top_k; a.norm_w = p_norm_w;
    // (the ids also go to the pair list in LDS: the grouping does not wait for them to come back from memory)
    for (int t = wave; t < T; t += GROUP_WAVES) route_wave_any(p_logits + (size_t)t * p_n_expert, a, t, lane, g_lds);
    __syncthreads();
    group_pairs(nullptr, T * p_top_k, p_n_expert, items, n_items, g_lds, ipairs);
}

int moe_router_group(const MoeRouteArgs &a, const float *x, int ldx, const float *norm_w, float eps, const float *W, int E,
                     float *logits, int T, int32_t *items, int32_t *n_items, int item_pairs, hipStream_t stream, uint16_t *planes, float *plane_scale) {
    if (T <= 0) return MESH_OK;
    if (!moe_router_group_supported(E, a.n_expert, a.top_k, T) || !logits)
        return fail(MESH_ERR_UNSUPPORTED, "moe: split router for hidden size %d / %d experts / %d tokens", E, a.n_expert, T);
    const dim3 grid((unsigned)((a.n_expert + SLICE_WAVES - 1) / SLICE_WAVES), (unsigned)T), block(SLICE_THREADS);
    MoeRouteArgs la = a;
    _Float16 *p = reinterpret_cast<_Float16 *>(planes);
    switch (E / 256) {
        case 2: MESH_LAUNCH(moe_router_slice_kernel<2>, grid, block, 0, stream, x, norm_w, W, logits, ldx, eps, a.n_expert, p, plane_scale); break;
        case 4: MESH_LAUNCH(moe_router_slice_kernel<4>, grid, block, 0, stream, x, norm_w, W, logits, ldx, eps, a.n_expert, p, plane_scale); break;
        case 8: MESH_LAUNCH(moe_router_slice_kernel<8>, grid, block, 0, stream, x, norm_w, W, logits, ldx, eps, a.n_expert, p, plane_scale); break;
        case 16: MESH_LAUNCH(moe_router_slice_kernel<16>, grid, block, 0, stream, x, norm_w, W, logits, ldx, eps, a.n_expert, p, plane_scale); break;
        default: return fail(MESH_ERR_UNSUPPORTED, "moe: fused router for hidden size %d", E);
    }
    MESH_LAUNCH_CHECK();
    la.logits = logits;
    const size_t smem = ((size_t)T * a.top_k + 2 * (size_t)a.n_expert) * sizeof(int32_t);
    MESH_LAUNCH(moe_route_group_kernel, dim3(1), dim3(GROUP_THREADS), smem, stream, la.logits, la.mask, la.ids, la.weights, T, la.n_expert, la.top_k, la.norm_w,
                                                                           items, n_items, item_pairs);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}
bool moe_router_group_supported(int E, int n_expert, int top_k, int T) {
    return moe_router_fused_supported(E, n_expert, top_k) && n_expert > ROUTER_WAVES && T >= 1 && T <= 64 &&
           ((size_t)T * top_k + 2 * (size_t)n_expert) * sizeof(int32_t) <= 28 * 1024;      // (plus 32 KB of logits rows in the same workgroup)
}

bool moe_group_supported(int n_pairs, int n_expert) {
    return n_pairs >= 1 && n_expert >= 1 && ((size_t)n_pairs + 2 * (size_t)n_expert) * sizeof(int32_t) <= 128 * 1024;
}

int moe_group(const int32_t *ids, int n_pairs, int n_expert, int32_t *items, int32_t *n_items, int item_pairs, hipStream_t stream) {
    if (!moe_group_supported(n_pairs, n_expert)) return fail(MESH_ERR_UNSUPPORTED, "moe: %d pairs over %d experts do not fit the grouping kernel", n_pairs, n_expert);
    static bool attr_set = false;
    if (!attr_set) {
        MESH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(moe_group_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024));
        attr_set = true;
    }
    const size_t smem = ((size_t)n_pairs + 2 * (size_t)n_expert) * sizeof(int32_t);
    MESH_LAUNCH(moe_group_kernel, dim3(1), dim3(GROUP_THREADS), smem, stream, ids, n_pairs, n_expert, items, n_items, item_pairs);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// out[t][i] = x[t][i] + sum_s w[t][s] * y[(t*top_k + s)][i]; out may be x
__global__ __launch_bounds__(256) void moe_combine_kernel(const float *x, float *out, const float *__restrict__ y,
                                                          const float *__restrict__ w, int n_embd, int top_k) {
    const int t = blockIdx.y;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_embd) return;
    float acc = x[(size_t)t * n_embd + i];
    for (int s = 0; s < top_k; ++s) acc = fmaf(w[(size_t)t * top_k + s], y[((size_t)t * top_k + s) * n_embd + i], acc);
    out[(size_t)t * n_embd + i] = acc;
}

int moe_combine(const float *x, float *out, const float *y, const float *w, int T, int n_embd, int top_k, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    MESH_LAUNCH(moe_combine_kernel, dim3((unsigned)((n_embd + 255) / 256), (unsigned)T), dim3(256), 0, stream, x, out, y, w, n_embd, top_k);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// the same with the rows of y at the slots of moe_sort: out[t][i] = x[t][i] + sum_s w[t][s] * y[slot_of_pair[t*top_k + s]][i], four columns a thread
__global__ __launch_bounds__(256) void moe_combine_slots_kernel(const float *x, float *out, const float *__restrict__ y, const float *__restrict__ w,
                                                                const int32_t *__restrict__ slot_of_pair, int n_embd, int top_k) {
    const int t = blockIdx.y;
    const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n_embd) return;
    float4 acc = *reinterpret_cast<const float4 *>(x + (size_t)t * n_embd + i);
    for (int s = 0; s < top_k; ++s) {
        const float ws = w[(size_t)t * top_k + s];
        const float4 v = *reinterpret_cast<const float4 *>(y + (size_t)slot_of_pair[(size_t)t * top_k + s] * n_embd + i);
        acc.x = fmaf(ws, v.x, acc.x); acc.y = fmaf(ws, v.y, acc.y); acc.z = fmaf(ws, v.z, acc.z); acc.w = fmaf(ws, v.w, acc.w);
    }
    *reinterpret_cast<float4 *>(out + (size_t)t * n_embd + i) = acc;
}

int moe_combine_slots(const float *x, float *out, const float *y, const float *w, const int32_t *slot_of_pair, int T, int n_embd, int top_k, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    if (n_embd % 4) return fail(MESH_ERR_INVALID, "moe_combine_slots: row length %d not a multiple of 4", n_embd);
    MESH_LAUNCH(moe_combine_slots_kernel, dim3((unsigned)((n_embd / 4 + 255) / 256), (unsigned)T), dim3(256), 0, stream, x, out, y, w, slot_of_pair, n_embd, top_k);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

// ---- pairs sorted by expert for the large-tile GEMM ------------------------------------------------------------
// One workgroup: counts per expert (LDS atomics), a scan over the experts for the first slot (a multiple of 16) and the
// tiles of each, then every pair takes the next free slot of its expert.  Which slot of its expert a pair gets
// depends on the order the atomics land in; nothing computed from the slots does (a column of a matrix product depends
// on that column alone, and the combine step finds its rows through slot_of_pair).
constexpr int SORT_THREADS = 1024;
__global__ __launch_bounds__(SORT_THREADS) void moe_sort_kernel(const int32_t *__restrict__ ids, int n_pairs, int n_expert, int cap_slots,
                                                                int32_t *__restrict__ slot_of_pair, int32_t *__restrict__ pair_of_slot,
                                                                int32_t *__restrict__ tiles, int32_t *__restrict__ counts) {
    extern __shared__ int32_t s_lds[];
    int32_t *s_cnt = s_lds, *s_off = s_cnt + n_expert, *s_full = s_off + n_expert, *s_rest = s_full + n_expert;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int e = tid; e < n_expert; e += SORT_THREADS) s_cnt[e] = 0;
    for (int sl = tid; sl < cap_slots; sl += SORT_THREADS) pair_of_slot[sl] = -1;
    __syncthreads();
    for (int p = tid; p < n_pairs; p += SORT_THREADS) atomicAdd(&s_cnt[ids[p]], 1);
    __syncthreads();
    if (wave == 0) {
        // exclusive prefixes over the experts: each lane sums a run of them, the runs are scanned across the wave.  [0]: padded
        // slots; [1..4]: tiles of more than 96, 64, 32 and 0 pairs.  The list begins with the largest tiles and ends with the
        // smallest: workgroups start in its order, and a long one that starts last is waited for with the chip idle.
        const int per = (n_expert + 63) / 64, e0 = lane * per;
        int mine[5] = {0, 0, 0, 0, 0}, run[5], base[5];
        for (int e = e0; e < e0 + per && e < n_expert; ++e) {
            const int c = s_cnt[e], rest = c & 127;
            mine[0] += (c + 15) & ~15;
            mine[1] += c >> 7;
#pragma unroll
            for (int k = 1; k < 5; ++k) mine[k] += rest && 4 - ((rest - 1) >> 5) == k ? 1 : 0;
        }
        int total = 0;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            const int in = wave_scan(mine[k]), sum = __builtin_amdgcn_readlane(in, 63);
            base[k] = k < 1 ? 0 : total;
            run[k] = base[k] + in - mine[k];
            if (k == 0) { if (lane == 0) counts[1] = sum; } else total += sum;
        }
        if (lane == 0) counts[0] = total;
        for (int e = e0; e < e0 + per && e < n_expert; ++e) {
            const int c = s_cnt[e], rest = c & 127;
            s_off[e] = run[0]; run[0] += (c + 15) & ~15;
            s_full[e] = run[1]; run[1] += c >> 7;
#pragma unroll
            for (int k = 1; k < 5; ++k)
                if (rest && 4 - ((rest - 1) >> 5) == k) s_rest[e] = run[k]++;
        }
    }
    __syncthreads();
    for (int e = tid; e < n_expert; e += SORT_THREADS) {
        const int cnt = s_cnt[e];
        for (int j = 0; j * 128 < cnt; ++j) {
            const int n = cnt - 128 * j < 128 ? cnt - 128 * j : 128;
            int32_t *tl = tiles + (size_t)(n == 128 ? s_full[e] + j : s_rest[e]) * 4;
            tl[0] = e; tl[1] = s_off[e] + 128 * j; tl[2] = n; tl[3] = 0;
        }
    }
    __syncthreads();
    for (int p = tid; p < n_pairs; p += SORT_THREADS) {
        const int e = ids[p];
        const int sl = atomicAdd(&s_off[e], 1);
        slot_of_pair[p] = sl;
        pair_of_slot[sl] = p;
    }
}

int moe_sort_slots(int n_pairs, int n_expert) { return (n_pairs + 15 * std::min(n_pairs, n_expert) + 15) / 16 * 16; }
int moe_sort_max_tiles(int n_pairs, int n_expert) { return n_pairs / 128 + std::min(n_pairs, n_expert); }

int moe_sort(const int32_t *ids, int n_pairs, int n_expert, const MoeSorted &out, hipStream_t stream) {
    if (n_pairs < 1 || n_expert < 1 || n_expert > 4096 || !ids || !out.slot_of_pair || !out.pair_of_slot || !out.tiles || !out.counts)
        return fail(MESH_ERR_INVALID, "moe_sort: bad arguments (%d pairs, %d experts)", n_pairs, n_expert);
    MESH_LAUNCH(moe_sort_kernel, dim3(1), dim3(SORT_THREADS), 4 * (size_t)n_expert * sizeof(int32_t), stream, ids, n_pairs, n_expert,
                moe_sort_slots(n_pairs, n_expert), out.slot_of_pair, out.pair_of_slot, out.tiles, out.counts);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

}  // namespace mesh
