// Gated recurrence over many tokens: a linear recurrence S = a S + b per channel, cut into windows of tokens and these into
// runs, one for each wave of a workgroup of 64 channels.
//
// The first launch composes each window's steps into (A, B), S_out = A S_in + B, or, when a sequence starts inside the window,
// into the state its last sequence leaves (a restart: S_out = B).  The second composes the windows before its own, a quarter a wave, and the
// runs before its own, and walks its run from there.  A call of one window (decode batches) needs the second launch only.
//
// Bound by memory.  A thread requests all its projections (16 in the first launch, 24 in the second) before it uses one: a loop
// that stores outputs between its loads has one token's in flight, a trip to memory a token.  900 tokens x 2048 channels
// (22 MB of projections): 14.8 -> 5.4 us and 24.8 -> 9.1.
//
// A sequence's starting state is read in the first launch where the sequence goes on into later windows: those may write
// its final state while this window still runs.  Within a window all starting states are read before the barrier, all final
// ones written behind it.
#include "act_math.hpp"
#include "rowops.hpp"

namespace mesh {

constexpr int GRU_RUN = 8, GRU_WAVES = 4, GRU_WINDOW = GRU_RUN * GRU_WAVES, GRU_THREADS = 64 * GRU_WAVES;

// A step or a row of them: S -> A S + B, or, where a sequence starts in the row, S -> B whatever S holds (another sequence's
// infinity, say): A is GRU_RESTART then, which no product of keeps is.  (A product that has underflowed to 0 is no restart: a NaN or
// an infinity of the sequence's own state stays in it, as it does token by token.)
constexpr float GRU_RESTART = -1.f;
struct GruStep { float A, B; };
__device__ __forceinline__ float gru_apply(const GruStep &s, float S) { return s.A == GRU_RESTART ? s.B : fmaf(s.A, S, s.B); }
__device__ __forceinline__ GruStep gru_then(const GruStep &first, const GruStep &s) {
    return {first.A == GRU_RESTART || s.A == GRU_RESTART ? GRU_RESTART : first.A * s.A, gru_apply(s, first.B)};
}

// The steps of tokens t0 .. t0 + GRU_RUN - 1 of channel c (identities from T on) and where sequences start among them.
struct GruRun {
    GruStep step[GRU_RUN];
    float init[GRU_RUN];            // the state a sequence that starts at this token starts from
    unsigned starts, ends;          // bit i: token t0 + i is its sequence's first / last one of the call
    __device__ __forceinline__ GruStep compose() const {
        GruStep r{1.f, 0.f};
#pragma unroll
        for (int i = 0; i < GRU_RUN; ++i) {
            if (starts >> i & 1) r = {GRU_RESTART, init[i]};
            r = gru_then(r, step[i]);
        }
        return r;
    }
};
// held: the starting state of the sequence that goes on past the window, from the launch before (null: it is read from the states)
__device__ __forceinline__ void gru_run(GruRun &run, const MinGruArgs &a, int T, int t0, int t_end, int c, const float *held) {
    const int W = a.width;
    float pz[GRU_RUN], px[GRU_RUN];
    int seq[GRU_RUN + 2];
#pragma unroll
    for (int i = 0; i < GRU_RUN; ++i) {
        const float *p = a.zxg + (size_t)(t0 + i < T ? t0 + i : T - 1) * 3 * W + c;
        pz[i] = p[0]; px[i] = p[W];
    }
#pragma unroll
    for (int i = 0; i < GRU_RUN + 2; ++i) {
        const int t = t0 - 1 + i;
        seq[i] = a.seq[t < 0 ? 0 : t < T ? t : T - 1];
    }
    const float bz = a.bias_z[c], bx = a.bias_x[c];
    run.starts = run.ends = 0;
#pragma unroll
    for (int i = 0; i < GRU_RUN; ++i) {
        const int t = t0 + i;
        run.init[i] = 0.f;
        if (t >= T) continue;
        if (t + 1 == T || seq[i + 2] != seq[i + 1]) run.ends |= 1u << i;
        if (t != 0 && seq[i] == seq[i + 1]) continue;
        run.starts |= 1u << i;
        if (a.pos[t] == 0) continue;
        bool last = held != nullptr;
        for (int u = t + 1; last && u < t_end; ++u) last = a.seq[u] == seq[i + 1];
        float v = last ? *held : a.state[(size_t)seq[i + 1] * W + c];
        asm volatile("" : "+v"(v));         // (waited for here, and not for all loads at the join of the rare branch)
        run.init[i] = v;
    }
#pragma unroll
    for (int i = 0; i < GRU_RUN; ++i) {
        const MinGruGate g = min_gru_gate(pz[i] + bz, px[i] + bx);
        run.step[i] = t0 + i < T ? GruStep{g.keep, g.in} : GruStep{1.f, 0.f};
    }
}

__global__ __launch_bounds__(GRU_THREADS) void min_gru_compose_kernel(const MinGruArgs a, int T) {
    __shared__ GruStep part[GRU_WAVES][64];
    __shared__ float s_init[GRU_WAVES][64];
    __shared__ unsigned s_starts[GRU_WAVES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = blockIdx.y, W = a.width;
    const int ch = blockIdx.x * 64 + lane, c = ch < W ? ch : W - 1;
    const int t1 = (w + 1) * GRU_WINDOW < T ? (w + 1) * GRU_WINDOW : T;
    GruRun run;
    gru_run(run, a, T, w * GRU_WINDOW + wave * GRU_RUN, t1, c, nullptr);
    float init = 0.f;
#pragma unroll
    for (int i = 0; i < GRU_RUN; ++i) init = run.starts >> i & 1 ? run.init[i] : init;
    part[wave][lane] = run.compose();
    s_init[wave][lane] = init;
    if (lane == 0) s_starts[wave] = run.starts;
    __syncthreads();
    if (wave || ch >= W) return;
    GruStep all{1.f, 0.f};
#pragma unroll
    for (int i = 0; i < GRU_WAVES; ++i) {
        all = gru_then(all, part[i][lane]);
        if (s_starts[i]) init = s_init[i][lane];
    }
    float *ws = a.ws + (size_t)w * 3 * W + ch;
    ws[0] = all.A; ws[W] = all.B; ws[2 * W] = init;
}

template <ActType ACT>
__global__ __launch_bounds__(GRU_THREADS) void min_gru_kernel(const MinGruArgs a, int T) {
    __shared__ GruStep before[GRU_WAVES][64], part[GRU_WAVES][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = blockIdx.y, W = a.width;
    const int ch = blockIdx.x * 64 + lane, c = ch < W ? ch : W - 1;
    const int t1 = (w + 1) * GRU_WINDOW < T ? (w + 1) * GRU_WINDOW : T, t0 = w * GRU_WINDOW + wave * GRU_RUN;
    float gate[GRU_RUN];
#pragma unroll
    for (int i = 0; i < GRU_RUN; ++i) gate[i] = a.zxg[((size_t)(t0 + i < T ? t0 + i : T - 1) * 3 + 2) * W + c];
    GruRun run;
    gru_run(run, a, T, t0, t1, c, gridDim.y > 1 ? a.ws + ((size_t)w * 3 + 2) * W + c : nullptr);
    // the windows before, a quarter a wave
    GruStep pre{1.f, 0.f};
    const int v1 = w * (wave + 1) / GRU_WAVES;
#pragma unroll 8
    for (int v = w * wave / GRU_WAVES; v < v1; ++v) pre = gru_then(pre, GruStep{a.ws[(size_t)v * 3 * W + c], a.ws[((size_t)v * 3 + 1) * W + c]});
    before[wave][lane] = pre;
    part[wave][lane] = run.compose();
    __syncthreads();
    float S = 0.f;
#pragma unroll
    for (int i = 0; i < GRU_WAVES; ++i) S = gru_apply(before[i][lane], S);
    for (int i = 0; i < wave; ++i) S = gru_apply(part[i][lane], S);
    if (ch >= a.ld) return;
#pragma unroll
    for (int i = 0; i < GRU_RUN; ++i) {
        if (t0 + i >= T) break;
        if (run.starts >> i & 1) S = run.init[i];
        S = gru_apply(run.step[i], S);
        const float v = ch < W ? S * act_silu(gate[i]) : 0.f;
        const size_t at = (size_t)(t0 + i) * a.ld + ch;
        if constexpr (ACT == ACT_BF16) static_cast<uint16_t *>(a.out)[at] = f32_to_bf16_bits(v);
        else static_cast<float *>(a.out)[at] = v;
        if ((run.ends >> i & 1) && ch < W) a.state[(size_t)a.seq[t0 + i] * W + ch] = S;
    }
}

size_t min_gru_workspace(int T, int width) { return (size_t)((T + GRU_WINDOW - 1) / GRU_WINDOW) * 3 * width; }

int min_gru(const MinGruArgs &a, int T, hipStream_t stream) {
    if (T <= 0) return MESH_OK;
    const int windows = (T + GRU_WINDOW - 1) / GRU_WINDOW;
    if (!a.zxg || !a.state || !a.out || a.ld < a.width || a.width < 1 || windows > 65535 || (windows > 1 && !a.ws)) return fail(MESH_ERR_INVALID, "min_gru: bad operands");
    const dim3 block(GRU_THREADS);
    if (windows > 1) {
        MESH_LAUNCH(min_gru_compose_kernel, dim3((unsigned)((a.width + 63) / 64), (unsigned)windows), block, 0, stream, a, T);
        MESH_LAUNCH_CHECK();
    }
    const dim3 grid((unsigned)((a.ld + 63) / 64), (unsigned)windows);
    if (a.act == ACT_BF16) MESH_LAUNCH((min_gru_kernel<ACT_BF16>), grid, block, 0, stream, a, T);
    else MESH_LAUNCH((min_gru_kernel<ACT_F32>), grid, block, 0, stream, a, T);
    MESH_LAUNCH_CHECK();
    return MESH_OK;
}

}  // namespace mesh
