// The choice of a token's experts, and the first products of the chosen ones for a few rows: shared by the kernels of the experts
// (block_experts.hip) and the launch that has attention beside them (block_attention_mixed.hip).
#pragma once

#include "block_stream.hpp"

namespace cg {

__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float activation(float g, float u, float limit, float slope) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g * (u + 1.0f) / (1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * slope * g));
}

// ---- the choice ------------------------------------------------------------------------------------------------------
// Every score is ranked against those it competes with: first a group's members, then the groups, then the members of the
// groups that count.  LDS: route_floats(experts, groups) floats.  Thread t of N; `chosen` and `weight` (LDS) are there after
// the last barrier, which is the whole workgroup's.
__host__ __device__ constexpr uint32_t route_floats(uint32_t experts, uint32_t groups) { return 2 * experts + 3 * groups; }
__device__ __forceinline__ bool beats(float a, uint32_t i, float b, uint32_t j) { return a > b || (a == b && i < j); }

template <int N>
__device__ void choose_experts(const ExpertsPlan &p, uint32_t row, float *lds, uint32_t *chosen, float *weight, const uint32_t t) {
    float *choice = lds, *own = lds + p.experts, *worth = own + p.experts; // worth: [groups][2], then [groups] whether it counts
    float *counts = worth + 2 * p.groups;
    const uint32_t size = p.experts / p.groups;
    for (uint32_t e = t; e < p.experts; e += N) {
        const float s = sigmoid(p.logits[(int64_t)row * p.experts + e]);
        own[e] = s;
        choice[e] = p.correction ? s + p.correction[e] : s;
    }
    for (uint32_t g = t; g < p.groups; g += N) worth[2 * g] = worth[2 * g + 1] = 0.0f; // (a group of one member)
    for (uint32_t i = t; i < p.top; i += N) { // (scores that are not numbers leave places untaken)
        chosen[i] = 0;
        weight[i] = 0.0f;
    }
    __syncthreads();
    if (p.keep < p.groups) {
        for (uint32_t e = t; e < p.experts; e += N) {
            const uint32_t g = e / size, first = g * size;
            const float mine = choice[e];
            uint32_t rank = 0;
            for (uint32_t j = first; j < first + size; j++) rank += beats(choice[j], j, mine, e);
            if (rank < 2) worth[2 * g + rank] = mine;
        }
        __syncthreads();
        for (uint32_t g = t; g < p.groups; g += N) {
            const float mine = worth[2 * g] + worth[2 * g + 1];
            uint32_t rank = 0;
            for (uint32_t j = 0; j < p.groups; j++) rank += beats(worth[2 * j] + worth[2 * j + 1], j, mine, g);
            counts[g] = rank < p.keep ? 1.0f : 0.0f;
        }
        __syncthreads();
        for (uint32_t e = t; e < p.experts; e += N)
            if (counts[e / size] == 0.0f) choice[e] = -INFINITY;
        __syncthreads();
    }
    for (uint32_t e = t; e < p.experts; e += N) {
        const float mine = choice[e];
        uint32_t rank = 0;
#pragma unroll 4
        for (uint32_t j = 0; j < p.experts; j++) rank += beats(choice[j], j, mine, e);
        if (rank < p.top) {
            chosen[rank] = e;
            weight[rank] = own[e];
        }
    }
    __syncthreads();
}

// A workgroup of kExpertThreads: four waves' columns (block x, per_wave each, one after the other) of row * top + choice (block y).
// LDS: route_bytes(p).
constexpr int kExpertThreads = 256, kExpertWaves = 4;
inline size_t route_bytes(const ExpertsPlan &p) { return (route_floats(p.experts, p.groups) + 2 * (size_t)p.top) * 4; }
template <bool BF16, bool VEC, int STEPS>
__device__ __forceinline__ void expert_first(const ExpertsPlan &p, const uint32_t per_wave, float *__restrict__ hidden, uint32_t *__restrict__ chosen_out, const uint32_t bx,
                                             const uint32_t by, float *const lds) {
    typedef Streamed<BF16, VEC> St;
    constexpr uint32_t W = St::W, SPAN = 64 * W;
    const uint32_t row = by / p.top, slot = by - row * p.top, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t *chosen = reinterpret_cast<uint32_t *>(lds + route_floats(p.experts, p.groups));
    float *weight = reinterpret_cast<float *>(chosen + p.top);
    // the row of h, this lane's values of it in registers where they fit
    float x[STEPS][W];
    auto take = [&](uint32_t k, float(&o)[W]) { // (clamped; zeros behind the last column)
        const int64_t at = (int64_t)row * p.width + min(k, p.width - W);
        if (p.h_fmt == kFmtBF16) {
#pragma unroll
            for (uint32_t i = 0; i < W; i++) o[i] = asf((uint32_t) static_cast<const uint16_t *>(p.h)[at + i] << 16);
        } else {
            St::input(static_cast<const float *>(p.h), at, o);
        }
#pragma unroll
        for (uint32_t i = 0; i < W; i++) o[i] = k < p.width ? o[i] : 0.0f;
    };
#pragma unroll
    for (int s = 0; s < STEPS; s++) take(s * SPAN + lane * W, x[s]);
    choose_experts<kExpertThreads>(p, row, lds, chosen, weight, threadIdx.x);
    const uint32_t e = chosen[slot];
    const float weigh = weight[slot];
    if (bx == 0 && threadIdx.x == 0) chosen_out[by] = e;
    const uint32_t f0 = (bx * kExpertWaves + wave) * per_wave;
    constexpr uint32_t EB = BF16 ? 2 : 4;
    for (uint32_t f = f0; f < min(f0 + per_wave, p.ff); f++) {
        const char *g = static_cast<const char *>(p.gate_up) + ((uint64_t)e * 2 * p.ff + f) * p.width * EB, *u = g + (uint64_t)p.ff * p.width * EB;
        float a = 0.0f, b = 0.0f;
        if (p.width <= STEPS * SPAN) {
            St wg[STEPS], wu[STEPS];
#pragma unroll
            for (int s = 0; s < STEPS; s++) { // (clamped: behind the last column x is zero)
                const uint32_t k = min(s * SPAN + lane * W, p.width - W);
                wg[s].load(g, k);
                wu[s].load(u, k);
            }
#pragma unroll
            for (int s = 0; s < STEPS; s++) {
                a = wg[s].dot(x[s], a);
                b = wu[s].dot(x[s], b);
            }
        } else {
            for (uint32_t k = lane * W; k < p.width; k += SPAN) {
                St wg, wu;
                wg.load(g, k);
                wu.load(u, k);
                float v[W];
                take(k, v);
                a = wg.dot(v, a);
                b = wu.dot(v, b);
            }
        }
        a = wave_total(a);
        b = wave_total(b);
        if (lane == 0) hidden[(uint64_t)by * p.ff + f] = weigh * activation(a, b, p.limit, p.slope);
    }
}

} // namespace cg
