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
#pragma unroll 8
            for (uint32_t j = first; j < first + size; j++) rank += beats(choice[j], j, mine, e);
            if (rank < 2) worth[2 * g + rank] = mine;
        }
        __syncthreads();
        for (uint32_t g = t; g < p.groups; g += N) {
            const float mine = worth[2 * g] + worth[2 * g + 1];
            uint32_t rank = 0;
#pragma unroll 4
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
#pragma unroll 16
        for (uint32_t j = 0; j < p.experts; j++) rank += beats(choice[j], j, mine, e);
        if (rank < p.top) {
            chosen[rank] = e;
            weight[rank] = own[e];
        }
    }
    __syncthreads();
}

// A workgroup of kExpertThreads: four waves' columns (block x, per_wave each, one after the other) of row * top + choice (block y).
// In front of the first weight lie the choice and its loads, 4 us: so the columns are cut for one round of workgroups, and a wave's next
// column is on its way while this one is multiplied.  The launch beside attention, 8 of 32 experts in bf16: 1024 columns of 2048 values
// 23.4 -> 20.5 us (67 MB, 13 us at the device's rate), 384 of 1024 12.4 -> 11.8.
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
    const uint32_t e = __builtin_amdgcn_readfirstlane(chosen[slot]);
    const float weigh = weight[slot];
    if (bx == 0 && threadIdx.x == 0) chosen_out[by] = e;
    const uint32_t f0 = (bx * kExpertWaves + __builtin_amdgcn_readfirstlane(wave)) * per_wave, f1 = min(f0 + per_wave, p.ff);
    if (f0 >= f1) return;
    constexpr uint32_t EB = BF16 ? 2 : 4;
    auto column = [&](uint32_t f) { return static_cast<const char *>(p.gate_up) + ((uint64_t)e * 2 * p.ff + f) * p.width * EB; };
    const uint64_t up = (uint64_t)p.ff * p.width * EB;
    auto put = [&](uint32_t f, float a, float b) {
        a = wave_total(a);
        b = wave_total(b);
        if (lane == 0) hidden[(uint64_t)by * p.ff + f] = weigh * activation(a, b, p.limit, p.slope);
    };
    if (p.width > STEPS * SPAN) {
        for (uint32_t f = f0; f < f1; f++) {
            const char *g = column(f);
            float a = 0.0f, b = 0.0f;
            for (uint32_t k = lane * W; k < p.width; k += SPAN) {
                St wg, wu;
                wg.load(g, k);
                wu.load(g + up, k);
                float v[W];
                take(k, v);
                a = wg.dot(v, a);
                b = wu.dot(v, b);
            }
            put(f, a, b);
        }
        return;
    }
    // the next column, or the second half of eight steps, is asked for before this one is multiplied
    constexpr int PART = STEPS < 4 ? STEPS : 4;
    struct Piece {
        St g[PART], u[PART];
    };
    auto ask = [&](uint32_t f, int first, Piece &c) {
        const char *g = column(f);
#pragma unroll
        for (int s = 0; s < PART; s++) { // (clamped: behind the last column x is zero)
            const uint32_t k = min((first + s) * SPAN + lane * W, p.width - W);
            c.g[s].load(g, k);
            c.u[s].load(g + up, k);
        }
    };
    auto use = [&](const int first, const Piece &c, float &a, float &b) {
#pragma unroll
        for (int s = 0; s < PART; s++) {
            a = c.g[s].dot(x[first + s], a);
            b = c.u[s].dot(x[first + s], b);
        }
    };
    Piece c0, c1;
    ask(f0, 0, c0);
    if constexpr (STEPS > PART) {
        for (uint32_t f = f0; f < f1; f++) {
            float a = 0.0f, b = 0.0f;
            ask(f, PART, c1);
            use(0, c0, a, b);
            if (f + 1 < f1) ask(f + 1, 0, c0);
            use(PART, c1, a, b);
            put(f, a, b);
        }
    } else {
        for (uint32_t f = f0; f < f1; f += 2) {
            float a = 0.0f, b = 0.0f, c = 0.0f, d = 0.0f;
            if (f + 1 < f1) ask(f + 1, 0, c1);
            use(0, c0, a, b);
            put(f, a, b);
            if (f + 1 >= f1) break;
            if (f + 2 < f1) ask(f + 2, 0, c0);
            use(0, c1, c, d);
            put(f + 1, c, d);
        }
    }
}

} // namespace cg
