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

// The choice by a wave alone, a lane to an expert: scores are ranked in registers, and nothing waits for LDS or a barrier.  At most 64 experts, their
// groups (where groups are dropped) of a power of two members.  (Every wave of a workgroup chooses for itself, so a comparison is three instructions:
// ties are resolved behind the ranks.)
__host__ __device__ inline bool wave_chooses(const ExpertsPlan &p) {
    const uint32_t size = p.experts / p.groups;
    return p.experts <= 64 && (p.keep >= p.groups || (size & (size - 1)) == 0);
}
struct WaveChoice {
    float logit, correction, own; // own: the lane's expert's score
    uint32_t rank;                // how many choices are better (none: the lane has no expert)
    __device__ __forceinline__ void ask(const ExpertsPlan &p, uint32_t row) { // (clamped, not tested: no load waits)
        const uint32_t e = min(threadIdx.x & 63, p.experts - 1);
        logit = p.logits[(int64_t)row * p.experts + e];
        correction = p.correction ? p.correction[e] : 0.0f;
    }
    template <int DIST> static __device__ __forceinline__ void best_two(float &first, float &second) {
        const float f = asf(across<DIST>(asu(first))), s = asf(across<DIST>(asu(second)));
        second = fmaxf(fminf(first, f), fmaxf(second, s));
        first = fmaxf(first, f);
    }
    static __device__ __forceinline__ float lane_of(float v, uint32_t lane) { return asf(__builtin_amdgcn_readlane(asu(v), lane)); }
    __device__ __forceinline__ void choose(const ExpertsPlan &p) {
        const uint32_t e = threadIdx.x & 63;
        own = sigmoid(logit);
        float choice = p.correction ? own + correction : own;
        if (p.keep < p.groups) {
            const uint32_t shift = __builtin_ctz(p.experts / p.groups), size = 1u << shift, g = e >> shift;
            float first = choice, second = size > 1 ? -INFINITY : 0.0f;
            if (size > 1) best_two<1>(first, second);
            if (size > 2) best_two<2>(first, second);
            if (size > 4) best_two<4>(first, second);
            if (size > 8) best_two<8>(first, second);
            if (size > 16) best_two<16>(first, second);
            if (size > 32) best_two<32>(first, second);
            const float worth = first + second;
            uint32_t before = 0;
            for (uint32_t j = 0; j < p.groups; j++) before += beats(lane_of(worth, j << shift), j, worth, g);
            if (before >= p.keep) choice = -INFINITY;
        }
        rank = 0;
#pragma unroll 8
        for (uint32_t j = 0; j < p.experts; j++) rank += lane_of(choice, j) > choice;
        if (e >= p.experts) rank = 64;
    }
    // the expert in a place and its weight (0 and 0 where scores that are not numbers leave the place untaken)
    __device__ __forceinline__ uint32_t in_place(uint32_t slot, float *weight) const {
        uint64_t there = 0;
        uint32_t r = slot; // equal choices share the first of their places and take them in the order of the experts
        while (!(there = __ballot(rank == r)) && r) r--;
        for (; r < slot; r++) there &= there - 1;
        const uint32_t e = there ? (uint32_t)__builtin_ctzll(there) : 0;
        *weight = there ? lane_of(own, e) : 0.0f;
        return e;
    }
};

// A workgroup of kExpertThreads: four waves' columns (block x, per_wave each, one after the other) of row * top + choice (block y).
// In front of the first weight lie the choice and its loads (3.0 us with barriers, 1.6 by waves, a third of it the way of the logits): so the columns are cut for one round of
// workgroups, and a wave's next column is on its way while this one is multiplied.  The launch beside attention, 8 of 32 experts in bf16: 1024 columns of 2048 values
// 23.4 -> 20.5 us (67 MB, 13 us at the device's rate), 384 of 1024 12.4 -> 11.8 (now, with mixed_step's loads all ahead, 9.4, and 7.7 to 8.1 with the choice by waves).
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
    const bool by_wave = wave_chooses(p);
    WaveChoice choice;
    if (by_wave) choice.ask(p, row);
    // the row of h, this lane's values of it in registers where they fit: words or pairs of bfloat16 patterns until the choice is made
    float x[STEPS][W];
    const bool narrow = p.h_fmt == kFmtBF16;
    typedef uint32_t __attribute__((aligned(2))) pair;
    auto ask_h = [&](uint32_t k, float(&o)[W]) { // (clamped)
        const int64_t at = (int64_t)row * p.width + min(k, p.width - W);
        if (narrow) {
            const uint16_t *const src = static_cast<const uint16_t *>(p.h) + at;
            if constexpr (W == 1) {
                o[0] = asf(src[0]);
            } else {
#pragma unroll
                for (uint32_t i = 0; i < W / 2; i++) o[i] = asf(reinterpret_cast<const pair *>(src)[i]);
            }
        } else {
            St::input(static_cast<const float *>(p.h), at, o);
        }
    };
    auto settle_h = [&](uint32_t k, float(&o)[W]) { // (zeros behind the last column)
        if (narrow) {
#pragma unroll
            for (int i = (int)W - 1; i >= 0; i--) o[i] = asf(W > 1 && i % 2 ? asu(o[i / 2]) & 0xFFFF0000u : asu(o[i / 2]) << 16);
        }
#pragma unroll
        for (uint32_t i = 0; i < W; i++) o[i] = k < p.width ? o[i] : 0.0f;
    };
#pragma unroll
    for (int s = 0; s < STEPS; s++) ask_h(s * SPAN + lane * W, x[s]);
    uint32_t e;
    float weigh;
    if (by_wave) {
        choice.choose(p);
        e = choice.in_place(slot, &weigh);
    } else {
        choose_experts<kExpertThreads>(p, row, lds, chosen, weight, threadIdx.x);
        e = __builtin_amdgcn_readfirstlane(chosen[slot]);
        weigh = weight[slot];
    }
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
                ask_h(k, v);
                settle_h(k, v);
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
#pragma unroll
    for (int s = 0; s < STEPS; s++) settle_h(s * SPAN + lane * W, x[s]);
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
