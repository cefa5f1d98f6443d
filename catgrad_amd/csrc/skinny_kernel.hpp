// What the kernels for one to eight rows of activations share: weights streamed from memory once.
//
// Such a launch takes a few microseconds: what surrounds the stream of weights is as long as the stream.  So nothing here waits but for
// memory: a workgroup's waves share k, every load is asked for at the start (activations and gains first: an RMS norm's sums are taken
// from them while the weights are on their way, by the launch that applies them), and one barrier is enough for the sums of the products
// and of the squares together.  An empty launch takes 2.6 us, and what is left above the stream is one trip to memory.
//
// Rows share the weights in registers, on the vector units (a 4x4x1 matrix instruction multiplies four rows at once, but then lanes have
// to be 16 bytes of one of four columns each; the sums it saves are not what takes the time).  Against kernels on that instruction, with a
// barrier for the norm's sums that the launch before had left, its power behind all of the weights and arguments of 1 KiB, us a launch in
// the steps of a model.  One row, Qwen3-0.6B shape: q, k and v 1024 -> 4096 6.5 and 5.1, gate and up 1024 -> 3072 7.7 and 6.5, the sums
// 2048 -> 1024 5.2 and 3.7, 3072 -> 1024 6.3 and 4.2, the vocabulary's product 1024 -> 151936 107 and 91 with its norm (6.9 TB/s);
// SmolLM2-135M shape: 576 -> 960 5.0 and 3.9, 576 -> 1536 5.5 and 4.1, the sums 3.7 and 2.9, 4.2 and 3.2.  Four rows, Llama-3.2-1B shape: q, k and v
// 2048 -> 3072 9.3 and 7.4, gate and up 2048 -> 8192 23.7 and 23.0, the sums 2048 -> 2048 5.8 and 5.1, 8192 -> 2048 15.6 and 13.3, the vocabulary's
// product 182 and 159.
#pragma once

#include "device_utils.hpp"
#include "skinny.hpp"

#include <type_traits>

namespace cg {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float divisor_of(const SkinnyInput &in, float squares) { return norm_divisor(squares, in.n_bits, in.eps_bits, in.exp_bits); }

// The sums of N values over a wave into dst[0 .. N)
template <int N, class Of> __device__ __forceinline__ void keep_lane_sums(float *dst, Of of) {
    const uint32_t lane = threadIdx.x & 63;
    if constexpr (N == 1) {
        const float v = wave_add<1>(of(0));
        if (lane == 0) dst[0] = v;
    } else if constexpr (N == 2) {
        const auto h = __builtin_amdgcn_permlane32_swap(asu(of(0)), asu(of(1)), false, false);
        float v = asf(fold_rows(asu(asf((uint32_t)h[0]) + asf((uint32_t)h[1])), AddWords{}));
        v = add_across<1>(add_across<2>(add_across<4>(add_across<8>(v))));
        if (lane % 32 == 0) dst[lane / 32] = v;
    } else {
        static_assert(N % 4 == 0, "four to a register");
#pragma unroll
        for (int i = 0; i < N; i += 4) {
            const float v = add_across<1>(add_across<2>(four_sums(of(i), of(i + 1), of(i + 2), of(i + 3))));
            if (lane % 16 == 0) dst[i + lane / 16] = v;
        }
    }
}

// A workgroup's W waves share k in runs of a W-th each, L trips of 256 values at most (more: further rounds, LOOP).  WHOLE: K is whole rounds.
// M: rows that the kernel holds (a lane has M * L * 4 activations and C * L * 4 weights in registers).
template <int M_, int L_, int W_, bool LOOP_, bool WHOLE_> struct Cut {
    static constexpr int M = M_, L = L_, W = W_;
    static constexpr bool LOOP = LOOP_, WHOLE = WHOLE_;
    static constexpr uint32_t kRound = L_ * W_ * 256;
};

// part[wave][m * C + c] = the wave's share of x[m] . row(c), squares[wave][m] of the norm's sum; `ask` is called in front of the weights' loads.
template <class T, int C, bool NORM, class RowOf, class Ask>
__device__ __forceinline__ void skinny_parts(const SkinnyInput &given, RowOf row, Ask ask, float (&part)[T::W][T::M * C], float (&squares)[T::W][T::M]) {
    constexpr int M = T::M;
    const uint32_t K = T::WHOLE && !T::LOOP ? T::kRound : given.k;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    float s[M][C] = {}, ss[M] = {};
    for (uint32_t k0 = 0; k0 < K; k0 += T::kRound) {
        const uint32_t left = min(K - k0, T::kRound), span = T::WHOLE ? T::L * 256 : (left + 4 * T::W - 1) / (4 * T::W) * 4;
        const uint32_t first = k0 + wave * span;
        uint32_t at[T::L];
        bool in[T::L];
#pragma unroll
        for (int i = 0; i < T::L; i++) {
            const uint32_t k = i * 256 + lane * 4;
            in[i] = T::WHOLE || (k < span && first + k < K);
            at[i] = T::WHOLE ? first + k : min(first + k, K - 4); // (clamped, not tested: no load waits for a test)
        }
        f4 xs[M][T::L], gm[NORM ? T::L : 1], w[C][T::L];
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float *const x = given.x + (M > 1 ? (int64_t)min((uint32_t)m, given.rows - 1) * given.pitch : 0);
#pragma unroll
            for (int i = 0; i < T::L; i++) xs[m][i] = *reinterpret_cast<const f4 *>(x + at[i]);
        }
        if constexpr (NORM) {
#pragma unroll
            for (int i = 0; i < T::L; i++) gm[i] = *reinterpret_cast<const f4 *>(given.gamma + at[i]);
        }
        if (k0 == 0) ask();
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int i = 0; i < T::L; i++) w[c][i] = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(row(c) + at[i]));
        __builtin_amdgcn_sched_barrier(0); // (what follows stays behind all of the loads)
#pragma unroll
        for (int i = 0; i < T::L; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float gain = 1.0f;
                if constexpr (NORM) gain = in[i] ? gm[i][e] : 0.0f;
#pragma unroll
                for (int m = 0; m < M; m++) {
                    float v = in[i] ? xs[m][i][e] : 0.0f;
                    if constexpr (NORM) {
                        ss[m] = fmaf(v, v, ss[m]);
                        v *= gain;
                    }
                    xs[m][i][e] = v;
                }
            }
#pragma unroll
        for (int i = 0; i < T::L; i++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int c = 0; c < C; c++) {
                    const float v = in[i] ? w[c][i][e] : 0.0f;
#pragma unroll
                    for (int m = 0; m < M; m++) s[m][c] = fmaf(xs[m][i][e], v, s[m][c]);
                }
        if constexpr (!T::LOOP) break;
    }
    keep_lane_sums<M * C>(part[wave], [&](int i) { return s[i / C][i % C]; });
    if constexpr (NORM) keep_lane_sums<M>(squares[wave], [&](int m) { return ss[m]; });
    __syncthreads();
}
// the waves' shares of one sum together, always in the same order
template <int W, int N> __device__ __forceinline__ float total(const float (&part)[W][N], uint32_t at) {
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < W; w += 2) s += part[w][at] + part[w + 1][at];
    return s;
}

// f(how the waves share K and the rows they hold, as a type)
template <class F> void with_cut(uint32_t rows, uint32_t K, F f) {
    auto go = [&](auto m, auto l, auto w, auto loop) {
        constexpr int M = decltype(m)::value, L = decltype(l)::value, W = decltype(w)::value;
        constexpr bool LOOP = decltype(loop)::value;
        if (K % (L * W * 256) == 0) f(Cut<M, L, W, LOOP, true>{});
        else f(Cut<M, L, W, LOOP, false>{});
    };
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 2> two{};
    constexpr std::integral_constant<int, 4> four{};
    constexpr std::integral_constant<int, 8> eight{};
    constexpr std::true_type loop{};
    constexpr std::false_type once{};
    auto more = [&](auto m) { // the activations' registers leave room for a trip each (4 x 8192 x 2048, back to back: four trips at once 15.2 us, two 14.4, one 13.5)
        if (K <= 1024) go(m, one, four, once);
        else if (K <= 2048) go(m, one, eight, once);
        else go(m, one, eight, loop);
    };
    if (rows > 4) more(eight);
    else if (rows > 2) more(four);
    else if (rows > 1) more(two);
    else if (K <= 1024) go(one, one, four, once); // one row: as much of K at once as there is
    else if (K <= 2048) go(one, two, four, once);
    else if (K <= 3072) go(one, std::integral_constant<int, 3>{}, four, once);
    else if (K <= 4096) go(one, four, four, once);
    else if (K <= 6144) go(one, std::integral_constant<int, 3>{}, eight, once); // (a fourth trip of idle lanes: the gated pair 1 x 4100 x 2052 18.8 us, 15.5 without, 1 x 5120 x 4608 35.9 and 30.4)
    else go(one, four, eight, loop);
}

inline int skinny_launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, what);
}

} // namespace
} // namespace cg
