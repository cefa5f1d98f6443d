// The linear layers of a decode step of one sequence: one row of activations, weights streamed from memory once.
//
// Such a launch takes a few microseconds: what surrounds the stream of weights is as long as the stream.  So nothing here waits but for
// memory: a workgroup's waves share k, every load is asked for at the start (activations and gains first: the RMS norm's sums are taken
// from them while the weights are on their way, by the launch that applies them), and one barrier is enough for the sums of the products
// and of the squares together.  Against the kernels of two to eight rows (matmul.hip: a barrier for the norm's sums that the launch before
// left, its power behind all of the weights, arguments of 1 KiB), us a launch in the steps of the Qwen3-0.6B shape: q, k and v 1024 -> 4096
// 6.5 and 5.1, gate and up 1024 -> 3072 7.7 and 6.5, the sums 2048 -> 1024 5.2 and 3.8, 3072 -> 1024 6.3 and 4.2, the vocabulary's
// product 1024 -> 151936 107 and 91 with its norm (6.9 TB/s); SmolLM2-135M shape: 576 -> 960 5.0 and 3.9, 576 -> 1536 5.5 and 4.1, the sums
// 3.7 and 2.9, 4.2 and 3.2.  An empty launch takes 2.6, and what is left above the stream is one trip to memory.
#include "one_row.hpp"
#include "device_utils.hpp"

#include <type_traits>

namespace cg {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

// pow(sum / n + eps, e) in the norm's own ops; a square root where e is one half, as in every model's norms (the power takes 0.7 us of a
// launch of 5; where they are not the same, at and below zero, it stays)
__device__ __forceinline__ float divisor_of(const OneRowInput &in, float squares) {
    const uint32_t mean = apply<kAdd, true>(apply<kDiv, true>(asu(squares), in.n_bits, 0, nullptr), in.eps_bits, 0, nullptr);
    if (in.exp_bits == 0x3F000000u && asf(mean) > 0.0f) return sqrtf(asf(mean));
    return asf(apply<kPow, true>(mean, in.exp_bits, 0, nullptr));
}

// The sums of C values over a wave: of s[r] in lane r * 64 / C
template <int C> __device__ __forceinline__ float lane_sums(const float (&s)[C]) {
    static_assert(C == 2 || C == 4, "two or four");
    if constexpr (C == 4) {
        return add_across<1>(add_across<2>(four_sums(s[0], s[1], s[2], s[3])));
    } else {
        const auto h = __builtin_amdgcn_permlane32_swap(asu(s[0]), asu(s[1]), false, false);
        float v = asf(fold_rows(asu(asf((uint32_t)h[0]) + asf((uint32_t)h[1])), AddWords{}));
        v = add_across<4>(add_across<8>(v));
        return add_across<1>(add_across<2>(v));
    }
}

// A workgroup's W waves share k in runs of a W-th each, L trips of 256 values at most (more: further rounds, LOOP).  WHOLE: K is whole trips.
template <int L_, int W_, bool LOOP_, bool WHOLE_> struct Cut {
    static constexpr int L = L_, W = W_;
    static constexpr bool LOOP = LOOP_, WHOLE = WHOLE_;
    static constexpr uint32_t kChunk = L_ * W_ * 256;
};

// part[wave][c] = the wave's share of x . row(c), squares[wave] of the norm's sum; `ask` is called in front of the weights' loads.
template <class T, int C, bool NORM, class RowOf, class Ask>
__device__ __forceinline__ void one_row_parts(const float *__restrict__ x, const float *__restrict__ gamma, const uint32_t k_given, RowOf row, Ask ask,
                                              float (&part)[T::W][C], float (&squares)[T::W]) {
    const uint32_t K = T::WHOLE && !T::LOOP ? T::kChunk : k_given;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    float s[C] = {}, ss = 0.0f;
    for (uint32_t k0 = 0; k0 < K; k0 += T::kChunk) {
        const uint32_t left = min(K - k0, T::kChunk), span = T::WHOLE ? T::L * 256 : (left + 4 * T::W - 1) / (4 * T::W) * 4;
        const uint32_t first = k0 + wave * span;
        uint32_t at[T::L];
        bool in[T::L];
#pragma unroll
        for (int i = 0; i < T::L; i++) {
            const uint32_t k = i * 256 + lane * 4;
            in[i] = T::WHOLE || (k < span && first + k < K);
            at[i] = T::WHOLE ? first + k : min(first + k, K - 4); // (clamped, not tested: no load waits for a test)
        }
        f4 xs[T::L], gm[NORM ? T::L : 1], w[C][T::L];
#pragma unroll
        for (int i = 0; i < T::L; i++) xs[i] = *reinterpret_cast<const f4 *>(x + at[i]);
        if constexpr (NORM) {
#pragma unroll
            for (int i = 0; i < T::L; i++) gm[i] = *reinterpret_cast<const f4 *>(gamma + at[i]);
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
                float v = in[i] ? xs[i][e] : 0.0f;
                if constexpr (NORM) {
                    ss = fmaf(v, v, ss);
                    v *= in[i] ? gm[i][e] : 0.0f;
                }
                xs[i][e] = v;
            }
#pragma unroll
        for (int i = 0; i < T::L; i++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int c = 0; c < C; c++) s[c] = fmaf(xs[i][e], in[i] ? w[c][i][e] : 0.0f, s[c]);
        if constexpr (!T::LOOP) break;
    }
    const float sums = lane_sums<C>(s);
    if (lane % (64 / C) == 0) part[wave][lane / (64 / C)] = sums;
    if constexpr (NORM) {
        ss = wave_add<1>(ss);
        if (lane == 0) squares[wave] = ss;
    }
    __syncthreads();
}
// the waves' shares of value c together, always in the same order
template <int W, int C> __device__ __forceinline__ float total(const float (&part)[W][C], uint32_t c) {
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < W; w += 2) s += part[w][c] + part[w + 1][c];
    return s;
}
template <int W> __device__ __forceinline__ float total(const float (&squares)[W]) {
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < W; w += 2) s += squares[w] + squares[w + 1];
    return s;
}

// Four columns a workgroup (4096 x 1024 with a norm, back to back: two 5.8, four 5.5, eight 5.6, sixteen 6.2; a wave per column or two without
// any barrier 5.8): two and the two half a head away, which the rotary embedding mixes them with, or four in a row.
template <class T, bool NORM> __global__ __launch_bounds__(T::W * 64) void one_row_group_kernel(const OneRowGroup g) {
    __shared__ float part[T::W][4], squares[T::W];
    uint32_t at = 0;
#pragma unroll
    for (int i = 1; i < kMaxOneRow; i++) at += (uint32_t)i < g.count && blockIdx.x >= g.p[i].first ? 1u : 0u;
    const OneRowProduct p = g.p[at];
    const uint32_t span = p.rope ? p.hd : 4, per = span / 4, block = blockIdx.x - p.first;
    const uint32_t n0 = block / per * span + block % per * 2, apart = span / 2;
    auto column = [&](uint32_t c) { return n0 + (c >> 1) * apart + (c & 1); };
    const uint32_t t = threadIdx.x & 3, col = column(t), d = col % p.hd;
    uint32_t cs = 0, sn = 0;
    one_row_parts<T, 4, NORM>(
        g.in.x, g.in.gamma, g.in.k, [&](int c) { return p.w + (int64_t)min(column(c), p.n - 1) * p.pitch; },
        [&] {
            if (p.rope && threadIdx.x < 4) {
                cs = p.cos[d];
                sn = p.sin[d];
            }
        },
        part, squares);
    if (threadIdx.x >= 4) return;
    float s = total(part, t);
    if constexpr (NORM) s = asf(apply<kDiv, true>(asu(s), asu(divisor_of(g.in, total(squares))), 0, nullptr));
    uint32_t v = asu(s);
    const uint32_t other = across<2>(v); // the column half a head away
    if (p.rope) { // lower half: rotate_half reads -x[d + hd / 2]; upper half: x[d - hd / 2]
        const uint32_t rot = t < 2 ? apply<kNeg, true>(other, 0, 0, nullptr) : other;
        v = apply<kAdd, true>(apply<kMul, true>(cs, v, 0, nullptr), apply<kMul, true>(sn, rot, 0, nullptr), 0, nullptr);
    }
    if (col < p.n) p.dst[(int64_t)(col / p.hd) * p.sh + d] = v;
}

// Two columns of either matrix a workgroup
template <class T, bool NORM> __global__ __launch_bounds__(T::W * 64) void one_row_gated_kernel(const OneRowGated g) {
    __shared__ float part[T::W][4], squares[T::W];
    const uint32_t n0 = blockIdx.x * 2;
    one_row_parts<T, 4, NORM>(
        g.in.x, g.in.gamma, g.in.k, [&](int c) { return (c < 2 ? g.wg : g.wu) + (int64_t)min(n0 + (c & 1), g.n - 1) * g.pitch; }, [] {}, part, squares);
    const uint32_t t = threadIdx.x;
    if (t >= 2 || n0 + t >= g.n) return;
    uint32_t gv = asu(total(part, t)), uv = asu(total(part, t + 2));
    if constexpr (NORM) {
        const uint32_t d = asu(divisor_of(g.in, total(squares)));
        gv = apply<kDiv, true>(gv, d, 0, nullptr);
        uv = apply<kDiv, true>(uv, d, 0, nullptr);
    }
    // the ops of the deferred program, in its order
    const uint32_t e = apply<kExp, true>(apply<kNeg, true>(gv, 0, 0, nullptr), 0, 0, nullptr);
    const uint32_t sg = apply<kDiv, true>(g.one, apply<kAdd, true>(g.one, e, 0, nullptr), 0, nullptr);
    g.dst[n0 + t] = apply<kMul, true>(apply<kMul, true>(gv, sg, 0, nullptr), uv, 0, nullptr);
}

// C columns a workgroup
template <class T, int C> __global__ __launch_bounds__(T::W * 64) void one_row_residual_kernel(const OneRowResidual r) {
    __shared__ float part[T::W][C], squares[T::W];
    const uint32_t n0 = blockIdx.x * C, t = threadIdx.x, col = min(n0 + t % C, r.n - 1);
    uint32_t term[4] = {};
    one_row_parts<T, C, false>(
        r.x, nullptr, r.k, [&](int c) { return r.w + (int64_t)min(n0 + c, r.n - 1) * r.pitch; },
        [&] { // the sum's other terms for the value this thread will store
            if (t < C) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if ((uint32_t)i != r.slot && (uint32_t)i < r.nterms) term[i] = r.term[i][col];
            }
        },
        part, squares);
    if (t >= C || n0 + t >= r.n) return;
    const uint32_t v = asu(total(part, t));
#pragma unroll
    for (int i = 0; i < 4; i++) term[i] = (uint32_t)i == r.slot ? v : term[i];
    uint32_t o;
    if (r.nterms == 2) {
        o = apply<kAdd, true>(term[0], term[1], 0, nullptr);
    } else {
        const uint32_t inner = apply<kAdd, true>(term[1], term[2], 0, nullptr);
        o = r.order == 0 ? apply<kAdd, true>(apply<kAdd, true>(term[0], inner, 0, nullptr), term[3], 0, nullptr)
                         : apply<kAdd, true>(term[0], apply<kAdd, true>(inner, term[3], 0, nullptr), 0, nullptr);
    }
    r.dst[n0 + t] = o;
}

// f(how the waves share K, as a type)
template <class F> void with_cut(uint32_t K, F f) {
    auto go = [&](auto l, auto w, auto loop) {
        constexpr int L = decltype(l)::value, W = decltype(w)::value;
        constexpr bool LOOP = decltype(loop)::value;
        if (K % (L * W * 256) == 0) f(Cut<L, W, LOOP, true>{});
        else f(Cut<L, W, LOOP, false>{});
    };
    constexpr std::integral_constant<int, 4> four{};
    if (K <= 1024) go(std::integral_constant<int, 1>{}, four, std::false_type{});
    else if (K <= 2048) go(std::integral_constant<int, 2>{}, four, std::false_type{});
    else if (K <= 3072) go(std::integral_constant<int, 3>{}, four, std::false_type{});
    else if (K <= 4096) go(four, four, std::false_type{});
    else go(four, std::integral_constant<int, 8>{}, std::true_type{});
}

} // namespace

int launch_one_row_group(cg_backend *be, OneRowGroup g) {
    uint32_t blocks = 0;
    for (uint32_t i = 0; i < g.count; i++) {
        g.p[i].first = blocks;
        blocks += (g.p[i].n + 3) / 4;
    }
    with_cut(g.in.k, [&](auto cut) {
        using T = decltype(cut);
        if (g.in.gamma) launch_kernel(one_row_group_kernel<T, true>, dim3(blocks), dim3(T::W * 64), 0, be->stream, g);
        else launch_kernel(one_row_group_kernel<T, false>, dim3(blocks), dim3(T::W * 64), 0, be->stream, g);
    });
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "one row's products launch");
}

int launch_one_row_gated(cg_backend *be, const OneRowGated &g) {
    with_cut(g.in.k, [&](auto cut) {
        using T = decltype(cut);
        const dim3 grid((g.n + 1) / 2), block(T::W * 64);
        if (g.in.gamma) launch_kernel(one_row_gated_kernel<T, true>, grid, block, 0, be->stream, g);
        else launch_kernel(one_row_gated_kernel<T, false>, grid, block, 0, be->stream, g);
    });
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "one row's gated products launch");
}

int launch_one_row_residual(cg_backend *be, const OneRowResidual &r) {
    with_cut(r.k, [&](auto cut) {
        using T = decltype(cut);
        // (two columns where four would leave fewer than four workgroups a compute unit: 1024 columns of 2048 values 3.62 and 3.76 us back to back)
        if (r.n >= 4 * 4 * (uint32_t)be->compute_units)
            launch_kernel(one_row_residual_kernel<T, 4>, dim3((r.n + 3) / 4), dim3(T::W * 64), 0, be->stream, r);
        else
            launch_kernel(one_row_residual_kernel<T, 2>, dim3((r.n + 1) / 2), dim3(T::W * 64), 0, be->stream, r);
    });
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "one row's product with residual launch");
}

} // namespace cg
