// Products of a few rows that share their left operand, with the rotary embedding and the write into a KV cache in the store.
#include "skinny_kernel.hpp"

namespace cg {
namespace {

// C columns a workgroup: half of them and those half a head away, which the rotary embedding mixes them with, or C in a row.
// (One row, 4096 x 1024 with a norm, back to back: four columns 5.5 us, eight 5.6, sixteen 6.2; a wave per column or two without any barrier 5.8.)
template <class T, int C, bool NORM> __global__ __launch_bounds__(T::W * 64) void skinny_group_kernel(const SkinnyGroup g) {
    __shared__ float part[T::W][T::M * C], squares[T::W][T::M];
    uint32_t at = 0;
#pragma unroll
    for (int i = 1; i < kMaxSkinny; i++) at += (uint32_t)i < g.count && blockIdx.x >= g.p[i].first ? 1u : 0u;
    const SkinnyProduct p = g.p[at];
    const uint32_t span = p.rope ? p.hd : C, per = span / C, block = blockIdx.x - p.first;
    const uint32_t n0 = block / per * span + block % per * (C / 2), apart = span / 2;
    auto column = [&](uint32_t c) { return n0 + c / (C / 2) * apart + c % (C / 2); };
    const uint32_t t = threadIdx.x % C, m = threadIdx.x / C, col = column(t), d = col % p.hd;
    uint32_t cs = 0, sn = 0;
    skinny_parts<T, C, NORM>(
        g.in, [&](int c) { return p.w + (int64_t)min(column(c), p.n - 1) * p.pitch; },
        [&] {
            if (p.rope && threadIdx.x < T::M * C) {
                cs = p.cos[d];
                sn = p.sin[d];
            }
        },
        part, squares);
    if (threadIdx.x >= T::M * C) return;
    float s = total(part, threadIdx.x);
    if constexpr (NORM) s = asf(apply<kDiv, true>(asu(s), asu(divisor_of(g.in, total(squares, m))), 0, nullptr));
    uint32_t v = asu(s);
    const uint32_t other = across<C / 2>(v); // the column half a head away
    if (p.rope) { // lower half: rotate_half reads -x[d + hd / 2]; upper half: x[d - hd / 2]
        const uint32_t rot = t < C / 2 ? apply<kNeg, true>(other, 0, 0, nullptr) : other;
        v = apply<kAdd, true>(apply<kMul, true>(cs, v, 0, nullptr), apply<kMul, true>(sn, rot, 0, nullptr), 0, nullptr);
    }
    if (col < p.n && m < g.in.rows) p.dst[(int64_t)m * p.sb + (int64_t)(col / p.hd) * p.sh + d] = v;
}

} // namespace

int launch_skinny_group(cg_backend *be, SkinnyGroup g) {
    bool wide = g.in.rows > 1; // eight columns share the rows' loads (4 x 2048 x 128256, back to back: 178 us, 163; 4 x 2048 x 3072: 7.2, 7.6)
    for (uint32_t i = 0; i < g.count; i++) wide = wide && g.p[i].n >= 8192 && !g.p[i].rope;
    const uint32_t C = wide ? 8 : 4;
    uint32_t blocks = 0;
    for (uint32_t i = 0; i < g.count; i++) {
        g.p[i].first = blocks;
        blocks += (g.p[i].n + C - 1) / C;
    }
    with_cut(g.in.rows, g.in.k, [&](auto cut) {
        using T = decltype(cut);
        auto launch = [&](auto kernel) { launch_kernel(kernel, dim3(blocks), dim3(T::W * 64), 0, be->stream, g); };
        if constexpr (T::M > 1) {
            if (wide && g.in.gamma) return launch(skinny_group_kernel<T, 8, true>);
            if (wide) return launch(skinny_group_kernel<T, 8, false>);
        }
        if (g.in.gamma) launch(skinny_group_kernel<T, 4, true>);
        else launch(skinny_group_kernel<T, 4, false>);
    });
    return skinny_launched("skinny products launch");
}

} // namespace cg
