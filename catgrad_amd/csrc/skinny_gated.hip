// The gated pair of an MLP block for a few rows.
#include "skinny_kernel.hpp"

namespace cg {
namespace {

// C / 2 columns of either matrix a workgroup
template <class T, int C, bool NORM> __global__ __launch_bounds__(T::W * 64) void skinny_gated_kernel(const SkinnyGated g) {
    constexpr uint32_t H = C / 2;
    __shared__ float part[T::W][T::M * C], squares[T::W][T::M];
    const uint32_t n0 = blockIdx.x * H;
    skinny_parts<T, C, NORM>(
        g.in, [&](uint32_t c) { return (c < H ? g.wg : g.wu) + (int64_t)min(n0 + c % H, g.n - 1) * g.pitch; }, [] {}, part, squares);
    const uint32_t m = threadIdx.x / H, c = threadIdx.x % H, n = n0 + c;
    if (m >= min((uint32_t)T::M, g.in.rows) || n >= g.n) return;
    uint32_t gv = asu(total(part, m * C + c)), uv = asu(total(part, m * C + H + c));
    if constexpr (NORM) {
        const uint32_t d = asu(divisor_of(g.in, total(squares, m)));
        gv = apply<kDiv, true>(gv, d, 0, nullptr);
        uv = apply<kDiv, true>(uv, d, 0, nullptr);
    }
    // the ops of the deferred program, in its order
    const uint32_t e = apply<kExp, true>(apply<kNeg, true>(gv, 0, 0, nullptr), 0, 0, nullptr);
    const uint32_t sg = apply<kDiv, true>(g.one, apply<kAdd, true>(g.one, e, 0, nullptr), 0, nullptr);
    g.dst[(uint64_t)m * g.n + n] = apply<kMul, true>(apply<kMul, true>(gv, sg, 0, nullptr), uv, 0, nullptr);
}

} // namespace

int launch_skinny_gated(cg_backend *be, const SkinnyGated &g) {
    with_cut(g.in.rows, g.in.k, [&](auto cut) {
        using T = decltype(cut);
        auto launch = [&](auto kernel, uint32_t h) { launch_kernel(kernel, dim3((g.n + h - 1) / h), dim3(T::W * 64), 0, be->stream, g); };
        if constexpr (T::M > 1) { // (4 x 2048 x 8192 twice, back to back: two columns of either 25.5 us, four 23.5; 4 x 1024 x 3072 twice: 7.1, 7.0)
            if (g.in.gamma) launch(skinny_gated_kernel<T, 8, true>, 4);
            else launch(skinny_gated_kernel<T, 8, false>, 4);
        } else {
            if (g.in.gamma) launch(skinny_gated_kernel<T, 4, true>, 2);
            else launch(skinny_gated_kernel<T, 4, false>, 2);
        }
    });
    return skinny_launched("skinny gated products launch");
}

} // namespace cg
