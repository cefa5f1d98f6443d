// A product of a few rows with the residual stream's sum in its store.
#include "skinny_kernel.hpp"

namespace cg {
namespace {

// C columns a workgroup
template <class T, int C> __global__ __launch_bounds__(T::W * 64) void skinny_residual_kernel(const SkinnyResidual r) {
    __shared__ float part[T::W][T::M * C], squares[T::W][T::M];
    const uint32_t n0 = blockIdx.x * C, m = threadIdx.x / C, n = n0 + threadIdx.x % C;
    const bool stores = m < min((uint32_t)T::M, r.in.rows) && n < r.n;
    const uint64_t at = (uint64_t)m * r.n + n;
    uint32_t term[4] = {};
    skinny_parts<T, C, false>(
        r.in, [&](uint32_t c) { return r.w + (int64_t)min(n0 + c, r.n - 1) * r.pitch; },
        [&] { // the sum's other terms for the value this thread will store
            if (stores) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if ((uint32_t)i != r.slot && (uint32_t)i < r.nterms) term[i] = r.term[i][at];
            }
        },
        part, squares);
    if (!stores) return;
    const uint32_t v = asu(total(part, threadIdx.x));
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
    r.dst[at] = o;
}

} // namespace

int launch_skinny_residual(cg_backend *be, const SkinnyResidual &r) {
    with_cut(r.in.rows, r.in.k, [&](auto cut) {
        using T = decltype(cut);
        auto launch = [&](auto kernel, uint32_t c) { launch_kernel(kernel, dim3((r.n + c - 1) / c), dim3(T::W * 64), 0, be->stream, r); };
        if constexpr (T::M == 1) { // (two columns where four would leave fewer than four workgroups a compute unit: 1024 columns of 2048 values 3.62 and 3.76 us back to back)
            if (r.n < 4 * 4 * (uint32_t)be->compute_units) return launch(skinny_residual_kernel<T, 2>, 2);
        }
        launch(skinny_residual_kernel<T, 4>, 4);
    });
    return skinny_launched("skinny product with residual launch");
}

} // namespace cg
