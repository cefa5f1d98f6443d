// Products of one to eight rows of activations with weight matrices whose rows have k contiguous: the linear layers of a decode step
// (skinny_group.hip, skinny_gated.hip, skinny_residual.hip on skinny_kernel.hpp; called by matmul.hip).
#pragma once

#include "common.hpp"

namespace cg {

// The left operand: rows of x, or their RMS norm x / pow(sum(x * x) / n + eps, e) * gamma (gamma not null).
struct SkinnyInput {
    const float *x, *gamma;
    int64_t pitch; // elements from one row of x to the next
    uint32_t rows, k, n_bits, eps_bits, exp_bits;
};
// Rows that the kernels take: K a multiple of 4, all rows of x and w at 16 bytes (as everywhere below)
inline bool takes_skinny(uint32_t M, uint32_t K) { return M >= 1 && M <= 8 && K % 4 == 0 && K > 256; }

// x . w^T: column n = head * hd + d of row m goes to dst[m * sb + head * sh + d], through the rotary embedding out[d] = cos[d] * v[d] +
// sin[d] * concat(-v[hd / 2 ..], v[.. hd / 2])[d] if `rope` (hd a multiple of 8, n of hd).
struct SkinnyProduct {
    const float *w;
    int64_t pitch; // elements from one row of w to the next
    uint32_t n, first; // columns; first workgroup (set by the launch)
    uint32_t *dst;
    int64_t sb, sh;
    const uint32_t *cos, *sin;
    uint32_t hd, rope;
};
constexpr int kMaxSkinny = 4;
struct SkinnyGroup {
    SkinnyInput in;
    SkinnyProduct p[kMaxSkinny];
    uint32_t count;
};
int launch_skinny_group(cg_backend *be, SkinnyGroup g);
// dst[m, n] = g * (1 / (one + exp(-g))) * u for g = x . wg^T, u = x . wu^T
struct SkinnyGated {
    SkinnyInput in;
    const float *wg, *wu;
    int64_t pitch;
    uint32_t n, one;
    uint32_t *dst;
};
int launch_skinny_gated(cg_backend *be, const SkinnyGated &g);
// dst[m, n] = a sum of 2 or 4 terms, term[slot] being x . w^T: t0 + t1, (t0 + (t1 + t2)) + t3 (order 0) or t0 + ((t1 + t2) + t3) (order 1)
struct SkinnyResidual {
    SkinnyInput in; // (without a norm)
    const float *w;
    int64_t pitch;
    uint32_t n;
    const uint32_t *term[4];
    uint32_t slot, order, nterms;
    uint32_t *dst;
};
int launch_skinny_residual(cg_backend *be, const SkinnyResidual &r);

} // namespace cg
