// Products of one row of activations with weight matrices whose rows have k contiguous: the linear layers of a decode step of one
// sequence (one_row.hip, called by matmul.hip).
#pragma once

#include "common.hpp"

namespace cg {

// x . w^T: column n = head * hd + d goes to dst[head * sh + d], through the rotary embedding out[d] = cos[d] * v[d] + sin[d] *
// concat(-v[hd / 2 ..], v[.. hd / 2])[d] if `rope` (hd a multiple of 8, n of hd).
struct OneRowProduct {
    const float *w;
    int64_t pitch; // elements from one row of w to the next
    uint32_t n, first; // columns; first workgroup (set by the launch)
    uint32_t *dst;
    int64_t sh;
    const uint32_t *cos, *sin;
    uint32_t hd, rope;
};
constexpr int kMaxOneRow = 4;
// The left operand: x, or its RMS norm x / pow(sum(x * x) / n + eps, e) * gamma (gamma not null).
struct OneRowInput {
    const float *x, *gamma;
    uint32_t k, n_bits, eps_bits, exp_bits;
};
struct OneRowGroup {
    OneRowInput in;
    OneRowProduct p[kMaxOneRow];
    uint32_t count;
};
// K a multiple of 4, all rows at 16 bytes (as everywhere below)
inline bool takes_one_row(uint32_t M, uint32_t K) { return M == 1 && K % 4 == 0 && K > 256; }
int launch_one_row_group(cg_backend *be, OneRowGroup g);
// dst[n] = g * (1 / (one + exp(-g))) * u for g = x . wg^T, u = x . wu^T
struct OneRowGated {
    OneRowInput in;
    const float *wg, *wu;
    int64_t pitch;
    uint32_t n, one;
    uint32_t *dst;
};
int launch_one_row_gated(cg_backend *be, const OneRowGated &g);
// dst[n] = a sum of 2 or 4 terms, term[slot] being x . w^T: t0 + t1, (t0 + (t1 + t2)) + t3 (order 0) or t0 + ((t1 + t2) + t3) (order 1)
struct OneRowResidual {
    const float *x, *w;
    int64_t pitch;
    uint32_t n, k;
    const uint32_t *term[4];
    uint32_t slot, order, nterms;
    uint32_t *dst;
};
int launch_one_row_residual(cg_backend *be, const OneRowResidual &r);

} // namespace cg
