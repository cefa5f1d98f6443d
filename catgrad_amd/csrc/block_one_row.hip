// The decoder blocks' products of one row of activations (one token of one sequence), for weights whose rows lie in 16-byte pieces: as
// in skinny_kernel.hpp a workgroup's waves share k, every load is asked for at the start, and one barrier is enough: what a norm multiplies a
// row by is a factor of the sums (for the polynomial one, of the sums of z, z^2, z^3 and 1 each).  Activations stay in 32 bits, also
// beside bfloat16 weights.  Against the kernels of up to four rows (block_rows.hip), us a launch in the steps of models of width 1024:
// 1024 -> 8328 with a norm, f32, 9.7 and 7.6; the sum of 2048 -> 1024 and of the polynomial norm's 3072 -> 1024, f32, 7.9 and 6.0; two products
// 1024 -> 4128 in bfloat16 4.7 and 3.9.
#include "blocks.hpp"
#include "device_utils.hpp"

#include <algorithm>
#include <type_traits>

namespace cg {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef f4 f4_words __attribute__((aligned(4))); // from any word's address
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sigmoid(float z) { // on the hardware's exp2 and reciprocal
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.44269504088896341f));
}

template <bool BF16> constexpr uint32_t kWide = BF16 ? 8 : 4; // values of k in a lane's 16 bytes of weights

// A wave's share of k of a row, L trips of 64 lanes: where each lane's values begin, and whether they are part of it.
template <bool BF16, int L> struct Share {
    uint32_t at[L];
    bool in[L];
    // wave `w` of `waves`; k a multiple of kWide, at most L * 64 * kWide * waves (loads behind the share are clamped, not tested)
    __device__ __forceinline__ Share(uint32_t w, uint32_t waves, uint32_t k) {
        constexpr uint32_t V = kWide<BF16>;
        const uint32_t span = (k + V * waves - 1) / (V * waves) * V, first = w * span;
#pragma unroll
        for (int i = 0; i < L; i++) {
            const uint32_t o = (i * 64 + (threadIdx.x & 63)) * V;
            in[i] = o < span && first + o < k;
            at[i] = min(first + o, k - V);
        }
    }
};
// A share of the activations (x | x2): in.k1 a multiple of kWide, rows at 16 bytes.
template <bool BF16, int L> struct Activations {
    float v[L][kWide<BF16>];
    __device__ __forceinline__ void ask(const ProductInput &in, const Share<BF16, L> &s) {
#pragma unroll
        for (int i = 0; i < L; i++) {
            const float *p = s.at[i] < in.k1 ? in.x.p + s.at[i] : in.x2.p + (s.at[i] - in.k1);
#pragma unroll
            for (uint32_t o = 0; o < kWide<BF16>; o += 4) {
                const f4 t = *reinterpret_cast<const f4 *>(p + o);
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][o + e] = t[e];
            }
        }
    }
    __device__ __forceinline__ void ask_gains(const float *gamma, const Share<BF16, L> &s) { // (at any word)
#pragma unroll
        for (int i = 0; i < L; i++)
#pragma unroll
            for (uint32_t o = 0; o < kWide<BF16>; o += 4) {
                const f4 t = *reinterpret_cast<const f4_words *>(gamma + s.at[i] + o);
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][o + e] = t[e];
            }
    }
    __device__ __forceinline__ void within(const Share<BF16, L> &s) { // zeros behind the share, whatever lies there
#pragma unroll
        for (int i = 0; i < L; i++)
#pragma unroll
            for (uint32_t e = 0; e < kWide<BF16>; e++) v[i][e] = s.in[i] ? v[i][e] : 0.0f;
    }
};
template <bool BF16, int L> struct WeightRow {
    u4 v[L];
    __device__ __forceinline__ void ask(const Weight &w, uint32_t n, const Share<BF16, L> &s) {
        const char *const row = static_cast<const char *>(w.p) + (int64_t)n * w.pitch * (BF16 ? 2 : 4);
#pragma unroll
        for (int i = 0; i < L; i++) v[i] = __builtin_nontemporal_load(reinterpret_cast<const u4 *>(row + (uint64_t)s.at[i] * (BF16 ? 2 : 4)));
    }
    __device__ __forceinline__ void within(const Share<BF16, L> &s) {
#pragma unroll
        for (int i = 0; i < L; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) v[i][e] = s.in[i] ? v[i][e] : 0;
    }
    __device__ __forceinline__ float at(int i, uint32_t e) const {
        if constexpr (BF16) return asf(e & 1 ? v[i][e / 2] & 0xFFFF0000u : v[i][e / 2] << 16);
        else return asf(v[i][e]);
    }
};

// The sum of four values over a wave: of s[r] in lanes 16 r .. 16 r + 15
__device__ __forceinline__ float lane_sums(const float (&s)[4]) { return add_across<1>(add_across<2>(four_sums(s[0], s[1], s[2], s[3]))); }

// ---- products that share a launch --------------------------------------------------------------------------------------
struct OneRowJob {
    ProductInput in;
    Weight w;
    const float *bias;
    float *out;
    float scale;
};
// Four columns to KW waves that share k, 4 / KW such groups a workgroup.  The first job on the first blocks0 workgroups.
template <bool BF16, int KW, int L> __global__ __launch_bounds__(256) void block_one_row_kernel(const OneRowJob j0, const OneRowJob j1, const uint32_t blocks0) {
    constexpr int GROUPS = 4 / KW;
    __shared__ float part[4][4], squares[4];
    const bool second = blockIdx.x >= blocks0;
    const OneRowJob &j = second ? j1 : j0;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t n0 = (blockIdx.x - (second ? blocks0 : 0)) * (4 * GROUPS), n_wave = n0 + wave / KW * 4;
    const Share<BF16, L> share(wave % KW, KW, j.w.k);
    Activations<BF16, L> x, gm;
    x.ask(j.in, share);
    if (j.in.gamma) gm.ask_gains(j.in.gamma, share);
    const uint32_t t = threadIdx.x, n = min(n0 + t % (4 * GROUPS), j.w.n - 1);
    const float bias = j.bias ? j.bias[n] : 0.0f;
    WeightRow<BF16, L> w[4];
#pragma unroll
    for (int c = 0; c < 4; c++) w[c].ask(j.w, min(n_wave + c, j.w.n - 1), share);
    __builtin_amdgcn_sched_barrier(0); // (what follows stays behind all of the loads)
    x.within(share);
    if (j.in.gamma) {
        gm.within(share);
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < L; i++)
#pragma unroll
            for (uint32_t e = 0; e < kWide<BF16>; e++) {
                ss = fmaf(x.v[i][e], x.v[i][e], ss);
                x.v[i][e] *= gm.v[i][e];
            }
        ss = wave_add<1>(ss);
        if (lane == 0) squares[wave] = ss;
    }
    float s[4] = {};
#pragma unroll
    for (int c = 0; c < 4; c++) {
        w[c].within(share);
#pragma unroll
        for (int i = 0; i < L; i++)
#pragma unroll
            for (uint32_t e = 0; e < kWide<BF16>; e++) s[c] = fmaf(x.v[i][e], w[c].at(i, e), s[c]);
    }
    const float sums = lane_sums(s);
    if (lane % 16 == 0) part[wave][lane / 16] = sums;
    __syncthreads();
    if (t >= 4 * GROUPS || n0 + t >= j.w.n) return;
    float v = 0.0f, q = 0.0f, factor = j.scale;
#pragma unroll
    for (int i = 0; i < KW; i++) v += part[t / 4 * KW + i][t % 4];
    if (j.in.gamma) {
#pragma unroll
        for (int i = 0; i < KW; i++) q += squares[i];
        factor /= sqrtf(q / (float)j.in.k + j.in.eps);
    }
    j.out[n] = v * factor + bias;
}

// ---- x + up to two products, gated -------------------------------------------------------------------------------------
constexpr int kResidualWaves = 8, kResidualColumns = 2;
template <bool BF16, int L, bool POLY> struct Branch {
    Activations<BF16, L> x;
    WeightRow<BF16, L> w[kResidualColumns];
    __device__ __forceinline__ void ask(const ResidualBranch &b, uint32_t n0, uint32_t width, const Share<BF16, L> &s) {
        x.ask(b.in, s);
#pragma unroll
        for (int c = 0; c < kResidualColumns; c++) w[c].ask(b.w, min(n0 + c, width - 1), s);
    }
    // part[c][term]: the wave's sums of z, z^2, z^3 and 1 (or of z), squares[term]: what the first three are scaled by
    __device__ __forceinline__ void sums(const Share<BF16, L> &s, float (&part)[kResidualColumns][4], float (&squares)[4]) {
        x.within(s);
#pragma unroll
        for (int c = 0; c < kResidualColumns; c++) w[c].within(s);
        float a[kResidualColumns][4] = {}, m[4] = {};
#pragma unroll
        for (int i = 0; i < L; i++)
#pragma unroll
            for (uint32_t e = 0; e < kWide<BF16>; e++) {
                const float z = x.v[i][e];
                if constexpr (POLY) {
                    const float z2 = z * z, z3 = z2 * z;
                    m[0] += z2;
                    m[1] = fmaf(z2, z2, m[1]);
                    m[2] = fmaf(z3, z3, m[2]);
#pragma unroll
                    for (int c = 0; c < kResidualColumns; c++) {
                        const float v = w[c].at(i, e);
                        a[c][0] = fmaf(z, v, a[c][0]);
                        a[c][1] = fmaf(z2, v, a[c][1]);
                        a[c][2] = fmaf(z3, v, a[c][2]);
                        a[c][3] += v;
                    }
                } else {
#pragma unroll
                    for (int c = 0; c < kResidualColumns; c++) a[c][0] = fmaf(z, w[c].at(i, e), a[c][0]);
                }
            }
        const uint32_t lane = threadIdx.x & 63;
        if constexpr (POLY) {
#pragma unroll
            for (int c = 0; c < kResidualColumns; c++) {
                const float v = lane_sums(a[c]);
                if (lane % 16 == 0) part[c][lane / 16] = v;
            }
            const float v = lane_sums(m);
            if (lane % 16 == 0) squares[lane / 16] = v;
        } else {
            static_assert(kResidualColumns == 2, "two sums to a register");
            const auto h = __builtin_amdgcn_permlane32_swap(asu(a[0][0]), asu(a[1][0]), false, false);
            float v = asf(fold_rows(asu(asf((uint32_t)h[0]) + asf((uint32_t)h[1])), AddWords{}));
            v = add_across<1>(add_across<2>(add_across<4>(add_across<8>(v))));
            if (lane % 32 == 0) part[lane / 32][0] = v;
        }
    }
};
// Two columns a workgroup of eight waves.  L0, L1: trips of the branches (L1 0: there is one).  POLY: the last one's polynomial norm.
template <bool BF16, int L0, int L1, bool POLY>
__global__ __launch_bounds__(kResidualWaves * 64) void block_one_row_residual_kernel(const Rows x, const ResidualBranch b0, const ResidualBranch b1, const uint32_t width,
                                                                                     float *__restrict__ out) {
    constexpr int NB = L1 ? 2 : 1;
    constexpr bool POLY0 = POLY && NB == 1, POLY1 = POLY && NB == 2;
    __shared__ float part[NB][kResidualWaves][kResidualColumns][4], squares[NB][kResidualWaves][4];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n0 = blockIdx.x * kResidualColumns;
    const Share<BF16, L0> s0(wave, kResidualWaves, b0.w.k);
    Branch<BF16, L0, POLY0> r0;
    // lane (column, term) of the first wave puts the sums together; what it needs besides is asked for first
    const uint32_t t = threadIdx.x, c = (t >> 2) % kResidualColumns, term = t & 3, n = min(n0 + c, width - 1);
    float xs = 0.0f, gate[NB] = {}, coef = 0.0f;
    if (t < 4 * kResidualColumns) {
        xs = x.p[n];
        if (b0.gate.p) gate[0] = b0.gate.p[n] + (b0.gate_bias ? b0.gate_bias[n] : 0.0f);
        if (NB > 1 && b1.gate.p) gate[NB - 1] = b1.gate.p[n] + (b1.gate_bias ? b1.gate_bias[n] : 0.0f);
        if (POLY) coef = (NB > 1 ? b1 : b0).in.poly[term];
    }
    r0.ask(b0, n0, width, s0);
    if constexpr (NB > 1) {
        const Share<BF16, L1 ? L1 : 1> s1(wave, kResidualWaves, b1.w.k);
        Branch<BF16, L1 ? L1 : 1, POLY1> r1;
        r1.ask(b1, n0, width, s1);
        __builtin_amdgcn_sched_barrier(0); // (what follows stays behind all of the loads)
        r0.sums(s0, part[0][wave], squares[0][wave]);
        r1.sums(s1, part[NB - 1][wave], squares[NB - 1][wave]);
    } else {
        __builtin_amdgcn_sched_barrier(0);
        r0.sums(s0, part[0][wave], squares[0][wave]);
    }
    __syncthreads();
    if (t >= 4 * kResidualColumns) return;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const ResidualBranch &br = b == 0 ? b0 : b1;
        float v = 0.0f;
        if (b == 0 ? POLY0 : POLY1) { // a lane per term
            float q = 0.0f;
#pragma unroll
            for (int i = 0; i < kResidualWaves; i++) {
                v += part[b][i][c][term];
                q += squares[b][i][term];
            }
            v *= term < 3 ? coef / sqrtf(q / (float)br.in.k + br.in.eps) : coef;
        } else { // a lane per quarter of the waves
#pragma unroll
            for (int i = 0; i < kResidualWaves; i += 4) v += part[b][i + term][c][0];
        }
        const float y = add_across<2>(add_across<1>(v));
        xs += br.gate.p ? sigmoid(gate[b]) * y : y;
    }
    if (term == 0 && n0 + c < width) out[n] = xs;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool rows_at_16(const ProductInput &in, const Weight &w) {
    const uint32_t v = w.fmt == kFmtBF16 ? 8 : 4;
    return w.k == in.k && w.k % v == 0 && w.pitch % v == 0 && aligned16(w.p) && in.k1 % v == 0 && aligned16(in.x.p) && (in.k1 >= in.k || aligned16(in.x2.p));
}
int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, what);
}

template <bool BF16> int linear(cg_backend *be, const OneRowJob &a, const OneRowJob &b, bool two) {
    const uint32_t trips = (a.w.k + 64 * kWide<BF16> - 1) / (64 * kWide<BF16>);
    auto go = [&](auto kw, auto l) {
        constexpr int KW = decltype(kw)::value, L = decltype(l)::value;
        constexpr uint32_t COLS = 16 / KW;
        const uint32_t b0 = (a.w.n + COLS - 1) / COLS, b1 = two ? (b.w.n + COLS - 1) / COLS : 0;
        launch_kernel((block_one_row_kernel<BF16, KW, L>), dim3(b0 + b1), dim3(256), 0, be->stream, a, b, b0);
    };
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 2> pair{};
    constexpr std::integral_constant<int, 4> four{};
    if (trips <= 1) go(one, one);
    else if (trips <= 2) go(pair, one);
    else if (trips <= 4) go(four, one);
    else if (trips <= 8) go(four, pair);
    else if (trips <= 12) go(four, std::integral_constant<int, 3>{});
    else go(four, four);
    return launched("one row's products");
}

} // namespace

// 4096 values of k (bfloat16: 8192) are what a workgroup's registers hold.
bool takes_block_one_row(const ProductInput &in, const Weight &w) {
    return !in.poly && w.k > 128 && w.k <= (w.fmt == kFmtBF16 ? 8192u : 4096u) && rows_at_16(in, w);
}
int launch_block_one_row(cg_backend *be, const ProductInput &in, const Weight &w, const float *bias, float scale, float *out) {
    const OneRowJob j{in, w, bias, out, scale};
    return w.fmt == kFmtBF16 ? linear<true>(be, j, j, false) : linear<false>(be, j, j, false);
}
int launch_block_one_row2(cg_backend *be, const ProductInput (&in)[2], const Weight (&w)[2], float *const (&out)[2]) {
    const OneRowJob a{in[0], w[0], nullptr, out[0], 1.0f}, b{in[1], w[1], nullptr, out[1], 1.0f};
    return w[0].fmt == kFmtBF16 ? linear<true>(be, a, b, true) : linear<false>(be, a, b, true);
}

static uint32_t residual_trips(const ResidualBranch &b) {
    const uint32_t trip = 64 * (b.w.fmt == kFmtBF16 ? 8 : 4) * kResidualWaves;
    return (b.w.k + trip - 1) / trip;
}
bool takes_block_one_row_residual(const ResidualBranch *br, int n) {
    if (n < 1 || n > 2 || (n == 2 && (br[0].w.fmt != br[1].w.fmt || br[0].in.poly))) return false;
    for (int i = 0; i < n; i++)
        if (br[i].in.gamma || !rows_at_16(br[i].in, br[i].w) || residual_trips(br[i]) > 4) return false;
    return true;
}
int launch_block_one_row_residual(cg_backend *be, const Rows &x, const ResidualBranch *br, int n, uint32_t width, float *out) {
    const uint32_t t0 = residual_trips(br[0]), t1 = n > 1 ? residual_trips(br[1]) : 0;
    const dim3 grid((width + kResidualColumns - 1) / kResidualColumns), block(kResidualWaves * 64);
    const bool poly = br[n - 1].in.poly != nullptr;
    auto go = [&](auto bf16, auto l0, auto l1, auto p) {
        launch_kernel((block_one_row_residual_kernel<decltype(bf16)::value, decltype(l0)::value, decltype(l1)::value, decltype(p)::value>), grid, block, 0, be->stream, x, br[0],
                      br[n - 1], width, out);
    };
    auto trips = [&](uint32_t t, auto f) {
        if (t <= 1) f(std::integral_constant<int, 1>{});
        else if (t <= 2) f(std::integral_constant<int, 2>{});
        else f(std::integral_constant<int, 4>{});
    };
    auto either = [&](bool b, auto f) {
        if (b) f(std::true_type{});
        else f(std::false_type{});
    };
    either(br[0].w.fmt == kFmtBF16, [&](auto bf16) {
        either(poly, [&](auto p) {
            trips(t0, [&](auto l0) {
                if (n == 1) go(bf16, l0, std::integral_constant<int, 0>{}, p);
                else trips(t1, [&](auto l1) { go(bf16, l0, l1, p); });
            });
        });
    });
    return launched("one row's residual sum");
}

} // namespace cg
