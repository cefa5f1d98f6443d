// C[b, M, N] = A[b, M, K] B[b, K, N] of 32-bit floats for more than eight rows, on the bfloat16 matrix instructions (split_tile.hpp).
//
// 8192 x 2048 x 8192: 1250 us = 220 TFLOP/s, where the 32-bit instructions took 1990 us = 138 (88 % of their peak); 1024 x 1024 x
// 3072: 53 against 74 us; 32 x 2048 x 8192: 22 against 46 us.  A few small shapes stay above the 32-bit instructions, whose tiles
// started sooner: with contiguous rows 100 x 576 x 1536 13.1 against 10.7, 4096 x 700 x 50 18.8 against 14.7 and 100 x 64 x 1024 6.6
// against 5.3; 333 x 1001 x 333 16.4 against 15.5.  The wide tile is bound by issuing: matrix pipes busy 66 % of the
// cycles at 1.77 GHz (64 SQ_VALU_MFMA_BUSY_CYCLES per instruction pair and GRBM_GUI_ACTIVE over the time); with one chain over all of
// k, without the additions of the chains' sums, 76 % at 1.74 GHz and 1150 us, but with sums off to one side.  Eight waves that share one
// 256 x 256 tile split a third less than two workgroups of four with 256 x 128 each and run 8 % faster.  Splitting by
// v_dot2c_f32_bf16 (one instruction for the shift and the subtraction): slower.
#include "gemm_args.hpp"
#include "split_tile.hpp"

#include <algorithm>
#include <cmath>

namespace cg {
namespace {

using namespace split;
constexpr int kThreads = 256;
constexpr uint32_t kXcds = 8, kGroupM = 8;

template <int WM, int WN, int MT, int NT, bool AF, bool BF, bool CARE>
__global__ __launch_bounds__(64 * WM * WN, 2) void split_gemm_kernel(const MmArgs a) {
    constexpr uint32_t BM = 32 * WM * MT, BN = 32 * WN * NT;
    extern __shared__ float lds_dyn[];
    // Workgroups are dealt round-robin to the XCDs: every XCD gets one run of tiles, walked down columns of kGroupM row tiles, so
    // that the tiles in flight on it share panels of both operands in its L2.
    const uint32_t tiles_n = (a.N + BN - 1) / BN, tiles_m = (a.M + BM - 1) / BM, ntiles = tiles_m * tiles_n;
    const uint32_t xcd = blockIdx.x % kXcds, q8 = ntiles / kXcds, r8 = ntiles % kXcds;
    const uint32_t lin = xcd * q8 + min(xcd, r8) + blockIdx.x / kXcds;
    const uint32_t group = lin / (kGroupM * tiles_n), in_group = lin % (kGroupM * tiles_n), first_m = group * kGroupM;
    const uint32_t gsize = min(tiles_m - first_m, kGroupM);
    const uint32_t m0 = (first_m + in_group % gsize) * BM, n0 = (in_group / gsize) * BN;
    int64_t pa, pb;
    batch_offsets(a, blockIdx.y, pa, pb);
    const uint32_t k0 = blockIdx.z * a.ksplit, K = a.ksplit ? min(a.K - k0, a.ksplit) : a.K;
    const TileSide oa = {a.A + pa + (int64_t)k0 * a.a_sk + (int64_t)m0 * a.a_sm, a.a_sk};
    const TileSide ob = {a.B + pb + (int64_t)k0 * a.b_sk + (int64_t)n0 * a.b_sn, a.b_sk};
    const int64_t sm = a.a_sm, sn = a.b_sn;
    float16v acc[MT][NT];
    product<WM, WN, MT, NT, AF, BF, CARE>(
        acc, (lds_char *)lds_dyn, oa, [=](uint32_t r) { return (int64_t)r * sm; }, min(a.M - m0, BM) - 1, ob, [=](uint32_t r) { return (int64_t)r * sn; },
        min(a.N - n0, BN) - 1, K);

    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), li = threadIdx.x % 32, lg = threadIdx.x % 64 / 32;
    const uint32_t wm = wave / WN * (32 * MT), wn = wave % WN * (32 * NT);
    uint32_t *const C = a.C + ((uint64_t)blockIdx.y * gridDim.z + blockIdx.z) * a.M * a.N + (uint64_t)m0 * a.N + n0;
    if (m0 + BM <= a.M && n0 + BN <= a.N && a.N < (1u << 20)) { // a lane's offset from addresses that all lanes share
        const uint32_t off = ((wm + 4 * lg) * a.N + wn + li) * 4;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const uint32_t *const to = C + (uint64_t)(i * 32 + 8 * (v / 4) + v % 4) * a.N + j * 32;
                    asm volatile("global_store_dword %0, %1, %2" ::"v"(off), "v"(acc[i][j][v]), "s"(to) : "memory");
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        return;
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const uint32_t col = wn + j * 32 + li;
            if (n0 + col < a.N) {
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const uint32_t row = wm + i * 32 + 8 * (v / 4) + 4 * lg + v % 4;
                    if (m0 + row < a.M) C[(uint64_t)row * a.N + col] = asu(acc[i][j][v]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
}

typedef void (*Kernel)(const MmArgs);
struct Tile {
    int bm, bn, threads;
    Kernel kernel[2][2]; // [rows of A fast][rows of B fast]
};
template <int WM, int WN, int MT, int NT, bool AF, bool BF, bool CARE> Kernel prepared() {
    Kernel k = &split_gemm_kernel<WM, WN, MT, NT, AF, BF, CARE>;
    const int lds = (int)lds_bytes(32 * WM * MT, 32 * WN * NT);
    return hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess ? k : nullptr;
}
// What a launch takes, in microseconds: before and behind the stages, a stage, and the share of a stage that each workgroup of a
// compute unit takes when there are several (they hide each other's waits).
struct Cost {
    double start, stage, share;
};
// In the order of `tiles`: the wide tile, the tile for what does not fill the device with it, two for a few rows, and the second
// one's twin for any alignment; 64 x 64 for k-contiguous operands, and its twin; 64 x 64 for operands with contiguous rows, which
// two waves turn in registers, and its twin.  Fitted to 474 shapes of 16 to 8192 rows in all layouts, every tile and cut timed: what this
// picks is 1 % above the fastest in the mean.
constexpr Cost kCost[9] = {{9.8, 1.64, 1.0}, {5.8, 0.70, 0.83}, {4.4, 0.61, 0.68}, {5.2, 0.42, 1.45}, {5.6, 1.44, 0.835},
                           {4.0, 0.37, 0.705}, {4.5, 0.68, 0.937}, {4.85, 0.40, 1.03}, {5.0, 0.817, 0.85}};
const Tile *tiles() {
#define CG_TILE(WM, WN, MT, NT, CARE)                                                                       \
    {32 * WM * MT, 32 * WN * NT, 64 * WM * WN, {{prepared<WM, WN, MT, NT, false, false, CARE>(), prepared<WM, WN, MT, NT, false, true, CARE>()}, \
                                  {prepared<WM, WN, MT, NT, true, false, CARE>(), prepared<WM, WN, MT, NT, true, true, CARE>()}}}
#define CG_SMALL_TILE(CARE) \
    {64, 64, 256, {{prepared<2, 2, 1, 1, false, false, CARE>(), nullptr}, {nullptr, nullptr}}}
#define CG_ROWS_TILE(CARE) \
    {64, 64, 128, {{nullptr, prepared<1, 2, 2, 1, false, true, CARE>()}, {prepared<1, 2, 2, 1, true, false, CARE>(), prepared<1, 2, 2, 1, true, true, CARE>()}}}
#define CG_LOW_TILE(WM, WN, MT, NT) \
    {32 * WM * MT, 32 * WN * NT, 64 * WM * WN, {{prepared<WM, WN, MT, NT, false, false, false>(), prepared<WM, WN, MT, NT, false, true, false>()}, {nullptr, nullptr}}}
    static const Tile t[9] = {CG_TILE(2, 4, 4, 2, false), CG_TILE(2, 2, 2, 2, false), CG_LOW_TILE(1, 4, 2, 1), CG_LOW_TILE(1, 4, 1, 2), CG_TILE(2, 2, 2, 2, true),
                              CG_SMALL_TILE(false), CG_SMALL_TILE(true), CG_ROWS_TILE(false), CG_ROWS_TILE(true)};
#undef CG_TILE
#undef CG_LOW_TILE
#undef CG_SMALL_TILE
#undef CG_ROWS_TILE
    return t;
}

// y[e] = the parts' sum, in their order
template <int VEC> __global__ __launch_bounds__(kThreads) void sum_splits_kernel(const float *part, float *y, uint32_t parts, uint32_t mn, uint64_t total) {
    const uint64_t e = ((uint64_t)blockIdx.x * kThreads + threadIdx.x) * VEC;
    if (e >= total) return;
    const float *p = part + e / mn * parts * mn + e % mn;
    if constexpr (VEC == 4) {
        float4v v = __builtin_nontemporal_load(reinterpret_cast<const float4v *>(p));
        for (uint32_t s = 1; s < parts; s++) v += __builtin_nontemporal_load(reinterpret_cast<const float4v *>(p + (uint64_t)s * mn));
        *reinterpret_cast<float4v *>(y + e) = v;
    } else {
        float v = *p;
        for (uint32_t s = 1; s < parts; s++) v += p[(uint64_t)s * mn];
        y[e] = v;
    }
}

} // namespace

int launch_split_gemm(cg_backend *be, MmArgs a, bool a_mfast, bool b_nfast) {
    const Tile *const all = tiles();
    // (byte offsets of a tile's loads in 32 bits; rows that are loaded four at a time come in fours)
    auto fits = [](bool fast, int64_t s_r, int64_t s_k, uint32_t rows) {
        return fast ? rows % 4 == 0 && s_k < (1ll << 25) : s_r < (1ll << 21);
    };
    const bool care = !a.a_vec || !a.b_vec || !fits(a_mfast, a.a_sm, a.a_sk, a.M) || !fits(b_nfast, a.b_sn, a.b_sk, a.N);
    auto count = [&](int t) { return (uint64_t)((a.M + all[t].bm - 1) / all[t].bm) * ((a.N + all[t].bn - 1) / all[t].bn) * a.batch; };
    const uint64_t mn = (uint64_t)a.M * a.N;
    // The tile, and over how many workgroups k is cut (at least 64 values each, partial results of at most 64 MB), by what the launch
    // takes: in us, 512 x 2048 x 2048 37 in four parts of 128 x 128 tiles, 45 in 16 of the wide one; 2048 x 2048 x 8192 342 with
    // the wide one, 401 without; 32 x 2048 x 8192 21 with 32 x 256, 34 with 128 x 128; 333 x 1536 x 576 16 with 64 x 64, 20 without; and where rows are contiguous, on the two-wave
    // tile and without it (before: on the 32-bit instructions), 100 x 64 x 1024 6.7 and 9.1 (5.2), 1500 x 700 x 50 15.6 and 19.8 (13.0).
    int t = -1;
    uint64_t splits = 1;
    double best = 0;
    auto consider = [&](int tile) {
        const Cost &c = kCost[tile];
        const uint64_t wgs = count(tile);
        for (uint64_t p = 1; p <= 16 && (p == 1 || (a.K / p >= 64 && p * a.batch * mn <= (16u << 20))); p++) {
            const uint32_t part = p > 1 ? (uint32_t)((a.K + p - 1) / p + 31) / 32 * 32 : a.K;
            if (p > 1 && (a.K + part - 1) / part != p) continue;
            const double rounds = std::ceil((double)(wgs * p) / be->compute_units), stages = c.stage * ((part + kDepth - 1) / kDepth);
            const double us = (tile == 0 ? rounds * (c.start + stages) : c.start + stages * std::max(1.0, c.share * rounds)) +
                              (p > 1 ? 2.15 + 0.19 * p + 1.05e-6 * p * a.batch * mn : 0.0);
            if (t < 0 || us < best) t = tile, splits = p, best = us;
        }
    };
    consider((a_mfast || b_nfast ? 7 : 5) + care);
    if (care) consider(4);
    else {
        consider(1);
        if (a.K % kDepth == 0) consider(0);
        if (!a_mfast && a.M <= 1024) consider(2);
        if (!a_mfast && a.M <= 32) consider(3);
    }
    // Few rows, or little work: without a second launch, where that is faster.  Up to four values of k are multiplied by the 32-bit
    // instructions alone (split_tile.hpp).
    if (!care && !a_mfast && !b_nfast && a.K % 4 == 0 && a.K > 4) {
        int high = 0;
        const double us = thin_gemm_cost(be, a, &high);
        if (high && us < best) return launch_thin_gemm(be, a, high);
    }
    const uint64_t tiles = count(t) / a.batch;
    if (tiles > 0x7FFFFFFFull) return fail(CG_ERR_UNSUPPORTED, "matmul: too many tiles");
    Kernel k = all[t].kernel[a_mfast][b_nfast];
    const uint32_t lds = lds_bytes(all[t].bm, all[t].bn);
    if (!k) return fail(CG_ERR_DEVICE, "matmul: cannot reserve %u bytes of LDS", lds);
    float *const y = reinterpret_cast<float *>(a.C);
    void *parts = nullptr;
    size_t cls = 0;
    if (splits > 1) {
        a.ksplit = (uint32_t)((a.K + splits - 1) / splits + 31) / 32 * 32;
        splits = (a.K + a.ksplit - 1) / a.ksplit;
    }
    if (splits > 1 && be->pool.alloc(a.batch * splits * mn * 4, &parts, &cls)) {
        (void)hipGetLastError();
        splits = 1; // no room for the parts: uncut
    }
    if (splits > 1) {
        a.C = static_cast<uint32_t *>(parts);
    } else {
        splits = 1;
        a.ksplit = 0;
    }
    launch_kernel(k, dim3((uint32_t)tiles, a.batch, (uint32_t)splits), dim3(all[t].threads), lds, be->stream, a);
    if (splits > 1) {
        const uint64_t total = mn * a.batch;
        const float *const from = static_cast<const float *>(parts);
        if (mn % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0)
            launch_kernel((sum_splits_kernel<4>), dim3((uint32_t)((total / 4 + kThreads - 1) / kThreads)), dim3(kThreads), 0, be->stream, from, y,
                               (uint32_t)splits, (uint32_t)mn, total);
        else
            launch_kernel((sum_splits_kernel<1>), dim3((uint32_t)((total + kThreads - 1) / kThreads)), dim3(kThreads), 0, be->stream, from, y,
                               (uint32_t)splits, (uint32_t)mn, total);
        be->pool.free(parts, cls); // stream-ordered
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "matmul launch");
}

} // namespace cg
